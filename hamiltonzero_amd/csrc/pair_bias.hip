// The trunk attention's coupling-bias producer, float32 products as six bfloat16 ones
// (split_f32.h, v_mfma_f32_16x16x32_bf16): per site pair (i, j) of a walker,
//     y   = x * (w * rsqrt(mean(x^2) + eps))           x = edge[b, i, j, :] (C channels)
//     h0  = y W_in + b_in                               (64 hidden)
//     h1  = h0 + gain * (silu(h0 W_1 + b_1) W_2 + b_2)
//     e   = (h1 W_out + b_out) / div                    (H heads)
// and, with a tangent edge_t, its forward-mode derivative, written straight into the
// attention kernels' bias layout: [B, N, H, N] / [B, N, N, H], or the compacted layout
// (e_blk > 0), where pair (i, j) of the walker's physical-site list goes to i * ceil4(n) + j
// of head h's block, so the attention reads n * ceil4(n) contiguous floats per (walker, head)
// instead of n rows of N.
//
// Orientation: every layer is computed transposed, features x pairs (features = the 16-row
// M blocks, 16 pairs = one N block), so the pairs are the columns of the B operand and the
// weights (split once per workgroup into LDS, as ready-made A fragments) the A operand. A
// layer's result C[feature 4g + r][pair c] of block m sits in lane (g, c) register r, and the two
// blocks 2s, 2s + 1 are exactly the eight values of the next layer's B operand in K step s if that
// layer's K order is permuted: slot j of lane group g multiplies feature 32 s + 16 (j / 4) + 4 g +
// j mod 4. The weight fragments are stored in that order, so the four layers chain in registers,
// split between layers, with no LDS round trip.
//
// The RMS scale r is a per-pair (column) scale and the norm weight w is folded into W_in's
// fragments: layer 1 runs on x and scales columns by r afterwards, so x streams straight from
// memory into the products while mean(x^2) (and, with a tangent, mean(x xdot)) accumulate
// alongside; the tangent of layer 1 is r xdot (w W_in) + rdot x (w W_in) with rdot = -0.5 r / v *
// 2 mean(x xdot).
//
// The weights' three parts (98 KB at C = 96, 32 heads) leave one workgroup per CU, of eight
// waves: two a SIMD, so one wave's splits and activations run under the other's products. A tile's
// 384 matrix instructions take 6144 cycles beside about 1400 vector instructions (5600 cycles);
// with two waves a SIMD they overlap by a third. 1024 walkers of 36 sites, C = 96, 32 heads, with
// tangent: 520 us (751 on the float32 matrix instruction), 572 where it zeroes the compacted layout's
// unfilled entries too. Of 495 us in one session: 250 with neither the products nor memory, 90 for
// the products beyond it, 95 for the loads and stores. Twelve waves spill and take 545 us.
//
// A tile is 16 pairs with their tangent (T = 1: N block 0 primal, N block 1 tangent) or 32
// pairs (T = 0). With a mask, only pairs whose key site is physical are computed (and, in
// the square-mask semantics, whose query site is physical too): a wave builds the walker's
// list of physical sites with a ballot, then walks the flattened (query, key) pair list.
// Each wave is persistent over (walker, part) items; a workgroup's waves share the staged weights.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mhsea_device.h"
#include "mhsea_launch.h"
#include "split_f32.h"

namespace hz {
namespace {

constexpr int kHid = 64;          // bias_mlp hidden width (trunk_attention_bias_hidden_dim)
constexpr int kPBWaves = 8;       // waves per workgroup
constexpr int kPBListN = 256;     // sites per walker the pair compaction handles

template <int C, int HB>
struct PBLds {
  // fragments, 16-byte units: [K step][M block][part][64 lanes]
  static constexpr int kBlock = 3 * 64;
  static constexpr int kF1 = 0;                            // W_in: C / 32 steps x 4 blocks
  static constexpr int kF2 = kF1 + C / 32 * 4 * kBlock;    // W_1: 2 x 4
  static constexpr int kF3 = kF2 + 8 * kBlock;             // W_2
  static constexpr int kF4 = kF3 + 8 * kBlock;             // W_out: 2 x HB
  static constexpr int kUnits = kF4 + 2 * HB * kBlock;
  // vectors, floats
  static constexpr int kBin = 0;
  static constexpr int kB1 = kBin + kHid;
  static constexpr int kB2 = kB1 + kHid;
  static constexpr int kBout = kB2 + kHid;
  static constexpr int kFloats = kBout + 16 * HB;
};

__device__ __forceinline__ float4 lds4(const float* base, int off) {
  return *reinterpret_cast<const float4*>(base + off);
}

__device__ __forceinline__ float comp(const float4& v, int u) {
  return u == 0 ? v.x : (u == 1 ? v.y : (u == 2 ? v.z : v.w));
}

// sigmoid(u) = 1 / (1 + 2^(-u log2 e)) on the hardware exp2 and reciprocal (about 1 ulp each;
// the exponent's rounding adds |u| 2^-24 relative): a few instructions instead of a
// full-precision expf and an IEEE division. u -> -inf gives 2^+inf = inf and 1/inf = 0.
__device__ __forceinline__ float sigmoid(float u) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(u * -1.44269504088896341f));
}

// The pairs of lane column c in tile t (N block cb): query site qi, key site qj, valid, and
// the pair's offset in a compacted (walker, head) block, row * ceil4(nk) + key (list order).
template <bool TAN>
__device__ __forceinline__ void tile_pairs(int t, int c, int npairs, int nk, bool rows_listed, bool keys_listed,
                                           const unsigned short* list, int qi[2], int qj[2], bool valid[2],
                                           int cpos[2]) {
  constexpr int TP = TAN ? 16 : 32;
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int q = TAN ? TP * t + c : TP * t + 16 * cb + c;
    valid[cb] = q < npairs;
    const int qq = valid[cb] ? q : 0;
    const int ii = qq / nk, jj = qq - ii * nk;
    qi[cb] = rows_listed ? list[ii] : ii;
    qj[cb] = keys_listed ? list[jj] : jj;
    cpos[cb] = ii * ((nk + 3) & ~3) + jj;
  }
}

// This lane's quarter (C / 4 channels) of the edge rows of its pairs (T = 1: the pair's edge
// and edge_t rows; T = 0: the rows of the two pairs).
template <int C, bool TAN>
__device__ __forceinline__ void load_rows(const float* edge_b, const float* edge_tb, int N, int g, const int qi[2],
                                          const int qj[2], const bool valid[2], float4 xin[2][C / 16]) {
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int src = TAN ? 0 : cb;
    const float* row = (TAN && cb == 1 ? edge_tb : edge_b) + (static_cast<int64_t>(qi[src]) * N + qj[src]) * C +
                       g * (C / 4);
#pragma unroll
    for (int v = 0; v < C / 16; ++v)
      xin[cb][v] = valid[src] ? *reinterpret_cast<const float4*>(row + 4 * v) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

// Splits one layer's weights into its fragments: w(k, o) the weight, k_of(step, g, j) the K order.
template <int KS, int MB, class W, class K>
__device__ __forceinline__ void stage_frags(v4u* dst, W w, K k_of) {
  for (int f = threadIdx.x; f < KS * MB * 64; f += blockDim.x) {
    const int lane = f & 63, m = (f >> 6) % MB, step = (f >> 6) / MB;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = w(k_of(step, lane >> 4, j), 16 * m + (lane & 15));
    const Split8 sp = split8(x);
    v4u* const d = dst + (step * MB + m) * (3 * 64) + lane;
    d[0] = sp.h;
    d[64] = sp.m;
    d[128] = sp.l;
  }
}

// out[m][cb] += W x[.][cb] over 64 features, the layers' registers as they stand.
template <int MB>
__device__ __forceinline__ void hidden_layer(const v4u* F, const v4f (&x)[4][2], v4f (&out)[MB][2]) {
#pragma unroll
  for (int step = 0; step < 2; ++step) {
    float x0[8], x1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      x0[j] = x[2 * step + (j >> 2)][0][j & 3];
      x1[j] = x[2 * step + (j >> 2)][1][j & 3];
    }
    mm_step<MB>(F + step * MB * (3 * 64), split8(x0), split8(x1), out);
  }
}

template <int C, int HB, bool TAN>
__global__ void __launch_bounds__(64 * kPBWaves, 2) pair_bias_kernel(PairBiasParams p) {
  using L = PBLds<C, HB>;
  constexpr int C4 = C / 4;    // channels per lane group
  constexpr int CG = C / 16;   // float4 groups per lane group
  constexpr int H = 16 * HB;
  constexpr int TP = TAN ? 16 : 32;  // pairs per tile
  __shared__ v4u frags[L::kUnits];
  __shared__ __attribute__((aligned(16))) float lds[L::kFloats];
  __shared__ unsigned short lists[kPBWaves][kPBListN];

  // ---- stage the weights as A fragments (once per workgroup) ----
  const auto hidden_k = [](int step, int g, int j) { return 32 * step + 16 * (j >> 2) + 4 * g + (j & 3); };
  stage_frags<C / 32, 4>(frags + L::kF1, [&](int k, int o) { return p.ln_w[k] * p.w_in[k * kHid + o]; },
                         [](int step, int g, int j) { return g * C4 + 8 * step + j; });
  stage_frags<2, 4>(frags + L::kF2, [&](int k, int o) { return p.w_1[k * kHid + o]; }, hidden_k);
  stage_frags<2, 4>(frags + L::kF3, [&](int k, int o) { return p.gain * p.w_2[k * kHid + o]; }, hidden_k);
  stage_frags<2, HB>(frags + L::kF4, [&](int k, int o) { return p.w_out[k * H + o]; }, hidden_k);
  for (int f = threadIdx.x; f < kHid; f += blockDim.x) {
    lds[L::kBin + f] = p.b_in[f];
    lds[L::kB1 + f] = p.b_1[f];
    lds[L::kB2 + f] = p.gain * p.b_2[f];
  }
  for (int f = threadIdx.x; f < H; f += blockDim.x) lds[L::kBout + f] = p.b_out[f];
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  unsigned short* list = lists[wave];
  const int N = p.N;
  const int64_t pair_stride = static_cast<int64_t>(N) * N;
  const bool use_list = p.mask != nullptr && N <= kPBListN;
  const float inv_c = 1.0f / static_cast<float>(C);
  // 1 / sqrt(d_head): exact for the power-of-two d_head the model uses (16), within 1 ulp of
  // the reference's division otherwise.
  const float inv_div = 1.0f / p.div;
  const int64_t total_waves = static_cast<int64_t>(gridDim.x) * kPBWaves;

  for (int64_t item = static_cast<int64_t>(blockIdx.x) * kPBWaves + wave; item < p.n_items; item += total_waves) {
    const int64_t b = item / p.parts;
    const int part = static_cast<int>(item - b * p.parts);

    // ---- the walker's physical sites ----
    int nk = N;
    bool keys_listed = false, rows_listed = false;
    if (use_list) {
      int n = 0;
      for (int s0 = 0; s0 < N; s0 += 64) {
        const int site = s0 + lane;
        const bool phys = site < N && p.mask[b * N + site] != 0;
        const uint64_t bal = __ballot(phys);
        if (phys) list[n + __popcll(bal & ((1ull << lane) - 1ull))] = static_cast<unsigned short>(site);
        n += __popcll(bal);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      // The entries of the walker's compacted blocks that no pair fills (the pad of each row, the
      // tail), zeroed while the matrix cores work: heads part, part + parts, ... of this item.
      if (p.zero_rest) {
        const int n4 = (n + 3) & ~3;
        for (int h = part; h < H; h += p.parts)
          for (int t = 0; t < (TAN ? 2 : 1); ++t) {
            float* const blk = (t == 0 ? p.e : p.e_t) + (b * H + h) * p.e_blk;
            for (int i = n * n4 + 4 * lane; i < p.e_blk; i += 256) *reinterpret_cast<v4f*>(blk + i) = zero4();
            for (int i = lane; i < n; i += 64)
              for (int j = n; j < n4; ++j) blk[i * n4 + j] = 0.f;
          }
      }
      if (n > 0) {
        nk = n;
        keys_listed = true;
        rows_listed = !p.key_mask;
      } else if (!p.key_mask) {
        continue;  // square mask, no physical site: the attention never reads this walker's bias
      }
    }
    const int nrows = rows_listed ? nk : N;
    const int npairs = nrows * nk;
    const int ntiles = (npairs + TP - 1) / TP;
    const int t0 = static_cast<int>(static_cast<int64_t>(ntiles) * part / p.parts);
    const int t1 = static_cast<int>(static_cast<int64_t>(ntiles) * (part + 1) / p.parts);

    const float* edge_b = p.edge + b * pair_stride * C;
    const float* edge_tb = TAN ? p.edge_t + b * pair_stride * C : nullptr;
    const bool cmp = p.e_blk > 0;
    const int64_t wstride = cmp ? p.e_blk * H : pair_stride * H;
    float* e_b = p.e + b * wstride;
    float* et_b = TAN ? p.e_t + b * wstride : nullptr;
    const int64_t hstride = cmp ? p.e_blk : p.e_sh;  // between heads (uniform)

    // The edge rows of the item's first tile; each tile then loads the next tile's rows.
    int qi[2], qj[2], cpos[2];
    bool valid[2];
    float4 xin[2][CG];
    if (t0 < t1) {
      tile_pairs<TAN>(t0, c, npairs, nk, rows_listed, keys_listed, list, qi, qj, valid, cpos);
      load_rows<C, TAN>(edge_b, edge_tb, N, g, qi, qj, valid, xin);
    }
    for (int t = t0; t < t1; ++t) {
      // The weight fragments are the same for every tile; an offset the compiler cannot see
      // through keeps their LDS reads inside the loop (hoisted, they would not fit the registers).
      int lz = 0;
      asm volatile("" : "+s"(lz));
      const float* W = lds + lz;
      const v4u* F = frags + lz + lane;

      // ---- layer 1: P = x (w W_in), with sum(x^2) and sum(x xdot) alongside ----
      v4f acc[4][2];
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m][0] = acc[m][1] = zero4();
      float s0 = 0.f, s1 = 0.f;  // sum x0^2; T = 1: sum x0 xdot, T = 0: sum x1^2
#pragma unroll
      for (int step = 0; step < C / 32; ++step) {
        float x0[8], x1[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x0[j] = comp(xin[0][2 * step + (j >> 2)], j & 3);
          x1[j] = comp(xin[1][2 * step + (j >> 2)], j & 3);
          s0 += x0[j] * x0[j];
          s1 += TAN ? x0[j] * x1[j] : x1[j] * x1[j];
        }
        mm_step<4>(F + L::kF1 + step * 4 * L::kBlock, split8_clamped(x0), split8_clamped(x1), acc);
      }
      s0 += __shfl_xor(s0, 16);
      s0 += __shfl_xor(s0, 32);
      s1 += __shfl_xor(s1, 16);
      s1 += __shfl_xor(s1, 32);
      const float v0 = s0 * inv_c + p.eps;
      const float r0 = 1.0f / sqrtf(v0);
      // T = 1: the tangent's column scale rdot; T = 0: the second pair block's scale
      const float r1 = TAN ? (2.0f * s1 * inv_c) * (-0.5f * r0 / v0) : 1.0f / sqrtf(s1 * inv_c + p.eps);
      // the next tile's rows, under the rest of this one
      int nqi[2] = {qi[0], qi[1]}, nqj[2] = {qj[0], qj[1]}, ncpos[2] = {cpos[0], cpos[1]};
      bool nvalid[2] = {false, false};
      if (t + 1 < t1) {
        tile_pairs<TAN>(t + 1, c, npairs, nk, rows_listed, keys_listed, list, nqi, nqj, nvalid, ncpos);
        load_rows<C, TAN>(edge_b, edge_tb, N, g, nqi, nqj, nvalid, xin);
      }
      v4f h[4][2];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float4 bi = lds4(W, L::kBin + 16 * m + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float P0 = acc[m][0][r], P1 = acc[m][1][r];
          h[m][0][r] = r0 * P0 + comp(bi, r);
          h[m][1][r] = TAN ? r0 * P1 + r1 * P0 : r1 * P1 + comp(bi, r);
        }
      }

      // ---- layer 2: a = silu(h0 W_1 + b_1) (and its tangent) ----
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m][0] = acc[m][1] = zero4();
      hidden_layer<4>(F + L::kF2, h, acc);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float4 b1 = lds4(W, L::kB1 + 16 * m + 4 * g);
        const float4 b2 = lds4(W, L::kB2 + 16 * m + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float u0 = acc[m][0][r] + comp(b1, r);
          const float s = sigmoid(u0);
          acc[m][0][r] = u0 * s;
          if (TAN) {
            acc[m][1][r] = acc[m][1][r] * (s + u0 * s * (1.0f - s));
          } else {
            const float u1 = acc[m][1][r] + comp(b1, r);
            acc[m][1][r] = u1 * sigmoid(u1);
          }
          h[m][0][r] += comp(b2, r);
          if (!TAN) h[m][1][r] += comp(b2, r);
        }
      }

      // ---- layer 3: h1 = h0 + gain b_2 + a (gain W_2), summed straight into h ----
      hidden_layer<4>(F + L::kF3, acc, h);

      // ---- layer 4: e = (h1 W_out + b_out) / div ----
      v4f o[HB][2];
#pragma unroll
      for (int m = 0; m < HB; ++m) o[m][0] = o[m][1] = zero4();
      hidden_layer<HB>(F + L::kF4, h, o);

      // ---- store: lane (g, c) holds heads 16 m + 4 g + r of its pair ----
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const int src = TAN ? 0 : cb;
        if (!valid[src]) continue;
        const int64_t at = cmp ? cpos[src]  // the pair's compacted position in each head's block
                               : static_cast<int64_t>(qi[src]) * p.e_sq + static_cast<int64_t>(qj[src]) * p.e_sk;
        float* const dst = (TAN && cb == 1 ? et_b : e_b) + at + 4 * g * hstride;
        const bool with_bias = !(TAN && cb == 1);
#pragma unroll
        for (int m = 0; m < HB; ++m) {
          const float4 bo = lds4(W, L::kBout + 16 * m + 4 * g);
          float val[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) val[r] = (o[m][cb][r] + (with_bias ? comp(bo, r) : 0.0f)) * inv_div;
          if (hstride == 1) {
            *reinterpret_cast<float4*>(dst + 16 * m) = make_float4(val[0], val[1], val[2], val[3]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[(16 * m + r) * hstride] = val[r];
          }
        }
      }
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        qi[cb] = nqi[cb];
        qj[cb] = nqj[cb];
        cpos[cb] = ncpos[cb];
        valid[cb] = nvalid[cb];
      }
    }
  }
}

template <int C, int HB>
hipError_t launch_pb(const PairBiasParams& p, bool tan, int64_t blocks, int cus, hipStream_t stream) {
  const int grid = static_cast<int>(blocks < cus ? blocks : cus);  // one workgroup per CU
  if (tan)
    hipLaunchKernelGGL((pair_bias_kernel<C, HB, true>), dim3(grid), dim3(64 * kPBWaves), 0, stream, p);
  else
    hipLaunchKernelGGL((pair_bias_kernel<C, HB, false>), dim3(grid), dim3(64 * kPBWaves), 0, stream, p);
  return hipGetLastError();
}

template <int C>
hipError_t launch_pb_c(const PairBiasParams& p, int H, bool tan, int64_t blocks, int cus, hipStream_t stream) {
  switch (H) {
    case 16: return launch_pb<C, 1>(p, tan, blocks, cus, stream);
    case 32: return launch_pb<C, 2>(p, tan, blocks, cus, stream);
    case 64: return launch_pb<C, 4>(p, tan, blocks, cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_pair_bias(PairBiasParams p, int C, int H, bool tan, hipStream_t stream) {
  int cus = 0;
  if (hipError_t err = device_cu_count(&cus); err != hipSuccess) return err;
  const int64_t waves = static_cast<int64_t>(cus) * kPBWaves;
  // Parts per walker: about four items per wave, each part at least four tiles.
  const int64_t tp = tan ? 16 : 32;
  const int64_t tiles = (static_cast<int64_t>(p.N) * p.N + tp - 1) / tp;
  int64_t parts = (4 * waves + p.B - 1) / p.B;
  parts = parts > tiles / 4 ? tiles / 4 : parts;
  parts = parts < 1 ? 1 : (parts > 4096 ? 4096 : parts);
  p.parts = static_cast<int>(parts);
  p.n_items = p.B * parts;
  const int64_t blocks = (p.n_items + kPBWaves - 1) / kPBWaves;
  switch (C) {
    case 32: return launch_pb_c<32>(p, H, tan, blocks, cus, stream);
    case 64: return launch_pb_c<64>(p, H, tan, blocks, cus, stream);
    case 96: return launch_pb_c<96>(p, H, tan, blocks, cus, stream);
    case 128: return launch_pb_c<128>(p, H, tan, blocks, cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace hz
