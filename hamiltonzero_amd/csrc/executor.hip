// The compiled per-walker executor's products: the quadrilinear merge of the tree levels and the
// factorized apply ((x V) o h) U of the leaf, merge and readout factors, float32 throughout, their
// products as sums of bfloat16 products (split_f32.h).
//
// Quadrilinear merge, out[m, iR + j] = sum_{k,l} T[i, j, k, l] a[m, iR + k] b[m, iR + l]:
// for one group i and each k the inner sum is a product with a contraction of length R = 32,
//     w_k[j, m] = sum_l T_i[j, k, l] b[m, iR + l],     out_i[m, j] = sum_k a[m, iR + k] w_k[j, m],
// so b is split once and stays in registers, T_i streams through LDS in chunks of four k (48 KB
// for two chunks), split as it is staged, and the outer sum is one multiply-add per element of
// w_k in the matrix cores' output layout (16 vector instructions per 12 matrix ones). The grouping is
// a (T b): where T b underflows float32 its bits are lost, where it overflows the sum is formed again
// as (a b) T. Bound by the
// matrix cores' power: 72% busy at 1.65 GHz, 206 TFLOP/s of float32 products at 32768 rows, G = 48
// (500 us; 1018 with the contraction over (k, l) on the float32 matrix instruction).
//
// Factorized apply: two launches of one tiled GEMM, C = A B with A [M, K], B [K, N]
// row-major; the first multiplies its result by the conditioner row of each output row
// (h[m mod h_rows], one row per tree node, broadcast over walkers) before storing, the
// second optionally adds a residual (the merge level's raw + apply(raw)). 177 TFLOP/s at 65536 rows
// of 1536 x 1024 x 1536 (123 with the float32 matrix instruction), 583 us at 16384 (866).
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "mhsea_device.h"
#include "mhsea_launch.h"
#include "split_f32.h"

// Workspace of hz_factorized_apply_noalloc: kApplyScratchFloats floats (32 MiB) per device,
// held from the library's first use on that device until the process ends. Every call on a
// device shares that device's array, so calls that overlap on one device race.
static __device__ __align__(256) float scratch[hz::kApplyScratchFloats];

namespace hz {
namespace {

// --------------------------------------------------------------------------------------
// Quadrilinear merge (R = 32)
// --------------------------------------------------------------------------------------
constexpr int kQR = 32;            // rank of the merge tensor
constexpr int kQK = 4;             // k per staged chunk of T_i

// Where row m's operands start in ua and ub, in floats. Plain rows (w = 0): m ld_in in both. Rows of
// the pair basis (w node pairs, nq basis rows per leaf, n leaves; see leaf_pair_level_kernel):
// m = (ci nq + cj) w + p takes basis row ci of leaf 2p from ua and cj of leaf 2p + 1 from ub, both
// [nq][n][ld_in].
struct MergeRows {
  int64_t ld_in;
  int w, nq, n;
  __device__ __forceinline__ void at(int64_t m, int64_t& a, int64_t& b) const {
    a = b = m * ld_in;
    if (w == 0) return;
    const int c = static_cast<int>(m / w), p = static_cast<int>(m - static_cast<int64_t>(c) * w);
    const int ci = c / nq, cj = c - ci * nq;
    a = (static_cast<int64_t>(ci) * n + 2 * p) * ld_in;
    b = (static_cast<int64_t>(cj) * n + 2 * p + 1) * ld_in;
  }
};

// A workgroup owns one group i, all 32 outputs j and 128 rows, 32 a wave. 160 registers leave three
// workgroups on a CU (two blocks of rows a wave share the T_i operands but need every register and
// spill: 375 against 246 us at 16384 rows, G = 48).
__global__ void __launch_bounds__(256, 3)
quadrilinear_merge_kernel(const float* __restrict__ T, const float* __restrict__ ua, const float* __restrict__ ub,
                          float* __restrict__ out, int64_t M, int G, MergeRows rows) {
  // [buffer][k][part][l half-block s][64 chunks of 8 l]: chunk (j, h) of block (k, s) at
  // 2 j + (h ^ (j / 4 mod 2)) + (2 k + s), mod 64, which spreads both the eight blocks a row's
  // stores go to and any 8 consecutive lanes of a read over the banks
  __shared__ v4u Ts[2][kQK][3][2][64];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int hh = lane >> 5, c = lane & 31;
  const int i = blockIdx.y;
  const int64_t m0 = (static_cast<int64_t>(blockIdx.x) * 4 + wave) * 32;
  const int64_t ld = static_cast<int64_t>(G) * kQR;  // floats per row of out

  // staging: thread t takes 16 consecutive l of (j = t / 8, k = t / 2 mod 4)
  const int sj = tid >> 3, sk = (tid >> 1) & 3, ss = tid & 1;
  const float* Tp = T + ((static_cast<int64_t>(i) * kQR + sj) * kQR + sk) * kQR + 16 * ss;
  float4 rt[4];
  auto tload = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) rt[u] = *reinterpret_cast<const float4*>(Tp + k0 * kQR + 4 * u);
  };
  auto tstore = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float x[8] = {rt[2 * h].x,     rt[2 * h].y,     rt[2 * h].z,     rt[2 * h].w,
                          rt[2 * h + 1].x, rt[2 * h + 1].y, rt[2 * h + 1].z, rt[2 * h + 1].w};
      const Split8 sp = split8(x);
      const int slot = (2 * sj + (h ^ ((sj >> 2) & 1)) + 2 * sk + ss) & 63;
      Ts[buf][sk][0][ss][slot] = sp.h;
      Ts[buf][sk][1][ss][slot] = sp.m;
      Ts[buf][sk][2][ss][slot] = sp.l;
    }
  };

  // this lane's row (past M the last): b split once, four values of a a chunk
  const int64_t row = m0 + c;
  int64_t ao, bo;
  rows.at(row < M ? row : M - 1, ao, bo);
  const float* const ar = ua + ao + i * kQR;
  const float* const br = ub + bo + i * kQR;
  bf16x8 bs[2][3];
  tload(0);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float4 v0 = *reinterpret_cast<const float4*>(br + 16 * s + 8 * hh);
    const float4 v1 = *reinterpret_cast<const float4*>(br + 16 * s + 8 * hh + 4);
    const float x[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    const Split8 sp = split8(x);
    bs[s][0] = as_bf16x8(sp.h);
    bs[s][1] = as_bf16x8(sp.m);
    bs[s][2] = as_bf16x8(sp.l);
  }
  v4f av = *reinterpret_cast<const v4f*>(ar);
  tstore(0);
  __syncthreads();

  v16f acc = v16f{};
  const int slot0 = 2 * c + (hh ^ ((c >> 2) & 1));
#pragma unroll 1
  for (int ch = 0; ch < kQR / kQK; ++ch) {
    const int buf = ch & 1;
    const bool more = ch + 1 < kQR / kQK;
    v4f an = av;
    if (more) {
      tload((ch + 1) * kQK);
      an = *reinterpret_cast<const v4f*>(ar + (ch + 1) * kQK);
    }
#pragma unroll
    for (int k = 0; k < kQK; ++k) {
      v16f w = v16f{};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int slot = (slot0 + 2 * k + s) & 63;
        bf16x8 t[3];
#pragma unroll
        for (int part = 0; part < 3; ++part) t[part] = as_bf16x8(Ts[buf][k][part][s][slot]);
#pragma unroll
        for (int e = 0; e < kSplitTerms; ++e) w = mfma32_bf16(t[kSplitA[e]], bs[s][kSplitB[e]], w);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = fmaf(w[e], av[k], acc[e]);
    }
    if (more) tstore(buf ^ 1);
    av = an;
    __syncthreads();
  }

  // element e: output j = 8 (e / 4) + 4 hh + e % 4 of row m0 + c
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 16; ++e) bad |= !finite_f32(acc[e]);
  if (__any(bad)) {  // formed again in float32, unless a NaN of the row's operands made them
    bool nan = false;
#pragma unroll
    for (int q = 0; q < kQR / 4; ++q) {
      const v4f x = *reinterpret_cast<const v4f*>(ar + 4 * q), y = *reinterpret_cast<const v4f*>(br + 4 * q);
#pragma unroll
      for (int u = 0; u < 4; ++u) nan |= x[u] != x[u] || y[u] != y[u];
    }
    bad = bad && !nan && row < M;
    if (__any(bad)) {
      const float* const tj = T + (static_cast<int64_t>(i) * kQR + c) * kQR * kQR + 4 * hh;
      v16f w = v16f{};
#pragma unroll 1
      for (int k = 0; k < kQR; ++k) {
        const float ak = ar[k];
        v4f t[4], y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          t[q] = *reinterpret_cast<const v4f*>(tj + k * kQR + 8 * q);
          y[q] = *reinterpret_cast<const v4f*>(br + 4 * hh + 8 * q);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int u = 0; u < 4; ++u) w = mfma32_f32(t[q][u], ak * y[q][u], w);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (bad && !finite_f32(acc[e])) acc[e] = w[e];
    }
  }
  if (row < M) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<v4f*>(out + row * ld + i * kQR + 8 * q + 4 * hh) =
          v4f{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
}

// --------------------------------------------------------------------------------------
// Tiled GEMM with epilogues
// --------------------------------------------------------------------------------------
constexpr int kBM = 128, kBN = 128, kBK = 16;

constexpr int kAhead = 2;  // K slices in flight in registers (even)

enum GemmEpi { kEpiPlain = 0, kEpiCond = 1, kEpiResidual = 2, kEpiRowMask = 3 };

// C[M, N] = A[M, K] B[K, N] (row-major); EPI: kEpiCond multiplies C[m, n] by
// h[((row0 + m) mod h_rows) * N + n] (row0: the first row's index in the caller's full
// row range, nonzero when the rows are processed in chunks); kEpiResidual adds res[m, n];
// kEpiRowMask multiplies row m by (mask[m] != 0), aux then being a uint8 mask.
// C may be the residual itself (each output entry reads its residual entry, then overwrites
// it, in one thread), so neither carries __restrict__. VEC: K is a multiple of 4 (16-byte loads
// of A); otherwise those loads are per element.
// Split K (gridDim.z > 1): workgroup z contracts k in [z K, min(z K + K, Ktot)) of A (row
// stride lda) and B and writes its partial product (EPI plain) at C + z cz.
//
// float32 products as six bfloat16 products (split_f32.h), K slices of 16 (one matrix step). A
// workgroup owns 128 rows x 128 columns, a wave 32 rows and every column: its rows of A go from
// memory to the wave's registers (8 consecutive k per lane, split there, so no two waves split
// the same row), the slice's columns of B through LDS, double-buffered, as their three bfloat16
// parts: a column is 2 chunks of 8 k (16 bytes, one operand read), chunk h of column n at
// h ^ ((n / 4) mod 2), which spreads any 8 consecutive lanes of a read or a store over all banks.
// Sums that are not finite are formed again on the float32 instruction, a wave's 32 x 32 block at a
// time, unless a NaN in the row of A made them: a diverged walker's row costs nothing, one with an
// infinity 0.4 ms where the wave comes last (16384 rows, K = 1536; 1.7 ms with a lane's own loop
// per sum).
// A thread stages 8 k of one column. Loads run kAhead slices ahead of their products (1024 rows,
// one workgroup to a CU: 202 us with one slice, 166 with two, 167 with four).
template <int EPI, bool VEC>
__global__ void __launch_bounds__(256, 3)
gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ Bm, float* C, const float* aux, int64_t M, int N,
                int K, int h_rows, int64_t row0, int lda, int Ktot, int64_t cz) {
  {
    const int kbeg = static_cast<int>(blockIdx.z) * K;
    A += kbeg;
    Bm += static_cast<int64_t>(kbeg) * N;
    C += static_cast<int64_t>(blockIdx.z) * cz;
    K = Ktot - kbeg < K ? Ktot - kbeg : K;
  }
  constexpr int kPart = 2 * kBN;  // 16-byte chunks of one part of B's slice
  __shared__ v4u smem[2][3 * kPart];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, c = lane & 31;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kBM + wave * 32;
  const int n0 = blockIdx.x * kBN;

  // Rows and columns past the matrix repeat its last (their sums are not stored).
  const float* const Ap = A + (m0 + c < M ? m0 + c : M - 1) * lda + 8 * hh;
  const int bc = tid & 127, bh = wave >> 1;  // this thread's column and k half of B's slice
  const int bn = n0 + bc < N ? n0 + bc : N - 1;
  const int bslot = 2 * bc + (bh ^ ((bc >> 2) & 1));
  float ra[kAhead][8], rb[kAhead][8];
  // a whole slice: no bounds, so nothing waits for these loads before they are staged
  auto gload = [&](int k0, float (&ra)[8], float (&rb)[8]) {
    if constexpr (VEC) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const v4f v = *reinterpret_cast<const v4f*>(Ap + k0 + 4 * u);
#pragma unroll
        for (int i = 0; i < 4; ++i) ra[4 * u + i] = v[i];
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) ra[u] = Ap[k0 + u];
    }
    const float* const bk = Bm + static_cast<int64_t>(k0 + 8 * bh) * N;
#pragma unroll
    for (int u = 0; u < 8; ++u) rb[u] = (bk + static_cast<int64_t>(u) * N)[bn];
  };
  // the last slice where K is not a multiple of 16, zeros past K
  auto gload_tail = [&](int k0, float (&ra)[8], float (&rb)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int ka = k0 + 8 * hh + u, kb = k0 + 8 * bh + u;
      ra[u] = ka < K ? Ap[k0 + u] : 0.f;
      rb[u] = kb < K ? Bm[static_cast<int64_t>(kb) * N + bn] : 0.f;
    }
  };
  bf16x8 af[3];
  auto stage = [&](int buf, const float (&ra)[8], const float (&rb)[8]) {
    const Split8 sa = split8(ra), sb = split8(rb);
    af[0] = as_bf16x8(sa.h);
    af[1] = as_bf16x8(sa.m);
    af[2] = as_bf16x8(sa.l);
    smem[buf][bslot] = sb.h;
    smem[buf][kPart + bslot] = sb.m;
    smem[buf][2 * kPart + bslot] = sb.l;
  };

  constexpr int NT = kBN / 32;
  v16f acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = v16f{};

  const int rd = 2 * c + (hh ^ ((c >> 2) & 1));  // this lane's chunk of column c of a block
  auto products = [&](int buf) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      bf16x8 bf[3];
#pragma unroll
      for (int part = 0; part < 3; ++part) bf[part] = as_bf16x8(smem[buf][part * kPart + 64 * nt + rd]);
#pragma unroll
      for (int s = 0; s < kSplitTerms; ++s) acc[nt] = mfma32_bf16(af[kSplitA[s]], bf[kSplitB[s]], acc[nt]);
    }
  };
  // Slice kt in LDS buffer kt mod 2 and, on its way there, register set kt mod kAhead; loads past
  // the last whole slice repeat it.
  const int nf = K / kBK;
  if (nf > 0) {
    auto at = [&](int kt) { return (kt < nf ? kt : nf - 1) * kBK; };
#pragma unroll
    for (int j = 0; j < kAhead; ++j) gload(at(j), ra[j], rb[j]);
    stage(0, ra[0], rb[0]);
    __syncthreads();
    for (int kt = 0; kt < nf; kt += kAhead) {
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        if (kt + j == nf) break;
        gload(at(kt + j + kAhead), ra[j], rb[j]);
        products(j & 1);
        stage((j + 1) & 1, ra[(j + 1) % kAhead], rb[(j + 1) % kAhead]);
        __syncthreads();
      }
    }
  }
  if (nf * kBK < K) {
    gload_tail(nf * kBK, ra[0], rb[0]);
    stage(0, ra[0], rb[0]);
    __syncthreads();
    products(0);
  }
  __syncthreads();  // smem is free for the epilogue

  // element i of block nt: row m0 + 8 (i / 4) + 4 hh + i % 4, column n0 + 32 nt + c
  auto row_of = [&](int i) { return m0 + 8 * (i >> 2) + 4 * hh + (i & 3); };
  uint32_t top = 0;  // (the largest magnitude: as 64 tests their masks would spill)
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t mag = __float_as_uint(acc[nt][i]) & 0x7fffffffu;
      top = top > mag ? top : mag;
    }
  if (__any(top >= 0x7f800000u)) {  // formed again in float32, unless a NaN in the row of A made them
    const float* const arow = Ap - 8 * hh;
    bool nan = false;
#pragma unroll 4
    for (int k = hh; k < K; k += 2) nan |= arow[k] != arow[k];
    const uint64_t lanes = __ballot(nan || m0 + c >= M);
    const unsigned rows = static_cast<unsigned>(lanes | (lanes >> 32)) >> (4 * hh);
    float* const mine = reinterpret_cast<float*>(&smem[0][0]) + wave * 1024 + lane;  // what stands
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int col = n0 + 32 * nt + c;
      bool again = false;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool stands = finite_f32(acc[nt][i]) || (rows >> (8 * (i >> 2) + (i & 3)) & 1u) != 0;
        again |= !stands;
        mine[64 * i] = stands ? acc[nt][i] : __builtin_inff();
      }
      if (!__any(again && col < N)) continue;
      acc[nt] = v16f{};
      const float* const bcol = Bm + (col < N ? col : N - 1);
#pragma unroll 1
      for (int k0 = 0; k0 < K; k0 += 16) {
        float x[8], y[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int k = k0 + 8 * hh + u, kc = k < K ? k : K - 1;
          const float xa = arow[kc], yb = bcol[static_cast<int64_t>(kc) * N];
          x[u] = k < K ? xa : 0.f;
          y[u] = k < K ? yb : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[nt] = mfma32_f32(x[u], y[u], acc[nt]);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float v = mine[64 * i];
        if (finite_f32(v) || v != v) acc[nt][i] = v;
      }
    }
  }
  unsigned hrow[16];
  if constexpr (EPI == kEpiCond) {
    const unsigned hbase = static_cast<unsigned>((row0 + m0) % h_rows);
#pragma unroll
    for (int i = 0; i < 16; ++i) hrow[i] = (hbase + static_cast<unsigned>(row_of(i) - m0)) % static_cast<unsigned>(h_rows);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int col = n0 + 32 * nt + c;
    if (col >= N) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t row = row_of(i);
      if (row >= M) continue;
      float v = acc[nt][i];
      if constexpr (EPI == kEpiCond) v *= aux[static_cast<int64_t>(hrow[i]) * N + col];
      if constexpr (EPI == kEpiResidual) v += aux[row * N + col];
      if constexpr (EPI == kEpiRowMask) v *= reinterpret_cast<const uint8_t*>(aux)[row] != 0 ? 1.f : 0.f;
      C[row * N + col] = v;
    }
  }
}

// Site-masked product C[m, :] = mask[m] != 0 ? A[m, :] B : 0 with the masked rows skipped.
// A workgroup takes kRM rows of A and one 128-column tile of C: its physical rows (in order)
// are compacted into the LDS tile, so only ceil(n / 16) row blocks are multiplied, and its
// masked rows of C are written as zeros. Wave w owns columns [32 w, 32 w + 32) of the tile for
// every row block. Workgroups are numbered so that the column tiles of one row block run on
// one XCD (one L2 holds their A rows). K and N are multiples of 4 (16-byte loads of A, stores of
// zeros). float32 products as six bfloat16 ones (split_f32.h): the slice's rows are split once, by
// all threads, into 48 KB of LDS that every wave reads; a wave's columns of B come from memory to its
// registers and are split there, a slice ahead of their products. Two workgroups of 50 KB and 244
// registers a CU, so one stages under the other's products. Bound by memory (its output alone is
// 134 MB) and the splits: 65536 rows, 36 of 64 physical, 256 x 512, y and its tangent 214 -> 155 us
// (the float32 matrix instruction was 53% busy).
constexpr int kRM = 256;  // 16 row blocks: the dispatch below instantiates 1..16
constexpr int kRK = 32;   // K per slice: one matrix step

__global__ void __launch_bounds__(256, 2)
gemm_rows_f32_kernel(const float* __restrict__ A, const float* __restrict__ Bm, float* __restrict__ C,
                     const uint8_t* __restrict__ mask, int64_t M, int N, int K, int ncol) {
  // a slice of A as ready operands, [row block][part][64 lanes]: slot s's chunk of lane group g at
  // lane 16 g + (s mod 16 ^ 2 g), which spreads any 8 consecutive lanes of a store or a read over
  // the banks
  __shared__ v4u As[kRM / 16 * 3 * 64];
  __shared__ int16_t prow[kRM], mrow[kRM];
  __shared__ int counts[8];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int64_t L = xcd_logical_block(blockIdx.x, gridDim.x);
  const int64_t m0 = (L / ncol) * kRM;
  const int n0 = static_cast<int>(L % ncol) * kBN;
  const int wn = wave * 32;

  // ---- this workgroup's physical and masked rows, each list in ascending order ---------
  const bool valid = m0 + tid < M;
  const bool phys = valid && mask[m0 + tid] != 0;
  const uint64_t pb = __ballot(phys), mb = __ballot(valid && !phys);
  const uint64_t below = (uint64_t(1) << lane) - 1;
  if (lane == 0) {
    counts[wave] = __popcll(pb);
    counts[4 + wave] = __popcll(mb);
  }
  __syncthreads();
  int pbase = 0, mbase = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    pbase += w < wave ? counts[w] : 0;
    mbase += w < wave ? counts[4 + w] : 0;
  }
  const int n = counts[0] + counts[1] + counts[2] + counts[3];
  const int nm = counts[4] + counts[5] + counts[6] + counts[7];
  if (phys) prow[pbase + __popcll(pb & below)] = static_cast<int16_t>(tid);
  if (valid && !phys) mrow[mbase + __popcll(mb & below)] = static_cast<int16_t>(tid);
  __syncthreads();

  // masked rows: the workgroup of column tile t writes the whole rows (every column) of the
  // masked rows i = t, t + ncol, ... of its row block, each row one contiguous run
  {
    const int t = static_cast<int>(L % ncol);
    const int nmine = nm > t ? (nm - t + ncol - 1) / ncol : 0;
    const int n4 = N / 4;
    for (int i = tid; i < nmine * n4; i += 256) {
      const int mi = t + (i / n4) * ncol;
      *reinterpret_cast<float4*>(C + (m0 + mrow[mi]) * N + 4 * (i % n4)) = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  if (n == 0) return;  // workgroup-uniform

  // the K loop and the stores for NMT = ceil(n / 16) row blocks, a compile-time count so
  // the products run without branches
  auto body = [&](auto nmt_c) {
    constexpr int NMT = decltype(nmt_c)::value;
    constexpr int NU = (NMT + 3) / 4;  // chunks of 8 k of one slot a thread stages
    // chunk it = tid + 256 u: slot it / 4, lane group it mod 4; slots past n are zero
    const int sg = tid & 3;
    const float* ap[NU];
    bool aok[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int slot = (tid >> 2) + 64 * u;
      aok[u] = slot < n;
      ap[u] = A + (m0 + prow[aok[u] ? slot : 0]) * K;
    }
    const int bn[2] = {n0 + wn + c < N ? n0 + wn + c : N - 1, n0 + wn + 16 + c < N ? n0 + wn + 16 + c : N - 1};
    float4 ra[NU][2];
    float rb[2][8];
    // zeros past K in A; B repeats its last row there
    auto gload = [&](int k0) {
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const int kk = k0 + 8 * sg + 4 * v;
          ra[u][v] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (aok[u] && kk < K) ra[u][v] = *reinterpret_cast<const float4*>(ap[u] + kk);
        }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int kk = k0 + 8 * g + j;
        const float* const br = Bm + static_cast<int64_t>(kk < K ? kk : K - 1) * N;
        rb[0][j] = br[bn[0]];
        rb[1][j] = br[bn[1]];
      }
    };
    auto sstore = [&]() {
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int slot = (tid >> 2) + 64 * u;
        const float x[8] = {ra[u][0].x, ra[u][0].y, ra[u][0].z, ra[u][0].w,
                            ra[u][1].x, ra[u][1].y, ra[u][1].z, ra[u][1].w};
        const Split8 sp = split8(x);
        v4u* const d = As + (slot >> 4) * (3 * 64) + 16 * sg + ((slot & 15) ^ (2 * sg));
        d[0] = sp.h;
        d[64] = sp.m;
        d[128] = sp.l;
      }
    };
    v4f acc[NMT][2];
#pragma unroll
    for (int mt = 0; mt < NMT; ++mt) acc[mt][0] = acc[mt][1] = zero4();
    const v4u* const rd = As + 16 * g + (c ^ (2 * g));
    gload(0);
    for (int k0 = 0; k0 < K; k0 += kRK) {
      if (k0 > 0) __syncthreads();  // the last slice's readers are done
      sstore();
      const Split8 b0 = split8(rb[0]), b1 = split8(rb[1]);
      __syncthreads();
      if (k0 + kRK < K) gload(k0 + kRK);
      mm_step<NMT>(rd, b0, b1, acc);
    }
    // lane (g, c) holds C[prow[16 mt + 4 g + r]][n0 + wn + 16 nt + c]
    bool bad = false;
#pragma unroll
    for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int slot = 16 * mt + 4 * g + r;
        const int64_t row = m0 + prow[slot < n ? slot : 0];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int col = n0 + wn + 16 * nt + c;
          bad |= !finite_f32(acc[mt][nt][r]);
          if (slot < n && col < N) C[row * N + col] = acc[mt][nt][r];
        }
      }
    // formed again in float32, unless a NaN in the row of A made them (a lane reads back only what it
    // stored)
    if (__any(bad)) {
#pragma unroll 1
      for (int mt = 0; mt < NMT; ++mt) {
        unsigned again = 0;  // element 4 nt + r
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int slot = 16 * mt + 4 * g + (e & 3), col = n0 + wn + 16 * (e >> 2) + c;
          if (slot < n && col < N && !finite_f32(C[(m0 + prow[slot]) * N + col])) again |= 1u << e;
        }
        if (!__any(again != 0)) continue;
        const int slot_a = 16 * mt + c;
        const float* const arow = A + (m0 + prow[slot_a < n ? slot_a : 0]) * K;
        bool nan = false;
#pragma unroll 4
        for (int k = 4 * g; k < K; k += 16) {
          const v4f x = *reinterpret_cast<const v4f*>(arow + k);
#pragma unroll
          for (int u = 0; u < 4; ++u) nan |= x[u] != x[u];
        }
        uint64_t lanes = __ballot(nan);
        lanes |= lanes >> 32;
        const unsigned rows = static_cast<unsigned>(lanes | (lanes >> 16)) >> (4 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (rows >> (e & 3) & 1) again &= ~(1u << e);
        if (!__any(again != 0)) continue;
        v4f w[2] = {zero4(), zero4()};
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += 16) {
          const int k = k0 + 4 * g;
          v4f x = zero4();
          if (k < K) x = *reinterpret_cast<const v4f*>(arow + k);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float* const br = Bm + static_cast<int64_t>(k < K ? k + u : 0) * N;
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) w[nt] = mfma16x4(x[u], k < K ? br[bn[nt]] : 0.f, w[nt]);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (again >> e & 1)
            C[(m0 + prow[16 * mt + 4 * g + (e & 3)]) * N + n0 + wn + 16 * (e >> 2) + c] = w[e >> 2][e & 3];
      }
    }
  };
  using std::integral_constant;
  switch ((n + 15) >> 4) {
    case 1: body(integral_constant<int, 1>{}); break;
    case 2: body(integral_constant<int, 2>{}); break;
    case 3: body(integral_constant<int, 3>{}); break;
    case 4: body(integral_constant<int, 4>{}); break;
    case 5: body(integral_constant<int, 5>{}); break;
    case 6: body(integral_constant<int, 6>{}); break;
    case 7: body(integral_constant<int, 7>{}); break;
    case 8: body(integral_constant<int, 8>{}); break;
    case 9: body(integral_constant<int, 9>{}); break;
    case 10: body(integral_constant<int, 10>{}); break;
    case 11: body(integral_constant<int, 11>{}); break;
    case 12: body(integral_constant<int, 12>{}); break;
    case 13: body(integral_constant<int, 13>{}); break;
    case 14: body(integral_constant<int, 14>{}); break;
    case 15: body(integral_constant<int, 15>{}); break;
    default: body(integral_constant<int, 16>{}); break;
  }
}

// Sum of the split-K partial products P[z] (z in order) with the GEMM's epilogue; N % 4 == 0.
// C may be the residual (aux): each element reads it, then overwrites it, in one thread.
template <int EPI>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ P, float* C, const float* aux,
                                                            int64_t M, int N, int S, int64_t cz, int h_rows,
                                                            int64_t row0) {
  const int64_t i4 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i4 >= M * N / 4) return;
  float4 v = *reinterpret_cast<const float4*>(P + 4 * i4);
  for (int z = 1; z < S; ++z) {
    const float4 w = *reinterpret_cast<const float4*>(P + z * cz + 4 * i4);
    v.x += w.x;
    v.y += w.y;
    v.z += w.z;
    v.w += w.w;
  }
  const int64_t row = 4 * i4 / N;
  const int col = static_cast<int>(4 * i4 - row * N);
  if constexpr (EPI == kEpiCond) {
    const float4 hv = *reinterpret_cast<const float4*>(aux + ((row0 + row) % h_rows) * N + col);
    v.x *= hv.x;
    v.y *= hv.y;
    v.z *= hv.z;
    v.w *= hv.w;
  }
  if constexpr (EPI == kEpiResidual) {
    const float4 rv = *reinterpret_cast<const float4*>(aux + row * N + col);
    v.x += rv.x;
    v.y += rv.y;
    v.z += rv.z;
    v.w += rv.w;
  }
  if constexpr (EPI == kEpiRowMask) {
    const float mk = reinterpret_cast<const uint8_t*>(aux)[row] != 0 ? 1.f : 0.f;
    v.x *= mk;
    v.y *= mk;
    v.z *= mk;
    v.w *= mk;
  }
  *reinterpret_cast<float4*>(C + 4 * i4) = v;
}

// One launch; parts > 1: split K.
template <int EPI>
hipError_t launch_tiles(const float* A, const float* B, float* C, const float* aux, int64_t M, int N, int kp, int parts,
                        int h_rows, int64_t row0, int K, int64_t cz, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((N + kBN - 1) / kBN), static_cast<unsigned>((M + kBM - 1) / kBM),
                  static_cast<unsigned>(parts));
  auto kern = K % 4 == 0 ? gemm_f32_kernel<EPI, true> : gemm_f32_kernel<EPI, false>;
  hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, A, B, C, aux, M, N, kp, h_rows, row0, K, K, cz);
  return hipGetLastError();
}

template <int EPI>
hipError_t launch_gemm(const float* A, const float* B, float* C, const float* aux, int64_t M, int N, int K,
                       int h_rows, int64_t row0, hipStream_t stream, float* split_ws = nullptr,
                       int64_t split_cap = 0) {
  // Split K where the tiles leave most CUs idle (the tree's deep levels: 1024-4096 rows,
  // 64-512 tiles of 96-step K chains): S parts of K into split_ws [S, M, N], then one pass
  // that sums the parts in order and applies the epilogue (deterministic).
  if (split_ws != nullptr && N % 4 == 0 && K % 4 == 0 && K >= 256) {
    int cus = 0;
    if (hipError_t err = device_cu_count(&cus); err != hipSuccess) return err;
    const int64_t tiles = static_cast<int64_t>((N + kBN - 1) / kBN) * ((M + kBM - 1) / kBM);
    const int64_t mn = M * N;
    int64_t S = tiles < cus ? (2 * cus + tiles - 1) / tiles : 1;
    S = S > 8 ? 8 : S;
    S = S > K / 128 ? K / 128 : S;
    S = S > split_cap / mn ? split_cap / mn : S;
    if (S >= 2) {
      const int kp = static_cast<int>(((K + S - 1) / S + kBK - 1) / kBK * kBK);
      const int parts = (K + kp - 1) / kp;
      if (hipError_t err = launch_tiles<kEpiPlain>(A, B, split_ws, nullptr, M, N, kp, parts, 1, 0, K, mn, stream);
          err != hipSuccess)
        return err;
      const int64_t n4 = mn / 4;
      hipLaunchKernelGGL((splitk_reduce_kernel<EPI>), dim3(static_cast<unsigned>((n4 + 255) / 256)), dim3(256), 0,
                         stream, split_ws, C, aux, M, N, parts, mn, h_rows, row0);
      return hipGetLastError();
    }
  }
  return launch_tiles<EPI>(A, B, C, aux, M, N, K, 1, h_rows, row0, K, 0, stream);
}

// One factorized apply over rows [row0, row0 + M) of the caller's range: x, residual and y
// point at row row0; work holds M x R floats; split_ws (split_cap floats, may be null) is free
// scratch for split-K partial products.
hipError_t apply_rows(const float* x, const float* V, const float* h, const float* U, const float* residual,
                      float* y, float* work, int64_t M, int d_in, int R, int d_out, int h_rows, int64_t row0,
                      hipStream_t stream, float* split_ws = nullptr, int64_t split_cap = 0) {
  hipError_t err = launch_gemm<kEpiCond>(x, V, work, h, M, R, d_in, h_rows, row0, stream, split_ws, split_cap);
  if (err != hipSuccess) return err;
  if (residual != nullptr)
    return launch_gemm<kEpiResidual>(work, U, y, residual, M, d_out, R, 1, 0, stream, split_ws, split_cap);
  return launch_gemm<kEpiPlain>(work, U, y, nullptr, M, d_out, R, 1, 0, stream, split_ws, split_cap);
}

// Device addresses of the no-alloc workspace, one per device, resolved on first use.
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxScratchDevices] = {};

// --------------------------------------------------------------------------------------
// Row epilogues of the executor, one wave per row of d floats (d a multiple of 4,
// d <= 64 * 4 * kRowVec): the leaf carriers' RMS normalisation, a level's rescale and
// opcode gate, and the readout's log|psi| and phase. Each row's sum of squares is reduced
// across the wave in a fixed order (results reproducible run to run).
// --------------------------------------------------------------------------------------
constexpr int kRowVec = 8;  // float4 per lane: rows up to 2048 floats

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__device__ __forceinline__ float sum_sq(const float4& v) { return v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w; }

// u[m, :] /= rms, s[m] = log(rms), rms = sqrt(mean(u[m]^2) + 1e-30)
__global__ void __launch_bounds__(256) normalize_rows_kernel(float* __restrict__ u, float* __restrict__ s, int64_t M,
                                                              int d) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  float4* ur = reinterpret_cast<float4*>(u + row * d);
  const int d4 = d / 4;
  float4 v[kRowVec];
  float ss = 0.f;
#pragma unroll
  for (int t = 0; t < kRowVec; ++t) {
    const int c4 = lane + 64 * t;
    v[t] = c4 < d4 ? ur[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
    ss += sum_sq(v[t]);
  }
  ss = wave_sum(ss);
  const float rms = sqrtf(ss / static_cast<float>(d) + 1e-30f);
#pragma unroll
  for (int t = 0; t < kRowVec; ++t) {
    const int c4 = lane + 64 * t;
    if (c4 < d4) ur[c4] = make_float4(v[t].x / rms, v[t].y / rms, v[t].z / rms, v[t].w / rms);
  }
  if (lane == 0) s[row] = logf(rms);
}

// One tree level's epilogue for output row m = (walker, node p), M = walkers x width:
//   scale = sqrt(mean(out[m]^2) + eps), candidate = out[m] / scale,
//   u'[m] = both * candidate + left * u[2m] + right * u[2m + 1]   (gates from opcode[p])
//   s'[m] = both * (s[2m] + s[2m + 1] + log(scale)) + left * s[2m] + right * s[2m + 1]
__global__ void __launch_bounds__(256) level_gate_kernel(const float* __restrict__ out, const float* __restrict__ u_in,
                                                          const float* __restrict__ s_in,
                                                          const uint8_t* __restrict__ opcodes, float* __restrict__ u_out,
                                                          float* __restrict__ s_out, int64_t M, int width, int d,
                                                          float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const int d4 = d / 4;
  const float4* orow = reinterpret_cast<const float4*>(out + row * d);
  const float4* lrow = reinterpret_cast<const float4*>(u_in + 2 * row * d);
  const float4* rrow = lrow + d4;
  float4 v[kRowVec];
  float ss = 0.f;
#pragma unroll
  for (int t = 0; t < kRowVec; ++t) {
    const int c4 = lane + 64 * t;
    v[t] = c4 < d4 ? orow[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
    ss += sum_sq(v[t]);
  }
  ss = wave_sum(ss);
  const float scale = sqrtf(ss / static_cast<float>(d) + eps);
  const int op = opcodes[row % width];
  const float both = op == 0 ? 1.f : 0.f, left = op == 1 ? 1.f : 0.f, right = op == 2 ? 1.f : 0.f;
  float4* urow = reinterpret_cast<float4*>(u_out + row * d);
#pragma unroll
  for (int t = 0; t < kRowVec; ++t) {
    const int c4 = lane + 64 * t;
    if (c4 < d4) {
      const float4 a = lrow[c4], b = rrow[c4];
      float4 r;
      r.x = both * (v[t].x / scale) + left * a.x + right * b.x;
      r.y = both * (v[t].y / scale) + left * a.y + right * b.y;
      r.z = both * (v[t].z / scale) + left * a.z + right * b.z;
      r.w = both * (v[t].w / scale) + left * a.w + right * b.w;
      urow[c4] = r;
    }
  }
  if (lane == 0) {
    const float sl = s_in[2 * row], sr = s_in[2 * row + 1];
    s_out[row] = both * (sl + sr + logf(scale)) + left * sl + right * sr;
  }
}

// log|psi| = 0.5 log(re^2 + im^2) + s_root, phase = atan2(im, re); psi [B, 2]
__global__ void __launch_bounds__(256) readout_kernel(const float* __restrict__ psi, const float* __restrict__ s_root,
                                                       float* __restrict__ log_abs, float* __restrict__ phase, int64_t B) {
  const int64_t b = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (b >= B) return;
  const float re = psi[2 * b], im = psi[2 * b + 1];
  log_abs[b] = 0.5f * logf(re * re + im * im) + s_root[b];
  phase[b] = atan2f(im, re);
}

// --------------------------------------------------------------------------------------
// The leaf and the first level through a basis of the walkers' inputs
// --------------------------------------------------------------------------------------
// Everything from a site's input q [nq] to the first merge is linear in q: the leaf carrier is
// u = sum_c q_c E[c], E[c] = ((W_q[c] V) o h) U, and a node of the first level is bilinear in the two
// leaves' inputs. So the leaf's and the first level's products run on nq rows per leaf and nq^2
// rows per pair instead of on every walker's rows. At 1024 walkers of 64 sites with nq = 4 the
// products fall from 65536 leaf and 32768 pair rows to 256 and 512.
// A sum over E itself would lose what the inputs cancel (a carrier kappa times smaller than its
// terms), and a node the product of what its two leaves cancel. So E is formed in 64 bits and each
// leaf's rows are made orthonormal there (orthonormal_basis_kernel): E[c] = sum_a R[a, c] Q[a] with
// mean(Q[a] Q[b]) = (a == b). A walker's coefficients y = R q are 64-bit sums, its carrier's rms is
// |y|, and the node is out = sum_ab (y_a / |y|) (y'_b / |y'|) O[a, b] with O the level's merge and
// residual apply of Q[a] and Q'[b]: terms of the node's own size, whatever q cancels. The node's
// error against 64 bits stays below 1e-6 for inputs that cancel by up to 1e5, where the products on
// every walker's rows lose 2.6e-3.
constexpr int kMaxBasis = 4;  // inputs per site the pair basis serves (one K step of the products)

typedef double v4d __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256) leaf_basis_kernel(const float* __restrict__ Wq, const float* __restrict__ V,
                                                         const float* __restrict__ h, double* __restrict__ out, int n,
                                                         int d_z, int R) {
  // out[(c n + s) R + r] = (sum_z W_q[c, z] V[z, r]) h[s, r]
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= R) return;
  const int c = blockIdx.y;
  double a = 0.0;
#pragma unroll 8
  for (int z = 0; z < d_z; ++z)
    a = fma(static_cast<double>(Wq[static_cast<int64_t>(c) * d_z + z]),
            static_cast<double>(V[static_cast<int64_t>(z) * R + r]), a);
  for (int s = blockIdx.z; s < n; s += gridDim.z)
    out[(static_cast<int64_t>(c) * n + s) * R + r] = a * h[static_cast<int64_t>(s) * R + r];
}

// C[M, N] = A[M, K] B[K, N] in 64 bits, B held in 32 (the leaf basis times the leaf's U). A workgroup
// owns 16 rows x 32 columns, its four waves every fourth K block of 16 each, summed through LDS in
// order. v_mfma_f64_16x16x4_f64, lane l = 16 g + c: A[row c][k g], B[k g][col c], C/D element r at
// [row g + 4 r][col c]; a lane's four k of a block are 4 g .. 4 g + 3 in both operands, its two columns
// neighbours. N is a multiple of 32. 34 us for 256 x 1536 x 1536 (15 at the 64-bit matrix rate): few
// workgroups, each waiting for its operands.
__global__ void __launch_bounds__(256) basis_gemm_f64_kernel(const double* __restrict__ A, const float* __restrict__ Bm,
                                                             double* __restrict__ C, int64_t M, int N, int K) {
  __shared__ double part[4][8][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * 16;
  const int n0 = blockIdx.x * 32;
  const double* const ar = A + (m0 + c < M ? m0 + c : M - 1) * K;  // rows past M repeat the last, not stored
  const float* const bc = Bm + n0 + 2 * c;
  v4d acc[2] = {v4d{0.0, 0.0, 0.0, 0.0}, v4d{0.0, 0.0, 0.0, 0.0}};
  auto step = [&](double a, float b0, float b1) {
    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, static_cast<double>(b0), acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, static_cast<double>(b1), acc[1], 0, 0, 0);
  };
  const int whole = K / 16;
  // this wave's blocks wave, wave + 4, ..., the operands of three in flight beside one's products
  constexpr int kDeep = 4;
  const int mine = (whole - wave + 3) >> 2;
  double a[kDeep][4];
  float2 b[kDeep][4];
  auto load = [&](int i, double (&a)[4], float2 (&b)[4]) {
    const int k0 = 16 * (wave + 4 * (i < mine ? i : mine - 1)) + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[j] = ar[k0 + j];
      b[j] = *reinterpret_cast<const float2*>(bc + static_cast<int64_t>(k0 + j) * N);
    }
  };
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < kDeep - 1; ++i) load(i, a[i], b[i]);
    for (int i0 = 0; i0 < mine; i0 += kDeep) {
#pragma unroll
      for (int i = 0; i < kDeep; ++i) {
        if (i0 + i == mine) break;
        load(i0 + i + kDeep - 1, a[(i + kDeep - 1) % kDeep], b[(i + kDeep - 1) % kDeep]);
#pragma unroll
        for (int j = 0; j < 4; ++j) step(a[i][j], b[i][j].x, b[i][j].y);
      }
    }
  }
  if (whole * 16 < K && wave == (whole & 3)) {  // the last K block, zeros past K
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 16 * whole + 4 * g + j;
      const float* const bk = bc + static_cast<int64_t>(k < K ? k : 0) * N;
      step(k < K ? ar[k] : 0.0, k < K ? bk[0] : 0.f, k < K ? bk[1] : 0.f);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    part[wave][2 * r][lane] = acc[0][r];
    part[wave][2 * r + 1][lane] = acc[1][r];
  }
  __syncthreads();
  // wave w stores element r = w of both blocks
  const int64_t row = m0 + g + 4 * wave;
  if (row < M) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = 2 * wave + j;
      C[row * N + n0 + 2 * c + j] = (part[0][e][lane] + part[1][e][lane]) + (part[2][e][lane] + part[3][e][lane]);
    }
  }
}

// One leaf's nq rows E (64 bits, [nq][n][d]) made orthonormal: Q [nq][n][d] in 32 bits with
// mean(Q_a Q_b) = (a == b), R [n][nq][nq] in 64 bits with E_c = sum_a R[a, c] Q_a (Gram-Schmidt, each
// row projected twice). A row whose rest is below 2^-40 of itself depends on the rows before it: its
// Q and its row of R are zeros, and what is left out is 2^-40 of E_c. One workgroup a leaf, a row
// eight values a thread; d <= 2048.
__global__ void __launch_bounds__(256) orthonormal_basis_kernel(const double* __restrict__ E, float* __restrict__ Q,
                                                                double* __restrict__ R, int n, int nq, int d) {
  constexpr int kPer = 8;
  __shared__ double red[2][4][kMaxBasis];
  const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double inv_d = 1.0 / static_cast<double>(d);
  int turn = 0;
  // mean over the row of NV products, in every thread
  auto means = [&](double (&v)[kMaxBasis], int count) {
#pragma unroll
    for (int i = 0; i < kMaxBasis; ++i)
      if (i < count)
        for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_xor(v[i], off);
    if (lane == 0)
#pragma unroll
      for (int i = 0; i < kMaxBasis; ++i) red[turn][wave][i] = v[i];
    __syncthreads();  // (two buffers: the last means' readers are behind this barrier)
#pragma unroll
    for (int i = 0; i < kMaxBasis; ++i)
      v[i] = ((red[turn][0][i] + red[turn][1][i]) + (red[turn][2][i] + red[turn][3][i])) * inv_d;
    turn ^= 1;
  };
  double basis[kMaxBasis][kPer];
  double* const Rs = R + static_cast<int64_t>(s) * nq * nq;
#pragma unroll
  for (int a = 0; a < kMaxBasis; ++a) {
    if (a >= nq) break;
    const int64_t at = (static_cast<int64_t>(a) * n + s) * d;
    double x[kPer], r[kMaxBasis] = {0.0, 0.0, 0.0, 0.0}, v[kMaxBasis] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int col = tid + 256 * i;
      x[i] = col < d ? E[at + col] : 0.0;
      v[0] = fma(x[i], x[i], v[0]);
    }
    means(v, 1);
    const double before = v[0];
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      if (a == 0) break;
#pragma unroll
      for (int b = 0; b < a; ++b) {
        v[b] = 0.0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) v[b] = fma(basis[b][i], x[i], v[b]);
      }
      means(v, a);
#pragma unroll
      for (int b = 0; b < a; ++b) {
        r[b] += v[b];
#pragma unroll
        for (int i = 0; i < kPer; ++i) x[i] = fma(-v[b], basis[b][i], x[i]);
      }
    }
    v[0] = 0.0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) v[0] = fma(x[i], x[i], v[0]);
    means(v, 1);
    // (also a row of zeros; not one with a value that is not finite, which stays so)
    const bool none = before < __builtin_huge_val() && v[0] <= before * 0x1p-80;
    const double norm = none ? 0.0 : sqrt(v[0]), inv = none ? 0.0 : 1.0 / norm;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      basis[a][i] = x[i] * inv;
      const int col = tid + 256 * i;
      if (col < d) Q[at + col] = static_cast<float>(basis[a][i]);
    }
    if (tid < nq) {  // column a of R, by row; zeros below the diagonal
      double v_r = tid == a ? norm : 0.0;
#pragma unroll
      for (int b = 0; b < a; ++b)
        if (tid == b) v_r = r[b];
      Rs[tid * nq + a] = v_r;
    }
  }
}

// The walkers' carriers after the first level, from the orthonormal basis Q, its pairs' nodes O and R:
// the leaf carriers' norms and coefficients, the node's sum, its rescale and its gate
// (normalize_rows_kernel and level_gate_kernel of the plain path). A workgroup owns 16 walkers of one
// node pair p, its waves a quarter of the columns each. Orientation: basis columns x walkers on
// v_mfma_f32_16x16x4_f32, the contraction over a (leaf) or, in four steps, over (a, b); the row of 16
// columns a lane's register holds is one 16-byte store, 64 bytes per walker. Two passes over the
// columns: the node's norm, the stores (the sums are formed again: the basis is in L2 and the
// products are few). 100 us at 1024 x 64 sites, 41 of them for the 201 MB of carriers it writes.
__global__ void __launch_bounds__(256) leaf_pair_level_kernel(const float* __restrict__ Q, const float* __restrict__ O,
                                                              const double* __restrict__ R, const float* __restrict__ q,
                                                              const uint8_t* __restrict__ opcodes,
                                                              float* __restrict__ u_out, float* __restrict__ s_out,
                                                              int64_t B, int n, int nq, int d, float eps) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int p = blockIdx.y, w = n / 2;
  const int64_t b = static_cast<int64_t>(blockIdx.x) * 16 + c;
  const bool ok = b < B;
  // this wave's columns, in steps of 32 (d is a multiple of 32)
  const int steps = d / 32;
  const int t0 = 32 * (steps * wave / 4), t1 = 32 * (steps * (wave + 1) / 4);
  __shared__ float part[4][16];  // per wave and walker: the node's sum of squares
  // y = R q of one leaf over its rms, which is sqrt(mean(u^2) + 1e-30) with mean(u^2) = |y|^2
  auto coefficients = [&](int leaf, float (&y)[kMaxBasis]) {
    const float* const qb = q + ((ok ? b : 0) * n + leaf) * nq;
    const double* const Rl = R + static_cast<int64_t>(leaf) * nq * nq;
    double yd[kMaxBasis], ss = 0.0;
#pragma unroll
    for (int a = 0; a < kMaxBasis; ++a) {
      yd[a] = 0.0;
#pragma unroll
      for (int i = 0; i < kMaxBasis; ++i)
        if (a < nq && i < nq) yd[a] = fma(Rl[a * nq + i], static_cast<double>(qb[i]), yd[a]);
      ss = fma(yd[a], yd[a], ss);
    }
    const double rms = sqrt(ss + 1e-30);
#pragma unroll
    for (int a = 0; a < kMaxBasis; ++a) y[a] = static_cast<float>(yd[a] / rms);
    return static_cast<float>(rms);
  };
  float yl[kMaxBasis], yr[kMaxBasis];
  const float rl = coefficients(2 * p, yl), rr = coefficients(2 * p + 1, yr);
  auto lane_of = [&](const float (&x)[kMaxBasis]) { return g == 0 ? x[0] : (g == 1 ? x[1] : (g == 2 ? x[2] : x[3])); };
  const float bl = lane_of(yl), br = lane_of(yr);
  float co[kMaxBasis];
#pragma unroll
  for (int s = 0; s < kMaxBasis; ++s) co[s] = yl[s] * br;
  // this lane group's basis row; past nq (coefficient 0) any row
  const int gr = g < nq ? g : 0;
  const float* Ql = Q + (static_cast<int64_t>(gr) * n + 2 * p) * d + c;
  const float* Qr = Ql + d;
  const float* Os[kMaxBasis];
#pragma unroll
  for (int s = 0; s < kMaxBasis; ++s) Os[s] = O + (static_cast<int64_t>((s < nq ? s : 0) * nq + gr) * w + p) * d + c;
  // the node's sum in columns t .. t + 31
  auto node = [&](int t, v4f (&o)[2]) {
    float a[2][kMaxBasis];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < kMaxBasis; ++s) a[j][s] = Os[s][t + 16 * j];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      o[j] = zero4();
#pragma unroll
      for (int s = 0; s < kMaxBasis; ++s) o[j] = mfma16x4(a[j][s], co[s], o[j]);
    }
  };
  float ss = 0.f;
  for (int t = t0; t < t1; t += 32) {
    v4f o[2];
    node(t, o);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) ss = fmaf(o[j][r], o[j][r], ss);
  }
  ss = group_sum(ss);
  if (g == 0) part[wave][c] = ss;
  __syncthreads();
  const float whole = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
  const float scale = sqrtf(whole / static_cast<float>(d) + eps);
  const float inv = 1.0f / scale;
  const int op = opcodes[p];
  const float both = op == 0 ? 1.f : 0.f, left = op == 1 ? 1.f : 0.f, right = op == 2 ? 1.f : 0.f;
  float* urow = u_out + ((ok ? b : 0) * w + p) * d + 4 * g;
  for (int t = t0; t < t1; t += 32) {
    v4f o[2];
    node(t, o);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[j][r] *= inv;
      if (op != 0) {
        const v4f ul = mfma16x4(Ql[t + 16 * j], bl, zero4()), ur = mfma16x4(Qr[t + 16 * j], br, zero4());
#pragma unroll
        for (int r = 0; r < 4; ++r) o[j][r] = both * o[j][r] + left * ul[r] + right * ur[r];
      }
      if (ok) *reinterpret_cast<v4f*>(urow + t + 16 * j) = o[j];
    }
  }
  if (ok && g == 0 && wave == 0) {
    const float sl = logf(rl), sr = logf(rr);
    s_out[b * w + p] = both * (sl + sr + logf(scale)) + left * sl + right * sr;
  }
}

// Whether the basis serves: at least one pair (and no more than a grid's second dimension), inputs
// that fit its one K step, and no more basis rows than walker rows, neither at the leaves (2 nq: the
// basis in 64 bits and its factors take half a leaf buffer each as floats) nor at the pairs (nq^2);
// R in 64 bits fits where z is not needed. At that line (nq = 4, fine-tune widths) the whole
// wavefunction takes 312 us for 16 walkers of 8 sites with it and 433 for 15 without, 522 and 653
// at 64 sites.
bool basis_serves(int64_t B, int n, int nq, int d_z) {
  const int64_t nq2 = static_cast<int64_t>(nq) * nq;
  return n > 1 && n / 2 <= 65535 && nq <= kMaxBasis && B >= nq2 && B >= 2 * nq && B * d_z >= 2 * nq2;
}

hipError_t launch_merge(const float* T, const float* ua, const float* ub, float* out, int64_t M, int G,
                        const MergeRows& rows, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((M + 127) / 128), static_cast<unsigned>(G));
  hipLaunchKernelGGL(quadrilinear_merge_kernel, grid, dim3(256), 0, stream, T, ua, ub, out, M, G, rows);
  return hipGetLastError();
}

// Workspace sections of the whole-wavefunction executor, in floats, each rounded up to 64
// floats (256 bytes).
struct WaveFnWorkspace {
  int64_t z, work, u0, u1, raw, s0, s1, psi, total;
  WaveFnWorkspace(int64_t B, int64_t n, int64_t d_z, int64_t r_leaf, int64_t d_m, int64_t r_merge, int64_t r_out) {
    auto up = [](int64_t x) { return (x + 63) / 64 * 64; };
    const int64_t half = n > 1 ? n / 2 : 1;
    int64_t wk = B * n * r_leaf;
    if (B * half * r_merge > wk) wk = B * half * r_merge;
    if (B * r_out > wk) wk = B * r_out;
    z = 0;
    work = z + up(B * n * d_z);
    u0 = work + up(wk);
    u1 = u0 + up(B * n * d_m);
    raw = u1 + up(B * half * d_m);
    s0 = raw + up(B * half * d_m);
    s1 = s0 + up(B * n);
    psi = s1 + up(B * half);
    total = psi + up(2 * B);
  }
};

}  // namespace

int64_t compiled_wavefunction_workspace_bytes(int64_t B, int64_t n, int64_t d_z, int64_t r_leaf, int64_t d_m,
                                              int64_t r_merge, int64_t r_out) {
  return WaveFnWorkspace(B, n, d_z, r_leaf, d_m, r_merge, r_out).total * static_cast<int64_t>(sizeof(float));
}

hipError_t launch_compiled_wavefunction(const WaveFnParams& p, hipStream_t stream) {
  const WaveFnWorkspace L(p.B, p.n, p.d_z, p.r_leaf, p.d_m, p.r_merge, p.r_out);
  float* ws = p.workspace;
  float *z = ws + L.z, *work = ws + L.work, *raw = ws + L.raw, *psi = ws + L.psi;
  float* u_buf[2] = {ws + L.u0, ws + L.u1};
  float* s_buf[2] = {ws + L.s0, ws + L.s1};
  // the carrier buffer a step does not use holds its split-K partial products
  const int64_t u_cap[2] = {L.u1 - L.u0, L.raw - L.u1};
  const int64_t rows = p.B * p.n;
  const int G = p.d_m / kQR;
  hipError_t err;
  int cur = 0, level = 0, width = p.n / 2;
  if (basis_serves(p.B, p.n, p.d_q, p.d_z)) {
    // E in 64 bits in the first carrier buffer (its left factor in work), Q in the second, R in z, the
    // first level's node basis in raw, carriers into the first
    const int64_t er = static_cast<int64_t>(p.d_q) * p.n, pr = static_cast<int64_t>(p.d_q) * p.d_q * width;
    double *const factor = reinterpret_cast<double*>(work), *const E = reinterpret_cast<double*>(u_buf[0]);
    double* const R = reinterpret_cast<double*>(z);
    hipLaunchKernelGGL(leaf_basis_kernel,
                       dim3(static_cast<unsigned>((p.r_leaf + 255) / 256), static_cast<unsigned>(p.d_q),
                            static_cast<unsigned>(p.n < 16 ? p.n : 16)),
                       dim3(256), 0, stream, p.q_weight, p.leaf_V, p.leaf_h, factor, p.n, p.d_z, p.r_leaf);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    hipLaunchKernelGGL(basis_gemm_f64_kernel,
                       dim3(static_cast<unsigned>(p.d_m / 32), static_cast<unsigned>((er + 15) / 16)), dim3(256), 0,
                       stream, factor, p.leaf_U, E, er, p.d_m, p.r_leaf);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    hipLaunchKernelGGL(orthonormal_basis_kernel, dim3(static_cast<unsigned>(p.n)), dim3(256), 0, stream, E, u_buf[1], R,
                       p.n, p.d_q, p.d_m);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    if ((err = launch_merge(p.merge_T, u_buf[1], u_buf[1], raw, pr, G, MergeRows{p.d_m, width, p.d_q, p.n}, stream)) !=
        hipSuccess)
      return err;
    if ((err = apply_rows(raw, p.merge_V, p.merge_h, p.merge_U, raw, raw, work, pr, p.d_m, p.r_merge, p.d_m, width, 0,
                          stream, u_buf[0], u_cap[0])) != hipSuccess)
      return err;
    hipLaunchKernelGGL(leaf_pair_level_kernel,
                       dim3(static_cast<unsigned>((p.B + 15) / 16), static_cast<unsigned>(width)), dim3(256), 0, stream,
                       u_buf[1], raw, R, p.q, p.opcodes, u_buf[0], s_buf[0], p.B, p.n, p.d_q, p.d_m, p.merge_eps);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    level = 1;
    width /= 2;
  } else {
    // leaf: z = q W_q; u = ((z V) o leaf_h[site]) U; carriers RMS-normalised, s = log rms
    if ((err = launch_gemm<kEpiPlain>(p.q, p.q_weight, z, nullptr, rows, p.d_z, p.d_q, 1, 0, stream)) != hipSuccess)
      return err;
    if ((err = apply_rows(z, p.leaf_V, p.leaf_h, p.leaf_U, nullptr, u_buf[0], work, rows, p.d_z, p.r_leaf, p.d_m, p.n,
                          0, stream, u_buf[1], u_cap[1])) != hipSuccess)
      return err;
    hipLaunchKernelGGL(normalize_rows_kernel, dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, stream,
                       u_buf[0], s_buf[0], rows, p.d_m);
    if ((err = hipGetLastError()) != hipSuccess) return err;
  }
  // levels: node pairs (2p, 2p + 1) merged into node p, widths n/2, n/4, ..., 1
  for (; width >= 1; ++level, width /= 2) {
    const int64_t m = p.B * width;
    const float* u_in = u_buf[cur];
    const float* h_level = p.merge_h + static_cast<int64_t>(level) * (p.n / 2) * p.r_merge;
    const uint8_t* ops = p.opcodes + static_cast<int64_t>(level) * (p.n / 2);
    if ((err = launch_merge(p.merge_T, u_in, u_in + p.d_m, raw, m, G, MergeRows{2 * static_cast<int64_t>(p.d_m), 0, 1, 1},
                            stream)) != hipSuccess)
      return err;
    // out = raw + ((raw V) o h_level[node]) U, written over raw
    if ((err = apply_rows(raw, p.merge_V, h_level, p.merge_U, raw, raw, work, m, p.d_m, p.r_merge, p.d_m, width, 0,
                          stream, u_buf[cur ^ 1], u_cap[cur ^ 1])) != hipSuccess)
      return err;
    hipLaunchKernelGGL(level_gate_kernel, dim3(static_cast<unsigned>((m + 3) / 4)), dim3(256), 0, stream, raw, u_in,
                       s_buf[cur], ops, u_buf[cur ^ 1], s_buf[cur ^ 1], m, width, p.d_m, p.merge_eps);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    cur ^= 1;
  }
  // readout: psi = ((u_root V) o readout_h) U, then log|psi| and phase
  if ((err = apply_rows(u_buf[cur], p.readout_V, p.readout_h, p.readout_U, nullptr, psi, work, p.B, p.d_m, p.r_out, 2,
                        1, 0, stream, u_buf[cur ^ 1], u_cap[cur ^ 1])) != hipSuccess)
    return err;
  hipLaunchKernelGGL(readout_kernel, dim3(static_cast<unsigned>((p.B + 255) / 256)), dim3(256), 0, stream, psi,
                     s_buf[cur], p.log_abs, p.phase, p.B);
  return hipGetLastError();
}

hipError_t launch_quadrilinear_merge(const float* T, const float* ua, const float* ub, float* out, int64_t M, int G,
                                     int64_t ld_in, hipStream_t stream) {
  return launch_merge(T, ua, ub, out, M, G, MergeRows{ld_in, 0, 1, 1}, stream);
}

hipError_t launch_factorized_apply(const float* x, const float* V, const float* h, const float* U,
                                   const float* residual, float* y, float* work, int64_t M, int d_in, int R, int d_out,
                                   int h_rows, hipStream_t stream) {
  return apply_rows(x, V, h, U, residual, y, work, M, d_in, R, d_out, h_rows, 0, stream);
}

hipError_t launch_out_proj(const float* y, const float* w_o, const uint8_t* mask, float* delta, int64_t M, int d_in,
                           int d_out, hipStream_t stream) {
  // The row-compacting kernel where its 256-row workgroups fill the chip; below that (few
  // rows, e.g. one large-N system's 4096 query rows: 64 workgroups for 256 CUs) the 128 x 128
  // tiled GEMM with the row mask in its epilogue runs twice the workgroups and multiplies the
  // masked rows too (the large-N tail's W_O on 4096 rows: about 93 -> 53 us).
  // At the line (16384 rows, 512 columns) the row kernel takes 29 us with 36 of 64 rows physical and
  // 40 with all, the tiled one 39 and 38; at 65536 rows 86 and 106 against 142 and 133.
  int cus = 0;
  if (hipError_t err = device_cu_count(&cus); err != hipSuccess) return err;
  const int64_t ncol = (d_out + kBN - 1) / kBN;
  const int64_t blocks = ncol * ((M + kRM - 1) / kRM);
  if (mask != nullptr && d_out % 4 == 0 && d_in % 4 == 0 && blocks >= cus) {
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_rows_f32_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, y, w_o, delta,
                       mask, M, d_out, d_in, static_cast<int>(ncol));
    return hipGetLastError();
  }
  if (mask != nullptr)
    return launch_gemm<kEpiRowMask>(y, w_o, delta, reinterpret_cast<const float*>(mask), M, d_out, d_in, 1, 0, stream);
  return launch_gemm<kEpiPlain>(y, w_o, delta, nullptr, M, d_out, d_in, 1, 0, stream);
}

static hipError_t apply_scratch_address(int device, float** ptr) {
  if (device < 0 || device >= kMaxScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device] == nullptr) {
    int current = -1;
    hipError_t err = hipGetDevice(&current);
    if (err != hipSuccess) return err;
    if (current != device && (err = hipSetDevice(device)) != hipSuccess) return err;
    // `scratch` names the array only inside kernels; host code uses this device's address.
    void* addr = nullptr;
    err = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
    if (current != device) {
      const hipError_t restore = hipSetDevice(current);
      if (err == hipSuccess) err = restore;
    }
    if (err != hipSuccess) return err;
    if (addr == nullptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = static_cast<float*>(addr);
  }
  *ptr = g_scratch_ptr[device];
  return hipSuccess;
}

hipError_t launch_factorized_apply_noalloc(const float* x, const float* V, const float* h, const float* U,
                                           const float* residual, float* y, int64_t M, int d_in, int R, int d_out,
                                           int h_rows, hipStream_t stream) {
  if (R > kApplyScratchMaxRank) return hipErrorInvalidValue;
  int device = -1;
  hipError_t err = hipStreamGetDevice(stream, &device);
  if (err != hipSuccess) return err;
  float* work = nullptr;
  if ((err = apply_scratch_address(device, &work)) != hipSuccess) return err;
  // Whole 128-row tiles of R floats per chunk; every workspace entry a chunk's second GEMM
  // reads is written by its first, so the array needs no clearing between calls.
  const int64_t chunk = kApplyScratchFloats / R / kBM * kBM;
  for (int64_t r0 = 0; r0 < M; r0 += chunk) {
    const int64_t rows = M - r0 < chunk ? M - r0 : chunk;
    err = apply_rows(x + r0 * d_in, V, h, U, residual == nullptr ? nullptr : residual + r0 * d_out, y + r0 * d_out,
                     work, rows, d_in, R, d_out, h_rows, r0, stream);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace hz
