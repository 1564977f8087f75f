"""GPU parity of the compiled executor's products (hz_quadrilinear_merge, hz_factorized_apply)
against the float64 oracle (oracle/executor_oracle.py), through the C ABI.

Tolerance: max-norm relative error <= 1e-5 (float32 inputs, float32 matrix-core products
and accumulation). Shapes cover the fine-tune model's (merge_dim 1536 = 48 groups of rank
32, merge_rank 1024, config.py:21-29,189-190) at reduced walker counts, row counts that are
not multiples of the tiles, one conditioner row per node and the readout's two outputs.
"""

import types

import numpy as np
import pytest
import torch

from oracle import executor_oracle as X

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _say(msg):
    print(f"[case] {msg}", flush=True)


def rel(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda()


@pytest.mark.parametrize("M,G", [(5, 2), (256, 48), (1000, 3), (2 * 32, 48)])
def test_quadrilinear_merge(M, G):
    from hamiltonzero_amd import executor

    _say(f"merge M={M} G={G}")
    rng = np.random.default_rng(M + G)
    R = 32
    T = (rng.standard_normal((G, R, R, R)) / R).astype(np.float32)
    a = rng.standard_normal((M, G * R)).astype(np.float32)
    b = rng.standard_normal((M, G * R)).astype(np.float32)
    got = executor.quadrilinear_merge(dev(T), dev(a), dev(b))
    torch.cuda.synchronize()
    assert rel(got.cpu().numpy(), X.quadrilinear_merge(T, a, b)) <= TOL


def test_quadrilinear_merge_leading_axes():
    from hamiltonzero_amd import executor

    _say("merge [walkers, nodes, G R]")
    rng = np.random.default_rng(11)
    G, R = 4, 32
    T = (rng.standard_normal((G, R, R, R)) / R).astype(np.float32)
    a = rng.standard_normal((3, 16, G * R)).astype(np.float32)
    b = rng.standard_normal((3, 16, G * R)).astype(np.float32)
    got = executor._compiled_quadrilinear_merge(dev(T), dev(a), dev(b))
    torch.cuda.synchronize()
    assert got.shape == (3, 16, G * R)
    assert rel(got.cpu().numpy(), X.quadrilinear_merge(T, a, b)) <= TOL


@pytest.mark.parametrize(
    "walkers,nodes,d_in,R,d_out,residual",
    [
        (2, 32, 96, 64, 48, False),         # small, tile remainders everywhere
        (8, 32, 1536, 1024, 1536, True),    # a merge level at the fine-tune ranks
        (3, 7, 130, 66, 18, False),         # sizes that are not multiples of 4
        (37, 1, 1536, 1024, 2, False),      # the readout: one conditioner row, psi = (re, im)
        (4, 64, 64, 1536, 1536, False),     # the leaf apply shape (rank 1536)
    ],
)
def test_factorized_apply(walkers, nodes, d_in, R, d_out, residual):
    from hamiltonzero_amd import executor

    _say(f"apply walkers={walkers} nodes={nodes} d_in={d_in} R={R} d_out={d_out} residual={residual}")
    rng = np.random.default_rng(walkers * 7 + nodes)
    x = rng.standard_normal((walkers, nodes, d_in)).astype(np.float32)
    V = (rng.standard_normal((d_in, R)) / np.sqrt(d_in)).astype(np.float32)
    U = (rng.standard_normal((R, d_out)) / np.sqrt(R)).astype(np.float32)
    h = rng.standard_normal((nodes, R)).astype(np.float32)
    res = rng.standard_normal((walkers, nodes, d_out)).astype(np.float32) if residual else None
    factor = types.SimpleNamespace(V=dev(V), U=dev(U))
    got = executor._factorized_apply(factor, dev(h), dev(x), None if res is None else dev(res))
    torch.cuda.synchronize()
    want = X.factorized_apply(V, U, h, x) + (0.0 if res is None else res)
    assert rel(got.cpu().numpy(), want) <= TOL


@pytest.mark.parametrize("M,d_in,R,d_out", [(1, 1, 1, 1), (127, 15, 16, 129), (129, 17, 33, 2), (128, 16, 32, 128), (5, 4, 260, 131)])
def test_factorized_apply_tile_edges(M, d_in, R, d_out):
    """One row, column or k either side of the 128 x 128 tiles and 16-deep slices; large and tiny
    magnitudes beside each other (each factor's terms keep their float32 bits: same bound)."""
    from hamiltonzero_amd import executor

    _say(f"apply edges M={M} d_in={d_in} R={R} d_out={d_out}")
    rng = np.random.default_rng(M + 3 * d_in + R)
    x = (rng.standard_normal((M, d_in)) * 10.0 ** rng.integers(-6, 7, size=(M, 1))).astype(np.float32)
    V, U = rng.standard_normal((d_in, R)).astype(np.float32), rng.standard_normal((R, d_out)).astype(np.float32)
    h = rng.standard_normal((1, R)).astype(np.float32)
    got = executor._factorized_apply(types.SimpleNamespace(V=dev(V), U=dev(U)), dev(h), dev(x)).cpu().numpy()
    want = X.factorized_apply(V, U, h, x)
    # per row: a float32 sum's bound scales with the sum of its terms' magnitudes
    terms = ((np.abs(x.astype(np.float64)) @ np.abs(V)) * np.abs(h)) @ np.abs(U)
    assert np.all(np.abs(got - want) <= 2.0**-24 * (d_in + R + 4) ** 0.5 * 4 * terms)


def test_products_of_values_the_split_does_not_hold():
    """Infinities, NaN and finite values above the largest bfloat16 (3.39e38): the sums are what
    float32 arithmetic gives, and only in the rows (and groups) that hold such a value."""
    from hamiltonzero_amd import executor

    _say("apply and merge, non-finite and largest values")
    rng = np.random.default_rng(3)
    M, d = 40, 48
    x = rng.random((M, d)).astype(np.float32) + 0.5
    V, U = (rng.random((d, d)).astype(np.float32) * 1e-3 + 1e-3 for _ in range(2))
    h = np.ones((1, d), np.float32)
    x[3, 7], x[9, 0], x[20, 40], x[33, 5] = np.inf, np.nan, 3.4e38, -np.inf
    fac = types.SimpleNamespace(V=dev(V), U=dev(U))
    got = executor._factorized_apply(fac, dev(h), dev(x)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = X.factorized_apply(V, U, h, x)
    assert np.all(np.isposinf(got[3])) and np.all(np.isneginf(got[33])) and np.all(np.isnan(got[9]))
    ok = [m for m in range(M) if m not in (3, 9, 33)]
    assert np.all(np.abs(got[ok] - want[ok]) <= TOL * np.abs(want[ok]))  # every term is positive

    G, R = 2, 32
    T = rng.random((G, R, R, R)).astype(np.float32)
    a, b = (rng.random((M, G * R)).astype(np.float32) + 0.5 for _ in range(2))
    a[3, 5], b[9, 40], a[20, 33], b[33, 1] = np.inf, np.nan, 3.4e38, -np.inf
    b[20] *= 1e-6
    got = executor.quadrilinear_merge(dev(T), dev(a), dev(b)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = X.quadrilinear_merge(T, a, b)
    assert np.all(np.isposinf(got[3, :R])) and np.all(np.isnan(got[9, R:])) and np.all(np.isneginf(got[33, :R]))
    mask = np.isfinite(want)
    assert np.all(np.isfinite(got) == mask) and np.all(np.abs(got[mask] - want[mask]) <= TOL * np.abs(want[mask]))


@pytest.mark.parametrize("M,d_in,R,d_out", [(1, 5, 3, 2), (33, 37, 50, 131), (129, 48, 260, 64)])
def test_sums_formed_again(M, d_in, R, d_out):
    """Rows with an infinity, a NaN or a value above the largest bfloat16, contraction lengths with
    every remainder, rows and columns past a tile: what float32 arithmetic gives in those rows, and
    every other row bit for bit what it is without them."""
    from hamiltonzero_amd import executor

    _say(f"sums formed again M={M} d_in={d_in} R={R} d_out={d_out}")
    rng = np.random.default_rng(M + d_in)
    x = rng.random((M, d_in)).astype(np.float32) + 0.5
    V = rng.random((d_in, R)).astype(np.float32) * 1e-3 + 1e-3
    U = rng.random((R, d_out)).astype(np.float32) * 1e-3 + 1e-3
    fac, h = types.SimpleNamespace(V=dev(V), U=dev(U)), dev(np.ones((1, R)))
    plain = executor._factorized_apply(fac, h, dev(x)).cpu().numpy()
    put = {0: np.inf, M // 2: 3.4e38, M - 1: -np.inf, M // 3: np.nan}
    for m, v in put.items():
        x[m, (3 * m) % d_in] = v
    got = executor._factorized_apply(fac, h, dev(x)).cpu().numpy()
    want = X.factorized_apply(V, U, np.ones((1, R)), x)  # every term of a row has one sign
    for m in range(M):
        if m not in put:
            assert np.array_equal(got[m], plain[m]), m
        elif np.isfinite(want[m]).all():
            assert np.all(np.abs(got[m] - want[m]) <= TOL * np.abs(want[m])), m
        else:
            assert np.array_equal(got[m], want[m].astype(np.float32), equal_nan=True), m


@pytest.mark.parametrize("value,most", [(float("nan"), 1.5), (float("inf"), 3.0)])
def test_a_row_that_is_not_finite_costs_little(value, most):
    """One walker among 16384 whose row holds a NaN (it has diverged, and carries it through every
    level): its sums need no second look and the products take their usual time. One with an
    infinity has its sums formed again by the whole wave (2.4 times the apply's time, two products;
    a serial loop over the contraction per sum took 3 to 5 times, for a NaN too)."""
    from hamiltonzero_amd import executor, kernels

    _say(f"cost of a row with {value}")
    gen = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    M, G, R = 16384, 48, 32
    T, a, b = rnd(G, R, R, R) / R, rnd(M, G * R), rnd(M, G * R)
    fac, h = types.SimpleNamespace(V=rnd(G * R, 1024) / 39, U=rnd(1024, G * R) / 32), rnd(1, 1024)
    y, w_o = rnd(1024, 64, 16, 16), rnd(256, 512) / 16
    mask = torch.arange(64, device="cuda")[None, :].expand(1024, 64) < 36
    calls = {
        "merge": (a, lambda x: executor.quadrilinear_merge(T, x, b)),
        "apply": (a, lambda x: executor._factorized_apply(fac, h, x)),
        "out_proj rows": (y, lambda x: kernels.gated_out_proj(x, w_o, mask=mask)[0]),
        "out_proj tiles": (y, lambda x: kernels.gated_out_proj(x, w_o)[0]),
    }

    def fastest(fn, x):
        times = []
        for _ in range(20):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            fn(x)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    for name, (x, fn) in calls.items():
        worse = x.clone()
        worse.view(-1, worse.shape[-1])[77, 5] = value
        clean, slow = fastest(fn, x), fastest(fn, worse)
        print(f"{name}: {clean * 1e3:.0f} us, with the row {slow * 1e3:.0f} us", flush=True)
        assert slow <= most * clean, (name, clean, slow)


def test_merge_level_products_compose():
    """One tree level's products as the executor chains them: merge, then the residual apply
    (execute.py:103-104), checked against the oracle's level up to the RMS rescale."""
    from hamiltonzero_amd import executor

    _say("merge level")
    rng = np.random.default_rng(21)
    G, R, Rm, W, B = 48, 32, 1024, 16, 4
    T = (rng.standard_normal((G, R, R, R)) / R).astype(np.float32)
    V = (rng.standard_normal((G * R, Rm)) / np.sqrt(G * R)).astype(np.float32)
    U = (rng.standard_normal((Rm, G * R)) / np.sqrt(Rm)).astype(np.float32)
    h = rng.standard_normal((W, Rm)).astype(np.float32)
    u = rng.standard_normal((B, 2 * W, G * R)).astype(np.float32)
    ul, ur = u[:, 0::2], u[:, 1::2]
    raw = executor.quadrilinear_merge(dev(T), dev(ul), dev(ur))
    out = executor.factorized_apply(types.SimpleNamespace(V=dev(V), U=dev(U)), dev(h), raw, raw)
    torch.cuda.synchronize()
    raw_ref = X.quadrilinear_merge(T, ul, ur)
    want = raw_ref + X.factorized_apply(V, U, h, raw_ref)
    assert rel(out.cpu().numpy(), want) <= TOL


def _wavefn_case(seed, B, n, d_q, d_z, R_leaf, G, R_merge, R_out, real):
    rng = np.random.default_rng(seed)
    R, dm = 32, G * 32
    f32 = lambda x: np.asarray(x, dtype=np.float32)  # noqa: E731
    w = lambda i, o: f32(rng.standard_normal((i, o)) / np.sqrt(i))  # noqa: E731
    if real == "all":
        leaf_real = np.ones(n, bool)
    else:
        leaf_real = rng.random(n) < (0.8 if real == "random" else 0.3)
        leaf_real[rng.integers(n)] = True
    p = dict(q=f32(rng.standard_normal((B, n, d_q))), q_weight=w(d_q, d_z), leaf_V=w(d_z, R_leaf),
             leaf_U=w(R_leaf, dm), leaf_h=f32(rng.standard_normal((n, R_leaf))),
             merge_T=f32(rng.standard_normal((G, R, R, R)) / R), merge_V=w(dm, R_merge), merge_U=w(R_merge, dm),
             readout_V=w(dm, R_out), readout_U=w(R_out, 2), readout_h=f32(rng.standard_normal(R_out)),
             merge_eps=1e-6)
    p["merge_h"] = [f32(rng.standard_normal((n >> (l + 1), R_merge))) for l in range(int(np.log2(n)))]
    p["opcodes"] = X.classify_opcodes(leaf_real) if n > 1 else []
    return p


def _readout_condition(p):
    """kappa_b = sum_r |m_r| (|U_r0| + |U_r1|) / |psi_b| from the oracle's root carriers."""
    z = np.asarray(p["q"], np.float64) @ p["q_weight"]
    u, s = X.normalize_leaf_carriers(X.factorized_apply(p["leaf_V"], p["leaf_U"], p["leaf_h"], z))
    for h, o in zip(p["merge_h"], p["opcodes"]):
        u, s = X.merge_level(p["merge_T"], p["merge_V"], p["merge_U"], h, p["merge_eps"], u, s, o)
    m = (u[:, 0] @ np.asarray(p["readout_V"], np.float64)) * p["readout_h"]
    U = np.asarray(p["readout_U"], np.float64)
    psi = m @ U
    return (np.abs(m) @ np.abs(U)).sum(axis=1) / np.hypot(psi[:, 0], psi[:, 1])


def _namespaces(p):
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    fac = lambda V, U: types.SimpleNamespace(V=t(V), U=t(U))  # noqa: E731
    kernel = types.SimpleNamespace(q_to_odd=types.SimpleNamespace(weight=t(p["q_weight"])),
                                   leaf_factors=(fac(p["leaf_V"], p["leaf_U"]),), merge_T=t(p["merge_T"]),
                                   merge_factors=(fac(p["merge_V"], p["merge_U"]),),
                                   readout_factors=(fac(p["readout_V"], p["readout_U"]),), merge_eps=p["merge_eps"])
    tree = types.SimpleNamespace(leaf_h=(t(p["leaf_h"]),), readout_h=(t(p["readout_h"]),), leaf_combiner_h=(),
                                 readout_combiner_h=(), merge_h=tuple(t(h) for h in p["merge_h"]),
                                 opcodes=tuple(t(o) for o in p["opcodes"]))
    return kernel, tree, t(p["q"])


@pytest.mark.parametrize(
    "B,n,d_q,d_z,R_leaf,G,R_merge,R_out,real",
    [
        (16, 64, 4, 32, 1536, 48, 1024, 64, "random"),  # the fine-tune sizes (config.py:21-29,189-190)
        (5, 8, 4, 40, 24, 4, 96, 8, "all"),
        (7, 16, 3, 30, 66, 2, 50, 6, "sparse"),          # sizes off the 4-float staging path
        (3, 1, 4, 32, 64, 3, 32, 16, "all"),             # one site: no merge level
        (300, 4, 4, 32, 128, 8, 64, 64, "random"),       # many walkers, shallow tree
    ],
)
def test_compiled_wavefunction_matches_oracle(B, n, d_q, d_z, R_leaf, G, R_merge, R_out, real):
    from hamiltonzero_amd import executor

    _say(f"wavefunction B={B} n={n} G={G} R_leaf={R_leaf} R_merge={R_merge} R_out={R_out} {real}")
    p = _wavefn_case(B * 3 + n, B, n, d_q, d_z, R_leaf, G, R_merge, R_out, real)
    kernel, tree, q = _namespaces(p)
    la, ph = executor.execute_wavefunction(kernel, tree, q)
    torch.cuda.synchronize()
    want_la, want_ph = X.execute_wavefunction(**p)
    # log|psi| and the phase carry psi's relative error. Where the readout's sum cancels,
    # kappa = sum_r |m_r| (|U_r0| + |U_r1|) / |psi| (m the conditioned readout row), that is
    # kappa times the float32 error of its terms (about 2e-7 kappa measured), so each walker
    # is allowed 1e-6 kappa on top of the max-norm bound.
    kappa = _readout_condition(p)
    dla = np.abs(la.cpu().numpy().astype(np.float64) - want_la)
    assert np.all(dla <= TOL * np.max(np.abs(want_la)) + 1e-6 * kappa), (dla.max(), kappa[np.argmax(dla)])
    dphi = np.abs(np.angle(np.exp(1j * (ph.cpu().numpy().astype(np.float64) - want_ph))))
    assert np.all(dphi <= TOL * np.pi + 1e-6 * kappa), (dphi.max(), kappa[np.argmax(dphi)])
    assert np.median(kappa) < 10  # most walkers are well conditioned: the bound is mostly the max-norm one


@pytest.mark.parametrize(
    "B,n,d_q,G,real",
    [
        (16, 2, 4, 2, "all"),      # the fewest walkers the pair basis serves (d_q^2), one pair
        (15, 2, 4, 2, "all"),      # one fewer: the plain path
        (9, 4, 3, 1, "random"),    # d_q below the basis width, 32 columns (three of four waves idle)
        (4, 8, 2, 3, "sparse"),    # 96 columns, carries and empty nodes
        (2, 4, 1, 2, "all"),
        (17, 8, 4, 5, "sparse"),   # a second, nearly empty block of walkers
        (70, 16, 5, 2, "random"),  # wider inputs: the plain path
    ],
)
def test_compiled_wavefunction_pair_basis(B, n, d_q, G, real):
    """The leaf and first level through the basis of the inputs (d_q <= 4, B >= max(d_q^2, 2 d_q)),
    at its edges, with the bound of the test above."""
    from hamiltonzero_amd import executor

    _say(f"wavefunction basis B={B} n={n} d_q={d_q} G={G} {real}")
    p = _wavefn_case(B * 5 + n + d_q, B, n, d_q, 20, 40, G, 36, 12, real)
    kernel, tree, q = _namespaces(p)
    la, ph = executor.execute_wavefunction(kernel, tree, q)
    torch.cuda.synchronize()
    want_la, want_ph = X.execute_wavefunction(**p)
    kappa = _readout_condition(p)
    dla = np.abs(la.cpu().numpy().astype(np.float64) - want_la)
    assert np.all(dla <= TOL * np.max(np.abs(want_la)) + 1e-6 * kappa), (dla.max(), kappa[np.argmax(dla)])
    dphi = np.abs(np.angle(np.exp(1j * (ph.cpu().numpy().astype(np.float64) - want_ph))))
    assert np.all(dphi <= TOL * np.pi + 1e-6 * kappa), (dphi.max(), kappa[np.argmax(dphi)])


@pytest.mark.parametrize("rows", ["1e-1", "1e-2", "1e-3", "equal", "zero"])
def test_pair_basis_of_inputs_that_cancel(rows):
    """Leaves whose inputs cancel: the rows of q_to_odd are a common vector and a part of size
    ``rows`` of their own, and a site's inputs sum to zero, so its carrier is about 1 / rows times
    smaller than the carriers of its single inputs. The same bound as for inputs that do not
    cancel: the carrier is a function of q to be evaluated, not of rounded sums. Rows that are
    equal, or zero, leave a basis of fewer rows."""
    from hamiltonzero_amd import executor

    _say(f"wavefunction basis, cancelling inputs, rows {rows}")
    B, n, d_q, G = 33, 4, 4, 4
    p = _wavefn_case(5, B, n, d_q, 32, 256, G, 128, 12, "all")
    rng = np.random.default_rng(9)
    if rows in ("equal", "zero"):
        p["q_weight"][2:] = p["q_weight"][0] if rows == "equal" else 0.0
    else:
        own = rng.standard_normal((d_q, 32)) * float(rows)
        p["q_weight"] = ((rng.standard_normal(32) + own) / 2).astype(np.float32)
        p["q"][..., 1], p["q"][..., 3] = -p["q"][..., 0], -p["q"][..., 2]
    kernel, tree, q = _namespaces(p)
    la, ph = executor.execute_wavefunction(kernel, tree, q)
    torch.cuda.synchronize()
    want_la, want_ph = X.execute_wavefunction(**p)
    kappa = _readout_condition(p)
    dla = np.abs(la.cpu().numpy().astype(np.float64) - want_la)
    assert np.all(dla <= TOL * np.max(np.abs(want_la)) + 1e-6 * kappa), (dla.max(), kappa[np.argmax(dla)])
    dphi = np.abs(np.angle(np.exp(1j * (ph.cpu().numpy().astype(np.float64) - want_ph))))
    assert np.all(dphi <= TOL * np.pi + 1e-6 * kappa), (dphi.max(), kappa[np.argmax(dphi)])


@pytest.mark.parametrize(
    "B,n,d_q,d_z,R_leaf,G",
    [
        (32, 4, 4, 1, 37, 2),    # R fills z to the last float; every leaf's basis has one row
        (31, 4, 4, 1, 37, 2),    # one walker fewer: it does not fit, the plain path
        (2, 2, 1, 1, 1, 1),      # the smallest of everything
        (18, 2, 3, 2, 15, 64),   # less than one K block; the widest carrier (2048); two rows of three
        (20, 16, 2, 3, 130, 33), # eight K blocks and a remainder, a row of 16 that is not full
        (17, 8, 4, 9, 80, 5),    # five whole K blocks: one wave has two
    ],
)
def test_pair_basis_sizes(B, n, d_q, d_z, R_leaf, G):
    """The leaf basis in 64 bits: contraction lengths either side of its blocks, column and row counts
    either side of its tiles, fewer independent rows than inputs, the workspace's exact fit."""
    from hamiltonzero_amd import executor

    _say(f"wavefunction basis sizes B={B} n={n} d_q={d_q} d_z={d_z} R_leaf={R_leaf} G={G}")
    p = _wavefn_case(B + n + R_leaf, B, n, d_q, d_z, R_leaf, G, 36, 12, "random")
    kernel, tree, q = _namespaces(p)
    la, ph = executor.execute_wavefunction(kernel, tree, q)
    torch.cuda.synchronize()
    want_la, want_ph = X.execute_wavefunction(**p)
    kappa = _readout_condition(p)
    dla = np.abs(la.cpu().numpy().astype(np.float64) - want_la)
    assert np.all(dla <= TOL * np.max(np.abs(want_la)) + 1e-6 * kappa), (dla.max(), kappa[np.argmax(dla)])
    dphi = np.abs(np.angle(np.exp(1j * (ph.cpu().numpy().astype(np.float64) - want_ph))))
    assert np.all(dphi <= TOL * np.pi + 1e-6 * kappa), (dphi.max(), kappa[np.argmax(dphi)])


@pytest.mark.parametrize("where", ["q", "leaf_U", "leaf_h"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_pair_basis_of_values_that_are_not_finite(where, value):
    """What is not finite stays so, and only where it belongs: one walker's input, or a weight (every
    walker) or one leaf's conditioner (every walker whose tree holds that leaf)."""
    from hamiltonzero_amd import executor

    _say(f"wavefunction basis, {value} in {where}")
    p = _wavefn_case(3, 20, 4, 4, 20, 40, 2, 36, 12, "all")
    kernel, tree, q = _namespaces(p)
    clean = [x.cpu().numpy() for x in executor.execute_wavefunction(kernel, tree, q)]
    p[where].reshape(-1)[(7 * 4 + 1) * 4 + 2 if where == "q" else 11] = value  # q: walker 7, site 1
    kernel, tree, q = _namespaces(p)
    got = [x.cpu().numpy() for x in executor.execute_wavefunction(kernel, tree, q)]
    hit = np.arange(20) == 7 if where == "q" else np.ones(20, bool)
    for a, b in zip(got, clean):
        assert np.all(np.isnan(a[hit])) and np.array_equal(a[~hit], b[~hit])


def test_compiled_wavefunction_structure_errors():
    from hamiltonzero_amd import executor

    _say("wavefunction structure errors")
    p = _wavefn_case(1, 2, 8, 4, 32, 64, 2, 32, 8, "all")
    kernel, tree, q = _namespaces(p)
    with pytest.raises(ValueError, match="one entry per tree level"):
        executor.execute_wavefunction(kernel, types.SimpleNamespace(**dict(vars(tree), opcodes=tree.opcodes[:-1])), q)
    with pytest.raises(ValueError, match="incompatible shrinking shape"):
        executor.execute_wavefunction(kernel, tree, q[:, :4])
    with pytest.raises(ValueError, match="does not accept combiners"):
        executor.execute_wavefunction(kernel, types.SimpleNamespace(**dict(vars(tree), leaf_combiner_h=(1,))), q)
