"""The autograd functions' handling of cotangents and tangents, without a GPU: the kernels are
replaced by functions that record what they are given and return tensors of the right shapes
(their numbers are compared in the GPU tests)."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from hamiltonzero_amd import _native
from hamiltonzero_amd import mhsea_tuned as MT

B, N, H, D = 2, 8, 4, 8


@pytest.fixture
def calls(monkeypatch):
    seen = []

    def fwd(q, k, v, mask, e=None, **_):
        seen.append(("fwd",))
        return torch.ones_like(q), torch.ones(B, N, H)

    def bwd(q, k, v, mask, lse, out, dout, e=None, **kw):
        seen.append(("bwd", dout))
        return torch.ones_like(q), torch.ones_like(q), None if e is None else torch.ones_like(e), torch.ones_like(q)

    def tangent(q, qt, kt, vt, et):
        seen.append(("jvp", qt, kt, vt, et))
        return torch.ones_like(q)

    def gated(q, k, v, mask, qt=None, kt=None, vt=None, e=None, et=None, **_):
        y = torch.ones(B, N, H // 2, D)
        return y, None if (qt, kt, vt, et) == (None,) * 4 else tangent(y, qt, kt, vt, et)

    for name, fn in {"mhsea_fwd": fwd, "mhsea_bwd": bwd, "mhsea_bwd_gated": bwd, "mhsea_fwd_jvp_gated": gated,
                     "gate_collapse": lambda out: out[:, :, : H // 2].clone(),
                     "mhsea_jvp": lambda q, k, v, m, o, l, qt=None, kt=None, vt=None, e=None, et=None, **_: tangent(
                         q, qt, kt, vt, et)}.items():
        monkeypatch.setattr(MT.kernels, name, fn)
    return seen


CALLS = {"attention": lambda *a: MT.mhsea_ad(*a)[0], "gated": MT.gated_edge_attention}


def operands(grad):
    shapes = ((B, N, H, D), (B, N, H, D), (B, N, H, N), (B, N, H, D))
    return [torch.randn(s).requires_grad_(grad) for s in shapes], torch.ones(B, N, dtype=torch.bool)


@pytest.mark.parametrize("call,cls", [("attention", MT._MhseaAD), ("gated", MT._GatedTrainAD)])
def test_reverse_mode_makes_no_cotangents_of_kept_outputs(calls, monkeypatch, call, cls):
    """The outputs that only serve the reverse mode (lse; for the collapse out too, 134 MB at
    [1024, 64, 32, 16]) get no zero-filled cotangents."""
    given, real = [], cls.backward
    monkeypatch.setattr(cls, "backward", staticmethod(lambda ctx, *d: (given.append(d), real(ctx, *d))[1]))
    xs, mask = operands(True)
    y = CALLS[call](*xs, mask)
    cot = torch.randn_like(y)
    grads = torch.autograd.grad(y, xs, cot)
    assert torch.equal(given[0][0], cot) and all(d is None for d in given[0][1:])
    assert torch.equal(calls[-1][1], cot) and all(torch.equal(g, torch.ones_like(x)) for g, x in zip(grads, xs))


def test_the_compacted_layout_has_no_reverse_mode(calls):
    """Its forward serves a call that wants a gradient; asking for the gradient is refused at once,
    without a second attention forward."""
    (q, k, _, v), mask = operands(True)
    e = torch.randn(B, H, N, N)
    y = MT.gated_edge_attention(q, k, e, v, mask, e_layout="compact")
    calls.clear()
    with pytest.raises(_native.HzError, match="no reverse mode"):
        torch.autograd.grad(y, q, torch.ones_like(y))
    assert not calls


@pytest.mark.parametrize("call", list(CALLS))
def test_an_undefined_cotangent_is_zero(calls, call):
    class NoGradient(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    xs, mask = operands(True)
    y = NoGradient.apply(CALLS[call](*xs, mask))
    torch.autograd.grad(y, xs, torch.ones_like(y))
    assert calls[-1][0] == "bwd" and torch.equal(calls[-1][1], torch.zeros_like(y))


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("call", list(CALLS))
def test_forward_mode_of_some_operands(calls, call, grad):
    """Tangents of q alone and of e alone, with and without a gradient wanted beside them."""
    for i, at in ((0, 1), (2, 4)):
        xs, mask = operands(grad)
        with fwAD.dual_level():
            t = torch.randn_like(xs[i])
            xs[i] = fwAD.make_dual(xs[i], t)
            y = CALLS[call](*xs, mask)
            assert torch.equal(fwAD.unpack_dual(y).tangent, torch.ones_like(fwAD.unpack_dual(y).primal))
        got = calls[-1]
        assert got[0] == "jvp" and torch.equal(got[at], t)
        assert all(x is None or not x.any() for j, x in enumerate(got) if j not in (0, at))
