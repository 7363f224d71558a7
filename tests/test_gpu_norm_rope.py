"""GPU parity of the one-launch RMSNorm (with the residual add) and per-head RMSNorm + RoPE against
the same formulas in float64. The kernels compute in fp32 and round once: half a step of the
storage dtype (2^-8 of the value or less in bf16, 2^-11 in fp16), plus the fp32 roundings (2^-21 of
the terms of a sum)."""

from __future__ import annotations

import pytest
import torch

from plastic_infer.kernel.norm_rope import add_rms_norm_rows, qk_norm_rope, rms_norm_rows

pytestmark = pytest.mark.gpu

STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _norm(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()


def _check(got, ref, terms, dtype):
    assert got.dtype == dtype and got.is_contiguous()
    bound = STEP[dtype] * ref.abs().clamp_min(2.0 ** -14) + 2.0 ** -21 * terms
    err = ((got.double().cpu() - ref).abs() / bound).max().item()
    assert err <= 1.0, err


@pytest.mark.parametrize("dtype", list(STEP))
@pytest.mark.parametrize("shape,offset", [((64, 2048), 0), ((1, 8), 0), ((3, 2050), 0),
                                          ((5, 1), 0), ((7, 4104), 0), ((4, 64), 1)])
def test_rms_norm(dev, dtype, shape, offset):
    g = torch.Generator().manual_seed(shape[1])
    n = shape[0] * shape[1]
    # offset 1: rows that start between vectors
    x = (torch.randn(n + 1, generator=g) * 3).to(dtype)[offset:n + offset].view(shape)
    y, w = torch.randn(shape, generator=g).to(dtype), torch.randn(shape[1], generator=g).to(dtype)
    xd = torch.empty(n + 1, dtype=dtype, device=dev)[offset:n + offset].view(shape)
    xd.copy_(x)
    ref = _norm(x, w)
    _check(rms_norm_rows(xd, w.to(dev)), ref, ref.abs(), dtype)
    s, h = add_rms_norm_rows(xd, y.to(dev), w.to(dev))
    assert torch.equal(s.cpu(), x + y)
    ref = _norm(x + y, w)
    _check(h, ref, ref.abs(), dtype)


def test_rms_norm_other_tensors(dev):
    """Strided rows and a weight of another dtype: as the plain formula gives them."""
    x = torch.randn(6, 40, device=dev).to(torch.bfloat16)
    w = torch.randn(20, device=dev)
    got = rms_norm_rows(x[:, ::2], w)
    assert got.dtype == torch.float32
    assert torch.allclose(got.double().cpu(), _norm(x[:, ::2].cpu(), w.cpu()), rtol=2e-2, atol=1e-2)
    assert rms_norm_rows(torch.empty(0, 20, device=dev), w).shape == (0, 20)


@pytest.mark.parametrize("dtype", list(STEP))
@pytest.mark.parametrize("B,Hq,Hkv,D,norm", [(64, 32, 4, 128, True), (1, 1, 1, 2, True),
                                             (3, 5, 3, 64, False), (2, 7, 1, 192, True)])
def test_qk_norm_rope(dev, dtype, B, Hq, Hkv, D, norm):
    g = torch.Generator().manual_seed(D)
    q, k = (torch.randn(B, h, D, generator=g).to(dtype) for h in (Hq, Hkv))
    cos, sin = (torch.randn(B, D, generator=g).to(dtype) for _ in range(2))
    ws = [torch.randn(D, generator=g).to(dtype) if norm else None for _ in range(2)]
    got = qk_norm_rope(q.to(dev), k.to(dev), *(None if w is None else w.to(dev) for w in ws),
                       cos.to(dev), sin.to(dev))
    for x, w, o in zip((q, k), ws, got):
        x = x.double() if w is None else _norm(x, w)
        c, s = cos.double()[:, None], sin.double()[:, None]
        a, b = x.chunk(2, -1)
        turned = torch.cat([-b, a], -1)
        _check(o, x * c + turned * s, (x * c).abs() + (turned * s).abs(), dtype)


def test_derivatives_pass_through(dev):
    """Values that autograd follows keep their derivatives, in reverse and in forward mode: those of
    the plain formulas (fp32: 2^-20 of the largest, sums of 40 terms in another order)."""
    def all_of(x, y, w, q, c, s):
        total, h = add_rms_norm_rows(x, y, w)
        qo, ko = qk_norm_rope(q, q, w[:16], w[:16], c, s)
        return [rms_norm_rows(x, w), total, h, qo, ko]

    def plain(x, y, w, q, c, s):
        def norm(x, w):
            return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w
        qn = norm(q, w[:16])
        a, b = qn.chunk(2, -1)
        qn = qn * c[:, None] + torch.cat([-b, a], -1) * s[:, None]
        return [norm(x, w), x + y, norm(x + y, w), qn, qn]

    g = torch.Generator().manual_seed(3)
    args = [torch.randn(s, generator=g).to(dev) for s in ((5, 40), (5, 40), (40,), (5, 3, 16),
                                                          (5, 16), (5, 16))]
    leaves = [a.clone().requires_grad_() for a in args]
    ref_leaves = [a.clone().requires_grad_() for a in args]
    weights = [torch.randn(o.shape, generator=g).to(dev) for o in plain(*args)]
    for f, v in ((all_of, leaves), (plain, ref_leaves)):
        sum((o * u).sum() for o, u in zip(f(*v), weights)).backward()
    for a, b in zip(leaves, ref_leaves):
        assert (a.grad - b.grad).abs().max() <= 2.0 ** -20 * b.grad.abs().max() * 40 ** 0.5
    with torch.autograd.forward_ad.dual_level():
        duals = [torch.autograd.forward_ad.make_dual(a, torch.ones_like(a)) for a in args]
        for o, r in zip(all_of(*duals), plain(*duals)):
            t, u = (torch.autograd.forward_ad.unpack_dual(x).tangent for x in (o, r))
            assert (t - u).abs().max() <= 2.0 ** -20 * u.abs().max() * 40 ** 0.5
    with torch.no_grad():   # nothing to follow: the kernels
        for o, r in zip(all_of(*leaves), plain(*leaves)):
            assert (o - r).abs().max() <= 2.0 ** -18 * r.abs().max()
