"""GPU parity of the fp32 matrix-core decode kernel (head_dim 64 and 128, fp32 pools, page sizes
other than 16, group sizes up to 16) against a 64-bit evaluation of the reference's decode
(src/plastic_infer/exec/attention.py:151-190), at the edges of its 64 / 128-token tiles.

Bars: scores, probabilities and sums are fp32, so a result is within 4e-6 of the row's largest
|v| (128-term fp32 dot products of N(0, 1) data and a convex combination of v) before it is rounded
once to the pool's dtype: one unit roundoff more for 16 bits (2^-8 / 2^-11 relative).
"""

from __future__ import annotations

import math

import pytest
import torch

from plastic_infer import _native as N
from plastic_infer.kernel import paged_decode_append_attention, paged_decode_attention
from plastic_infer.kernel.paged_kv import decode_workspace_bytes

pytestmark = pytest.mark.gpu

ROUNDOFF = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _reference(q, kp, vp, bt, lens, bad):
    """64-bit decode; tokens on pages in `bad` (row, page index) are no keys."""
    B, Hq, D = q.shape
    P, Hkv = kp.shape[3], kp.shape[1]
    out = torch.zeros(B, Hq, D, dtype=torch.float64)
    for b, n in enumerate(lens.tolist()):
        keep = [t for t in range(n) if (b, t // P) not in bad]
        if not keep:
            continue
        t = torch.tensor(keep)
        pg = bt[b].long()[t // P]
        k, v = (x[pg, :, :, t % P].double() for x in (kp, vp))       # [n, Hkv, D]
        qh = q[b].double().view(Hkv, Hq // Hkv, D)
        p = torch.softmax(qh @ k.permute(1, 2, 0) / math.sqrt(D), -1)
        out[b] = (p @ v.permute(1, 0, 2)).reshape(Hq, D)
    return out


@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("dtype,D,P,G", [
    (torch.float32, 128, 16, 1), (torch.float32, 64, 4, 7), (torch.float32, 128, 12, 16),
    (torch.bfloat16, 64, 16, 4), (torch.bfloat16, 128, 32, 4), (torch.float16, 64, 8, 3),
    (torch.float16, 128, 16, 9), (torch.bfloat16, 128, 8, 16)])
def test_decode_f32_tile_edges(dev, dtype, D, P, G, append):
    Hkv, lens = 2, [1, 3, 63, 64, 65, 127, 128, 129, 0, 700, 2500, 255, 256, 257, 40, 130]
    g = torch.Generator().manual_seed(D + P + G)
    n_pages = [(n + P - 1) // P for n in lens]
    total = sum(n_pages) + 3
    perm = torch.randperm(total, generator=g)
    bt = torch.full((len(lens), max(n_pages)), -1, dtype=torch.int32)
    off = 0
    for b, n in enumerate(n_pages):
        bt[b, :n] = perm[off:off + n].to(torch.int32)
        off += n
    kp = torch.randn(total, Hkv, D, P, generator=g).to(dtype)
    vp = torch.randn(total, Hkv, D, P, generator=g).to(dtype)
    q = torch.randn(len(lens), Hkv * G + 2, D, generator=g).to(dtype)[:, :Hkv * G]
    kn = torch.randn(len(lens), Hkv, D, generator=g).to(dtype)
    vn = torch.randn(len(lens), Hkv, D, generator=g).to(dtype)
    lens_t = torch.tensor(lens, dtype=torch.int32)
    for b, n in enumerate(lens):                  # stale slots past the end hold NaN / Inf
        if n % P:
            kp[bt[b, n // P], :, :, n % P:] = float("nan")
            vp[bt[b, n // P], :, :, n % P:] = float("inf")
    bad = {(10, 3), (14, 0)} | {(14, i) for i in range(n_pages[14])}
    bt_call = bt.clone()
    for b, i in bad:                              # row 10 loses a page, row 14 all of them
        bt_call[b, i] = total if i % 2 else -1
    assert N.query("pia_paged_decode_split_scratch_bytes", Hkv * G, Hkv, D, P,
                   N.dtype_code(dtype)) > 0
    gk, gv = kp.to(dev), vp.to(dev)
    args = (q.to(dev), gk, gv, bt_call.to(dev), lens_t.to(dev))
    if append:
        for b, n in enumerate(lens):
            if n and (b, (n - 1) // P) not in bad:
                kp[bt[b, (n - 1) // P], :, :, (n - 1) % P] = kn[b]
                vp[bt[b, (n - 1) // P], :, :, (n - 1) % P] = vn[b]
                gk[bt[b, (n - 1) // P], :, :, (n - 1) % P] = float("nan")
                gv[bt[b, (n - 1) // P], :, :, (n - 1) % P] = float("inf")
        out = paged_decode_append_attention(*args, kn.to(dev), vn.to(dev)).cpu()
        for got, want in ((gk, kp), (gv, vp)):
            assert torch.equal(got.cpu().nan_to_num(7.0), want.nan_to_num(7.0))
    else:
        out = paged_decode_attention(*args).cpu()
    ref = _reference(q, kp, vp, bt, lens_t, bad)
    assert not out[8].any() and not out[14].any()
    err = (out.double() - ref).abs()
    assert (err <= ROUNDOFF[dtype] * 1.01 * ref.abs() + 4e-6 * 4.0).all(), err.max().item()
    # the same call without scratch (general kernel) agrees within both kernels' error
    if not append:
        alone = torch.empty(q.shape, dtype=dtype, device=dev)
        N.call("pia_paged_decode_attention", alone.data_ptr(), args[0].data_ptr(),
               args[0].stride(0), gk.data_ptr(), gv.data_ptr(), args[3].data_ptr(), bt.shape[1],
               args[4].data_ptr(), len(lens), Hkv * G, Hkv, D, P, total, 1.0 / math.sqrt(D),
               N.dtype_code(dtype), None, 0, N.stream_of(dev))
        diff = (alone.cpu().double() - out.double()).abs()
        assert (diff <= 2.02 * ROUNDOFF[dtype] * ref.abs() + 2 * 4e-6 * 4.0).all()


@pytest.mark.parametrize("dtype", list(ROUNDOFF))
def test_decode_f32_infinite_values(dev, dtype):
    """V holds infinities: the result is that infinity (never infinity - infinity) for one key and
    for many."""
    q = torch.randn(2, 8, 64).to(dtype).to(dev)
    kp, vp = (torch.randn(40, 2, 64, 16).to(dtype).to(dev) for _ in range(2))
    vp[0, :, 5, 0] = float("-inf")
    vp[3, :, 9, :8] = float("inf")
    bt = torch.tensor([[0] + [1] * 19, [3] + list(range(4, 23))], dtype=torch.int32, device=dev)
    out = paged_decode_attention(q, kp, vp, bt, torch.tensor([1, 300], dtype=torch.int32,
                                                             device=dev)).cpu()
    assert torch.equal(out[0].view(2, 4, 64), vp[0, :, :, 0].cpu().view(2, 1, 64).expand(-1, 4, -1))
    assert (out[1, :, 9] == float("inf")).all()
    assert out[1, :, torch.arange(64) != 9].isfinite().all()


@pytest.mark.parametrize("dtype,D,P,G", [
    (torch.float32, 128, 16, 2), (torch.bfloat16, 64, 16, 4), (torch.float16, 128, 32, 16),
    (torch.bfloat16, 128, 16, 4), (torch.float16, 128, 16, 1), (torch.bfloat16, 128, 16, 8),
    (torch.float32, 128, 16, 65)])
def test_decode_nan_score_reaches_its_rows(dev, dtype, D, P, G):
    """A NaN in an admissible key makes the rows of its kv head NaN, whether the sequence is cut over
    waves (rows 0, 1: more steps than one wave's share) or not (row 2), and no other row."""
    Hkv, lens, at = 2, [3000, 2900, 40, 700], [5, 2899, 3, None]
    n_pages = [(n + P - 1) // P for n in lens]
    bt = torch.zeros(len(lens), max(n_pages), dtype=torch.int32)
    for b, n in enumerate(n_pages):
        bt[b, :n] = torch.arange(n) + sum(n_pages[:b])
    g = torch.Generator().manual_seed(G)
    kp, vp = (torch.randn(sum(n_pages), Hkv, D, P, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(len(lens), Hkv * G, D, generator=g).to(dtype)
    for b, t in enumerate(at):
        if t is not None:
            kp[bt[b, t // P], 0, 7, t % P] = float("nan")
    out = paged_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), bt.to(dev),
                                 torch.tensor(lens, dtype=torch.int32, device=dev)).cpu()
    out = out.view(len(lens), Hkv, G, D)
    for b, t in enumerate(at):
        assert out[b, 0].isnan().all() if t is not None else out[b, 0].isfinite().all(), b
        assert out[b, 1].isfinite().all(), b


def _small_call(dev, dtype, D, P):
    g = torch.Generator().manual_seed(D)
    kp, vp = (torch.randn(30, 2, D, P, generator=g).to(dtype).to(dev) for _ in range(2))
    q = torch.randn(2, 8, D, generator=g).to(dtype).to(dev)
    bt = torch.arange(30, dtype=torch.int32, device=dev).view(2, 15)
    return q, kp, vp, bt, torch.tensor([201, 37], dtype=torch.int32, device=dev)


@pytest.mark.parametrize("dtype,D,P", [(torch.float32, 128, 32), (torch.bfloat16, 64, 16)])
def test_decode_f32_leaves_the_callers_workspace(dev, dtype, D, P):
    """decode_workspace_bytes is 0 for these shapes: a workspace passed all the same (one a program
    shares between streams, say) is not written."""
    args = _small_call(dev, dtype, D, P)
    assert decode_workspace_bytes(2, 8, 2, D, P, 15) == 0
    assert N.query("pia_paged_decode_split_scratch_bytes", 8, 2, D, P, N.dtype_code(dtype)) > 0
    ws = torch.full((1 << 26,), 0xAB, dtype=torch.uint8, device=dev)
    out = paged_decode_attention(*args, workspace=ws)
    assert bool((ws == 0xAB).all())
    assert torch.equal(out, paged_decode_attention(*args))


@pytest.mark.parametrize("dtype,D,P", [(torch.float32, 128, 32), (torch.bfloat16, 64, 16)])
def test_decode_f32_without_memory_for_scratch(dev, dtype, D, P, monkeypatch):
    """A pool that leaves no memory for the scratch: the kernel that takes none runs."""
    args = _small_call(dev, dtype, D, P)
    want = paged_decode_attention(*args)
    empty = torch.empty

    def none_left(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no memory left")
        return empty(*a, **kw)

    monkeypatch.setattr(torch, "empty", none_left)
    got = paged_decode_attention(*args)
    monkeypatch.undo()
    diff = (got.double() - want.double()).abs()   # both within the bars above of the exact result
    assert (diff <= 2.02 * ROUNDOFF[dtype] * want.double().abs() + 2 * 4e-6 * 4.0).all()
