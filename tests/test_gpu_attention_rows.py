"""GPU parity of the fp32-precision kernel for several query rows per sequence (fp32 pools,
head_dim 64, other page and group sizes) against a 64-bit evaluation of the reference's attention
with the causal offset rule (src/plastic_infer/exec/runner_paged.py:36-95), at the edges of its
16-row blocks and 64 / 128-token tiles, and with non-finite values that only some rows see.

Bars: as test_gpu_decode_f32: 4e-6 of the largest |v| (about 4), plus one unit roundoff of a 16-bit
result.
"""

from __future__ import annotations

import math

import pytest
import torch

from plastic_infer.kernel import paged_attention

pytestmark = pytest.mark.gpu

ROUNDOFF = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _reference(q, kp, vp, bt, kv_lens, rows, offs, bad):
    Hq, D = q.shape[1:]
    P, Hkv = kp.shape[3], kp.shape[1]
    out = torch.zeros(q.shape, dtype=torch.float64)
    r = 0
    for b, n_rows in enumerate(rows):
        n = int(kv_lens[b])
        t = torch.arange(n)
        pg = bt[b].long()[t // P] if n else t
        k, v = (x[pg, :, :, t % P].double() for x in (kp, vp))       # [n, Hkv, D]
        dead = torch.tensor([(b, int(i) // P) in bad for i in t], dtype=torch.bool)
        for s in range(n_rows):
            see = n if offs is None else max(0, min(n, int(offs[b]) + s + 1))
            keep = ~dead & (t < see)
            if keep.any():
                qh = q[r].double().view(Hkv, Hq // Hkv, D)
                p = torch.softmax(qh @ k[keep].permute(1, 2, 0) / math.sqrt(D), -1)
                out[r] = (p @ v[keep].permute(1, 0, 2)).reshape(Hq, D)
            r += 1
    return out


def _case(dtype, D, P, G, lens, rows, Hkv=2):
    g = torch.Generator().manual_seed(7 * D + P + G)
    n_pages = [(n + P - 1) // P for n in lens]
    perm = torch.randperm(sum(n_pages) + 3, generator=g)
    bt = torch.full((len(lens), max(n_pages)), -1, dtype=torch.int32)
    off = 0
    for b, n in enumerate(n_pages):
        bt[b, :n] = perm[off:off + n].to(torch.int32)
        off += n
    kp, vp = (torch.randn(len(perm), Hkv, D, P, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(sum(rows), Hkv * G, D, generator=g).to(dtype)
    for b, n in enumerate(lens):                  # stale slots past the end hold NaN / Inf
        if n % P:
            kp[bt[b, n // P], :, :, n % P:] = float("nan")
            vp[bt[b, n // P], :, :, n % P:] = float("inf")
    return q, kp, vp, bt, torch.tensor(lens, dtype=torch.int32)


def _cu(rows):
    return torch.tensor([0] + torch.tensor(rows).cumsum(0).tolist(), dtype=torch.int32)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,D,P,G", [
    (torch.float32, 128, 16, 2), (torch.float32, 64, 4, 7), (torch.float32, 128, 12, 20),
    (torch.bfloat16, 64, 16, 4), (torch.bfloat16, 128, 32, 1), (torch.float16, 64, 8, 3),
    (torch.float16, 128, 16, 7)])
def test_rows_block_and_tile_edges(dev, dtype, D, P, G, causal):
    lens = [63, 64, 65, 129, 257, 40, 700, 0, 20, 300]
    rows = [63, 1, 17, 16, 33, 40, 5, 3, 0, 15]
    offs = [0, 63, 48, 113, 224, 0, 650, 0, 0, -4]   # the last: rows before any key
    q, kp, vp, bt, lens_t = _case(dtype, D, P, G, lens, rows)
    bad = {(6, 1), (5, 0)}
    call_bt = bt.clone()
    call_bt[6, 1], call_bt[5, 0] = -1, kp.shape[0]
    offs_t = torch.tensor(offs, dtype=torch.int32)
    out = paged_attention(q.to(dev), kp.to(dev), vp.to(dev), call_bt.to(dev), lens_t.to(dev),
                          cu_q=_cu(rows).to(dev),
                          q_pos_offsets=offs_t.to(dev) if causal else None).cpu()
    ref = _reference(q, kp, vp, bt, lens_t, rows, offs if causal else None, bad)
    err = (out.double() - ref).abs()
    assert (err <= 1.01 * ROUNDOFF[dtype] * ref.abs() + 4e-6 * 4.0).all(), err.max().item()


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 64),
                                     (torch.bfloat16, 64), (torch.float16, 64)])
def test_rows_non_finite_values_reach_only_the_rows_that_see_them(dev, dtype, D):
    """V of two tokens is Inf / NaN: rows before them stay finite and exact, rows at or after
    them get the reference's Inf / NaN."""
    lens, rows = [200], [40]
    q, kp, vp, bt, lens_t = _case(dtype, D, 16, 4, lens, rows)
    for tok, val in ((175, float("inf")), (190, float("nan"))):
        vp[bt[0, tok // 16], :, 3:7, tok % 16] = val
    out = paged_attention(q.to(dev), kp.to(dev), vp.to(dev), bt.to(dev), lens_t.to(dev),
                          cu_q=_cu(rows).to(dev),
                          q_pos_offsets=torch.tensor([160], dtype=torch.int32, device=dev)).cpu()
    ref = _reference(q, kp, vp, bt, lens_t, rows, [160], set())
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    # a single key: its probability is 1 and the result is its V, infinities included
    vp[bt[0, 0], :, 5, 0] = float("-inf")
    one = paged_attention(q[:1].to(dev), kp.to(dev), vp.to(dev), bt.to(dev),
                          torch.ones(1, dtype=torch.int32, device=dev)).cpu()
    assert torch.equal(one.view(1, 2, 4, D), vp[bt[0, 0], :, :, 0].view(1, 2, 1, D).expand(-1, -1, 4, -1))
    ok = ref.isfinite()
    err = (out.double() - ref)[ok].abs()
    assert (err <= 1.01 * ROUNDOFF[dtype] * ref[ok].abs() + 4e-6 * 4.0).all(), err.max().item()


def test_one_row_per_sequence_and_trailing_rows(dev):
    """Without cu_q row b belongs to sequence b; rows past cu_q's end belong to the last one."""
    lens = [1, 64, 500, 0, 129]
    q, kp, vp, bt, lens_t = _case(torch.float32, 128, 16, 4, lens, [1] * 5)
    args = (kp.to(dev), vp.to(dev), bt.to(dev), lens_t.to(dev))
    out = paged_attention(q.to(dev), *args).cpu()
    ref = _reference(q, kp, vp, bt, lens_t, [1] * 5, None, set())
    assert (out.double() - ref).abs().max() <= 4e-6 * 4.0
    cu = torch.tensor([0, 1, 2, 3, 3, 4], dtype=torch.int32)
    out = paged_attention(q.to(dev), *args, cu_q=cu.to(dev)).cpu()
    ref = _reference(q, kp, vp, bt, lens_t, [1, 1, 1, 0, 2], None, set())
    assert (out.double() - ref).abs().max() <= 4e-6 * 4.0
