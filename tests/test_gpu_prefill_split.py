"""GPU parity of the multi-row attention kernel's three shapes (256-row items, 128-row items, and
128-row items whose keys two wave groups share) and of its work list over the XCDs, against the
same attention in float64. Bar: the probabilities' and the output's rounding to the storage dtype,
2^-8 each of the largest |V| in bf16 (2^-11 in fp16)."""

from __future__ import annotations

import math

import pytest
import torch

from plastic_infer.kernel import paged_attention

pytestmark = pytest.mark.gpu

P, D = 16, 128


def _case(dev, rows, ctx, Hq, Hkv, dtype, seed=0, width=0):
    g = torch.Generator().manual_seed(seed)
    kv = [r + c for r, c in zip(rows, ctx)]
    n = [(x + P - 1) // P for x in kv]
    pages = sum(n) + 3
    perm = torch.randperm(pages, generator=g).to(torch.int32)
    bt = torch.full((len(rows), max(max(n), width)), -1, dtype=torch.int32)
    off = 0
    for b, k in enumerate(n):
        bt[b, :k] = perm[off:off + k]
        off += k
    kp, vp = (torch.randn(pages, Hkv, D, P, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(sum(rows), Hq, D, generator=g).to(dtype)
    cu = torch.zeros(len(rows) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(rows), 0)
    return q, kp, vp, bt, torch.tensor(kv, dtype=torch.int32), cu, \
        torch.tensor(ctx, dtype=torch.int32)


def _ref(q, kp, vp, bt, kv, cu, ctx):
    out = torch.empty(q.shape, dtype=torch.float64)
    Hq, Hkv = q.shape[1], kp.shape[1]
    for b, n in enumerate(kv.tolist()):
        ids = bt[b, :(n + P - 1) // P].long()
        k, v = (x[ids].double().permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :n] for x in (kp, vp))
        r0, r1 = int(cu[b]), int(cu[b + 1])
        hide = torch.arange(n)[None] > int(ctx[b]) + torch.arange(r1 - r0)[:, None]
        for h in range(Hq):
            s = q[r0:r1, h].double() @ k[h * Hkv // Hq].t() / math.sqrt(D)
            out[r0:r1, h] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ v[h * Hkv // Hq]
    return out


# 50 pages: the launch of two wave groups where items are few, which share keys from six tiles on
@pytest.mark.parametrize("width", [0, 50])
@pytest.mark.parametrize("rows,ctx,Hq,Hkv,dtype", [
    # few items: one tile, an odd count of tiles, a group without a tile for the first rows,
    # ragged sequences; kv heads that do and do not divide over the XCDs
    ([5], [0], 32, 8, torch.bfloat16),
    ([64], [65], 8, 8, torch.float16),
    ([33, 4, 130], [0, 700, 63], 24, 3, torch.bfloat16),
    ([300], [129], 16, 2, torch.float16),
    ([17, 1, 90], [250, 0, 1], 28, 7, torch.bfloat16),
    # 128-row items on their own
    ([260, 300, 200, 250], [0, 5, 64, 300], 32, 8, torch.bfloat16),
    # 256-row items (512 or more of them)
    ([520] * 5 + [600, 3], [0, 64, 1, 0, 0, 100, 0], 64, 64, torch.float16),
])
def test_prefill_shapes(dev, rows, ctx, Hq, Hkv, dtype, width):
    args = _case(dev, rows, ctx, Hq, Hkv, dtype, width=width)
    q, kp, vp, bt, kv, cu, off = (x.to(dev) for x in args)
    got = paged_attention(q, kp, vp, bt, kv, cu_q=cu, q_pos_offsets=off).double().cpu()
    tol = 2.0 * args[2].abs().max().item() * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
    assert (got - _ref(*args)).abs().max().item() <= tol


def test_shared_keys_nonfinite(dev):
    """A NaN or infinite key or value reaches the rows that see it and no other row; a row with no key
    at all is zero. In the launch of two wave groups, an item of three tiles (one group's)."""
    rows, ctx, Hq, Hkv = [70], [100], 8, 8
    q, kp, vp, bt, kv, cu, off = _case(dev, rows, ctx, Hq, Hkv, torch.bfloat16, 3, 50)
    clean = _ref(q, kp, vp, bt, kv, cu, off)
    kp[bt[0, 10].long(), 1, 5, 9] = math.nan      # token 169: tile 2, the last row only
    kp[bt[0, 4].long(), 2, 7, 0] = math.nan       # token 64: tile 1, every row
    dev_args = [x.to(dev) for x in (q, kp, vp, bt, kv, cu, off)]
    got = paged_attention(*dev_args[:5], cu_q=dev_args[5], q_pos_offsets=dev_args[6]).cpu()
    assert bool(got[69, 1].isnan().all()) and bool(got[:, 2].isnan().all())
    keep = torch.ones(70, 8, dtype=torch.bool)
    keep[69, 1] = keep[:, 2] = False
    tol = 2.0 * vp.abs().max().item() * 2 ** -8
    assert (got.double()[keep] - clean[keep]).abs().max().item() <= tol
    dev_args[4] = torch.zeros_like(dev_args[4])   # no keys
    got = paged_attention(*dev_args[:5], cu_q=dev_args[5], q_pos_offsets=dev_args[6])
    assert bool((got == 0).all())


@pytest.mark.parametrize("rows,ctx,Hq,Hkv,dtype", [
    # 11, 12, 13 and 14 tiles of 64 keys: the last that one group takes, an even and an odd count
    # for two; a last tile of one key; items of one call on either side, with the early rows of an
    # item short of its last tiles
    ([40], [660], 8, 8, torch.bfloat16),
    ([40], [728], 32, 8, torch.float16),
    ([33, 5], [736, 800], 16, 2, torch.bfloat16),
    ([300, 20, 130], [640, 100, 702], 28, 7, torch.bfloat16),
])
def test_keys_shared_by_two_groups(dev, rows, ctx, Hq, Hkv, dtype):
    args = _case(dev, rows, ctx, Hq, Hkv, dtype, 5, 50)
    q, kp, vp, bt, kv, cu, off = (x.to(dev) for x in args)
    got = paged_attention(q, kp, vp, bt, kv, cu_q=cu, q_pos_offsets=off).double().cpu()
    tol = 2.0 * args[2].abs().max().item() * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
    assert (got - _ref(*args)).abs().max().item() <= tol


def test_shared_keys_nonfinite_long(dev):
    """A NaN key in either group's tiles of an item that two groups share."""
    q, kp, vp, bt, kv, cu, off = _case(dev, [70], [900], 8, 8, torch.bfloat16, 3)
    clean = _ref(q, kp, vp, bt, kv, cu, off)
    kp[bt[0, 60].long(), 1, 5, 9] = math.nan      # token 969: tile 15 (group 1), the last row only
    kp[bt[0, 32].long(), 2, 7, 0] = math.nan      # token 512: tile 8 (group 0), every row
    got = paged_attention(*(x.to(dev) for x in (q, kp, vp, bt, kv)), cu_q=cu.to(dev),
                          q_pos_offsets=off.to(dev)).cpu()
    assert bool(got[69, 1].isnan().all()) and bool(got[:, 2].isnan().all())
    keep = torch.ones(70, 8, dtype=torch.bool)
    keep[69, 1] = keep[:, 2] = False
    tol = 2.0 * vp.abs().max().item() * 2 ** -8
    assert (got.double()[keep] - clean[keep]).abs().max().item() <= tol


@pytest.mark.parametrize("rows,ctx", [([300], [0]), ([17, 150, 301], [100, 0, 200]), ([90], [600])])
def test_table_width_changes_nothing(dev, rows, ctx):
    """A block table wider than its sequences need (a program with tables of one width): the same
    bits, so the same split of the keys, which goes by the keys there are."""
    q, kp, vp, bt, kv, cu, off = (x.to(dev) for x in _case(dev, rows, ctx, 32, 8, torch.bfloat16))
    wide = torch.full((len(rows), 512), -1, dtype=torch.int32, device=dev)
    wide[:, :bt.shape[1]] = bt
    assert torch.equal(paged_attention(q, kp, vp, bt, kv, cu_q=cu, q_pos_offsets=off),
                       paged_attention(q, kp, vp, wide, kv, cu_q=cu, q_pos_offsets=off))


@pytest.mark.parametrize("rows,ctx,Hq,Hkv,dtype", [
    # kv heads that XCDs share (4, 10, 6, 3 heads: two, four, four, eight XCDs a head): sequences alike,
    # dealt out in runs; of equal rows but other contexts, and of other rows, item by item
    ([70] * 4, [30] * 4, 32, 4, torch.bfloat16),
    ([130] * 2, [300, 290], 16, 4, torch.float16),
    ([65] * 8, [0] * 8, 20, 10, torch.bfloat16),
    ([33] * 4, [100] * 4, 48, 6, torch.bfloat16),
    ([40] * 8, [16] * 8, 12, 3, torch.float16),
    ([70] * 4, [0, 600, 10, 300], 32, 4, torch.bfloat16),
    ([1, 139, 70, 70], [0, 0, 64, 1], 20, 10, torch.bfloat16),
    ([50] * 3, [20] * 3, 12, 3, torch.bfloat16),
    # equal chunks whose 256-row items fill the compute units once (a line in the launch)
    ([512] * 4, [0] * 4, 32, 8, torch.bfloat16),
    ([1024], [1200], 64, 8, torch.bfloat16),
])
def test_work_lists(dev, rows, ctx, Hq, Hkv, dtype):
    args = _case(dev, rows, ctx, Hq, Hkv, dtype, 9)
    q, kp, vp, bt, kv, cu, off = (x.to(dev) for x in args)
    got = paged_attention(q, kp, vp, bt, kv, cu_q=cu, q_pos_offsets=off).double().cpu()
    tol = 2.0 * args[2].abs().max().item() * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
    assert (got - _ref(*args)).abs().max().item() <= tol
