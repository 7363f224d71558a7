"""GPU parity of decode attention on fp16 pools. fp16 at head_dim 128 / page size 16 runs the
same kernels as bf16 (paged_decode_stream for Hq / Hkv in {1, 2, 4}, paged_decode_mfma for 8):
the scores, the online softmax and the P . V sums in fp32, the probabilities rounded to fp16
(bf16 for bf16 pools) as the operands of the P . V products, the output rounded to fp16. The
reference runs its torch path in the pools' dtype (src/plastic_infer/exec/attention.py:151-190,
src/plastic_infer/exec/runner_paged.py:112-129, 251-255).

Bars: the pools after an append call equal the oracle's write of the new rows bit for bit
(OP.scatter_slots), with the new tokens' slots holding NaN / Inf before the call; outputs are
within 5e-3 of the oracle (fp16 keeps 11 significant bits: the rounding of a probability to
fp16 moves an output of magnitude <= ~1 by at most a few 1e-4, against 2e-2 for bf16's 8).
"""

from __future__ import annotations

import pytest
import torch

import oracle.paged_kv as OP
from plastic_infer.kernel import paged_decode_append_attention, paged_decode_attention
from plastic_infer.kernel.paged_kv import decode_workspace_bytes
from test_gpu_append_decode import _case, _check
from test_gpu_attention import oracle_max_err_all_rows, qwen3_8b_b256_inputs

pytestmark = pytest.mark.gpu

FP16_TOL = 5e-3


@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_fp16_append_decode_groups_and_edge_lengths(dev, G):
    """Lengths around page (16) and step (128) boundaries; the append call against the oracle
    and against kv_scatter + paged_decode_attention on the same fp16 inputs."""
    Hkv = 8 if G < 8 else 4
    lens = [1, 15, 16, 17, 127, 128, 129, 511, 512, 513, 1024, 1100]
    q, kp, vp, bt, lens_t, kn, vn = _case(60 + G, lens, Hkv * G, Hkv, 1200, dtype=torch.float16)
    _check(dev, q, kp, vp, bt, lens_t, kn, vn, 16, tol=FP16_TOL)


@pytest.mark.parametrize("G,lens", [
    (4, [8192]),                 # one segment per kv head, cut over many waves and merged
    (1, [8191, 3]),
    (2, [0, 4097, 0, 129, 0]),   # empty sequences between and around long ones
    (8, [8192]),
    (8, [0, 4097, 0, 129, 0]),
])
def test_fp16_decode_long_sequences_split_over_waves(dev, G, lens):
    Hkv = 8
    q, kp, vp, bt, lens_t, _, _ = _case(70 + G, lens, Hkv * G, Hkv, 1100, dtype=torch.float16)
    out = paged_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), bt.to(dev),
                                 lens_t.to(dev)).cpu()
    assert out.dtype == torch.float16
    live = lens_t > 0
    assert not out[~live].any()
    ref = OP.decode_batch(q[live], kp, vp, bt[live].clamp(min=0), lens_t[live], 16)
    err = (out[live].float() - ref.float()).abs().max().item()
    assert err <= FP16_TOL, err


@pytest.mark.parametrize("G", [4, 8])
def test_fp16_decode_stale_tail_tokens(dev, G):
    """Tokens past a sequence's length on its last page hold NaN (K) and Inf (V): they are not
    keys, so the output stays finite and equal to the oracle's over the first L tokens."""
    Hkv = 4
    lens = [37, 200, 1000, 4093]
    q, kp, vp, bt, lens_t, _, _ = _case(80 + G, lens, Hkv * G, Hkv, 400, dtype=torch.float16)
    ref = OP.decode_batch(q, kp, vp, bt.clamp(min=0), lens_t, 16)
    for b, L in enumerate(lens):
        page = int(bt[b, (L - 1) // 16])
        kp[page, :, :, L % 16:] = float("nan")
        vp[page, :, :, L % 16:] = float("inf")
    out = paged_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), bt.to(dev),
                                 lens_t.to(dev)).cpu()
    assert torch.isfinite(out.float()).all()
    err = (out.float() - ref.float()).abs().max().item()
    assert err <= FP16_TOL, err


def test_fp16_append_qwen3_8b_b256_full_shape(dev):
    """The decode step of the benchmark at full size on fp16 pools: one
    paged_decode_append_attention call (B = 256, L ~ U[512, 8192], a 160k-page pool, seed 2),
    the new tokens' slots poisoned first; the pools bit-exact against the oracle's write over
    the whole pool and all 256 rows against the oracle's decode."""
    P = 16
    q, kp, vp, bt, lens, n_pages, page, offset, slots, k_new, v_new = qwen3_8b_b256_inputs(
        dev, torch.float16)
    pg, of = page.to(dev), offset.to(dev)
    kp[pg, :, :, of] = float("nan")
    vp[pg, :, :, of] = float("inf")
    kb, vb = kp.cpu(), vp.cpu()
    out = paged_decode_append_attention(q, kp, vp, bt.to(dev), lens.to(torch.int32).to(dev),
                                        k_new, v_new)
    OP.scatter_slots(k_new.cpu(), v_new.cpu(), kb, vb, slots.tolist())
    assert torch.equal(kp.cpu(), kb), "K pool differs from the oracle's write"
    assert torch.equal(vp.cpu(), vb), "V pool differs from the oracle's write"
    del kb, vb
    worst = oracle_max_err_all_rows(out.cpu(), q, kp, vp, bt, lens, n_pages, P)
    assert worst <= FP16_TOL, worst


@pytest.mark.parametrize("lens", [
    [130], [900], [1000], [3001],           # 2, 8, 8 and 24 pieces per head, each wave one step
    [700, 5, 1100, 129, 0, 2000],           # fewer and more than eight pieces in one launch
    [2000] * 24,                            # several steps a wave, both ends of its range cut
])
@pytest.mark.parametrize("dtype,G", [(torch.float16, 4), (torch.bfloat16, 8), (torch.float32, 2)])
def test_arrivals_from_any_workspace(dev, dtype, G, lens):
    """Cut segments are merged once whatever the counters hold: a workspace of any content, and the
    same one after calls of other shapes. Every call gives the same bits; with the tolerance of the
    files of the three kernels against the oracle."""
    Hkv = 8
    need = sum((n + 15) // 16 for n in lens) + 8
    q, kp, vp, bt, lens_t, _, _ = _case(80 + G, lens, Hkv * G, Hkv, need, dtype=dtype)
    args = [x.to(dev) for x in (q, kp, vp, bt, lens_t)]
    size = decode_workspace_bytes(len(lens), Hkv * G, Hkv, 128, 16, bt.shape[1])
    g = torch.Generator(device=dev).manual_seed(G)
    outs = [paged_decode_attention(*args)]
    for fill in (0, 0xFF, None):
        ws = torch.randint(0, 256, (size,), generator=g, device=dev, dtype=torch.uint8) \
            if fill is None else torch.full((size,), fill, dtype=torch.uint8, device=dev)
        for _ in range(3):
            outs.append(paged_decode_attention(*args, workspace=ws))
            paged_decode_attention(args[0][:1], *args[1:3], args[3][:1], args[4][:1], workspace=ws)
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    live = lens_t > 0
    ref = OP.decode_batch(q[live], kp, vp, bt[live].clamp(min=0), lens_t[live], 16)
    tol = {torch.float16: FP16_TOL, torch.bfloat16: 2e-2, torch.float32: 1e-5}[dtype]
    assert (outs[0].cpu()[live].float() - ref.float()).abs().max().item() <= tol
