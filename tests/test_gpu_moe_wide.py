"""GPU parity of the expert GEMM for many routes per expert (moe_gemm_wide) at the edges of its row
tiles, K stages, column tiles and work lists, and of the one-launch permute plan, against the
oracle. Bars as in test_gpu_fused_experts.py: fp32 sums in another order, then one rounding."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle.fused_experts as OF
import oracle.moe_route as OM
from plastic_infer.kernel import moe_align_block_size, moe_expert_gemm
from plastic_infer.kernel.moe_ops import moe_sum_reduce
from plastic_infer.moe.fused import (
    fused_experts_decode_impl, fused_experts_impl, routed_ffn_routes)

pytestmark = pytest.mark.gpu


def _mostly_equal(got: torch.Tensor, ref: torch.Tensor, what: str):
    got, ref = got.float().cpu(), ref.float().cpu()
    diff = got != ref
    assert diff.float().mean().item() < 0.01, what
    if diff.any():
        rel = ((got - ref).abs() / ref.abs().clamp_min(1e-2))[diff].max().item()
        assert rel <= 4 * 2 ** -7, f"{what}: relative difference {rel}"


def _ids(rows_of_expert, T, k, seed):
    """Routes [T, k] that give expert e exactly rows_of_expert[e] of them, the rest -1."""
    flat = np.concatenate([np.full(n, e) for e, n in enumerate(rows_of_expert)])
    assert flat.size <= T * k
    flat = np.concatenate([flat, np.full(T * k - flat.size, -1)])
    return torch.tensor(np.random.default_rng(seed).permutation(flat).reshape(T, k),
                        dtype=torch.int32)


@pytest.mark.parametrize("rows,T,k,H,I,dtype,activation,on_input", [
    # 64-row tiles (mean 18.75): none, one, 16 / 17 / 64 / 65 rows, an expert of four tiles
    ([0, 1, 15, 16, 17, 63, 64, 65, 255] + [15] * 119, 300, 8, 328, 72, torch.bfloat16, "silu",
     False),
    # 128-row tiles (mean 80), K of whole stages and of one element vector more
    ([127, 128, 129, 0, 300] + [60] * 27, 320, 8, 320, 200, torch.float16, "gelu", True),
    # 192-row tiles (mean 150), short K: stages past its end
    ([191, 192, 193, 385] + [80] * 12, 600, 4, 64, 136, torch.bfloat16, "gelu_tanh", False),
    # 320-row tiles (mean 512): 319 / 320 / 321 rows and three tiles
    ([319, 320, 321, 700, 1], 600, 4, 136, 264, torch.bfloat16, "silu", True),
    # over 64 experts per XCD's work list
    ([4] * 599 + [4], 300, 8, 72, 40, torch.float16, "silu", False),
])
def test_wide_expert_gemms(dev, rows, T, k, H, I, dtype, activation, on_input):
    E, numel = len(rows), T * k
    g = torch.Generator().manual_seed(E)
    x = torch.randn(T, H, generator=g).to(dtype)
    w1 = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dtype)
    w2 = (torch.randn(E, H, I, generator=g) * 0.05).to(dtype)
    tw = torch.rand(T, k, generator=g)
    ids = _ids(rows, T, k, E)
    live = (ids >= 0).view(-1)
    _, rc2, rc3 = OF.fused_experts(x, w1, w2, tw, ids.clamp_min(0), activation, on_input,
                                   return_intermediate=True)
    rc2, rc3 = torch.from_numpy(rc2).view(numel, I), torch.from_numpy(rc3).view(numel, H)
    s, e, npp = moe_align_block_size(ids.to(dev), 16, E)
    twd = tw.to(dev)
    # a wider output row than its columns, and rows of dropped routes left alone
    out = torch.full((numel, I + 3), 7.0, dtype=dtype, device=dev)
    c2 = moe_expert_gemm(x.to(dev), w1.to(dev), twd, s, e, npp, 16, numel, k,
                         activation=activation, mul_routed_weight=on_input, out=out[:, :I])
    _mostly_equal(c2.cpu()[live], rc2[live], "first GEMM + activation")
    assert bool((out.cpu()[~live] == 7.0).all()) and bool((out[:, I:] == 7.0).all())
    c3 = moe_expert_gemm(rc2.to(dtype).to(dev), w2.to(dev), twd, s, e, npp, 16, numel, 1,
                         mul_routed_weight=not on_input)
    _mostly_equal(c3.cpu()[live], rc3[live], "second GEMM")


@pytest.mark.parametrize("n_rows,K", [(100, 328), (250, 64), (257, 640)])
def test_wide_odd_columns(dev, n_rows, K):
    """Output columns that are no multiple of a store's eight."""
    T, k, E = 520, 4, 8
    g = torch.Generator().manual_seed(n_rows)
    a = torch.randn(T * k, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(E, n_rows, K, generator=g) * 0.05).to(torch.bfloat16)
    ids = torch.randint(0, E, (T, k), generator=g).to(torch.int32)
    s, e, npp = moe_align_block_size(ids.to(dev), 16, E)
    got = moe_expert_gemm(a.to(dev), w.to(dev), None, s, e, npp, 16, T * k, 1)
    ref = torch.stack([w[x].float() @ r for x, r in zip(ids.view(-1).tolist(), a.float())])
    _mostly_equal(got, ref.to(torch.bfloat16), "odd columns")


@pytest.mark.parametrize("T,k,E,skew", [(1, 1, 1, 0), (128, 8, 2, 0), (512, 8, 255, 1),
                                        (129, 8, 2047, 0), (512, 8, 2048, 0), (205, 5, 300, 1)])
def test_one_launch_plan(dev, T, k, E, skew):
    """The plan of up to 4096 routes: rounds of 1024, waves that share an expert, and either side
    of the largest expert count that has per-wave counters."""
    rng = np.random.default_rng(T + E)
    ids = rng.integers(-1, E + 2, size=(T, k)).astype(np.int32)
    if skew:                                    # most routes to one expert
        ids[rng.random((T, k)) < 0.8] = E - 1
    rs, re, rnpp, rpos = OM.moe_align_block_size(ids, 16, E)
    s, e, npp, pos = moe_align_block_size(torch.tensor(ids, device=dev), 16, E,
                                          return_route_pos=True)
    assert int(npp.item()) == rnpp
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(e.cpu().numpy()[:rnpp // 16], re[:rnpp // 16])
    assert np.array_equal(pos.cpu().numpy(), rpos)


@pytest.mark.parametrize("T,dtype,on_input", [(1, torch.float16, False), (37, torch.bfloat16, True),
                                              (700, torch.bfloat16, False), (9, torch.float32, True)])
def test_ffn_call(dev, T, dtype, on_input):
    """The whole FFN call: strided hidden rows, a caller's activation buffer and route rows, routes
    of no expert left alone, and the result over its own input; all the same bits."""
    H, I, E, k = 264, 72, 9, 3
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H + 8, generator=g).to(dtype).to(dev)[:, :H]
    w1 = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dtype).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.05).to(dtype).to(dev)
    tw, ids = torch.rand(T, k, generator=g).to(dev), torch.randint(-1, E, (T, k), generator=g)
    ids = ids.to(torch.int32).to(dev)
    routes = [torch.full((T, k, H), 7.0, dtype=dtype, device=dev) for _ in range(2)]
    act = torch.empty(T * k, I + 8, dtype=dtype, device=dev)[:, :I]
    routed_ffn_routes(x, w1, w2, tw, ids, routes[0], "gelu", on_input)
    routed_ffn_routes(x, w1, w2, tw, ids, routes[1], "gelu", on_input, act_buffer=act)
    assert torch.equal(routes[0], routes[1])
    assert bool((routes[0][ids < 0] == 7.0).all())
    ref, _, _ = OF.fused_experts(x.cpu(), w1.cpu(), w2.cpu(), tw.cpu(), ids.cpu().clamp_min(0),
                                 "gelu", on_input, return_intermediate=True)
    full = ids.clamp_min(0)
    out = fused_experts_decode_impl(x.contiguous(), w1, w2, tw, full, "gelu", on_input)
    err = (out.cpu().float() - ref.float()).abs().max() / ref.float().abs().max()
    assert err < (2e-5 if dtype == torch.float32 else 1e-2)
    xc = x.contiguous()
    assert fused_experts_impl(xc, w1, w2, tw, full, "gelu", on_input) is xc
    assert torch.equal(xc, out)
    with pytest.raises(ValueError):
        routed_ffn_routes(x, w1, w2[:, :, :64].contiguous(), tw, ids, routes[0], "gelu", on_input)
    with pytest.raises(ValueError):
        routed_ffn_routes(x, w1, w2, tw, ids, routes[0], "gelu", on_input, act_buffer=act[:, :64])


@pytest.mark.parametrize("T", [3, 400])
def test_ffn_fewer_second_matrices(dev, T):
    """w2 with fewer experts than w1: the experts it lacks (and the id one past w1's) give zero rows,
    the others the rows of a call with all of w2, routes of no expert stay as they are."""
    H, I, E, E2, k = 128, 64, 6, 4, 2
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    w1 = (torch.randn(E, 2 * I, H, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    tw = torch.rand(T, k, generator=g).to(dev)
    ids = torch.randint(-1, E + 1, (T, k), generator=g).to(torch.int32).to(dev)
    full, part = (torch.full((T, k, H), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    routed_ffn_routes(x, w1, w2, tw, ids, full)
    routed_ffn_routes(x, w1, w2[:E2].contiguous(), tw, ids, part)
    assert bool((part[ids < 0] == 7.0).all())
    assert not bool(part[ids >= E2].any())
    held = (ids >= 0) & (ids < E2)
    err = (part[held].float() - full[held].float()).abs().max()
    assert err <= 2.0 ** -7 * full[held].float().abs().max()   # one rounding step: other sum order


@pytest.mark.parametrize("E,n_rows,K,activation,line", [
    (32, 2 * 3072, 1000, "silu", 2), (64, 2304, 1408, None, 2),    # no streaming kernel for this K
    (64, 2048, 1104, None, 7), (64, 2048, 1000, None, 8), (64, 2 * 2048, 264, "silu", 14),
    (128, 2048, 768, None, 9), (64, 2 * 1024, 2048, "gelu_tanh", 10),   # one for this
    (64, 3072, 512, None, 12), (32, 2 * 1024, 3072, "silu", 12), (64, 2 * 512, 1024, "gelu", 14),
])
def test_either_side_of_the_line(dev, E, n_rows, K, activation, line):
    """Calls of one route fewer and of as many as the wide kernel takes."""
    g = torch.Generator(device=dev).manual_seed(K)
    w = (torch.randn(E, n_rows, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    for numel in (line * E - 1, line * E):
        a = torch.randn(numel, K, generator=g, device=dev).to(torch.bfloat16)
        ids = torch.randint(0, E, (numel, 1), generator=g, device=dev, dtype=torch.int32)
        s, e, npp = moe_align_block_size(ids, 16, E)
        got = moe_expert_gemm(a, w, None, s, e, npp, 16, numel, 1, activation=activation)
        ref = torch.empty(numel, n_rows, device=dev)
        for x in range(E):
            at = (ids.view(-1) == x).nonzero().view(-1)
            ref[at] = a[at].float() @ w[x].float().t()
        bound = 0.0
        if activation:
            gate, up = ref.to(torch.bfloat16).float().chunk(2, -1)

            def f(x):
                return torch.nn.functional.silu(x) if activation == "silu" else \
                    torch.nn.functional.gelu(x, approximate="tanh" if activation == "gelu_tanh"
                                             else "none")

            # a first sum on the other side of a rounding point: one step (2^-7) of the gate or of up
            step = torch.maximum((f(gate * (1 + 2 ** -7)) - f(gate)).abs(),
                                 (f(gate * (1 - 2 ** -7)) - f(gate)).abs())
            ref = f(gate) * up
            bound = step * up.abs() * (1 + 2 ** -7) + ref.abs() * 2 ** -7
        diff = (got.float() - ref).abs()
        # one step of the result's own, and fp32 sums of K products in another order (2^-20 of ~K^0.5)
        assert bool((diff <= bound + ref.abs() * 2 ** -7 + 2 ** -20 * K ** 0.5).all()), numel
        assert (got != ref.to(torch.bfloat16)).float().mean().item() < 0.01, numel


@pytest.mark.parametrize("T", [40, 1100])
def test_bank_of_several_layers(dev, T):
    """One layer's experts among the slots of a larger bank: the same results with and without the
    number of a layer's experts, whole or in the two parts of a split call."""
    E, used, k, H, I = 256, 32, 4, 128, 96
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    w1 = (torch.randn(E, 2 * I, H, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    tw = torch.rand(T, k, generator=g).to(dev)
    ids = torch.randint(100, 100 + used, (T, k), generator=g).to(torch.int32).to(dev)
    plain = fused_experts_decode_impl(x, w1, w2, tw, ids)
    told = fused_experts_decode_impl(x, w1, w2, tw, ids, layer_experts=used)
    _mostly_equal(told, plain, "layer_experts")
    rows = torch.empty(T, k, H, dtype=torch.bfloat16, device=dev)
    for part in (ids < 110, ids >= 110):
        routed_ffn_routes(x, w1, w2, tw, torch.where(part, ids, -1), rows, layer_experts=used)
    out = torch.empty_like(x)
    moe_sum_reduce(rows, out)
    assert torch.equal(out, told)
