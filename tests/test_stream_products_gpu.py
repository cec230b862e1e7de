"""The products of at most 64 rows that bring everything through shared memory, at the edges of tiles of 16 rows, of workgroups'
columns and of their rings, from the weight row by row and from its tile-major copy.  The one of many columns and the gated one have
the bits of the few-row kernels, which take the same operands where they begin at odd places; the one whose wavefronts meet
has a stack of its own pieces, whose sum in order a whole result is."""
import math

import pytest
import torch

from wllm_amd.kernels import ops
from wllm_amd.kernels.hip_backend import HipBackend

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(m, n, k, halves=1):
    torch.manual_seed(41)
    w = (torch.randn(halves * n, k, device=DEV) / math.sqrt(k)).bfloat16()
    flat = torch.randn(m * k + 8, device=DEV).bfloat16()
    x, odd = flat[:m * k].view(m, k), torch.empty(m * k + 1, device=DEV, dtype=torch.bfloat16)[1:].view(m, k)
    odd.copy_(x)
    return x, odd, w, ops.tile_weight(w, halves)


@pytest.mark.parametrize("n,k", [(12289, 1024), (12300, 2048), (20000, 512)])
def test_split_products(n, k):
    splits = HipBackend.skinny_split(n, k)
    assert splits > 1 and k % (64 * splits) == 0 and HipBackend.piece_split(n, k) == (0, 0)
    for m in (1, 16, 17, 33, 64):
        x, odd, w, tiles = operands(m, n, k)
        assert HipBackend.stream_takes(x.data_ptr(), w.data_ptr(), m, n, k, splits)
        assert not HipBackend.stream_takes(odd.data_ptr(), w.data_ptr(), m, n, k, splits)
        want = torch.empty(splits, m, n, device=DEV)
        ops.linear(odd, w, want, tiles)
        for t in (None, tiles):
            stack = torch.full((splits + 1, m, n), 7.0, device=DEV)
            ops.linear(x, w, stack[:splits], t)
            assert torch.equal(stack[:splits], want) and bool((stack[splits] == 7.0).all()), f"{m} rows, copy {t is not None}"
        for dtype in (torch.bfloat16, torch.float32):
            whole, whole_odd = torch.full((m + 1, n), 7.0, device=DEV, dtype=dtype), torch.empty(m, n, device=DEV, dtype=dtype)
            ops.linear(x, w, whole[:m], tiles)
            ops.linear(odd, w, whole_odd, tiles)
            assert torch.equal(whole[:m], whole_odd) and bool((whole[m] == 7.0).all())
    assert float((want.sum(0).double() - x.double() @ w.double().T).abs().max()) <= k / 32 * 8 * 2 ** -23


# one, two and three bands a workgroup, two to sixteen pieces, columns that fill no band, pieces whose steps of 64 keys the four
# wavefronts share unevenly
@pytest.mark.parametrize("n,k", [(2048, 2048), (2560, 2048), (2568, 768), (100, 4096), (3072, 24576), (2047, 16384), (40, 1024), (10304, 2048),
                                 (6145, 1152), (130, 3072), (2048, 5632), (3000, 1408)])
def test_products_whose_wavefronts_meet(n, k):
    pieces, _ = HipBackend.piece_split(n, k)
    assert pieces > 1
    for m in (1, 15, 16, 17, 33, 48, 49, 64):
        x, odd, w, tiles = operands(m, n, k)
        assert ops.linear_splits(m, n, k, torch.bfloat16) == pieces
        x[m // 2] *= 100.0          # (a row is its own product)
        odd.copy_(x)
        exact = x.double() @ w.double().T
        # float32 sums of K products: each step of 32 keys, wavefront and piece rounds a partial sum below 8 (800) deviations
        bound = (k / 32 + 8) * 8 * 2 ** -23 * x.double().square().mean(1, keepdim=True).sqrt()
        first = None
        for t in (None, tiles):
            stack = torch.full((pieces + 1, m, n), 7.0, device=DEV)
            ops.linear(x, w, stack[:pieces], t)
            assert bool((stack[pieces] == 7.0).all()) and bool(((stack[:pieces].double().sum(0) - exact).abs() <= bound).all())
            first = stack[:pieces].clone() if first is None else first
            assert torch.equal(stack[:pieces], first), "the copy of the weight has the bits of the weight"
            part = k // pieces
            for p in range(pieces):
                want = x[:, p * part:(p + 1) * part].double() @ w[:, p * part:(p + 1) * part].double().T
                assert bool(((stack[p].double() - want).abs() <= bound).all()), f"piece {p}"
            whole = first[0].clone()
            for p in first[1:]:
                whole += p
            for dtype in (torch.bfloat16, torch.float32):
                out = torch.full((m + 1, n), 7.0, device=DEV, dtype=dtype)
                ops.linear(x, w, out[:m], t)
                assert torch.equal(out[:m], whole.to(dtype)) and bool((out[m] == 7.0).all()), f"{m} rows, {dtype}"
            # operands that begin at odd places take the few-row kernels, in the same pieces
            other, out = torch.empty(pieces, m, n, device=DEV), torch.empty(m, n, device=DEV)
            ops.linear(odd, w, other, t)
            ops.linear(odd, w, out, t)
            assert bool(((other - first).abs() <= 2 * bound).all()) and bool(((out.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("act", ["gelu_tanh", "silu", ops.ClampedSwish(1.5, 1.702, 1.0)], ids=["gelu_tanh", "silu", "clamped"])
@pytest.mark.parametrize("inter,k", [(16384, 2048), (250, 128), (777, 384), (64, 2048), (1000, 3072)])
def test_gated_products(act, inter, k):
    for m in (33, 48, 49, 64):
        x, odd, w, tiles = operands(m, inter, k, halves=2)
        want = torch.empty(m, inter, device=DEV, dtype=torch.bfloat16)
        scratch = torch.empty(m, 2 * inter, device=DEV, dtype=torch.bfloat16)
        ops.gated_linear(odd, w, want, act, scratch, tiles)
        wider = torch.full((m, inter + 24), 7.0, device=DEV, dtype=torch.bfloat16)
        for t in (None, tiles):
            for out in (torch.empty(m, inter, device=DEV, dtype=torch.bfloat16), wider[:, 8:8 + inter]):
                ops.gated_linear(x, w, out, act, scratch, t)
                assert torch.equal(out, want), f"{m} rows, copy {t is not None}"
        assert bool((wider[:, :8] == 7.0).all()) and bool((wider[:, 8 + inter:] == 7.0).all())


@pytest.mark.parametrize("half,k", [(300, 128), (4096, 2048)])
def test_squared_relu_of_two_halves(half, k):
    for m in (33, 64):
        x, odd, w, tiles = operands(m, half, k, halves=2)
        want, out = (torch.empty(m, 2 * half, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        ops.activated_linear(odd, w, want, "squared_relu", paired_tiles=tiles)
        for t in (None, tiles):
            ops.activated_linear(x, w, out, "squared_relu", paired_tiles=t)
            assert torch.equal(out, want)
