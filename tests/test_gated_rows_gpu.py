"""The gated product of few rows with x whole in shared memory: its rows have the bits that the same rows have in a call of more rows,
which other kernels take (33 to 64 rows through shared memory; 16 rows of 2,048 and more keys, chunks of x)."""
import math

import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(m, inter, k):
    torch.manual_seed(53)
    w = (torch.randn(2 * inter, k, device=DEV) / math.sqrt(k)).bfloat16()
    return torch.randn(m, k, device=DEV).bfloat16(), w, ops.tile_weight(w, 2)


# (13 rows of 2,048 keys and 8 of 3,072 are the most that go whole)
@pytest.mark.parametrize("act", ["gelu_tanh", "silu", ops.ClampedSwish(1.5, 1.702, 1.0)], ids=["gelu_tanh", "silu", "clamped"])
@pytest.mark.parametrize("inter,k", [(16384, 2048), (250, 128), (777, 384), (33, 640), (1000, 3072), (64, 4096)])
def test_rows_have_the_bits_of_more_rows(act, inter, k):
    x, w, tiles = operands(40, inter, k)
    scratch = torch.empty(40, 2 * inter, device=DEV, dtype=torch.bfloat16)
    want = torch.empty(40, inter, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, want, act, scratch, tiles)
    for first, m in ((0, 1), (3, 2), (1, 8), (5, 9), (7, 13), (2, 14), (4, 16), (0, 17), (6, 32)):
        for t in (None, tiles):
            wider = torch.full((m + 1, inter + 24), 7.0, device=DEV, dtype=torch.bfloat16)
            out = wider[:m, 8:8 + inter]
            ops.gated_linear(x[first:first + m], w, out, act, scratch[:m], t)
            assert torch.equal(out, want[first:first + m]), f"{m} rows, copy {t is not None}"
            wider[:m, 8:8 + inter] = 7.0
            assert bool((wider == 7.0).all()), f"{m} rows"


@pytest.mark.parametrize("half,k", [(300, 128), (4096, 2048)])
def test_squared_relu_of_two_halves(half, k):
    x, w, tiles = operands(40, half, k)
    want = torch.empty(40, 2 * half, device=DEV, dtype=torch.bfloat16)
    ops.activated_linear(x, w, want, "squared_relu", paired_tiles=tiles)
    for first, m in ((0, 1), (3, 13), (4, 20)):
        for t in (None, tiles):
            out = torch.empty(m, 2 * half, device=DEV, dtype=torch.bfloat16)
            ops.activated_linear(x[first:first + m], w, out, "squared_relu", paired_tiles=t)
            assert torch.equal(out, want[first:first + m])


@pytest.mark.parametrize("inter,k", [(16384, 2048), (250, 3072), (1000, 5120)])
def test_norm_on_load_has_the_bits_of_more_rows(inter, k):
    _, w, tiles = operands(1, inter, k)
    residual = torch.randn(16, k, device=DEV) * 3
    norm_w = torch.randn(k, device=DEV) * 0.2
    sumsq = residual.square().view(16, -1, 16).sum(-1).contiguous()
    want = torch.empty(16, inter, device=DEV, dtype=torch.bfloat16)
    for t in (None, tiles):
        ops.gated_linear(ops.NormOnLoad(residual, sumsq, norm_w, 1e-6, 1.0, torch.bfloat16), w, want, "gelu_tanh", None, t)
        for first, m in ((0, 1), (3, 2), (1, 5), (5, 8), (7, 9), (2, 13), (1, 14)):
            rows = slice(first, first + m)
            out = torch.full((m + 1, inter), 7.0, device=DEV, dtype=torch.bfloat16)
            ops.gated_linear(ops.NormOnLoad(residual[rows].clone(), sumsq[rows].clone(), norm_w, 1e-6, 1.0, torch.bfloat16), w, out[:m],
                             "gelu_tanh", None, t)
            assert torch.equal(out[:m], want[rows]) and bool((out[m] == 7.0).all()), f"{m} rows, copy {t is not None}"


def test_a_row_that_is_not_finite_stays_alone():
    x, w, tiles = operands(9, 256, 512)
    want, out = (torch.empty(9, 256, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    scratch = torch.empty(9, 512, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, want, "silu", scratch, tiles)
    bad = x.clone()
    bad[4, 100], bad[8, 3] = float("nan"), float("inf")
    ops.gated_linear(bad, w, out, "silu", scratch, tiles)
    others = [0, 1, 2, 3, 5, 6, 7]
    assert torch.equal(out[others], want[others]) and bool(torch.isnan(out[4]).all()) and not bool(torch.isfinite(out[8].float()).all())
