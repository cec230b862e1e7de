"""float32 products made of bfloat16 parts (`split_product.h`): how far they are off, numbers of any size, infinities and NaN, and tiles of every height."""
import math

import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product(x, w, tiles=None):
    out = torch.full((x.shape[0] + 1, w.shape[0]), 7.0, device=DEV)
    ops.linear(x, w, out[:-1], tiles)
    assert bool((out[-1] == 7.0).all())
    return out[:-1]


# at most 64 rows (row-major and tile-major), tiles of 2 to 8 blocks of 16 rows, K axes that end inside a step of 32 and inside a segment of 512
@pytest.mark.parametrize("m", [1, 17, 64, 65, 81, 97, 128, 145, 333, 600])
@pytest.mark.parametrize("n,k", [(2048, 2048), (70, 1036), (33000, 516), (130, 52), (16, 4)])
def test_off_by_less_than_a_chain_of_float32_sums(m, n, k):
    torch.manual_seed(63)
    x = torch.randn(m, k, device=DEV) * torch.exp2(torch.randint(-12, 12, (m, 1), device=DEV).float())
    w = torch.randn(n, k, device=DEV) / math.sqrt(k)
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # six sums a step of 32 keys and one a segment, each rounded to (or cut off at) 2^-23, and what the split leaves out, 2^-25
    bound = (6 * math.ceil(min(k, 512) / 32) + math.ceil(k / 512)) * 2.0 ** -23 + 2.0 ** -25
    got = product(x, w)
    assert bool(((got.double() - exact).abs() <= bound * size).all())
    if m <= 64:
        assert torch.equal(product(x, w, ops.tile_weight(w)), got)
    # in the 2-norm no further off than float32 products added one by one (three quarters of a unit a step of the chain, at random)
    ref = float((got.double() - exact).norm() / exact.norm())
    assert ref <= 2.0 ** -24 * (1.0 + 0.75 * math.sqrt(min(k, 512)))


@pytest.mark.parametrize("m", [5, 64, 100, 333])
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -60, 2.0 ** 60, 2.0 ** 115])
def test_numbers_of_any_size(m, scale):
    """The parts have float32's range: what they leave to the last bit lies above bfloat16's smallest numbers down to 2^-110."""
    torch.manual_seed(64)
    x = torch.randn(m, 640, device=DEV)
    w = torch.randn(300, 640, device=DEV)
    got, want = product(x * scale, w), product(x, w) * scale
    # (at 2^-100 the smallest of x are below 2^-110)
    assert bool(((got - want).abs() <= (2.0 ** -24 if scale < 2.0 ** -90 else 0.0) * scale * (x.abs() @ w.abs().T)).all())


@pytest.mark.parametrize("m", [3, 64, 70, 200, 333])
@pytest.mark.parametrize("n,k", [(2048, 2048), (33000, 516), (30, 40)])
def test_what_is_not_finite_reaches_its_rows_and_columns_alone(m, n, k):
    torch.manual_seed(65)
    x = torch.randn(m, k, device=DEV)
    w = torch.randn(n, k, device=DEV) / math.sqrt(k)
    clean = product(x, w)
    x[1, 3], x[m - 1, k - 1], x[2, k // 2] = math.inf, math.nan, -math.inf
    w[n - 2, 0], w[5, k - 2] = math.nan, math.inf
    w[9, 3] = 0.0                                              # infinity times nothing
    x[0, 2], w[12, 2] = 3.4e38, 1e-3                           # finite, and beyond bfloat16's largest number
    got = product(x, w)
    # infinities and NaN as 64 bits have them, where no sum of finite numbers leaves float32 (x[0, 2] by columns of w[:, 2] of a size below one)
    exact = x.double() @ w.double().T
    assert bool((w[:, 2].abs() < 0.9).all())
    assert torch.equal(torch.isnan(got), torch.isnan(exact)) and torch.equal(got[torch.isinf(exact)].double(), exact[torch.isinf(exact)])
    touched_rows = torch.tensor([0, 1, 2, m - 1], device=DEV)
    touched_columns = torch.tensor([5, 9, 12, n - 2], device=DEV)
    rows = torch.ones(m, dtype=torch.bool, device=DEV).index_fill_(0, touched_rows, False)
    columns = torch.ones(n, dtype=torch.bool, device=DEV).index_fill_(0, touched_columns, False)
    assert torch.equal(got[rows][:, columns], clean[rows][:, columns])
    finite = torch.isfinite(exact)
    size = torch.nan_to_num(x.double().abs(), posinf=0.0) @ torch.nan_to_num(w.double().abs(), posinf=0.0).T
    # (those made again are a chain of a segment's products: 512 + k / 512 roundings)
    assert bool(((got.double() - exact).abs()[finite] <= (512 + k / 512) * 2.0 ** -23 * size[finite]).all())
    if m <= 64:
        assert torch.equal(torch.nan_to_num(product(x, w, ops.tile_weight(w)), nan=1.5), torch.nan_to_num(got, nan=1.5))
