"""float32 products whose last tile of rows is part full: the blocks without rows are left out, the bits stay."""
import math

import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows at which the last tile of 64 or 128 has one row, one block of 16, one more, or all but one; products whole and cut along K
@pytest.mark.parametrize("n,k", [(32768, 512), (2048, 2048), (2568, 1540), (300, 16384), (8200, 1028)])
def test_rows_have_the_bits_of_whole_tiles(n, k):
    torch.manual_seed(57)
    w = torch.randn(n, k, device=DEV) / math.sqrt(k)
    x = torch.randn(512, k, device=DEV)
    whole = torch.empty(512, n, device=DEV)
    ops.linear(x, w, whole)
    # one rounding a product and sum, sums of 512 keys and then of the segments: 512 + k / 512 roundings of half a unit each, in a chain
    bound = (512 + k / 512) * 2.0 ** -24
    exact = x[:8].double() @ w.double().T
    assert bool(((whole[:8].double() - exact).abs() <= bound * (x[:8].double().abs() @ w.double().abs().T)).all())
    for m in (65, 66, 79, 80, 81, 95, 97, 112, 127, 129, 145, 160, 161, 193, 222, 257, 260, 289, 333, 369, 400, 450, 511):
        out = torch.full((m + 1, n), 7.0, device=DEV)
        ops.linear(x[:m], w, out[:m])
        assert torch.equal(out[:m], whole[:m]) and bool((out[m] == 7.0).all()), f"{m} rows"
