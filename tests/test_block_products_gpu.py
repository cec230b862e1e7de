"""Products of some hundred to two thousand rows in tiles of one round, against the product in 64 bits, and their rows against each other."""
import math

import pytest
import torch

from wllm_amd.kernels import ops
from wllm_amd.kernels.hip_backend import HipBackend

DEV = "cuda"


def test_the_rule():
    takes = HipBackend.block_tile
    assert takes(64, 2048, 2048) is None and takes(65, 2048, 2048) == (64, 64) and takes(100, 2048, 2080) is None
    assert takes(512, 2048, 2048) == (64, 64) and takes(513, 2048, 2048) == (128, 64) and takes(1025, 2048, 2048) == (192, 64)
    assert takes(1537, 2048, 2048) == (128, 128) and takes(2049, 2048, 2048) == (192, 128) and takes(3073, 2048, 2048) is None
    assert takes(512, 64, 2048) == (64, 64) and takes(513, 64, 2048) is None and takes(513, 1024, 2048) is not None
    assert takes(448, 2048, 4096) is None and takes(449, 2048, 4096) == (64, 64) and takes(512, 2048, 4160) is None
    assert takes(100, 0, 2048) is None and takes(100, 2048, 0) is None and takes(0, 2048, 2048) is None
    for rows in (65, 300, 1111, 2048):
        for n in (1, 2048, 2568, 6144):
            tile = takes(rows, n, 2048)
            assert tile is None or -(-rows // tile[0]) * -(-n // tile[1]) <= HipBackend.COMPUTE_UNITS


# by tile: its edges in rows and columns, ragged columns (rows of 16 bytes or not), the fewest stages up to more than the ring, an odd number of them
@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(2048, 64), (2568, 128), (1030, 192), (3328, 320), (2047, 448), (2048, 2048), (64, 768), (1, 640)])
def test_products_and_their_rows(n, k):
    torch.manual_seed(59)
    w = (torch.randn(n, k, device=DEV) / math.sqrt(k)).bfloat16()
    x = torch.randn(2048, k, device=DEV).bfloat16()
    exact, scale = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    seen = {}
    for m in (65, 127, 128, 129, 191, 193, 256, 257, 500, 512, 513, 700, 1024, 1025, 1300, 1537, 2048):
        tile = HipBackend.block_tile(m, n, k)
        if tile is None:
            continue
        out = torch.full((m + 1, n), 7.0, device=DEV, dtype=torch.bfloat16)
        ops.linear(x[:m], w, out[:m])
        # a chain of k float32 sums (half a unit in the last place each of at most the absolute products' sum), and one rounding to bfloat16
        bound = k * 2.0 ** -24 * scale[:m] + 2.0 ** -8 * exact[:m].abs() + 1e-30
        assert bool(((out[:m].double() - exact[:m]).abs() <= bound).all()) and bool((out[m] == 7.0).all()), f"{m} rows, {tile}"
        for other, first in seen.items():
            assert torch.equal(out[:min(m, 65)], first[:65]), f"{m} rows, tiles {tile} and {other}"
        seen[tile] = out[:m].clone()
    assert seen


@pytest.mark.gpu
def test_a_row_and_a_column_that_are_not_finite_stay_alone():
    torch.manual_seed(60)
    x, w = torch.randn(200, 192, device=DEV).bfloat16(), torch.randn(1100, 192, device=DEV).bfloat16()
    want, out = (torch.empty(200, 1100, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.linear(x, w, want)
    bad_x, bad_w = x.clone(), w.clone()
    bad_x[199, 191], bad_x[70, 3], bad_w[1099, 5] = float("nan"), float("inf"), float("nan")
    ops.linear(bad_x, bad_w, out)
    rows = [r for r in range(200) if r not in (70, 199)]
    assert torch.equal(out[rows, :1099], want[rows, :1099]) and bool(torch.isnan(out[:, 1099]).all()) and bool(torch.isnan(out[199]).all())


@pytest.mark.gpu
def test_results_at_any_address_and_captured():
    torch.manual_seed(61)
    x, w = torch.randn(333, 2048, device=DEV).bfloat16(), (torch.randn(2048, 2048, device=DEV) / 45).bfloat16()
    want = torch.empty(333, 2048, device=DEV, dtype=torch.bfloat16)
    ops.linear(x, w, want)
    flat = torch.full((333 * 2048 + 16,), 7.0, device=DEV, dtype=torch.bfloat16)
    for offset in (1, 4, 8):
        flat.fill_(7.0)
        ops.linear(x, w, flat[offset:offset + 333 * 2048].view(333, 2048))
        assert torch.equal(flat[offset:offset + 333 * 2048].view(333, 2048), want)
        assert bool((flat[:offset] == 7.0).all()) and bool((flat[offset + 333 * 2048:] == 7.0).all())
    # operands at odd addresses go to the library, as before
    odd = torch.empty(333 * 2048 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(333, 2048).copy_(x)
    out = torch.empty_like(want)
    ops.linear(odd, w, out)
    assert bool(((out.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 1e-3).all())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        ops.linear(x, w, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
