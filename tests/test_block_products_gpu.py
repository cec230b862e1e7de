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


# the most rows that the rule has, by columns
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile", [(3072, 2048, 192, (192, 128)), (2305, 2047, 448, (192, 128)), (6144, 1024, 128, (192, 128)), (5000, 1100, 64, (192, 128))])
def test_products_of_many_rows(m, n, k, tile):
    assert HipBackend.block_tile(m, n, k) == tile
    torch.manual_seed(66)
    w, x = (torch.randn(n, k, device=DEV) / math.sqrt(k)).bfloat16(), torch.randn(m, k, device=DEV).bfloat16()
    out = torch.full((m + 1, n), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.linear(x, w, out[:m])
    exact = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -8 * exact.abs() + 1e-30        # (as above)
    assert bool(((out[:m].double() - exact).abs() <= bound).all()) and bool((out[m] == 7.0).all())


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


def odd_copy(t):
    return torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)[1:].view(t.shape).copy_(t)


def test_the_rules_of_gated_products_and_stacks():
    gated, stack = HipBackend.block_gated_tile, HipBackend.block_split_tile
    assert gated(64, 16384, 2048) is None and gated(128, 16384, 2048) == (128, 128) and gated(129, 16384, 2048) == (192, 128)
    assert gated(256, 16384, 2048) == (256, 128) and gated(257, 16384, 2048) is None and gated(100, 16385, 2048) is None
    assert gated(65, 4096, 2048) == (64, 64) and gated(512, 4096, 2048) == (128, 128) and gated(1500, 4096, 2048) is None
    assert gated(100, 4096, 4160) is None and gated(100, 4096, 2080) is None and gated(100, 0, 2048) is None
    assert stack(65, 2048, 16384, 8) == (128, 64) and stack(164, 2048, 16384, 8) == (192, 64) and stack(256, 2048, 16384, 8) == (128, 128)
    assert stack(257, 2048, 16384, 16) is None and stack(200, 3072, 24576, 16) is None and stack(100, 2048, 192, 4) is None


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["gelu_tanh", "silu", ops.ClampedSwish(1.5, 1.702, 1.0)], ids=["gelu_tanh", "silu", "clamped"])
@pytest.mark.parametrize("inter,k", [(16384, 2048), (4096, 1984), (250, 64), (777, 192), (33, 320)])
def test_gated_products_have_the_bits_of_other_tiles(act, inter, k):
    """Operands at odd addresses go in tiles of 256 x 256, whose gate up to 256 rows is as exact and whose sums go in the same order."""
    torch.manual_seed(62)
    w = (torch.randn(2 * inter, k, device=DEV) / math.sqrt(k)).bfloat16()
    for m in (65, 100, 128, 129, 191, 192, 193, 256):
        assert HipBackend.block_gated_tile(m, inter, k) is not None
        x = torch.randn(m, k, device=DEV).bfloat16()
        scratch = torch.empty(m, 2 * inter, device=DEV, dtype=torch.bfloat16)
        want, out = (torch.full((m + 1, inter), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        ops.gated_linear(odd_copy(x), w, want[:m], act, scratch)
        ops.gated_linear(x, w, out[:m], act, scratch)
        assert torch.equal(out, want), f"{m} rows"


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["gelu_tanh", "silu"])
@pytest.mark.parametrize("m,inter,k", [(257, 4096, 2048), (385, 1000, 192), (512, 4096, 2048), (600, 250, 64), (1030, 778, 128), (5003, 90, 320),
                                       (16384, 32, 64), (300, 512, 3072), (700, 500, 4096)])
def test_gated_products_of_more_rows(act, m, inter, k):
    assert HipBackend.block_gated_tile(m, inter, k) is not None
    torch.manual_seed(63)
    x, w = torch.randn(m, k, device=DEV).bfloat16(), (torch.randn(2 * inter, k, device=DEV) / math.sqrt(k)).bfloat16()
    wide = torch.full((m, inter + 16), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, wide[:, 8:8 + inter], act, torch.empty(m, 2 * inter, device=DEV, dtype=torch.bfloat16))
    gate, up = (x.double() @ w.double().T).split(inter, 1)
    f = torch.nn.functional
    exact = (f.gelu(gate, approximate="tanh") if act == "gelu_tanh" else f.silu(gate)) * up
    # sums of deviation one, each off by at most k roundings of half a unit of numbers below 8: both factors (slope of the gate below 1.2), the gate's
    # own arithmetic (a few units of 2^-24), and one rounding to bfloat16
    off = k * 2.0 ** -24 * 8
    bound = 1.2 * off * (up.abs() + gate.abs() + off) + 2.0 ** -20 * exact.abs() + 2.0 ** -8 * exact.abs() + 1e-6
    assert bool(((wide[:, 8:8 + inter].double() - exact).abs() <= bound).all())
    assert bool((wide[:, :8] == 7.0).all()) and bool((wide[:, 8 + inter:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("half,k", [(300, 128), (4096, 2048)])
def test_squared_relu_of_two_halves(half, k):
    torch.manual_seed(64)
    w = (torch.randn(2 * half, k, device=DEV) / math.sqrt(k)).bfloat16()
    for m in (65, 192, 256):
        x = torch.randn(m, k, device=DEV).bfloat16()
        want, out = (torch.empty(m, 2 * half, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        ops.activated_linear(odd_copy(x), w, want, "squared_relu")
        ops.activated_linear(x, w, out, "squared_relu")
        assert torch.equal(out, want), f"{m} rows"


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(2048, 16384), (2047, 8192), (1030, 8192), (64, 8192)])
def test_stacks_have_the_bits_of_other_tiles(n, k):
    torch.manual_seed(65)
    w, taken = (torch.randn(n, k, device=DEV) / math.sqrt(k)).bfloat16(), 0
    for m in (65, 128, 129, 192, 193, 256):
        s = ops.linear_splits(m, n, k, torch.bfloat16)
        if s == 1 or HipBackend.wide_splits(n, k, m) > 1 or HipBackend.block_split_tile(m, n, k, s) is None:
            continue
        taken += 1
        x = torch.randn(m, k, device=DEV).bfloat16()
        want, out = (torch.full((s + 1, m, n), 7.0, device=DEV) for _ in range(2))
        ops.linear(odd_copy(x), w, want[:s])
        ops.linear(x, w, out[:s])
        assert torch.equal(out, want), f"{m} rows in {s} pieces"
        flat = torch.full((s * m * n + 5,), 7.0, device=DEV)
        ops.linear(x, w, flat[3:3 + s * m * n].view(s, m, n))
        assert torch.equal(flat[3:3 + s * m * n].view(s, m, n), want[:s]) and bool((flat[:3] == 7.0).all()) and bool((flat[-2:] == 7.0).all())
    assert taken
