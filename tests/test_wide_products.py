"""The product in tiles of 256 x 256: which sizes go to it (on the CPU), and its results at the edges of its tiles, stages and
pieces of the K axis, for operands that begin anywhere, without room for partial sums, and captured (on the GPU)."""
import math

import pytest
import torch

from kernel_emulation import EmulatedKernels
from wllm_amd.kernels import ops
from wllm_amd.kernels.hip_backend import HipBackend
from wllm_amd.parts.common import project

DEV = "cuda"


def test_rules_keep_to_what_the_kernel_takes():
    """A piece has at least 512 keys and a launch one round of workgroups; sizes that the kernel refuses go elsewhere."""
    taken = 0
    for rows in (65, 128, 129, 255, 256, 257, 511, 512, 513, 1500, 4096, 4097, 20000):
        for n in (1, 48, 200, 2047, 2048, 3072, 8192, 10304, 16384):
            for k in (64, 2048, 8192, 8256, 8200, 16384, 24576):
                s = HipBackend.wide_splits(n, k, rows)
                tiles = -(-rows // 256) * -(-n // 256)
                assert s == 1 or (rows > 128 and k >= 8192 and k % 64 == 0 and k // s >= 512 and tiles * s <= 256)
                for takes in (HipBackend.wide_takes(rows, n, k), HipBackend.wide_gated_takes(rows, n, k)):
                    assert not takes or (rows > 128 and k % 64 == 0)
                taken += s > 1
    assert taken > 50
    assert HipBackend.wide_splits(2048, 16384, 2048) == 4 and HipBackend.wide_splits(2048, 16384, 257) == 16
    for rows, n, k in ((2 ** 20, 10304, 2048), (1500, 2 ** 21 + 8, 1024)):      # 4 GiB of operands
        assert not HipBackend.wide_takes(rows, n, k) and not HipBackend.wide_gated_takes(rows, n, k)


def test_a_product_without_room_for_its_partial_sums_is_made_whole():
    class Ctx:
        def buffer(self, name, shape, dtype):
            if len(shape) == 3:
                raise torch.OutOfMemoryError("no room")
            return torch.empty(shape, dtype=dtype)

    x, w = torch.randn(3, 4096).bfloat16(), torch.randn(32, 4096).bfloat16() / 64
    kernels = EmulatedKernels()
    kernels.splits = 2
    with ops.use_backend(kernels):
        assert ops.linear_splits(3, 32, 4096, torch.bfloat16) > 1
        out = project(Ctx(), "product", x, w)
    assert out.shape == (3, 32) and torch.allclose(out.float(), x.float() @ w.float().T, rtol=2 ** -7, atol=1e-4)


def operands(m, n, k, offset=0):
    def matrix(rows, scale):
        flat = torch.empty(rows * k + offset, device=DEV, dtype=torch.bfloat16)
        flat.copy_(torch.randn(rows * k + offset, device=DEV) * scale)
        return flat[offset:].view(rows, k)
    torch.manual_seed(31)
    return matrix(m, 1.0), matrix(n, 1.0 / math.sqrt(k))


def sums(x, w):
    """The product in 64 bits, and how far float32 sums over K may be off: every step of 32 keys rounds a partial sum (of
    numbers whose sum has deviation one: below 8) by 2^-24, twice over for the order inside a step."""
    return x.double() @ w.double().T, x.shape[1] / 32 * 8 * 2 ** -23


def check_bf16(got, want, slack):
    assert bool(torch.isfinite(got).all())
    over = (got.double() - want).abs() - 2 ** -8 * want.abs() - slack
    assert float(over.max()) <= 0, f"off by {float(over.max())} more than rounding explains"


def activated(gate, up, act):
    if isinstance(act, ops.ClampedSwish):
        g, u = gate.clamp(max=act.limit), up.clamp(-act.limit, act.limit)
        return g * torch.sigmoid(act.slope * g) * (u + act.shift)
    g = torch.nn.functional.gelu(gate, approximate="tanh") if act == "gelu_tanh" else torch.nn.functional.silu(gate)
    return g * up


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["gelu_tanh", "silu", ops.ClampedSwish(1.5, 1.702, 1.0)], ids=["gelu_tanh", "silu", "clamped"])
@pytest.mark.parametrize("m,inter,k,offset", [
    (129, 16384, 64, 0), (256, 16259, 128, 0),          # one row tile, one and two stages, columns that fill no vector
    (400, 16004, 192, 0), (512, 16384, 2048, 0),        # two row tiles, a multiple of four columns
    (1500, 16390, 64, 0), (2100, 12000, 320, 3),        # several tiles a workgroup, two bands of row tiles; operands at odd places
])
def test_gated_product(act, m, inter, k, offset):
    assert HipBackend.wide_gated_takes(m, inter, k)
    x, w = operands(m, 2 * inter, k, offset)
    wide = torch.full((m + 1, inter), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, wide[:m], act, torch.empty(m, 2 * inter, device=DEV, dtype=torch.bfloat16))
    both, slack = sums(x, w)
    gate, up = both[:, :inter], both[:, inter:]
    # (a gate's derivative is at most 1.2, or the slope's times that; both streams carry the sums' error, and the
    # hardware's exponential and reciprocal a few ulp)
    want = activated(gate, up, act)
    check_bf16(wide[:m], want, 2 * slack * (1 + gate.abs() + up.abs()) + 2 ** -20 * want.abs())
    assert bool((wide[m] == 7.0).all())


@pytest.mark.gpu
def test_gated_product_into_a_band_of_columns():
    m, inter, k = 1500, 16384, 64
    x, w = operands(m, 2 * inter, k)
    scratch = torch.empty(m, 2 * inter, device=DEV, dtype=torch.bfloat16)
    want = torch.empty(m, inter, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, want, "silu", scratch)
    wider = torch.full((m, inter + 24), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.gated_linear(x, w, wider[:, 8:8 + inter], "silu", scratch)
    assert torch.equal(wider[:, 8:8 + inter], want)
    assert bool((wider[:, :8] == 7.0).all()) and bool((wider[:, 8 + inter:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,half,k", [(200, 16384, 64), (600, 10876, 128), (1500, 16388, 64)])
def test_squared_relu_of_two_halves(m, half, k):
    assert HipBackend.wide_gated_takes(m, half, k)
    x, w = operands(m, 2 * half, k)
    out = torch.full((m + 1, 2 * half), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.activated_linear(x, w, out[:m], "squared_relu")
    both, slack = sums(x, w)
    check_bf16(out[:m], both.clamp(min=0) ** 2, 2 * slack * (1 + both.abs()))
    assert bool((out[m] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,offset", [
    (129, 3072, 24576, 0), (257, 2048, 8192, 0), (512, 2047, 8192, 0),      # 16 pieces of 24 and of 8 stages; odd columns
    (1500, 2050, 8256, 0), (2049, 2052, 8192, 5), (4096, 2048, 8192, 0),    # pieces of unequal length, nine row tiles
])
def test_product_in_pieces_of_the_k_axis(m, n, k, offset):
    s = ops.linear_splits(m, n, k, torch.bfloat16)
    assert s > 1 and s == HipBackend.wide_splits(n, k, m)
    x, w = operands(m, n, k, offset)
    stack = torch.full((s * m * n + 4,), 7.0, device=DEV)
    ops.linear(x, w, stack[:s * m * n].view(s, m, n))
    parts, total = stack[:s * m * n].view(s, m, n), 0
    for part in parts:
        total = total + part
    want, slack = sums(x, w)
    assert float((total.double() - want).abs().max()) <= slack and bool((stack[s * m * n:] == 7.0).all())
    for dtype in (torch.float32, torch.bfloat16):
        whole = torch.full((m + 1, n), 7.0, device=DEV, dtype=dtype)
        ops.linear(x, w, whole[:m])
        assert torch.equal(whole[:m], total.to(dtype)) and bool((whole[m] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,offset", [(1024, 10304, 64, 0), (2040, 5130, 192, 0), (1000, 12289, 128, 1), (3000, 10300, 2048, 0)])
def test_product_of_columns_that_fill_no_tiles(m, n, k, offset):
    assert HipBackend.wide_takes(m, n, k)
    x, w = operands(m, n, k, offset)
    out = torch.full((m + 1, n), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.linear(x, w, out[:m])
    check_bf16(out[:m], *sums(x, w))
    assert bool((out[m] == 7.0).all())


@pytest.mark.gpu
def test_product_without_room_for_partial_sums(monkeypatch):
    m, n, k = 300, 2048, 8192
    x, w = operands(m, n, k)
    out, refused = torch.empty(m, n, device=DEV, dtype=torch.bfloat16), []
    assert ops.linear_splits(m, n, k, torch.bfloat16) > 1

    def full(*args, **kwargs):
        refused.append(args)
        raise torch.OutOfMemoryError("no room")
    monkeypatch.setattr(torch, "empty", full)
    ops.linear(x, w, out)
    monkeypatch.undo()
    assert len(refused) == 1
    check_bf16(out, *sums(x, w))


@pytest.mark.gpu
def test_captured_products_replay():
    m, inter, k = 160, 16384, 2048
    x, w = operands(m, 2 * inter, k)
    down = (torch.randn(3072, inter, device=DEV) / 128).bfloat16()
    act, scratch = (torch.empty(m, c, device=DEV, dtype=torch.bfloat16) for c in (inter, 2 * inter))
    s = ops.linear_splits(m, 3072, inter, torch.bfloat16)
    stack = torch.empty(s, m, 3072, device=DEV)

    def step():
        ops.gated_linear(x, w, act, "gelu_tanh", scratch)
        ops.linear(act, down, stack)
    assert HipBackend.wide_gated_takes(m, inter, k) and s == HipBackend.wide_splits(3072, inter, m) > 1
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for seed in range(3):
        x.copy_(torch.randn(m, k, device=DEV, generator=torch.Generator(DEV).manual_seed(seed)))
        step()
        want = act.clone(), stack.clone()
        act.zero_()
        stack.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(act, want[0]) and torch.equal(stack, want[1])
