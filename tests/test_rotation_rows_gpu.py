"""Rotation and cache write with a bias or partial sums on both sides of the lines at which another kernel takes them, and at sizes that
are never its: a token has the same bits on either side, and agrees with the emulation of the contract."""
import pytest
import torch

import test_kernels_gpu as kernels
from wllm_amd.kernels import library, ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("with_bias,splits", [(True, 0), (False, 1), (False, 3), (True, 8)])
@pytest.mark.parametrize("nh,nkv,d,rot,line,crossed", [
    (8, 1, 256, 256, 64, True), (32, 8, 128, 128, 64, True), (16, 4, 128, 128, 42, True), (40, 40, 64, 32, 11, True), (60, 10, 40, 40, 13, True),
    (130, 4, 20, 16, 7, True), (8, 1, 256, 256, 128, False), (3, 3, 64, 32, 128, False), (5, 1, 20, 8, 128, False), (2, 2, 40, 40, 128, False)])
def test_both_sides_of_the_line(nh, nkv, d, rot, line, crossed, with_bias, splits, dtype):
    n, ps, width = line + 1, 6, (nh + 2 * nkv) * d
    by_heads = library.load().wllm_rope_by_heads
    assert by_heads(line, nh, nkv, d, rot, ps) == int(crossed) and by_heads(line + 1, nh, nkv, d, rot, ps) == 0
    g = torch.Generator(device="cpu").manual_seed(3)
    rows = torch.randn(n, width, generator=g).to(dtype).to(DEV)
    parts = torch.randn(splits, n, width, generator=g).to(DEV) if splits else None
    bias = (torch.randn(width, generator=g) * 0.3).to(DEV) if with_bias else None
    positions = torch.randint(0, 5000, (n,), generator=g, dtype=torch.int32).to(DEV)
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot))).to(DEV)
    pages = n // ps + 4
    slots = torch.randperm(pages * ps, generator=g)[:n].to(torch.int32).to(DEV)

    def run(count):
        qkv, cache = rows[:count].clone(), torch.zeros(pages, 2, nkv, ps * d, dtype=dtype, device=DEV)
        some = parts[:, :count].contiguous() if splits else None
        ops.rope_and_cache_write(qkv, bias, positions[:count].contiguous(), inv_freq, slots[:count].contiguous(), cache, num_heads=nh,
                                 num_kv_heads=nkv, head_dim=d, page_size=ps, parts=some)
        return qkv, cache

    many, few, one = run(n), run(line), run(1)
    assert torch.equal(many[0][:line], few[0]) and torch.equal(many[0][:1], one[0])
    last = (int(slots[line]) // ps, int(slots[line]) % ps)
    keys, values = (c.view(pages, nkv, -1) for c in (many[1][:, 0], many[1][:, 1]))
    keys.view(pages, nkv, ps, d)[last[0], :, last[1]] = 0           # the token that only the longer call has
    values.view(pages, nkv, d, ps)[last[0], :, :, last[1]] = 0
    assert torch.equal(many[1], few[1])
    with ops.use_backend(kernels.EmulatedKernels(precise=True)):
        want = run(line)
    kernels.close(few[0], want[0], dtype, "rows")
    kernels.close(few[1], want[1], dtype, "pages")
