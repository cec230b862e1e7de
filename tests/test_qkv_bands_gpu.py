"""The joint projection, rotation and cache write where a pair of bands is two workgroups (up to 128 pairs) and where it is one: the
smallest launch, both sides of the line, tokens of one and of two tiles, against the emulation of the contract."""
import math

import pytest
import torch

import test_kernels_gpu as kernels
from wllm_amd.kernels import ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("m", [1, 16, 17, 32])
@pytest.mark.parametrize("k,nh,nkv,d", [(96, 1, 1, 32),         # 3 pairs
                                        (288, 30, 1, 128),      # 128: the last launch in halves
                                        (288, 41, 1, 96),       # 129
                                        (64, 66, 1, 64)])       # 136
def test_halves_and_whole_bands(k, nh, nkv, d, m, tiled):
    dtype, ps, width = torch.bfloat16, 8, (nh + 2 * nkv) * d
    assert ops.qkv_rope_takes(m, dtype, k, d, d)

    def make():
        g = torch.Generator(device="cpu").manual_seed(5)
        x = torch.randn(m, k, generator=g).to(dtype).to(DEV)
        w = (torch.randn(width, k, generator=g) / math.sqrt(k)).to(dtype).to(DEV)
        bias = (torch.randn(width, generator=g) * 0.3).to(DEV)
        positions = torch.randint(0, 3000, (m,), generator=g, dtype=torch.int32).to(DEV)
        inv_freq = (1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).to(DEV)
        pages = m + 3
        slots = torch.randperm(pages * ps, generator=g)[:m].to(torch.int32).to(DEV)
        cache = torch.zeros(pages, 2, nkv, ps * d, dtype=dtype, device=DEV)
        qkv = torch.zeros(m, width, dtype=dtype, device=DEV)
        return [x, w, qkv, bias, positions, inv_freq, slots, cache], dict(
            num_heads=nh, num_kv_heads=nkv, head_dim=d, page_size=ps, tiles=ops.tile_weight(w) if tiled else None)

    got, want = kernels.both("qkv_rope", make, dtype)
    kernels.close(got[2], want[2], dtype, "rotated queries, keys and values")
    kernels.close(got[7], want[7], dtype, "pages")
    assert (got[7] != 0).sum() == (want[7] != 0).sum(), "only the tokens' slots are written"


# More than eight steps of 32 keys a wavefront, so that its registers are filled again: 2,080 keys are nine steps for some, 4,096 sixteen
@pytest.mark.gpu
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("k", [2080, 4096])
def test_halves_have_the_bits_of_whole_bands(k, tiled):
    """The first 20 heads of 34 by themselves are 88 pairs of bands, in halves; all of them 136, whole."""
    dtype, ps, d = torch.bfloat16, 8, 128
    torch.manual_seed(6)
    w = (torch.randn(36 * d, k, device=DEV) / math.sqrt(k)).to(dtype)
    x, bias = torch.randn(32, k, device=DEV).to(dtype), torch.randn(36 * d, device=DEV) * 0.3
    inv_freq = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float32, device=DEV) / d))
    positions = torch.randint(0, 3000, (32,), dtype=torch.int32, device=DEV)

    def run(m, heads):
        rows = (heads + 2) * d
        qkv, cache = torch.zeros(m, rows, dtype=dtype, device=DEV), torch.zeros(m, 2, 1, ps * d, dtype=dtype, device=DEV)
        part = w[:rows].contiguous()
        ops.qkv_rope(x[:m], part, qkv, bias[:rows].contiguous(), positions[:m].contiguous(), inv_freq,
                     torch.arange(m, dtype=torch.int32, device=DEV) * ps, cache, num_heads=heads, num_kv_heads=1, head_dim=d, page_size=ps,
                     tiles=ops.tile_weight(part) if tiled else None)
        return qkv

    for m in (1, 16, 17, 32):
        assert torch.equal(run(m, 20)[:, :20 * d], run(m, 34)[:, :20 * d]), f"{m} tokens"
