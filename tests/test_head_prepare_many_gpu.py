"""Heads of many tokens in one launch (a workgroup walks groups of heads, values copied by columns of a page): the bits of the same tokens in
launches of few (a workgroup a group of heads, values a token at a time)."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,nh,nkv,d,rot,ps,own_values,bias_width", [
    (511, 9, 2, 64, 32, 16, True, 0), (512, 9, 2, 64, 32, 16, True, 100), (517, 7, 5, 256, 256, 16, True, 0), (1025, 5, 1, 12, 8, 3, True, 0),
    (2049, 17, 1, 256, 64, 32, False, 0), (2051, 3, 2, 32, 32, 16, True, 5 * 32), (1400, 2, 1, 20, 8, 8, True, 3 * 20 + 7), (2100, 21, 1, 128, 0, 16, True, 0)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_many_tokens_have_the_bits_of_few(dtype, n, nh, nkv, d, rot, ps, own_values, bias_width, interleaved):
    g = torch.Generator().manual_seed(n + d)
    width = (nh + (2 if own_values else 1) * nkv) * d + 8
    rows = torch.randn(n, width, generator=g).to(dtype).to(DEV)
    bias = torch.randn(bias_width, generator=g).to(DEV) if bias_width else None
    positions = torch.randint(0, 5000, (n,), generator=g, dtype=torch.int32).to(DEV)
    pages = n // ps + 3
    slots = torch.randperm(pages * ps, generator=g)[:n].to(torch.int32)
    slots[: n // 2] = torch.arange(n // 2, dtype=torch.int32) + 1 if ps > 3 else slots[: n // 2]      # half of them in order, which may repeat the others':
    slots = torch.where(torch.arange(n) % 50 == 7, torch.full_like(slots, -1), slots).to(DEV)       # some are stored nowhere
    seen, first = set(), torch.full((n,), -1, dtype=torch.int32)                                    # (only a slot's first token keeps it)
    for t, s in enumerate(slots.tolist()):
        if s >= 0 and s not in seen:
            seen.add(s)
            first[t] = s
    slots = first.to(DEV)
    inv_freq = (1.0 / (1e4 ** (torch.arange(0, rot, 2).float() / rot))).to(DEV) if rot else None
    weights = torch.rand(2, d, generator=g).to(DEV) + 0.5
    options = dict(num_heads=nh, num_kv_heads=nkv, head_dim=d, page_size=ps, interleaved=interleaved, values_are_keys=not own_values,
                   norm_eps=1e-6 if nh % 2 else None, head_norm=(weights[0], weights[1], 1e-5) if nkv == 2 else None,
                   q_temperature=(0.1, 1000) if d == 256 else None)
    many, few = rows.clone(), rows.clone()
    cache_many, cache_few = (torch.full((pages, 2, nkv, ps * d), 3.0, dtype=dtype, device=DEV) for _ in range(2))
    ops.head_prepare(many, bias, positions, inv_freq, slots, cache_many, **options)
    for t0 in range(0, n, 100):
        t1 = min(n, t0 + 100)
        ops.head_prepare(few[t0:t1], bias, positions[t0:t1], inv_freq, slots[t0:t1], cache_few, **options)
    assert torch.equal(many, few)
    assert torch.equal(cache_many, cache_few)
