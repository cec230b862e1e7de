"""Kernels of a row each (the gated norms of groups and of heads) that take many rows another way: the bits of the same rows in
launches of few.  Against 64 bits: a bfloat16 result is rounded by 2^-9 of itself, what was computed in float32 takes some dozen roundings of 2^-24 and an
exponential."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,groups,size", [(256, 8, 512), (700, 3, 200), (2048, 1, 256), (517, 5, 513), (300, 7, 1024), (1100, 2, 1), (690, 3, 1025)])
def test_gated_norm_of_groups(dtype, n, groups, size):
    g = torch.Generator().manual_seed(n)
    width = groups * size
    y = (torch.randn(n, width, generator=g) * 2).to(DEV)
    row = torch.randn(n, width + 6, generator=g).to(dtype).to(DEV)
    weight = (1 + 0.2 * torch.randn(width, generator=g)).to(DEV)
    many, few = (torch.zeros(n, width, dtype=dtype, device=DEV) for _ in range(2))
    ops.gated_group_norm(y, row[:, 5:5 + width], weight, many, groups, 1e-5)
    step = max(1, 2047 // groups)
    for t in range(0, n, step):
        ops.gated_group_norm(y[t:t + step], row[t:t + step, 5:5 + width], weight, few[t:t + step], groups, 1e-5)
    assert torch.equal(many, few)
    z = row[:, 5:5 + width].double()
    v = (y.double() * z * torch.sigmoid(z)).view(n, groups, size)
    exact = (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-5)).reshape(n, width) * weight.double()
    bound = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18) * exact.abs() + 1e-7
    assert ((many.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,heads,dim", [(256, 16, 128), (1400, 3, 129), (4100, 1, 64), (820, 5, 256), (700, 6, 257), (1030, 4, 7)])
@pytest.mark.parametrize("activation", ["sigmoid", "silu", "none"])
def test_gated_norm_of_heads(dtype, n, heads, dim, activation):
    g = torch.Generator().manual_seed(n + dim)
    y = (torch.randn(n, heads * dim, generator=g) * 3).to(DEV)
    row = torch.randn(n, heads * dim + 3, generator=g).to(dtype).to(DEV)
    weight = (1 + 0.2 * torch.randn(heads * dim, generator=g)).to(DEV)
    nq, floor = (torch.randn(n, heads, generator=g).to(DEV), torch.rand(n, heads, generator=g).to(DEV)) if heads % 2 else (None, None)
    many, few = (torch.zeros(n, heads * dim, dtype=dtype, device=DEV) for _ in range(2))
    step = max(1, 4095 // heads)
    for t0, t1, out in [(0, n, many)] + [(t, min(n, t + step), few) for t in range(0, n, step)]:
        ops.head_norm_gate(y[t0:t1], None if activation == "none" else row[t0:t1, 3:], weight, out[t0:t1], heads=heads, eps=1e-6, activation=activation,
                           scale=0.5, **({} if nq is None else dict(nq=nq[t0:t1], floor=floor[t0:t1], den_eps=1e-6)))
    assert torch.equal(many, few)
    v = y.double().view(n, heads, dim)
    if nq is not None:
        v = v / (torch.maximum(nq.abs(), floor) + 1e-6).double()[..., None]
    exact = (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6)).reshape(n, -1) * weight.double() * 0.5
    z = row[:, 3:].double()
    exact = exact * (1 if activation == "none" else torch.sigmoid(z) if activation == "sigmoid" else z * torch.sigmoid(z))
    bound = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18) * exact.abs() + 1e-7
    assert ((many.double() - exact).abs() <= bound).all()
