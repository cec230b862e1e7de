"""Decoded tokens over pages of 16 and of powers of two from 32 on, whose addresses are worked out a wavefront, against pages of 8 and 24, whose are a lane's."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
SEGS = [(1, 1), (1, 31), (1, 33), (1, 128), (1, 129), (2, 300), (1, 1000)]


def attend(ps, nh, nkv, d, segs, window, rows, keys, values, **options):
    g = torch.Generator().manual_seed(7)
    counts = [-(-c // ps) for _, c in segs]
    order = (torch.randperm(sum(counts), generator=g) + 1).tolist()
    table = torch.zeros(len(segs), max(counts), dtype=torch.int32)
    cache = torch.full((sum(counts) + 1, 2, nkv, ps * d), float("nan"), dtype=torch.bfloat16)     # stale slots and page 0: NaN
    kview, vview = cache[:, 0].unflatten(2, (ps, d)), cache[:, 1].unflatten(2, (d, ps))
    for s, (_, c) in enumerate(segs):
        for p in range(counts[s]):
            table[s, p] = at = order.pop()
            part = slice(p * ps, min(c, (p + 1) * ps))
            kview[at, :, :part.stop - part.start] = keys[s][part].transpose(0, 1)
            vview[at, :, :, :part.stop - part.start] = values[s][part].permute(1, 2, 0)
    q_len, ctx = (torch.tensor([x[i] for x in segs], dtype=torch.int32) for i in (0, 1))
    n = int(q_len.sum())
    tok_seg = torch.repeat_interleave(torch.arange(len(segs), dtype=torch.int32), q_len.long())
    out = torch.full((n, nh * d), 7.0, dtype=torch.bfloat16, device=DEV)
    plan = ops.plan_paged_attention(q_len.numpy(), ctx.numpy(), num_heads=nh, num_kv_heads=nkv, head_dim=d, page_size=ps,
                                    window=window if "chunk" not in options else -options["chunk"], dtype=torch.bfloat16, device=DEV)
    assert plan is not None and plan.num_prefill == 0
    ops.paged_attention(rows, cache.to(DEV), table.to(DEV), tok_seg.to(DEV), (torch.cumsum(q_len, 0, dtype=torch.int32) - q_len).to(DEV),
                        q_len.to(DEV), ctx.to(DEV), out, num_heads=nh, num_kv_heads=nkv, head_dim=d, page_size=ps, scale=d ** -0.5,
                        window=window, max_q_len=int(q_len.max()), max_ctx_len=int(ctx.max()), plan=plan, **options)
    return out


@pytest.mark.parametrize("nh,nkv,d", [(8, 1, 256), (6, 2, 96), (16, 16, 32), (40, 2, 128), (5, 5, 64)])
@pytest.mark.parametrize("window,options", [(0, {}), (50, {}), (0, {"chunk": 70}), (0, {"softcap": 20.0}), (0, {"exact_weights": True})])
def test_pages_of_any_size_have_the_same_bits(nh, nkv, d, window, options):
    torch.manual_seed(66)
    segs = [(q if q * (nh // nkv) <= 16 else 1, c) for q, c in SEGS]          # (short segments all)
    n = sum(q for q, _ in segs)
    rows = torch.randn(n, (nh + 2 * nkv) * d, device=DEV).bfloat16()
    keys = [torch.randn(c, nkv, d).bfloat16() for _, c in SEGS]
    values = [torch.randn(c, nkv, d).bfloat16() for _, c in SEGS]
    want = attend(8, nh, nkv, d, segs, window, rows, keys, values, **options)
    assert bool(torch.isfinite(want.float()).all())
    for ps in (16, 24, 32, 64, 256):
        got = attend(ps, nh, nkv, d, segs, window, rows, keys, values, **options)
        assert torch.equal(got, want), f"pages of {ps}"
    # the last segment by itself against 64 bits
    q, k, v = rows[-1, :nh * d].double().view(nh, d), keys[-1].to(DEV).double(), values[-1].to(DEV).double()
    c = SEGS[-1][1]
    low = max(0, c - window) if window else (c - 1) // 70 * 70 if "chunk" in options else 0
    for h in range(nh):
        s = k[low:, h // (nh // nkv)] @ q[h] * d ** -0.5
        if "softcap" in options:
            s = 20.0 * torch.tanh(s / 20.0)
        exact = torch.softmax(s, 0) @ v[low:, h // (nh // nkv)]
        # weights and the result rounded to bfloat16, and a cap by the hardware's exponential
        assert float((want[-1, h * d:(h + 1) * d].double() - exact).abs().max()) <= 2.0 ** -8 * 2 * float(v[low:].abs().max())
