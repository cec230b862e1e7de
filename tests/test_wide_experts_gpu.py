"""The experts' products in tiles of two of the plan's tiles of 128 rows: experts whose rows end at, before and behind the
edges of a half and of a whole tile, columns that fill no vector, operands that begin anywhere, inputs with a weight, and
more tiles than one launch takes."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def of_experts(counts, top=1):
    """Assignments of which expert e has counts[e], mixed."""
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])
    return ids[torch.randperm(ids.shape[0], generator=torch.Generator().manual_seed(1))].view(-1, top).to(DEV)


def plan_of(ids, experts):
    plan = torch.full((ops.moe_plan_size(ids.numel(), experts, 128),), -7, dtype=torch.int32, device=DEV)
    ops.moe_plan(ids, plan, experts, 128)
    return plan


def bf16_tensor(*shape, scale=1.0, offset=0):
    size = 1
    for s in shape:
        size *= s
    flat = torch.empty(size + offset, dtype=torch.bfloat16, device=DEV)
    flat.copy_(torch.randn(size + offset, device=DEV) * scale)
    return flat[offset:].view(*shape)


@pytest.mark.parametrize("counts,top,width,ff,offset", [
    ([1, 128, 129, 256, 257, 384, 0, 385], 1, 64, 64, 0),
    ([127, 0, 255, 2], 2, 192, 200, 0),                         # 200 and 100 columns: the last tiles hold few
    ([300, 700], 1, 320, 75, 0),                                # columns that fill no vector
    ([513, 130, 1, 900], 4, 128, 640, 3),
])
@pytest.mark.parametrize("act_name", ["silu", "gelu_tanh"])
def test_both_products(counts, top, width, ff, offset, act_name):
    torch.manual_seed(3)
    experts, ids = len(counts), of_experts(counts, top)
    n = ids.shape[0]
    plan = plan_of(ids, experts)
    x, w_up = bf16_tensor(n, width, offset=offset), bf16_tensor(experts, 2 * ff, width, scale=width ** -0.5, offset=offset)
    in_weights = torch.rand(n, top, device=DEV) + 0.5
    flat = ids.view(-1).long()
    rows = x.double().repeat_interleave(top, dim=0)
    for factor in (None, in_weights):
        act = torch.full((n * top + 1, ff), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_experts_up(x, w_up, plan, act[:n * top], top, act_name, 128, in_weights=factor)
        want = torch.empty(n * top, ff, dtype=torch.float64, device=DEV)
        for e in range(experts):
            of = flat == e
            up = rows[of] @ w_up[e].double().T
            if factor is not None:
                up *= factor.view(-1)[of, None].double()
            gate = torch.nn.functional.silu(up[:, :ff]) if act_name == "silu" else torch.nn.functional.gelu(up[:, :ff], approximate="tanh")
            want[of] = gate * up[:, ff:]
        # one rounding to bfloat16, and float32 sums of at most 640 products whose partial sums stay below 16
        over = (act[:n * top].double() - want).abs() - 2 ** -8 * want.abs() - 640 / 32 * 16 * 2 ** -22
        assert float(over.max()) <= 0 and bool((act[n * top] == 7.0).all())
    if ff % 64:
        return
    # the second product reads what the first wrote
    w_down = bf16_tensor(experts, width, ff, scale=ff ** -0.5, offset=offset)
    weights = torch.rand(n, top, device=DEV)
    h = act[:n * top].contiguous()
    for weighted in (True, False):
        out = torch.full((top, n, width), float("nan"), device=DEV)
        ops.moe_experts_down(h, w_down, plan, weights, out, 128, weighted=weighted)
        got = out.transpose(0, 1).reshape(n * top, width).double()
        for e in range(experts):
            of = flat == e
            want = h[of].double() @ w_down[e].double().T
            if weighted:
                want *= weights.view(-1)[of, None].double()
            if want.numel():
                # (a partial sum rounds by 2^-24 of its size, at most that of the largest result and a half more, every 32 keys)
                assert float((got[of] - want).abs().max()) <= ff / 32 * 1.5 * (1 + float(want.abs().max())) * 2 ** -23


def test_more_tiles_than_a_launch_takes():
    """16,000 tiles of the plan a launch: the rows behind them are made by a second one."""
    torch.manual_seed(4)
    n, width, ff = 2_060_000, 64, 64
    ids = (torch.arange(n, device=DEV, dtype=torch.int32) % 3 == 0).int().view(n, 1)
    plan = plan_of(ids, 2)
    assert int(plan[0]) > 16000
    x, w_up, w_down = bf16_tensor(n, width), bf16_tensor(2, 2 * ff, width, scale=0.125), bf16_tensor(2, width, ff, scale=0.125)
    act = torch.full((n, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_experts_up(x, w_up, plan, act, 1, "silu", 128)
    out = torch.full((1, n, width), float("nan"), device=DEV)
    ops.moe_experts_down(act, w_down, plan, torch.ones(n, 1, device=DEV), out, 128)
    for e in range(2):
        of = ids.view(-1) == e
        up = x[of].float() @ w_up[e].float().T
        want = torch.nn.functional.silu(up[:, :ff]) * up[:, ff:]
        assert float(((act[of].float() - want).abs() - 2 ** -8 * want.abs()).max()) <= 1e-4
        assert float((out[0, of] - act[of].float() @ w_down[e].float().T).abs().max()) <= 1e-4      # (float32 sums of 64 numbers in two orders)
