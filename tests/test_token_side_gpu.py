"""A layer's token input in one launch: the same bits as the three operations that make it."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("rows,hidden,dim", [(1, 2048, 64), (8, 2048, 64), (16, 1536, 64), (11, 640, 64), (5, 2048, 32), (15, 1920, 32),
                                             (3, 128, 64), (9, 384, 32)])
def test_one_launch_gives_what_three_give(rows, hidden, dim, tiled):
    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g).bfloat16().to(DEV)
    w_gate = (torch.randn(dim, hidden, generator=g) * hidden ** -0.5).bfloat16().to(DEV)
    w_proj = (torch.randn(hidden, dim, generator=g) * dim ** -0.5).bfloat16().to(DEV)
    table = torch.randn(70, 3 * dim + 4, generator=g).bfloat16().to(DEV)
    ids = torch.randint(0, 70, (rows,), generator=g, dtype=torch.int32).to(DEV)
    ids[0] = 69
    t_gate, t_proj = (ops.tile_weight(w_gate), ops.tile_weight(w_proj)) if tiled else (None, None)
    col0 = 2 * dim + 4 if rows % 2 else dim
    gate, bent = torch.empty(rows, dim, dtype=x.dtype, device=DEV), torch.empty(rows, dim, dtype=x.dtype, device=DEV)
    for name in ops.ACTIVATIONS:
        assert ops.token_side_takes(x, w_gate, w_proj, table)
        got = torch.full((rows + 1, hidden), 7.0, dtype=x.dtype, device=DEV)
        ops.token_side(x, w_gate, ids, table, col0, w_proj, got[:rows], name, t_gate, t_proj)
        want = torch.empty(rows, hidden, dtype=x.dtype, device=DEV)
        ops.linear(x, w_gate, gate, t_gate)
        ops.gated_lookup(gate, ids, table, col0, bent, name)
        ops.linear(bent, w_proj, want, t_proj)
        assert (got[rows] == 7).all()
        if hidden >= 512:       # the few-row product has two pieces of the K axis, too
            assert torch.equal(got[:rows], want), (name, (got[:rows].float() - want.float()).abs().max())
        # against 64 bits: the bent gate is rounded twice (2^-9 each, its own rounding to the gate's slope of at most 1.13), the result once; sums in float32
        act = torch.nn.functional.gelu if name == "gelu_tanh" else torch.nn.functional.silu
        z = x.double() @ w_gate.double().T
        entry = table.double()[ids.long(), col0:col0 + dim]
        inner = (act(z, approximate="tanh") if name == "gelu_tanh" else act(z)) * entry
        exact = inner @ w_proj.double().T
        slack = (1.13 * z.abs() * entry.abs() + inner.abs()) * 2.0 ** -9 * 1.05
        bound = slack @ w_proj.double().abs().T + 2.0 ** -9 * 1.05 * exact.abs() + 1e-4
        assert ((got[:rows].double() - exact).abs() <= bound).all()


def test_what_it_does_not_take():
    x = torch.zeros(17, 2048, dtype=torch.bfloat16, device=DEV)
    w, p, table = x.new_zeros(64, 2048), x.new_zeros(2048, 64), x.new_zeros(5, 64)
    assert not ops.token_side_takes(x, w, p, table)                                          # rows
    assert ops.token_side_takes(x[:16], w, p, table)
    assert not ops.token_side_takes(x[:1], w[:48], p[:, :48].contiguous(), table)            # the band
    assert not ops.token_side_takes(x[:1].float(), w.float(), p.float(), table.float())      # the type
    assert not ops.token_side_takes(x.new_zeros(1, 2176), x.new_zeros(64, 2176), x.new_zeros(2176, 64), table)
    off = x.new_zeros(2049)[1:].view(1, 2048)
    assert not ops.token_side_takes(off, w, p, table)                                        # the address
