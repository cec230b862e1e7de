"""Prompt portions and decoded tokens in one launch: lists of items shorter than a run of 64 workgroups, of whole runs, and with
what is left of the one or the other, by head size and option.  The results have the bits of the two launches, and are held against
the emulation of the contract."""
import pytest
import torch

import test_kernels_gpu as kernels
from wllm_amd.kernels import hip_backend, ops

DEV = "cuda"


def test_the_rule():
    takes = hip_backend.HipBackend.portions_beside
    assert takes(64, 8) and takes(128, 16) and takes(256, 256)
    assert not takes(96, 16) and not takes(256, 4) and not takes(128, 24)


@pytest.mark.gpu
@pytest.mark.parametrize("option", ["plain", "softcap", "sinks", "exact_weights", "window", "chunk"])
@pytest.mark.parametrize("nh,nkv,d,ps,segs", [
    (8, 1, 256, 16, [(17, 17), (1, 1)]),                                            # an item or two of either kind
    (8, 1, 256, 16, [(300, 333), (70, 500)] + [(1, 40 + i) for i in range(70)]),    # less than a run of portions, a run and some tokens
    (4, 4, 64, 8, [(400, 410)] + [(1, 200)] * 3),                                   # the other way round
    (8, 4, 128, 32, [(130, 700), (1, 300), (33, 65)] + [(1, 500 + i) for i in range(40)]),      # runs of both, some of each left
    (64, 64, 64, 16, [(64, 64), (1, 100)]),                                         # 64 items of either kind
    (64, 64, 64, 16, [(270, 270)] + [(1, 100 + i) for i in range(5)]),              # 320 of either, heads of 64: a run of 256 each, and some left
])
def test_together_as_apart(nh, nkv, d, ps, segs, option, monkeypatch):
    window = {"window": 100, "chunk": -70}.get(option, 0)
    options = {"softcap": {"softcap": 3.0}, "sinks": {"sinks": torch.linspace(-2.0, 3.0, nh, device=DEV)},
               "exact_weights": {"exact_weights": True}, "chunk": {"chunk": 70}}.get(option, {})
    args, kwargs = kernels._attention_case(torch.bfloat16, nh, nkv, d, ps, segs, max(window, 0), seed=11)
    ref_args = [a.clone() for a in args]
    kw = dict(kernels._with_plan(args, dict(kwargs, window=window)), window=max(window, 0), **options)
    assert kw["plan"].num_prefill and kw["plan"].num_items and kw["plan"].prefill_rows == 64
    ops.paged_attention(*args, **kw)
    together = args[7].clone()
    args[7].fill_(9.0)
    monkeypatch.setattr(hip_backend.HipBackend, "portions_beside", staticmethod(lambda *a: False))
    ops.paged_attention(*args, **kw)
    assert torch.equal(together, args[7])
    with ops.use_backend(kernels.EmulatedKernels(precise=True)):
        ops.paged_attention(*ref_args, **kwargs, **options)
    kernels.close(together, ref_args[7], torch.bfloat16, option)
