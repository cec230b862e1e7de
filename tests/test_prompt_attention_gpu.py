"""The attention kernel for long prompts (blocks of 128 rows, two groups of wavefronts that take the blocks of keys in turn)
against the emulation of its contract, with NaN in the slots of pages that are no request's: rows that fill no block, one
block of keys, pieces of odd and even numbers of blocks, masks of every kind, heads by group, softcap, sinks and the weights
of 16 bits.  The rule that sends a step to it is checked on its own (on the CPU)."""
import numpy as np
import pytest
import torch

import test_kernels_gpu as kernels
from wllm_amd.kernels import attention_plan, hip_backend, ops

DEV = "cuda"


def test_the_rule_takes_long_prompts_only():
    def pays(segs, nh, nkv, window=0):
        return attention_plan.prompt_kernel_pays([q for q, _ in segs], [c for _, c in segs], nh // nkv, nkv, window)

    assert pays([(2048, 2048)], 8, 1) and pays([(512, 8192)], 8, 1) and pays([(1500, 1500)], 16, 16) and pays([(2048, 2048)], 8, 1, 4096)
    assert pays([(2048, 2048), (1, 700)], 8, 1)
    assert not pays([(1500, 1500)], 8, 1)                      # 2,270 groups of 32 keys
    assert not pays([(1000, 1000)] * 8, 8, 1)                  # none of them long
    assert not pays([(4096, 4096)], 8, 1, 300)                 # a window keeps the spans short
    assert not pays([(1, 8000)] * 64, 8, 1) and not pays([(2, 9000)], 8, 1)        # decoded tokens and a few rows
    assert not pays([], 8, 1)


@pytest.fixture
def always(monkeypatch):
    monkeypatch.setattr(hip_backend, "prompt_kernel_pays", lambda *a: True)
    return monkeypatch


SHAPES = [
    (8, 1, 16, [(3, 3), (5, 40), (16, 16)], 0),                          # a block of 128 rows that is mostly empty, one block of keys
    (8, 1, 16, [(37, 37), (17, 33), (1, 300), (2, 65)], 0),              # last blocks of keys that are partly stale, decoded tokens beside
    (8, 1, 16, [(300, 300)], 0),
    (4, 4, 32, [(129, 129), (70, 500)], 0),                              # no grouping: a block's rows far apart
    (6, 2, 64, [(100, 260), (43, 43)], 0),                               # a group of 3: tiles that end inside a token
    (5, 1, 128, [(90, 400)], 0),
    (8, 1, 16, [(200, 700)], 100),                                       # a window, first blocks below it
    (16, 1, 256, [(60, 900)], 40),
]


@pytest.mark.gpu
@pytest.mark.parametrize("piece", [0, 1, 2, 3])
@pytest.mark.parametrize("nh,nkv,ps,segs,window", SHAPES)
def test_against_the_emulation(nh, nkv, ps, segs, window, piece, always):
    """`piece`: groups of 32 keys a workgroup gets at most (0: as planned)."""
    if piece:
        always.setattr(attention_plan, "prefill_piece_length", lambda *a, **k: piece)
    plan = kernels._check_matrix_cores(nh, nkv, 256, ps, segs, window)
    assert plan.prefill_rows == 128 and plan.num_prefill > 0


@pytest.mark.gpu
@pytest.mark.parametrize("option", ["softcap", "sinks", "exact_weights", "chunk"])
def test_options(option, always):
    segs = [(100, 350), (33, 33)]
    options = {"softcap": {"softcap": 3.0}, "sinks": {"sinks": torch.linspace(-2.0, 3.0, 8, device=DEV)},
               "exact_weights": {"exact_weights": True}, "chunk": {"chunk": 70}}[option]
    args, kwargs = kernels._attention_case(torch.bfloat16, 8, 2, 256, 16, segs, 0, seed=5)
    ref_args = [a.clone() for a in args]
    # (a plan takes one number for the mask: chunks of positions are negative)
    kw = dict(kernels._with_plan(args, dict(kwargs, window=-options.get("chunk", 0))), window=0)
    assert kw["plan"].prefill_rows == 128
    ops.paged_attention(*args, **kw, **options)
    with ops.use_backend(kernels.EmulatedKernels(precise=True)):
        ops.paged_attention(*ref_args, **kwargs, **options)
    kernels.close(args[7], ref_args[7], torch.bfloat16, option)


@pytest.mark.gpu
def test_a_maximum_that_grows_late(always):
    """Scores that climb block by block: past the slack that a row's reference is allowed, and just below it; the last key
    carries nearly all of the weight."""
    for step in (0.2, 5.0, 40.0):
        args, kwargs = kernels._attention_case(torch.bfloat16, 8, 1, 256, 16, [(64, 640)], 0, seed=9)
        qkv, cache, bt = args[0], args[1], args[2]
        q = torch.nn.functional.normalize(torch.ones(256, device=DEV), dim=0)
        qkv[:, :8 * 256] = (q * 16).repeat(8).bfloat16()
        keys = cache[:, 0].view(cache.shape[0], 1, 16, 256)
        for k in range(640):
            keys[int(bt[0, k // 16]), 0, k % 16] = (q * (step * (k // 32))).bfloat16()
        ref_args = [a.clone() for a in args]
        kw = kernels._with_plan(args, kwargs)
        assert kw["plan"].prefill_rows == 128
        ops.paged_attention(*args, **kw)
        with ops.use_backend(kernels.EmulatedKernels(precise=True)):
            ops.paged_attention(*ref_args, **kwargs)
        kernels.close(args[7], ref_args[7], torch.bfloat16, f"scores that climb by {step}")


@pytest.mark.gpu
def test_no_further_off_than_the_kernel_of_shorter_prompts(monkeypatch):
    """The same step by both kernels against float64: weights relative to a maximum that lags lose nothing."""
    errors = []
    for rule in (lambda *a: True, lambda *a: False):
        monkeypatch.setattr(hip_backend, "prompt_kernel_pays", rule)
        args, kwargs = kernels._attention_case(torch.bfloat16, 8, 1, 256, 16, [(400, 1400)], 0, seed=13)
        ref_args = [a.clone() for a in args]
        ops.paged_attention(*args, **kernels._with_plan(args, kwargs))
        with ops.use_backend(kernels.EmulatedKernels(precise=True)):
            ops.paged_attention(*ref_args, **kwargs)
        want = ref_args[7].double()
        errors.append(float((args[7].double() - want).norm() / want.norm()))
    assert errors[0] <= 1.1 * errors[1], errors      # (a tenth: which way single roundings fall)


@pytest.mark.gpu
def test_one_long_prompt_as_planned():
    plan = kernels._check_matrix_cores(8, 1, 256, 16, [(2048, 2048), (1, 50)], 0)
    assert plan.prefill_rows == 128 and plan.num_prefill > 200 and np.all(plan.prefill_items[:, 5].cpu().numpy() >= -1)
