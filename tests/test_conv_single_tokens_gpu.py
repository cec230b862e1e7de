"""The causal convolution of steps of a token a segment and fewer, one launch that keeps the carried rows too: the bits of the launches of longer
segments, fed whole."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("channels,taps", [(6144, 4), (300, 4), (70, 1), (513, 2), (64, 7)])
def test_tokens_one_by_one_give_what_whole_segments_give(dtype, channels, taps):
    g = torch.Generator().manual_seed(channels + taps)
    segments, length, offset = 5, 9, 6
    inp = torch.randn(segments * length, channels + 3, generator=g).to(dtype).to(DEV)
    weight, bias = (torch.randn(channels, taps, generator=g) * 0.5).to(DEV), (torch.randn(channels, generator=g) * 0.2).to(DEV)
    slots = torch.randperm(7, generator=g)[:segments].to(torch.int32).to(DEV)
    start = torch.randn(7, offset + (taps - 1) * channels + 2, generator=g).to(DEV)

    def run(state, rows, lengths):
        """lengths: a segment's tokens of this call, from row `rows[segment]` on."""
        q_len = torch.tensor(lengths, dtype=torch.int32)
        q_start = (torch.cumsum(q_len, 0) - q_len).to(torch.int32)
        x = torch.cat([inp[r:r + k] for r, k in zip(rows, lengths)]) if sum(lengths) else inp[:0]
        out = torch.zeros(x.shape[0], channels, dtype=dtype, device=DEV)
        seg = torch.repeat_interleave(torch.arange(segments, dtype=torch.int32), q_len.long())
        ops.causal_conv(x[:, 2:2 + channels], weight, bias, state, offset, seg.to(DEV), q_start.to(DEV), q_len.to(DEV), slots, out)
        return out.split(lengths)

    whole, parts = start.clone(), start.clone()
    want = run(whole, [s * length for s in range(segments)], [length] * segments)
    at, got = [s * length for s in range(segments)], [[] for _ in range(segments)]
    for lengths in ([1, 1, 1, 1, 1], [2, 0, 1, 1, 1], [0, 3, 0, 1, 0], [5, 0, 0, 0, 0], [0, 0, 0, 0, 1], [1, 1, 1, 1, 1]):     # tokens <= segments
        for s, out in enumerate(run(parts, at, lengths)):
            got[s].append(out)
            at[s] += lengths[s]
    for s in range(segments):
        left = length - (at[s] - s * length)
        assert torch.equal(torch.cat(got[s]), want[s][:length - left]), s
    while any(at[s] < (s + 1) * length for s in range(segments)):
        lengths = [int(at[s] < (s + 1) * length) for s in range(segments)]
        for s, out in enumerate(run(parts, at, lengths)):
            assert torch.equal(out, want[s][at[s] - s * length:at[s] - s * length + lengths[s]])
            at[s] += lengths[s]
    assert torch.equal(parts, whole)
