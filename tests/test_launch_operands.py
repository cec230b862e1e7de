"""What a launch is handed, without a GPU: every address it gets belongs to a tensor that is still held when it is made."""
import ctypes
import weakref

import pytest
import torch

from wllm_amd.kernels import ops


@pytest.fixture
def chunks_from_64(monkeypatch):
    monkeypatch.setattr(ops, "ssm_chunk_from", lambda heads, groups: 64)
    monkeypatch.setattr(ops, "memory_chunk_from", lambda heads, value_dim, row_decays: 64)


class Launches:
    """A backend whose launches end in a function that only looks at the arguments of the entry point."""

    def __init__(self, look):
        self.look = look

    def run_registered(self, op, args, kwargs):
        op.launch(lambda *arguments: self.look(op, arguments), 0, *args, **kwargs)


def _ints(*values):
    return torch.tensor(values, dtype=torch.int32)


def _scan(kind, n, **extra):
    heads, d = 2, 16
    state, seg = torch.zeros(3, heads * d * d + heads * d), (_ints(0), _ints(n), _ints(1))
    if kind == "space":
        xbc, vectors = torch.zeros(n, heads * d + 2 * d, dtype=torch.bfloat16), [torch.zeros(heads) for _ in range(3)]
        ops.ssm_scan(xbc, torch.zeros(n, heads, dtype=torch.bfloat16), *vectors, state, *seg, torch.zeros(n, heads * d), heads=heads,
                     groups=1, state_size=d, head_dim=d, **extra)
    else:
        ops.memory_scan(torch.zeros(2, n, heads * d), torch.zeros(n, heads * d, dtype=torch.bfloat16), None, torch.zeros(heads), state,
                        *seg, torch.zeros(n, heads * d), heads=heads, head_dim=d, value_dim=d, **extra)


@pytest.mark.parametrize("kind", ["space", "memory"])
def test_scratch_that_a_scan_makes_is_held_until_its_launch(kind, monkeypatch, chunks_from_64):
    """The scratch of a recurrence walked in chunks (the fourth argument from the end) is a tensor that something refers to
    when the launch is made: else its memory is the allocator's again before a kernel has run."""
    made, empty, seen = [], torch.empty, []

    def recorded(*args, **kwargs):
        t = empty(*args, **kwargs)
        made.append((t.data_ptr(), weakref.ref(t)))
        return t

    def look(op, arguments):
        address = getattr(arguments[-4], "value", arguments[-4])
        seen.append(address)
        assert any(at == address and ref() is not None for at, ref in made), "the scratch was given back before the launch"
        return 0
    monkeypatch.setattr(torch, "empty", recorded)
    with ops.use_backend(Launches(look)):
        _scan(kind, 80)
    assert seen and seen[0]


@pytest.mark.parametrize("kind", ["space", "memory"])
def test_a_scan_uses_the_callers_scratch_and_refuses_less_than_it_needs(kind, chunks_from_64):
    size = ops.ssm_chunk_size(80, 1, 2, 1, 16, torch.bfloat16) if kind == "space" else ops.memory_chunk_size(80, 1, 2, 16, 16, torch.bfloat16, False)
    mine = torch.zeros(size)
    with ops.use_backend(Launches(lambda op, arguments: seen.append(arguments[-4]) or 0)):
        seen = []
        _scan(kind, 80, chunks=mine)
        assert seen == [mine.data_ptr()]
        for wrong in (mine[:-1], mine.double(), torch.zeros(size, 2)[:, 0]):
            with pytest.raises(ops.KernelShapeError):
                _scan(kind, 80, chunks=wrong)
        assert len(seen) == 1
    assert ops.ssm_chunk_size(63, 1, 2, 1, 16, torch.bfloat16) == 0 == ops.memory_chunk_size(96, 96, 2, 16, 16, torch.bfloat16, False)
    assert ops.ssm_chunk_size(80, 1, 2, 1, 16, torch.float32) == 0 == ops.memory_chunk_size(80, 1, 2, 16, 16, torch.float32, False)


@pytest.mark.parametrize("kind", ["space", "memory"])
def test_a_scan_without_room_for_its_scratch_is_walked_token_by_token(kind, monkeypatch, chunks_from_64):
    seen, empty = [], torch.empty

    def full(size, *args, **kwargs):
        if isinstance(size, int):                  # (the chunks' scratch; the steps' has three axes)
            raise torch.OutOfMemoryError("no room")
        return empty(size, *args, **kwargs)
    monkeypatch.setattr(torch, "empty", full)
    with ops.use_backend(Launches(lambda op, arguments: seen.append(arguments[-4:-2]) or 0)):
        _scan(kind, 80)
    assert seen == [(None, 0)]


@pytest.mark.parametrize("handle", [0, 0x7F0012345678])
def test_a_registered_launch_is_handed_the_stream_as_a_pointer(handle, monkeypatch):
    """The launch that a part registers gets the step's stream as a ctypes pointer, whatever the framework's own get."""
    from wllm_amd.kernels import hip_backend
    seen = []
    monkeypatch.setattr(ops, "_REGISTERED", dict(ops._REGISTERED))
    backend = hip_backend.HipBackend.__new__(hip_backend.HipBackend)
    backend._registered, backend.lib = {}, type("Library", (), {"an_entry": staticmethod(lambda: 0)})()
    monkeypatch.setattr(backend, "_stream", lambda: handle, raising=False)
    ops.register_op("a_parts_own", entry_point="an_entry", argtypes=[], launch=lambda fn, stream: seen.append(stream) or 0)
    with ops.use_backend(backend):
        ops.call("a_parts_own")
    assert isinstance(seen[0], ctypes.c_void_p) and seen[0].value == (handle or None)


@pytest.mark.parametrize("kind,first", [("space", 64), ("memory", 128)])
def test_a_scan_is_walked_in_chunks_from_where_they_pay(kind, first):
    """The tokens from which a segment takes chunks go to the launch, and a step without such a segment has none of it."""
    with ops.use_backend(Launches(lambda op, arguments: seen.append(arguments[-4:-1]) or 0)):
        seen = []
        for n, extra in ((first - 1, {}), (first, {}), (first, {"longest": first - 1}), (first + 40, {"longest": first, "shortest": 5})):
            _scan(kind, n, **extra)
    assert [begin for _, begin, _ in seen] == [0, first, 0, first] and [bool(chunks) for chunks, _, _ in seen] == [False, True, False, True]
    assert seen[-1][2] == 5
    assert [ops.ssm_chunk_from(h, g) for h, g in ((16, 1), (17, 1), (64, 1), (65, 1), (64, 8))] == [64, 128, 128, 130, 64]
    sizes = ((4, 512), (8, 64), (8, 65), (16, 128), (8, 256), (1, 511))
    assert [ops.memory_chunk_from(h, v, True) for h, v in sizes] == [96, 128, 192, 192, 192, 128]
    assert [ops.memory_chunk_from(h, v, False) for h, v in sizes] == [160, 128, 256, 256, 192, 128]


def test_where_pieces_of_few_rows_products_are_joined():
    """By rows and keys: every band of columns reads the rows for itself."""
    from wllm_amd.kernels.hip_backend import HipBackend
    takes = HipBackend.joined_takes
    assert takes(16, 2048, 16, 6144) and not takes(17, 2048, 16, 6144) and takes(12, 2048, 16, 8192) and not takes(1, 2048, 16, 8224)
    assert takes(24, 2048, 16, 4096) and not takes(25, 2048, 16, 4096) and takes(64, 2048, 2, 768) and not takes(64, 2048, 2, 2048)
