"""The native way to the entry points, without a GPU: what a call hands on, what it refuses, and the look at operands."""
import ctypes
import subprocess

import pytest
import torch

from wllm_amd.kernels import library, ops

SOURCE = r"""
#include <stdio.h>
static char out[512];
extern "C" const char* text() { return out; }
extern "C" int mixed(void* a, int b, float c, long long d, void* e, int f, int g, float h, int i, void* j, float k, long long l, int m) {
    snprintf(out, sizeof(out), "%lld %d %g %lld %lld %d %d %g %d %lld %g %lld", (long long)a, b, c, d, (long long)e, f, g, h, i, (long long)j, k, l);
    return m;
}
extern "C" int many(int a0, int a1, int a2, int a3, int a4, int a5, long long a6, int a7, int a8, int a9, float f0, float f1, float f2, float f3,
                    float f4, float f5, float f6, float f7, void* last) {
    return a0 + 2 * a1 + 3 * a2 + 4 * a3 + 5 * a4 + 6 * a5 + 7 * (int)a6 + 8 * a7 + 9 * a8 + 10 * a9 +
           (int)(f0 + 2 * f1 + 3 * f2 + 4 * f3 + 5 * f4 + 6 * f5 + 7 * f6 + 8 * f7) + (last ? 1000 : 0);
}
"""


@pytest.fixture(scope="module")
def door():
    return library.door()


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    folder = tmp_path_factory.mktemp("functions")
    (folder / "f.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(folder / "f.cpp"), "-o", str(folder / "f.so")], check=True)
    lib = ctypes.CDLL(str(folder / "f.so"))
    lib.text.restype = ctypes.c_char_p
    return lib


def entry(door, fn, codes):
    return door.Entry(ctypes.cast(fn, ctypes.c_void_p).value, codes)


def test_arguments_arrive_as_through_ctypes(door, functions):
    codes, of = "pifl" + "pii" + "fipfli", {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_longlong, "f": ctypes.c_float}
    functions.mixed.argtypes = [of[c] for c in codes]
    call = entry(door, functions.mixed, codes)
    for args in ((4096, -3, 1.5, -(1 << 40), None, 7, True, 2, -9, ctypes.c_void_p(17), -0.25, 1 << 50, -12),
                 ((1 << 63) + 5, (1 << 31) - 1, 0.0, (1 << 63) - 1, ctypes.c_void_p(0), -(1 << 31), 0, 3.0, 1, 0, 1e30, 0, 5)):
        want = functions.mixed(*args), functions.text()
        assert (call(*args), functions.text()) == want
    numbers = list(range(1, 11))
    floats = [float(v) for v in range(1, 9)]
    want = sum((i + 1) * v for i, v in enumerate(numbers)) + sum((i + 1) * int(v) for i, v in enumerate(floats)) + 1000
    assert entry(door, functions.many, "iiiiiiliii" + "f" * 8 + "p")(*numbers, *floats, 64) == want


def test_what_an_entry_refuses(door, functions):
    args = (4096, -3, 1.5, 0, None, 7, 1, 2, -9, 17, -0.25, 0, -12)
    call = entry(door, functions.mixed, "piflpiifipfli")
    for at, value, error in ((0, "x", TypeError), (0, 1.5, TypeError), (0, -1, OverflowError), (1, 1 << 31, OverflowError), (1, 2.5, TypeError),
                             (2, "y", TypeError), (3, 1 << 63, OverflowError), (1, torch.zeros(2), (TypeError, ValueError))):
        with pytest.raises(error):
            call(*args[:at], value, *args[at + 1:])
    for wrong in (args[:-1], args + (0,)):
        with pytest.raises(TypeError):
            call(*wrong)
    with pytest.raises(TypeError):
        call(*args[:-1], last=1)
    for address, codes in ((0, "p"), (1, "q"), (1, "p" * 41), (1, "f" * 9), (1, "i" * 49)):
        with pytest.raises(ValueError):
            door.Entry(address, codes)


def test_the_look_at_an_operand_is_the_plain_ones(door):
    asked = []

    def slow(*args, **kwargs):
        asked.append((args, kwargs))
        return "slow"
    dense = door.make_dense(slow)
    t = torch.zeros(4, 8)
    both = (torch.float32, torch.bfloat16)
    for args in ((t, "t", torch.float32), (t, "t", both), (t, "t", torch.float32, (4, 8)), (t, "t", both, t.shape), (t[0], "t", both, (8,)),
                 (torch.zeros(0, 3), "t", torch.float32, (0, 3)), (torch.tensor(1.0), "t", torch.float32, ())):
        assert dense(*args) is None
    assert not asked
    unusual = [((t, "t", torch.bfloat16), {}), ((t.t(), "t", torch.float32), {}), ((t, "t", torch.float32, (4, 9)), {}), ((t, "t", torch.float32, (4,)), {}),
               ((t, "t", torch.float32, (4, 8, 1)), {}), ((None, "t", torch.float32), {}), ((t, "t", torch.float32, [4, 8]), {}), ((3, "t", both), {}),
               ((t, "t", torch.float32, (4, 1 << 70)), {}), ((t.to_sparse(), "t", torch.float32), {}), ((t, "t"), {"dtype": torch.float32})]
    for args, kwargs in unusual:
        assert dense(*args, **kwargs) == "slow"
    assert len(asked) == len(unusual)


def test_addresses_and_places(door):
    t = torch.zeros(4, 8)
    assert door.address(t) == t.data_ptr() and door.address(t[1:, 3:]) == t.data_ptr() + 44 and door.address(None) is None
    with pytest.raises(TypeError):
        door.address(4)

    class Elsewhere(RuntimeError):
        pass
    on_gpu = door.make_on_gpu(Elsewhere)
    assert on_gpu() is None and on_gpu(None, None) is None
    with pytest.raises(Elsewhere, match="not on the GPU"):
        on_gpu(None, t)
    with pytest.raises(TypeError):
        on_gpu(None, 3)
    with pytest.raises(TypeError):
        door.make_on_gpu(t)


def test_operands_of_the_wrong_kind_are_named():
    """Through whichever of the two looks is in use."""
    t = torch.zeros(4, 8)
    for args, message in (((t, "x", torch.bfloat16), "x: dtype torch.float32, expected torch.bfloat16"), ((t.t(), "x", torch.float32), "x: must be contiguous"),
                          ((t, "x", torch.float32, (4, 9)), r"x: shape \(4, 8\), expected \(4, 9\)"), ((None, "x", torch.float32), "x: expected a tensor")):
        with pytest.raises(ops.KernelShapeError, match=message):
            ops._dense(*args)


# ---- which build of the module is loaded, and what happens without one --------------------------------------------------------------

@pytest.fixture
def elsewhere(tmp_path, monkeypatch):
    """A package folder and a temporary folder that hold no build, in a process that has loaded none."""
    (tmp_path / "package").mkdir()
    monkeypatch.setattr(library, "PACKAGE_DIR", str(tmp_path / "package"))
    monkeypatch.setattr(library.tempfile, "tempdir", str(tmp_path))
    monkeypatch.setattr(library, "_loaded", {})
    return tmp_path / "package"


def a_build_that_fails(monkeypatch):
    monkeypatch.setattr(library, "_door_command", lambda hipcc, target: ["/bin/sh", "-c", "echo no headers >&2; exit 1"])


@pytest.mark.parametrize("of", ["torch", "abi", "interpreter", "source"])
def test_a_build_for_something_else_is_not_loaded(of, elsewhere, monkeypatch):
    """The module is compiled against headers of torch and of the interpreter: one for others would look for a tensor's fields in the wrong
    places, so it is none."""
    here = library._door_places()[0]
    with open(here, "w") as f:
        f.write("a build that would be taken")
    if of == "torch":
        monkeypatch.setattr(torch, "__version__", "9.9.9")
    elif of == "abi":
        monkeypatch.setattr(torch._C, "_GLIBCXX_USE_CXX11_ABI", not torch._C._GLIBCXX_USE_CXX11_ABI)
    elif of == "interpreter":
        monkeypatch.setattr(library.sysconfig, "get_config_var", lambda name: "cpython-399")
    else:
        (elsewhere / "launch_door.cpp").write_text("// another")
        monkeypatch.setattr(library, "SOURCE_DIR", str(elsewhere))
    assert here not in library._door_places()
    a_build_that_fails(monkeypatch)
    assert library.built_door() is None and library.door() is None


def test_a_module_that_cannot_be_loaded_is_built_again(elsewhere):
    """And importing the operations needs none."""
    here = library._door_places()[0]
    for name in (here, here.replace(".so", "0.so").rsplit(".", 2)[0] + ".0123456789ab.so"):
        with open(name, "w") as f:
            f.write("no module")
    assert library.built_door() is None
    door = library.door()
    assert door is not None and door.address(None) is None
    assert [p.name for p in elsewhere.iterdir()] == [here.rsplit("/", 1)[1]]         # what older sources left is gone


def test_the_kernels_are_built_without_the_module(elsewhere, monkeypatch, capsys):
    """Where the module cannot be compiled (no headers, another processor) the kernels are, as if there were none."""
    (elsewhere / "one.hip").write_text('extern "C" __attribute__((visibility("default"))) int one() { return 1; }\n')
    (elsewhere / "launch_door.cpp").write_text("#error no")
    monkeypatch.setattr(library, "SOURCE_DIR", str(elsewhere))
    a_build_that_fails(monkeypatch)
    path = library.build(source_dir=str(elsewhere))
    assert ctypes.CDLL(path).one() == 1 and library.door() is None
    assert "calls go through ctypes: no headers" in capsys.readouterr().err


@pytest.fixture
def a_backend(monkeypatch):
    """Makes one as it would be made on a GPU, and undoes at the end of the test what it changes."""
    from wllm_amd.kernels import hip_backend
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    before = ops._address
    for module, name, plain in ((ops, "_dense", ops._plain_dense), (ops, "_address", plain_address), (hip_backend, "_ptr", plain_address)):
        monkeypatch.setattr(module, name, plain)
    ops._use_address(plain_address)
    yield hip_backend.HipBackend
    ops._use_address(before)


def plain_address(t):
    return t.data_ptr() if t is not None else None


def test_a_backend_brings_the_native_look_at_operands(door, a_backend, monkeypatch):
    """Also in a process that imported the operations before there was a build."""
    from wllm_amd.kernels import hip_backend
    backend = a_backend()
    assert type(backend.lib.wllm_split_sum) is door.Entry and type(backend._on_gpu).__name__ == "Bound"
    assert type(ops._dense).__name__ == "Bound" and ops._address is hip_backend._ptr is door.address
    seen = []
    monkeypatch.setattr(ops, "_use_address", seen.append)
    ops.use_native(door)
    assert seen == [door.address]


def test_a_backend_without_the_module_calls_through_ctypes(a_backend, monkeypatch):
    from wllm_amd.kernels import hip_backend
    monkeypatch.setattr(hip_backend, "door", lambda: None)
    backend = a_backend()
    assert isinstance(backend.lib.wllm_split_sum, ctypes._CFuncPtr) and backend.lib.wllm_split_sum.argtypes[-1] is ctypes.c_void_p
    assert ops._dense is ops._plain_dense and hip_backend._ptr is plain_address
    with pytest.raises(hip_backend.KernelError, match="not on the GPU"):
        backend._on_gpu(None, torch.zeros(2))
    op = next(o for o in ops._REGISTERED.values() if o.own)
    assert backend._entry(getattr(backend.lib.raw, op.entry_point), op.argtypes) is getattr(backend.lib.raw, op.entry_point)


def test_registered_launches_take_the_address_that_is_in_use():
    t, seen = torch.zeros(3, 4, dtype=torch.bfloat16), []
    try:
        ops._use_address(lambda x: seen.append(x) or 7)
        assert ops._REGISTERED["activation"].launch(lambda *args: args, 0, t, t, "silu")[:2] == (7, 7) and len(seen) == 2
    finally:
        ops._use_address(ops._address)
