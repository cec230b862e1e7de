"""Building and loading the kernel library.

The kernels under `wllm_amd/csrc` are compiled with hipcc for gfx950 into one
shared library, `wllm_amd/libwllm_kernels.so`, whose `extern "C"` entry points
are called with raw device pointers and a stream.  The kernels are compiled against nothing of
torch; beside them `csrc/launch_door.cpp`, host code alone, becomes a CPython module
(`door()`) through which the framework's own calls go, since ctypes would take half
as long for each as the launch itself.  The module is compiled against the interpreter's and torch's
headers, so its file's name says for which of them it is; where it cannot be built, ctypes does its
work.  A build takes about a minute from nothing.

`load()` loads the library if it is built from the present sources and builds it
first if not (a line is printed per compiled file, so that a first call in a
fresh checkout shows what it is doing).  If the package folder cannot be
written to, the build goes to a folder under the system's temporary directory.
"""
from __future__ import annotations

import contextlib
import ctypes
import hashlib
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
import time
from concurrent.futures import ThreadPoolExecutor
from importlib import util
from typing import Optional

PACKAGE_DIR = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE_DIR = os.path.join(PACKAGE_DIR, "csrc")
LIBRARY_NAME = "libwllm_kernels.so"
DOOR_SOURCE, DOOR_NAME = "launch_door.cpp", "launch_door"
ARCH = "gfx950"
# Packed float32 instructions are switched off for all device code.  The first 16 words of a kernel's arguments are in scalar registers when its wavefronts
# start: loaded by the kernel itself they are a trip to memory in front of everything else, in each of a step's 131 to 292 launches (decode steps at Gemma-2B
# sizes of 1 / 8 / 64 requests 1,311 / 1,401 / 2,161 to 1,293 / 1,375 / 2,113 us, Tokuvik's of 8 2,052 to 1,998, Duvozen's of 24 2,674 to 2,629).
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-mllvm", "-amdgpu-kernarg-preload-count=16", "-fvisibility=hidden", "-Wno-unused-command-line-argument"]


class KernelLibraryMissing(RuntimeError):
    """The kernel library is not built and cannot be built here."""


def sources(source_dir: str = SOURCE_DIR) -> list:
    return sorted(f for f in os.listdir(source_dir) if f.endswith(".hip"))


def _fingerprint(source_dir: str = SOURCE_DIR) -> str:
    """Of the flags and of every source and header of the folder (and, for a folder of kernels that
    is not the framework's own, of the framework's headers it may include)."""
    h = hashlib.sha256()
    h.update(" ".join(FLAGS).encode())
    folders = [source_dir] if os.path.samefile(source_dir, SOURCE_DIR) else [source_dir, SOURCE_DIR]
    for folder in folders:
        for name in sorted(os.listdir(folder)):
            if name.endswith(".h") or (folder == source_dir and name.endswith(".hip")):
                h.update(name.encode())
                with open(os.path.join(folder, name), "rb") as f:
                    h.update(f.read())
    return h.hexdigest()


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.isfile(cand) and os.access(cand, os.X_OK):
            return cand
    raise KernelLibraryMissing("hipcc was not found (looked at $HIPCC, PATH and /opt/rocm/bin); "
                               "the kernel library cannot be built")


def _writable(folder: str) -> bool:
    try:
        os.makedirs(folder, exist_ok=True)
        probe = os.path.join(folder, f".probe{os.getpid()}")
        with open(probe, "w"):
            pass
        os.remove(probe)
        return True
    except OSError:
        return False


def _locations(fingerprint: str, source_dir: str = SOURCE_DIR, library_name: str = LIBRARY_NAME) -> list:
    """(library path, object folder) candidates, beside the sources first (the framework's own
    library lies in the package folder, one level above its sources)."""
    fallback = os.path.join(tempfile.gettempdir(), f"wllm_amd_build_{os.getuid()}_{fingerprint[:16]}")
    beside = PACKAGE_DIR if os.path.samefile(source_dir, SOURCE_DIR) else source_dir
    return [(os.path.join(beside, library_name), os.path.join(source_dir, "_build")),
            (os.path.join(fallback, library_name), os.path.join(fallback, "obj"))]


def _is_current(lib_path: str, fingerprint: str) -> bool:
    stamp = lib_path + ".stamp"
    if not (os.path.isfile(lib_path) and os.path.isfile(stamp)):
        return False
    with open(stamp, "r", encoding="utf-8") as f:
        return f.read().strip() == fingerprint


def _door_command(hipcc: str, target: str) -> list:
    """Compiles the module of `DOOR_SOURCE`: host code, against the interpreter's and torch's headers."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    include = [a for folder in [sysconfig.get_paths()["include"]] + include_paths() for a in ("-isystem", folder)]
    return [hipcc, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"] + include + [
            os.path.join(SOURCE_DIR, DOOR_SOURCE), "-o", target] + [f"-L{p}" for p in library_paths()] + [
            "-ltorch_python", "-ltorch_cpu", "-lc10"]         # (found where `import torch` has loaded them)


def _door_places() -> list:
    """Where the module lies, beside the kernel library first.  Its name holds a hash of what it is compiled against (the interpreter, and
    torch, whose inline accessors know how a tensor is laid out) and one of its source: a file of that name can be loaded, and a build for
    another torch or interpreter is left alone."""
    import torch
    host = "\n".join([sys.version, str(sysconfig.get_config_var("SOABI")), torch.__version__, str(getattr(torch.version, "git_version", "")),
                      str(torch._C._GLIBCXX_USE_CXX11_ABI)])
    with open(os.path.join(SOURCE_DIR, DOOR_SOURCE), "rb") as f:
        source = f.read()
    name = ".".join([DOOR_NAME, hashlib.sha256(host.encode()).hexdigest()[:12], hashlib.sha256(source).hexdigest()[:12], "so"])
    return [os.path.join(PACKAGE_DIR, name), os.path.join(tempfile.gettempdir(), f"wllm_amd_build_{os.getuid()}_door", name)]


def build_door(verbose: bool = True) -> Optional[str]:
    """Compiles the module and returns its path; None, with a line that says why, where that is not possible here (no compiler, no headers
    of the interpreter or of torch, another processor): the kernels don't need it."""
    def say(msg: str) -> None:
        if verbose:
            print(f"[wllm_amd build] {msg}", file=sys.stderr, flush=True)

    path = next((p for p in _door_places() if _writable(os.path.dirname(p))), None)
    if path is None:
        say(f"no writable place for {DOOR_NAME}: calls go through ctypes")
        return None
    t0, tmp = time.time(), f"{path}.tmp{os.getpid()}"
    try:
        r = subprocess.run(_door_command(_hipcc(), tmp), capture_output=True, text=True)
        failure = r.stderr[-4000:] if r.returncode != 0 else ""
    except (KernelLibraryMissing, OSError, ImportError) as e:
        failure = str(e)
    if failure or not os.path.isfile(tmp):
        say(f"{DOOR_SOURCE} cannot be built here, calls go through ctypes: {failure or 'no module came out'}")
        if os.path.isfile(tmp):
            os.remove(tmp)
        return None
    os.replace(tmp, path)
    # (builds of older sources for the same interpreter and torch; a process that has one loaded keeps it)
    of_host = os.path.basename(path).rsplit(".", 2)[0] + "."
    for name in os.listdir(os.path.dirname(path)):
        if name.startswith(of_host) and name.endswith(".so") and name != os.path.basename(path):
            with contextlib.suppress(FileNotFoundError):
                os.remove(os.path.join(os.path.dirname(path), name))
    say(f"built {path} in {time.time() - t0:.0f} s")
    return path


def build(verbose: bool = True, force: bool = True, source_dir: str = SOURCE_DIR, library_name: str = LIBRARY_NAME) -> str:
    """Compiles every source of the folder for gfx950 and links the library; returns its path.
    The framework's headers are on the include path of any folder."""
    fingerprint = _fingerprint(source_dir)
    hipcc = _hipcc()
    lib_path = obj_dir = None
    for cand_lib, cand_obj in _locations(fingerprint, source_dir, library_name):
        if _writable(os.path.dirname(cand_lib)) and _writable(cand_obj):
            lib_path, obj_dir = cand_lib, cand_obj
            break
    if lib_path is None:
        raise KernelLibraryMissing("no writable place for the kernel library (beside its sources and the temporary folder)")
    if not force and _is_current(lib_path, fingerprint):
        return lib_path
    names = sources(source_dir)
    env = dict(os.environ)
    env.setdefault("TMPDIR", tempfile.gettempdir())
    t0 = time.time()

    def say(msg: str) -> None:
        if verbose:
            print(f"[wllm_amd build] {msg}", file=sys.stderr, flush=True)

    say(f"compiling {len(names)} kernel files of {source_dir} for {ARCH} with {hipcc}")

    def compile_one(name: str):
        obj = os.path.join(obj_dir, name[:-4] + ".o")
        cmd = [hipcc] + FLAGS + ["-I", source_dir, "-I", SOURCE_DIR, "-c", os.path.join(source_dir, name), "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True, env=env)
        return name, obj, r

    objects = []
    with ThreadPoolExecutor(max_workers=min(8, max(1, len(names)))) as pool:
        door_run = pool.submit(build_door, verbose) if os.path.samefile(source_dir, SOURCE_DIR) else None
        for name, obj, r in pool.map(compile_one, names):
            if r.returncode != 0:
                raise KernelLibraryMissing(f"hipcc failed on {name}:\n{r.stderr[-4000:]}")
            say(f"compiled {name} ({time.time() - t0:.0f} s)")
            objects.append(obj)
    tmp = lib_path + f".tmp{os.getpid()}"
    r = subprocess.run([hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objects,
                       capture_output=True, text=True, env=env)
    if r.returncode != 0:
        raise KernelLibraryMissing(f"linking the kernel library failed:\n{r.stderr[-4000:]}")
    os.replace(tmp, lib_path)
    with open(lib_path + ".stamp", "w", encoding="utf-8") as f:
        f.write(fingerprint)
    if door_run is not None:
        door_run.result()
    say(f"built {lib_path} in {time.time() - t0:.0f} s")
    return lib_path


_loaded: dict = {}


def built_door():
    """The module of `launch_door.cpp` if it is built from the present source for this interpreter and this torch and can be loaded, else
    None: nothing is built for it."""
    if DOOR_NAME not in _loaded:
        import torch  # noqa: F401  (the module's symbols of torch)
        for path in _door_places():
            if not os.path.isfile(path):
                continue
            spec = util.spec_from_file_location(DOOR_NAME, path)
            try:
                module = util.module_from_spec(spec)
                spec.loader.exec_module(module)
            except ImportError:
                continue
            _loaded[DOOR_NAME] = module
            break
    return _loaded.get(DOOR_NAME)


def door():
    """The module of `launch_door.cpp`, built first when there is none that can be loaded; None where it cannot be built."""
    module = built_door()
    if module is None and (path := build_door()) is not None:
        module = built_door()
        if module is None:
            print(f"[wllm_amd build] {path} cannot be loaded, calls go through ctypes", file=sys.stderr, flush=True)
    return module


def load(verbose: bool = True, source_dir: str = SOURCE_DIR, library_name: str = LIBRARY_NAME) -> ctypes.CDLL:
    """The loaded library of a folder of kernels (the framework's own by default); built first when
    no build of the present sources exists.  A part that brings kernels of its own keeps them in a
    folder of `.hip` files and loads them with `load(source_dir=..., library_name=...)`: the same
    compiler flags, the framework's headers on the include path, the library beside the sources."""
    key = (os.path.realpath(source_dir), library_name)
    if key in _loaded:
        return _loaded[key]
    fingerprint = _fingerprint(source_dir)
    path = None
    for cand_lib, _ in _locations(fingerprint, source_dir, library_name):
        if _is_current(cand_lib, fingerprint):
            path = cand_lib
            break
    if path is None:
        path = build(verbose=verbose, source_dir=source_dir, library_name=library_name)
    try:
        lib = ctypes.CDLL(path)
    except OSError as e:
        raise KernelLibraryMissing(f"{path} cannot be loaded: {e}") from e
    lib.wllm_path = path
    _loaded[key] = lib
    return lib
