"""Builds and loads the HIP libraries, one shared object per source file under `csrc/`.

A library is compiled with hipcc for gfx950 the first time something in it is called and
kept beside the package (`minfer_amd/_lib/`); a hash of its sources decides whether a
built file is still current.  There is no other backend: if a library can neither be
loaded nor built, the call raises.
"""
from __future__ import annotations

import ctypes
import hashlib
import os
import shutil
import subprocess
import sys
import threading
import time
from typing import Dict, List

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc")
LIB_DIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "_lib")

# library name -> source file; HEADERS: what each includes (default: common.h).  A `.cpp` source is
# host code only and is built with the host compiler.  EXTENSIONS: those that are Python modules against torch's headers
# (`load_extension`).
LIBRARIES: Dict[str, str] = {
    "host_random": "host_random.cpp",
    "host_call": "host_call.cpp",
    "elementwise": "elementwise.hip",
    "gemm_f32": "gemm_f32.hip",
    "gemm_bf16": "gemm_bf16.hip",
    "attn_tokens_f32": "attn_tokens_f32.hip",
    "attn_prompt_f32": "attn_prompt_f32.hip",
    "attn_decode_bf16": "attn_decode_bf16.hip",
    "attn_prefill_bf16": "attn_prefill_bf16.hip",
    "attn_latent": "attn_latent.hip",
    "attn_latent_mfma": "attn_latent_mfma.hip",
    "recurrence": "recurrence.hip",
    "linear_attention": "linear_attention.hip",
    "attn_capped": "attn_capped.hip",
    "attn_capped_mfma": "attn_capped_mfma.hip",
    "attn_normed": "attn_normed.hip",
    "gated_recurrence": "gated_recurrence.hip",
    "moe": "moe.hip",
    "sampling": "sampling.hip",
    "probe": "probe.hip",
}
EXTENSIONS = {"host_call": "mf_host_call"}
# library name -> extra -D definitions (variants of one source compiled for given sizes, see `variant`)
DEFINES: Dict[str, List[str]] = {}
HEADERS = {"host_random": ["random_normal.h"],
           "host_call": [],
           "elementwise": ["common.h", "random_normal.h"],
           "attn_tokens_f32": ["common.h", "attn_tokens_impl.h"],
           "attn_prompt_f32": ["common.h", "attn_tokens_impl.h"],
           "attn_decode_bf16": ["common.h", "attn_tokens_impl.h", "noalloc.h"],
           "attn_capped": ["common.h", "attn_tokens_impl.h"],
           "attn_capped_mfma": ["common.h", "attn_tokens_impl.h"]}

HIPCC_FLAGS = ["-O3", "--offload-arch=gfx950", "-fPIC", "-shared", "-std=c++17",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               # a kernel's first arguments come in registers: with the trip to memory for them in front, a split product of 40 rows with the
               # kernel that adds its parts 10.0 us (896 x 4,864), 9.65 so; 11.4 and 10.7 (2,560 x 2,048, 100 rows)
               "-mllvm", "-amdgpu-kernarg-preload-count=14",
               "-Wno-unused-command-line-argument"]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", "-ffp-contract=off", "-Wno-unknown-pragmas"]


class KernelBuildError(RuntimeError):
    pass


def _host_flags(name: str) -> List[str]:
    """What a host library is compiled with; for an extension also where torch's and Python's headers and torch's
    libraries are."""
    if name not in EXTENSIONS:
        return HOST_FLAGS
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    return HOST_FLAGS + ["-I" + os.path.join(root, "include"), "-I" + sysconfig.get_paths()["include"],
                         f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-L" + os.path.join(root, "lib"),
                         "-ltorch_python", "-ltorch_cpu", "-lc10"]


def _stamp_flags(name: str) -> List[str]:
    """What besides its sources decides whether a built file is current: the flags, and for an extension the versions of
    the interpreter and torch."""
    if name not in EXTENSIONS:
        return HOST_FLAGS if is_host_library(name) else HIPCC_FLAGS
    import torch
    return HOST_FLAGS + [sys.version, torch.__version__]


def variant(base: str, **sizes: int) -> str:
    """Registers (once) and names the library that is `base`'s source compiled with the given
    sizes as definitions (`-DNAME=value`): kernels whose tiles and register arrays depend on a
    model's sizes are built for the sizes at hand the first time a model with them runs."""
    name = base + "".join(f"_{k.lower()}{int(v)}" for k, v in sorted(sizes.items()))
    if name not in LIBRARIES:
        LIBRARIES[name] = LIBRARIES[base]
        DEFINES[name] = DEFINES.get(base, []) + [f"-D{k}={int(v)}" for k, v in sorted(sizes.items())]
        if base in HEADERS:
            HEADERS[name] = HEADERS[base]
        _note_variant(base, sizes)
    return name


def _variants_file() -> str:
    return os.path.join(lib_dir(), "variants.txt")


def _note_variant(base: str, sizes: Dict[str, int]) -> None:
    """Keeps the variants that were ever asked for beside the built files, so that `build_all`
    builds them again with the rest."""
    line = base + " " + " ".join(f"{k}={int(v)}" for k, v in sorted(sizes.items()))
    try:
        have = open(_variants_file()).read().splitlines() if os.path.exists(_variants_file()) else []
        if line not in have:
            with open(_variants_file(), "a") as f:
                f.write(line + "\n")
    except OSError:
        pass


def known_variants() -> List[str]:
    """Registers the variants listed beside the built files and returns their names."""
    names = []
    if os.path.exists(_variants_file()):
        for line in open(_variants_file()).read().splitlines():
            parts = line.split()
            if parts and parts[0] in LIBRARIES:
                names.append(variant(parts[0], **{k: int(v) for k, v in (p.split("=") for p in parts[1:])}))
    return names


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise KernelBuildError("hipcc not found (looked at $HIPCC, PATH and /opt/rocm/bin): the HIP "
                           "kernels cannot be built and there is no other backend")


def is_host_library(name: str) -> bool:
    return LIBRARIES[name].endswith(".cpp")


def _host_compiler() -> str:
    for cand in (os.environ.get("CXX"), shutil.which("g++"), shutil.which("c++"), shutil.which("clang++")):
        if cand and (os.path.exists(cand) or shutil.which(cand)):
            return cand
    raise KernelBuildError("no host C++ compiler found (looked at $CXX, g++, c++, clang++)")


def source_hash(name: str) -> str:
    h = hashlib.sha256()
    h.update(" ".join(_stamp_flags(name) + DEFINES.get(name, [])).encode())
    for fname in [LIBRARIES[name]] + HEADERS.get(name, ["common.h"]):
        with open(os.path.join(CSRC, fname), "rb") as f:
            h.update(fname.encode())
            h.update(f.read())
    return h.hexdigest()


def lib_dir() -> str:
    """Beside the package; a per-user folder under the temporary directory when the package
    folder cannot be written (a read-only checkout)."""
    global LIB_DIR
    try:
        os.makedirs(LIB_DIR, exist_ok=True)
        if os.access(LIB_DIR, os.W_OK):
            return LIB_DIR
    except OSError:
        pass
    import tempfile
    alt = os.path.join(tempfile.gettempdir(), f"minfer_amd_lib_{os.getuid()}")
    os.makedirs(alt, exist_ok=True)
    have = os.path.join(os.path.dirname(CSRC), "_lib")
    if os.path.isdir(have):           # built files that came with the checkout still count
        for f in os.listdir(have):
            if not os.path.exists(os.path.join(alt, f)):
                shutil.copy(os.path.join(have, f), os.path.join(alt, f))
    LIB_DIR = alt
    return LIB_DIR


def lib_path(name: str) -> str:
    return os.path.join(lib_dir(), f"libmf_{name}.so")


def is_current(name: str) -> bool:
    so, stamp = lib_path(name), lib_path(name) + ".hash"
    if not (os.path.exists(so) and os.path.exists(stamp)):
        return False
    with open(stamp) as f:
        return f.read().strip() == source_hash(name)


def _say(msg: str) -> None:
    print(f"[minfer_amd] {msg}", file=sys.stderr, flush=True)


def compile_library(name: str, quiet: bool = False) -> str:
    """Compiles one library; prints a line at start and every 15 s while hipcc runs."""
    so = lib_path(name)
    tmp = f"{so}.{os.getpid()}.tmp"
    if is_host_library(name):
        flags = _host_flags(name)
        libs = [f for f in flags if f.startswith("-l")]
        cmd = [_host_compiler()] + [f for f in flags if f not in libs] + ["-I", CSRC, os.path.join(CSRC, LIBRARIES[name]), "-o", tmp] + libs
    else:
        cmd = [_hipcc()] + HIPCC_FLAGS + DEFINES.get(name, []) + ["-I", CSRC, os.path.join(CSRC, LIBRARIES[name]), "-o", tmp]
    if not quiet:
        _say(f"compiling {LIBRARIES[name]}" + ("" if is_host_library(name) else " for gfx950") + " ...")
    t0 = time.time()
    env = dict(os.environ)
    env.setdefault("TMPDIR", "/tmp")
    proc = subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, env=env, cwd=lib_dir())
    done = threading.Event()

    def ticker():
        while not done.wait(15.0):
            _say(f"  still compiling {LIBRARIES[name]} ({time.time() - t0:.0f} s)")
    th = threading.Thread(target=ticker, daemon=True)
    th.start()
    out = proc.communicate()[0].decode(errors="replace")
    done.set()
    if proc.returncode != 0:
        if os.path.exists(tmp):
            os.remove(tmp)
        lines = [l for l in out.splitlines() if "packed-fp32-ops" not in l]
        raise KernelBuildError(f"{os.path.basename(cmd[0])} failed on {LIBRARIES[name]}:\n" + "\n".join(lines[-60:]))
    os.replace(tmp, so)
    with open(so + ".hash", "w") as f:
        f.write(source_hash(name))
    if not quiet:
        _say(f"built {os.path.basename(so)} in {time.time() - t0:.1f} s")
    return so


def build_all(force: bool = True, jobs: int = 4) -> List[str]:
    """Compiles every library and every sized variant asked for before (always, when `force`), a few
    at a time."""
    known_variants()
    names = [n for n in LIBRARIES if force or not is_current(n)]
    errors, lock = [], threading.Lock()
    pending = list(names)

    def worker():
        while True:
            with lock:
                if not pending:
                    return
                n = pending.pop(0)
            try:
                compile_library(n)
            except Exception as e:  # collected and raised together below
                with lock:
                    errors.append(e)
    threads = [threading.Thread(target=worker) for _ in range(max(1, min(jobs, len(names))))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise KernelBuildError("\n".join(str(e) for e in errors))
    return [lib_path(n) for n in names]


_loaded: Dict[str, ctypes.CDLL] = {}
_load_lock = threading.Lock()
_modules: Dict[str, object] = {}


def load_extension(name: str):
    """The Python module built from an extension's source, compiled first if it is missing or its source changed."""
    import importlib.machinery
    import importlib.util
    with _load_lock:
        module = _modules.get(name)
        if module is None:
            if not is_current(name):
                compile_library(name)
            loader = importlib.machinery.ExtensionFileLoader(EXTENSIONS[name], lib_path(name))
            spec = importlib.util.spec_from_file_location(EXTENSIONS[name], lib_path(name), loader=loader)
            try:
                module = importlib.util.module_from_spec(spec)
                loader.exec_module(module)
            except ImportError as e:
                raise KernelBuildError(f"cannot load {lib_path(name)}: {e}") from None
            _modules[name] = module
        return module


def load(name: str) -> ctypes.CDLL:
    """The loaded library, compiled first if it is missing or its sources changed."""
    lib = _loaded.get(name)
    if lib is not None:
        return lib
    with _load_lock:
        if name in _loaded:
            return _loaded[name]
        if name not in LIBRARIES:
            raise KernelBuildError(f"unknown kernel library {name!r}")
        if not is_current(name):
            compile_library(name)
        try:
            lib = ctypes.CDLL(lib_path(name))
        except OSError as e:
            raise KernelBuildError(f"cannot load {lib_path(name)}: {e}") from None
        _loaded[name] = lib
        return lib
