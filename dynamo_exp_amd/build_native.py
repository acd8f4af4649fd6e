"""In-tree native build for dynamo_exp_amd.

Two extension modules are produced next to the Python sources (so they travel
with the tree to a machine that only runs them):

* ``dynamo_exp_amd/_C_kernels*.so`` -- hand-written HIP kernels for gfx950
  (RMSNorm, RoPE + paged-KV write, SiLU-gate, embedding, paged attention
  prefill/decode, sampling, KV block copy/pack).  Compiled with
  ``hipcc --offload-arch=gfx950``; exposes raw-pointer launchers via pybind11 so
  the Python side never pays torch-extension compile time and the kernels are
  free of any torch ABI coupling.
* ``dynamo_exp_amd/_C_runtime*.so`` -- host-only C++20 runtime pieces (xxh3
  block hashing, radix KV indexer, two-part codec, block pool).

The build is incremental (mtime based) and parallel.  ``python -m
dynamo_exp_amd.build_native`` or ``__graft_entry__.build()`` drive it.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG.parent / "build" / "native"
EXT = sysconfig.get_config_var("EXT_SUFFIX") or ".so"
ARCH = os.environ.get("DX_OFFLOAD_ARCH", "gfx950")


def _py_includes() -> list[str]:
    import pybind11

    return [f"-I{pybind11.get_include()}", f"-I{sysconfig.get_paths()['include']}"]


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"native build failed: {' '.join(cmd[:3])} ... ({cmd[-1]})")
    elif verbose and r.stderr.strip():
        sys.stderr.write(r.stderr)


def _stale(out: Path, deps: list[Path]) -> bool:
    if not out.exists():
        return True
    t = out.stat().st_mtime
    return any(d.stat().st_mtime > t for d in deps)


def _headers(d: Path) -> list[Path]:
    return sorted(d.glob("*.h"))


# attn_prefill: scores are finite or -inf by construction, so fmax needs no NaN
# quieting (IEEE mode off: v_max3 without a v_mul canonicalize per score).
# decode_attention: one wave a SIMD has registers of both kinds; without the
# option all matrix products' accumulators are of the second kind, and those
# of shared rows were copied to and fro in every tile (600 instructions of 1770).
PER_FILE_FLAGS = {"attn_prefill.hip": ["-fno-honor-nans", "-mno-amdgpu-ieee"],
                  "decode_attention.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}


def _kernel_flags(src_dir: Path) -> list[str]:
    return [
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-ffp-contract=fast",
        "-munsafe-fp-atomics",
        "-Wno-unused-result",
        "-DNDEBUG",
        f"-I{src_dir}",
    ] + _py_includes()


# No HIP source is built with packed-fp32 instruction selection: some forms of v_pk_{add,mul,fma}_f32 have given
# wrong results on this hardware.  A device-side feature, so only for sources compiled as HIP.
HIP_FLAGS = ["-x", "hip", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def verify_kernels(names: list[str] | None = None, jobs: int = 8) -> dict[str, str]:
    """Compile the device side of the HIP sources in csrc/kernels, and of the
    mixers with code generation options of their own, with LLVM's machine
    verifier (``-mllvm -verify-machineinstrs``) and return {file: error} for
    the ones it rejects.  ROCm 7.2 had a sub-register liveness
    miscompile in attn_decode.hip ("No live subrange at use": V-row registers
    reused as temporaries, wrong output in the G = 1 instance only) that the
    verifier reports at compile time; the normal build does not run it."""
    import tempfile

    srcs = sorted((CSRC / "kernels").glob("*.hip")) + [s for s in sorted((CSRC / "mixers").glob("*.hip")) if s.name in PER_FILE_FLAGS]
    srcs = [s for s in srcs if names is None or s.name in names]
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    bad: dict[str, str] = {}
    with tempfile.TemporaryDirectory() as td:
        def one(s: Path):
            flags = [f for f in _kernel_flags(s.parent) if f != "-fPIC"]
            cmd = [hipcc, *flags, *HIP_FLAGS, *PER_FILE_FLAGS.get(s.name, []), "--cuda-device-only", "-c", str(s),
                   "-o", str(Path(td) / (s.name + ".o")), "-mllvm", "-verify-machineinstrs"]
            r = subprocess.run(cmd, capture_output=True, text=True)
            if r.returncode != 0:
                lines = [ln for ln in (r.stdout + r.stderr).splitlines()
                         if "Bad machine code" in ln or "- function:" in ln or "error" in ln]
                bad[s.name] = "\n".join(lines[:12])

        with ThreadPoolExecutor(max(1, jobs)) as ex:
            list(ex.map(one, srcs))
    return bad


def build_kernels(verbose: bool = False, jobs: int = 8) -> Path:
    src_dir = CSRC / "kernels"
    out = PKG / f"_C_kernels{EXT}"
    objdir = BUILD / "kernels"
    objdir.mkdir(parents=True, exist_ok=True)
    srcs = sorted(src_dir.glob("*.hip")) + sorted(src_dir.glob("*.cpp"))
    hdrs = _headers(src_dir)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    flags = _kernel_flags(src_dir)
    objs = []
    todo = []
    for s in srcs:
        o = objdir / (s.name + ".o")
        objs.append(o)
        if _stale(o, [s, Path(__file__)] + hdrs):
            extra = list(HIP_FLAGS) if s.suffix == ".hip" else []
            extra += PER_FILE_FLAGS.get(s.name, [])
            todo.append([hipcc, *flags, *extra, "-c", str(s), "-o", str(o)])
    with ThreadPoolExecutor(max(1, jobs)) as ex:
        list(ex.map(lambda c: _run(c, verbose), todo))
    if todo or _stale(out, objs):
        _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(out), *map(str, objs)], verbose)
    return out


def build_mixers(verbose: bool = False, jobs: int = 8) -> Path:
    """_C_mixers: the kernels of the layer-listed (hybrid) models
    (csrc/mixers): multi-stream residual + norm, head prep + paged cache
    write, row attention, gated activations.  A module of its own, so a
    process that serves only such a model builds and loads nothing else."""
    src_dir = CSRC / "mixers"
    out = PKG / f"_C_mixers{EXT}"
    objdir = BUILD / "mixers"
    objdir.mkdir(parents=True, exist_ok=True)
    srcs = sorted(src_dir.glob("*.hip")) + sorted(src_dir.glob("*.cpp"))
    hdrs = _headers(src_dir) + [CSRC / "kernels" / "common.h"]
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    flags = _kernel_flags(src_dir)
    objs, todo = [], []
    for s in srcs:
        o = objdir / (s.name + ".o")
        objs.append(o)
        if _stale(o, [s, Path(__file__)] + hdrs):
            extra = list(HIP_FLAGS) if s.suffix == ".hip" else []
            extra += PER_FILE_FLAGS.get(s.name, [])
            todo.append([hipcc, *flags, *extra, "-c", str(s), "-o", str(o)])
    with ThreadPoolExecutor(max(1, jobs)) as ex:
        list(ex.map(lambda c: _run(c, verbose), todo))
    if todo or _stale(out, objs):
        _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(out), *map(str, objs)], verbose)
    return out


def build_runtime(verbose: bool = False, jobs: int = 8) -> Path:
    src_dir = CSRC / "runtime"
    out = PKG / f"_C_runtime{EXT}"
    objdir = BUILD / "runtime"
    objdir.mkdir(parents=True, exist_ok=True)
    srcs = sorted(src_dir.glob("*.cpp"))
    hdrs = _headers(src_dir)
    cxx = os.environ.get("CXX", "g++")
    san = os.environ.get("DX_SANITIZE", "")  # e.g. "address,undefined" or "thread"
    flags = ["-O3", "-std=c++20", "-fPIC", "-Wall", "-Wno-unused-function", f"-I{src_dir}"] + _py_includes()
    if san:
        flags = ["-O1", "-g", f"-fsanitize={san}", "-fno-omit-frame-pointer"] + flags[1:]
    objs, todo = [], []
    for s in srcs:
        o = objdir / (s.name + (f".{san.replace(',', '_')}" if san else "") + ".o")
        objs.append(o)
        if _stale(o, [s] + hdrs):
            todo.append([cxx, *flags, "-c", str(s), "-o", str(o)])
    with ThreadPoolExecutor(max(1, jobs)) as ex:
        list(ex.map(lambda c: _run(c, verbose), todo))
    link = [cxx, "-shared", "-fPIC", "-o", str(out), *map(str, objs), "-lpthread"]
    if san:
        link.insert(1, f"-fsanitize={san}")
    if todo or _stale(out, objs):
        _run(link, verbose)
    return out


def build_capi(verbose: bool = False) -> Path:
    """libdynamo_llm_capi.so: C ABI for external engines' KV events
    (include/dynamo_exp_amd/kv_events.h)."""
    src = CSRC / "capi" / "kv_events.cpp"
    out = PKG / "libdynamo_llm_capi.so"
    hdr = PKG / "include" / "dynamo_exp_amd" / "kv_events.h"
    if _stale(out, [src, hdr, CSRC / "runtime" / "xxh3.h"]):
        cxx = os.environ.get("CXX", "g++")
        _run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", f"-I{PKG / 'include'}", "-o", str(out),
              str(src), "-lpthread"], verbose)
    return out


def build_ctrld(verbose: bool = False) -> Path:
    """bin/dx-ctrld: the native control-plane server (csrc/ctrld)."""
    srcs = [CSRC / "ctrld" / "ctrld.cpp", CSRC / "ctrld" / "msgpack.h"]
    out = PKG / "bin" / "dx-ctrld"
    if _stale(out, srcs):
        out.parent.mkdir(exist_ok=True)
        cxx = os.environ.get("CXX", "g++")
        flags = ["-O2", "-std=c++17", "-Wall", "-Wextra", "-Wno-unused-parameter"]
        san = os.environ.get("DX_SANITIZE")
        if san:
            flags += [f"-fsanitize={san}", "-fno-omit-frame-pointer", "-g"]
        _run([cxx, *flags, "-o", str(out), str(srcs[0])], verbose)
    return out


def build_all(verbose: bool = False) -> list[Path]:
    jobs = int(os.environ.get("MAX_JOBS", "8"))
    jobs = max(1, min(jobs, 16))
    return [build_runtime(verbose, jobs), build_capi(verbose), build_ctrld(verbose), build_kernels(verbose, jobs),
            build_mixers(verbose, jobs)]


if __name__ == "__main__":
    for p in build_all(verbose="-v" in sys.argv):
        print("built", p)
