"""In-tree build of the native core `ollama_operator_amd/_C*.so` for gfx950.

hipcc compiles every `csrc/**/*.hip` (device code) and `csrc/**/*.cpp` (host code: loader,
executor, pybind11 bindings) in parallel, incrementally, then links one shared object against the
HIP runtime that torch ships (same SONAME, so one runtime instance per process). No torch headers
are used, which keeps a full rebuild to well under a minute on 8 cores.

    python build_native.py [--clean] [--jobs N]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import glob
import os
import subprocess
import sys
import sysconfig

ROOT = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(ROOT, "csrc")
CPU_SRC = os.path.join(CSRC, "cpu")
STACK_SRC = os.path.join(CSRC, "stack")
BUILD = os.path.join(ROOT, "build", "native")
STACK_BUILD = os.path.join(ROOT, "build", "stack")
DEBUG_BUILD = os.path.join(ROOT, "build", "debug")
ARCH = os.environ.get("OMX_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# HIP device code is compiled without packed-float32 instructions: the compiler forms them from ordinary float code, and
# some of their forms have given wrong results now and then
NO_PK_F32 = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _ext_suffix() -> str:
    return sysconfig.get_config_var("EXT_SUFFIX") or ".so"


def target_path() -> str:
    return os.path.join(ROOT, "ollama_operator_amd", "_C" + _ext_suffix())


def _torch_lib() -> str | None:
    try:
        import importlib.util
        spec = importlib.util.find_spec("torch")
        if spec and spec.origin:
            d = os.path.join(os.path.dirname(spec.origin), "lib")
            if os.path.exists(os.path.join(d, "libamdhip64.so")):
                return d
    except Exception:
        pass
    return None


def _headers() -> list[str]:
    return glob.glob(os.path.join(CSRC, "**", "*.h"), recursive=True) + [os.path.abspath(__file__)]  # and the flags here


def _needs(obj: str, src: str, hdr_mtime: float) -> bool:
    if not os.path.exists(obj):
        return True
    m = os.path.getmtime(obj)
    return m < os.path.getmtime(src) or m < hdr_mtime


DEBUG_FLAGS = ["-O1", "-g", "-DOMX_DEBUG_KERNELS"]


def _core_sources() -> list[str]:
    return sorted(s for s in glob.glob(os.path.join(CSRC, "**", "*.hip"), recursive=True) +
                  glob.glob(os.path.join(CSRC, "**", "*.cpp"), recursive=True)
                  if not s.startswith(CPU_SRC + os.sep)  # the CPU backend is its own module (build_cpu)
                  and not s.startswith(STACK_SRC + os.sep))  # and so is the stack executor (build_stack)


def _stack_sources() -> list[str]:
    srcs = sorted(glob.glob(os.path.join(STACK_SRC, "*.hip")) + glob.glob(os.path.join(STACK_SRC, "*.cpp")))
    return srcs + [os.path.join(CSRC, "kernels", "sampling.hip")]


def units(srcs: list[str], build_dir: str, opt: list[str]) -> list[tuple[str, str, list[str]]]:
    """(source, object, command) of each translation unit."""
    import pybind11
    common = [*opt, "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I", CSRC, "-I", pybind11.get_include(), "-I",
              sysconfig.get_paths()["include"], "-Wno-unused-result"]
    out = []
    for s in srcs:
        obj = os.path.join(build_dir, os.path.relpath(s, CSRC).replace(os.sep, "_") + ".o")
        if s.endswith(".hip"):
            cmd = [HIPCC, *common, *NO_PK_F32, "-c", s, "-o", obj]
        else:  # host-only translation unit
            cmd = [HIPCC, *common, "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-c", s, "-o", obj,
                   "-fvisibility=hidden"]
        out.append((s, obj, cmd))
    return out


def all_units() -> list[tuple[str, str, list[str]]]:
    """Every translation unit that hipcc compiles for the release modules."""
    return units(_core_sources(), BUILD, ["-O3"]) + units(_stack_sources(), STACK_BUILD, ["-O3"])


def _compile(todo: list[tuple[str, str, list[str]]], jobs: int, verbose: bool, what: str) -> None:
    def run(item):
        s, _, cmd = item
        r = subprocess.run(cmd, capture_output=True, text=True)
        return s, r.returncode, r.stdout + r.stderr, " ".join(cmd)

    failed = []
    if todo:
        with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
            for s, rc, out, cmd in ex.map(run, todo):
                if rc != 0:
                    failed.append((s, out, cmd))
                elif verbose:
                    print("compiled", os.path.relpath(s, ROOT))
    if failed:
        for s, out, cmd in failed:
            sys.stderr.write(f"--- {s}\n{cmd}\n{out}\n")
        raise RuntimeError(f"{what} build failed ({len(failed)} translation units)")


def _link(objs: list[str], out: str, libs: list[str], what: str) -> None:
    """Linked beside the target, then renamed: a reader of the tree (a test, a tree snapshot) never sees a half-written library."""
    tmp = out + ".tmp"
    link = [HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs, "-lpthread"]
    tl = _torch_lib()
    if tl:
        link += [f"-L{tl}", f"-Wl,-rpath,{tl}"]
    r = subprocess.run([*link, *libs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} link failed:\n" + " ".join([*link, *libs]) + "\n" + r.stdout + r.stderr)
    os.replace(tmp, out)


def build(jobs: int | None = None, clean: bool = False, verbose: bool = False, debug: bool = False,
          sources: list[str] | None = None) -> str:
    """debug: the in-kernel bounds assertions (OMX_KASSERT) and -O1 -g, objects in build/debug and the
    module in build/debug/ollama_operator_amd (put that directory first on sys.path to load it).
    sources: compile only these csrc-relative translation units (no link), e.g. for a build check."""
    build_dir = DEBUG_BUILD if debug else BUILD
    os.makedirs(build_dir, exist_ok=True)
    if clean:
        for f in glob.glob(os.path.join(build_dir, "*.o")):
            os.remove(f)
    srcs = _core_sources() if sources is None else [os.path.join(CSRC, x) for x in sources]
    hdr_mtime = max((os.path.getmtime(h) for h in _headers()), default=0.0)
    all_ = units(srcs, build_dir, DEBUG_FLAGS if debug else ["-O3"])
    objs = [obj for _, obj, _ in all_]
    todo = [u for u in all_ if _needs(u[1], u[0], hdr_mtime)]
    _compile(todo, jobs or min(8, os.cpu_count() or 4), verbose, "native")
    if sources is not None:
        return build_dir
    out = target_path()
    if debug:
        os.makedirs(os.path.join(build_dir, "ollama_operator_amd"), exist_ok=True)
        out = os.path.join(build_dir, "ollama_operator_amd", os.path.basename(out))
    if not os.path.exists(out) or todo or any(os.path.getmtime(o) > os.path.getmtime(out) for o in objs):
        # hipBLASLt for the large-M prefill GEMM (csrc/runtime/blas.cpp): torch's copy when present
        # (one instance per process), else the ROCm one
        tl = _torch_lib()
        torch_has = tl and os.path.exists(os.path.join(tl, "libhipblaslt.so"))
        _link(objs, out, ["-lhipblaslt"] + ([] if torch_has else ["-L/opt/rocm/lib"]), "native")
    return out


def stack_target_path() -> str:
    return os.path.join(ROOT, "ollama_operator_amd", "_stack" + _ext_suffix())


def build_stack(verbose: bool = False, force: bool = False) -> str:
    """`ollama_operator_amd/_stack*.so`: the kernels and step executor of layer-list models (csrc/stack) with
    the on-device sampler (csrc/kernels/sampling.hip). Its own small library: a checkout that serves only
    such a model compiles these few files (about a minute), not the quantised-GEMV families of `_C`."""
    os.makedirs(STACK_BUILD, exist_ok=True)
    hdr_mtime = max((os.path.getmtime(h) for h in _headers()), default=0.0)
    all_ = units(_stack_sources(), STACK_BUILD, ["-O3"])
    objs = [obj for _, obj, _ in all_]
    todo = [u for u in all_ if force or _needs(u[1], u[0], hdr_mtime)]
    _compile(todo, min(8, max(1, len(todo))), verbose, "stack module")
    out = stack_target_path()
    if not os.path.exists(out) or todo or any(os.path.getmtime(o) > os.path.getmtime(out) for o in objs):
        _link(objs, out, [], "stack module")
    return out


def cpu_target_path() -> str:
    return os.path.join(ROOT, "ollama_operator_amd", "_cpu" + _ext_suffix())


def build_cpu(verbose: bool = False) -> str:
    """`ollama_operator_amd/_cpu*.so`: the CPU serving backend (csrc/cpu), host compiler only (no HIP
    runtime dependency, so it loads on a CPU-only node). AVX2 + FMA + F16C baseline, OpenMP threads."""
    import pybind11
    srcs = sorted(glob.glob(os.path.join(CPU_SRC, "*.cpp")))
    hdrs = glob.glob(os.path.join(CPU_SRC, "*.h"))
    out = cpu_target_path()
    newest = max(os.path.getmtime(f) for f in srcs + hdrs)
    if os.path.exists(out) and os.path.getmtime(out) >= newest:
        return out
    cxx = os.environ.get("CXX", "g++")
    cmd = [cxx, "-O3", "-std=c++17", "-fPIC", "-shared", "-fopenmp", "-mavx2", "-mfma", "-mf16c",
           "-fvisibility=hidden", "-I", CPU_SRC, "-I", pybind11.get_include(), "-I", sysconfig.get_paths()["include"],
           *srcs, "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("CPU backend build failed:\n" + " ".join(cmd) + "\n" + r.stdout + r.stderr)
    if verbose:
        print("built", os.path.relpath(out, ROOT))
    return out


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--clean", action="store_true")
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("--cpu-only", action="store_true", help="build only the CPU backend module")
    ap.add_argument("--stack", action="store_true", help="build only the stack executor's module")
    ap.add_argument("--debug", action="store_true",
                    help="kernels with in-kernel bounds assertions (OMX_KASSERT), -O1 -g, into build/debug")
    a = ap.parse_args()
    if a.stack:
        print(build_stack(verbose=True))
        sys.exit(0)
    if not a.debug:
        print(build_stack(verbose=True))
    if not a.debug:
        print(build_cpu(verbose=True))
    if not a.cpu_only:
        print(build(a.jobs, a.clean, verbose=True, debug=a.debug))
