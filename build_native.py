"""In-tree build of the native core `ollama_operator_amd/_C*.so` for gfx950.

hipcc compiles every `csrc/**/*.hip` (device code) and `csrc/**/*.cpp` (host code: loader,
executor, pybind11 bindings) in parallel, those whose content, headers or command changed, then
links one shared object against the HIP runtime that torch ships (same SONAME, so one runtime
instance per process). A full rebuild takes four to five minutes on 8 cores.

    python build_native.py [--clean] [--jobs N]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import glob
import hashlib
import os
import re
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
DEBUG_FLAGS = ["-O1", "-g", "-DOMX_DEBUG_KERNELS"]
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


def _hash(*parts: str | bytes) -> str:
    h = hashlib.sha256()
    for x in parts:
        x = x if isinstance(x, bytes) else x.encode()
        h.update(len(x).to_bytes(8, "little") + x)
    return h.hexdigest()


def _read(path: str) -> bytes:
    with open(path, "rb") as f:
        return f.read()


def _unit_text(src: str) -> list[bytes]:
    """A unit's source and all headers of the tree that it includes, directly or not, by name and content."""
    seen: dict[str, bytes] = {}
    todo = [os.path.abspath(src)]
    while todo:
        f = todo.pop()
        if f in seen:
            continue
        seen[f] = _read(f)
        for name in re.findall(rb'^[ \t]*#[ \t]*include[ \t]*"([^"]+)"', seen[f], re.M):
            for d in (os.path.dirname(f), CSRC):
                h = os.path.normpath(os.path.join(d, name.decode()))
                if os.path.exists(h):
                    todo.append(h)
                    break
    return [x for f in sorted(seen) for x in (os.path.relpath(f, CSRC).encode(), seen[f])]


# A product (object, library) is current when the record beside it names what it was made of and the product itself, both by
# content: times say nothing about an object that was copied, touched or compiled while a header changed.
def _current(product: str, inputs: str, record: str) -> bool:
    if not os.path.exists(product) or not os.path.exists(record):
        return False
    return _read(record).decode().split() == [inputs, _hash(_read(product))]


def _record(product: str, inputs: str, record: str) -> None:
    if os.path.exists(product):
        with open(record, "w") as f:
            f.write(f"{inputs} {_hash(_read(product))}\n")


def _core_sources() -> list[str]:
    srcs = [s for s in glob.glob(os.path.join(CSRC, "**", "*.hip"), recursive=True) +
            glob.glob(os.path.join(CSRC, "**", "*.cpp"), recursive=True)
            if not s.startswith(CPU_SRC + os.sep)  # the CPU backend is its own module (build_cpu)
            and not s.startswith(STACK_SRC + os.sep)]  # and so is the stack executor (build_stack)
    long = ("gemv8.hip", "gemv.hip")  # four and three minutes: a build lasts as long as they do if they start first
    return sorted(srcs, key=lambda s: (os.path.basename(s) not in long, s))


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


def _compile(all_: list[tuple[str, str, list[str]]], jobs: int, verbose: bool, what: str, force: bool = False) -> None:
    version, todo = "/opt/rocm/.info/version", []
    compiler = _read(version) if os.path.exists(version) else b""
    for s, obj, cmd in all_:
        inputs = _hash(compiler, *_unit_text(s), *cmd)
        if force or not _current(obj, inputs, obj + ".sha256"):
            todo.append((s, obj, cmd, inputs))

    def run(item):
        s, obj, cmd, inputs = item
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode == 0:
            _record(obj, inputs, obj + ".sha256")
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


def _link(objs: list[str], out: str, libs: list[str], what: str, record: str) -> None:
    """Linked beside the target, then renamed: a reader of the tree (a test, a tree snapshot) never sees a half-written library."""
    inputs = _hash(*(_hash(_read(o)) for o in objs), *libs)
    if _current(out, inputs, record):
        return
    tmp = out + ".tmp"
    link = [HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs, "-lpthread"]
    tl = _torch_lib()
    if tl:
        link += [f"-L{tl}", f"-Wl,-rpath,{tl}"]
    r = subprocess.run([*link, *libs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} link failed:\n" + " ".join([*link, *libs]) + "\n" + r.stdout + r.stderr)
    os.replace(tmp, out)
    _record(out, inputs, record)


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
    all_ = units(srcs, build_dir, DEBUG_FLAGS if debug else ["-O3"])
    _compile(all_, jobs or min(8, os.cpu_count() or 4), verbose, "native")
    if sources is not None:
        return build_dir
    out = target_path()
    if debug:
        os.makedirs(os.path.join(build_dir, "ollama_operator_amd"), exist_ok=True)
        out = os.path.join(build_dir, "ollama_operator_amd", os.path.basename(out))
    # hipBLASLt for the large-M prefill GEMM (csrc/runtime/blas.cpp): torch's copy when present
    # (one instance per process), else the ROCm one
    tl = _torch_lib()
    torch_has = tl and os.path.exists(os.path.join(tl, "libhipblaslt.so"))
    _link([obj for _, obj, _ in all_], out, ["-lhipblaslt"] + ([] if torch_has else ["-L/opt/rocm/lib"]), "native",
          os.path.join(build_dir, "module.sha256"))
    return out


def stack_target_path() -> str:
    return os.path.join(ROOT, "ollama_operator_amd", "_stack" + _ext_suffix())


def build_stack(verbose: bool = False, force: bool = False) -> str:
    """`ollama_operator_amd/_stack*.so`: the kernels and step executor of layer-list models (csrc/stack) with
    the on-device sampler (csrc/kernels/sampling.hip). Its own small library: a checkout that serves only
    such a model compiles these few files (about a minute), not the quantised-GEMV families of `_C`."""
    os.makedirs(STACK_BUILD, exist_ok=True)
    all_ = units(_stack_sources(), STACK_BUILD, ["-O3"])
    _compile(all_, min(8, len(all_)), verbose, "stack module", force)
    out = stack_target_path()
    _link([obj for _, obj, _ in all_], out, [], "stack module", os.path.join(STACK_BUILD, "module.sha256"))
    return out


def cpu_target_path() -> str:
    return os.path.join(ROOT, "ollama_operator_amd", "_cpu" + _ext_suffix())


def build_cpu(verbose: bool = False) -> str:
    """`ollama_operator_amd/_cpu*.so`: the CPU serving backend (csrc/cpu), host compiler only (no HIP
    runtime dependency, so it loads on a CPU-only node). AVX2 + FMA + F16C baseline, OpenMP threads."""
    import pybind11
    srcs = sorted(glob.glob(os.path.join(CPU_SRC, "*.cpp")))
    hdrs = sorted(glob.glob(os.path.join(CPU_SRC, "*.h")))
    out = cpu_target_path()
    cxx = os.environ.get("CXX", "g++")
    cmd = [cxx, "-O3", "-std=c++17", "-fPIC", "-shared", "-fopenmp", "-mavx2", "-mfma", "-mf16c",
           "-fvisibility=hidden", "-I", CPU_SRC, "-I", pybind11.get_include(), "-I", sysconfig.get_paths()["include"],
           *srcs, "-o", out]
    inputs, record = _hash(*(_read(f) for f in srcs + hdrs), *cmd), os.path.join(ROOT, "build", "cpu.sha256")
    if _current(out, inputs, record):
        return out
    os.makedirs(os.path.dirname(record), exist_ok=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("CPU backend build failed:\n" + " ".join(cmd) + "\n" + r.stdout + r.stderr)
    _record(out, inputs, record)
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
