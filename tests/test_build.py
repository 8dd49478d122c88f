"""The native modules build from the tracked sources: every translation unit of `build_native.py`, compiled from a copy that holds
only what git knows, passes the compiler's front end (host and gfx950). Objects in build/ play no part."""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import build_native  # noqa: E402

HIPCC = pytest.mark.skipif(not os.path.exists(build_native.HIPCC), reason="needs hipcc")


def _tracked(folder):
    r = subprocess.run(["git", "ls-files", "-z", folder], cwd=ROOT, capture_output=True, text=True)
    return [f for f in r.stdout.split("\0") if f] if r.returncode == 0 else []


@HIPCC
def test_every_unit_of_the_tracked_sources_compiles(tmp_path, monkeypatch):
    files = _tracked("csrc")
    if not files:
        pytest.skip("no git checkout")
    for f in files:
        dst = tmp_path / f
        dst.parent.mkdir(parents=True, exist_ok=True)
        shutil.copyfile(os.path.join(ROOT, f), dst)
    csrc = str(tmp_path / "csrc")
    for name, value in (("CSRC", csrc), ("CPU_SRC", os.path.join(csrc, "cpu")), ("STACK_SRC", os.path.join(csrc, "stack"))):
        monkeypatch.setattr(build_native, name, value)
    units = build_native.all_units()
    assert len(units) > 30 and all(s.startswith(csrc) and csrc in cmd for s, _, cmd in units)

    def check(unit):
        src, obj, cmd = unit
        cmd = [c for c in cmd if c not in ("-c", "-o", obj)] + ["-fsyntax-only", "-w"]
        r = subprocess.run(cmd, capture_output=True, text=True)
        return os.path.relpath(src, csrc), r.returncode, r.stderr[-2000:]

    with cf.ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 4)) as ex:
        failed = [x for x in ex.map(check, units) if x[1] != 0]
    assert not failed, failed


@pytest.fixture
def small(tmp_path, monkeypatch):
    """A tree of two units over two headers, and a compiler that writes down what it is asked for."""
    csrc = tmp_path / "csrc"
    (csrc / "kernels").mkdir(parents=True)
    (csrc / "kernels" / "a.hip").write_text('#include "k.h"\n')
    (csrc / "b.cpp").write_text("#include <vector>\n")
    (csrc / "kernels" / "k.h").write_text('#include "kernels/deep.h"\n')
    (csrc / "kernels" / "deep.h").write_text("struct P { int x; };\n")
    (tmp_path / "ollama_operator_amd").mkdir()
    for name, value in (("ROOT", str(tmp_path)), ("CSRC", str(csrc)), ("CPU_SRC", str(csrc / "cpu")),
                        ("STACK_SRC", str(csrc / "stack")), ("BUILD", str(tmp_path / "build"))):
        monkeypatch.setattr(build_native, name, value)
    ran = []

    def run(cmd, **kw):
        out = cmd[cmd.index("-o") + 1]
        ran.append(os.path.basename(out))
        with open(out, "w") as f:
            f.write(" ".join(cmd))
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build_native.subprocess, "run", run)

    def build():
        ran.clear()
        build_native.build(jobs=1)
        return sorted(ran)

    return csrc, build


LIB = "_C" + build_native._ext_suffix() + ".tmp"


def _age(path, seconds):
    t = os.path.getmtime(path) + seconds
    os.utime(path, (t, t))


def test_build_decides_by_content(small):
    csrc, build = small
    obj = os.path.join(build_native.BUILD, "kernels_a.hip.o")
    assert build() == [LIB, "b.cpp.o", "kernels_a.hip.o"]
    assert build() == []
    # a header changed, its time and the objects' say otherwise (the objects were touched afterwards)
    (csrc / "kernels" / "deep.h").write_text("struct P { long x; };\n")
    for o in (obj, os.path.join(build_native.BUILD, "b.cpp.o")):
        _age(o, 3600)
    assert build() == ["kernels_a.hip.o"]  # (this compiler's output is the same: nothing to link)
    # a newer time alone is no change
    _age(csrc / "kernels" / "deep.h", 7200)
    assert build() == []
    # an object from elsewhere, newer than everything
    with open(obj, "w") as f:
        f.write("another")
    _age(obj, 9000)
    assert build() == ["kernels_a.hip.o"]
    # a module from elsewhere
    with open(build_native.target_path(), "w") as f:
        f.write("another")
    _age(build_native.target_path(), 9000)
    assert build() == [LIB]


def test_build_follows_flags(small, monkeypatch):
    _, build = small
    build()
    monkeypatch.setattr(build_native, "NO_PK_F32", ["-other"])
    assert build() == [LIB, "kernels_a.hip.o"]
