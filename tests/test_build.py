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
