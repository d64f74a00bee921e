"""A slot's instance and triangle (csrc/pbr_slot.h) against integer division on
the host, up to the instance count from which the band kernel leaves a batch
to the tile kernels.  A limit of 2^24 instances must be caught."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "native" / "slot_check.cpp"
HDR = ROOT / "pybatchrender_amd" / "csrc" / "pbr_slot.h"
LIMIT = "constexpr uint32_t kMaxInstances = 1u << 22;"


def _run(tmp: Path, header: Path) -> subprocess.CompletedProcess:
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    cpp = tmp / "slot_check.cpp"
    cpp.write_text(SRC.read_text().replace("../../pybatchrender_amd/csrc/pbr_slot.h", str(header)))
    exe = tmp / "slot_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-o", str(exe), str(cpp)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)


def test_slot_split_matches_division(tmp_path):
    res = _run(tmp_path, HDR)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 10_000_000


def test_larger_limit_is_caught(tmp_path):
    bad = tmp_path / "pbr_slot_bad.h"
    text = HDR.read_text()
    assert LIMIT in text
    bad.write_text(text.replace(LIMIT, LIMIT.replace("22", "24")))
    res = _run(tmp_path, bad)
    assert res.returncode == 1 and res.stdout.startswith("mismatch"), res.stdout


def test_band_dispatch_keeps_the_limit():
    """The band path's plan refuses nodes beyond the limit."""
    plan = (ROOT / "pybatchrender_amd" / "csrc" / "pbr_bands.hip").read_text()
    plan = plan[plan.index("bool bands_plan("):]
    assert "pbr_slot::kMaxInstances" in plan[:plan.index("\n}\n")]
