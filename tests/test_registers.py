"""The build's check that no transport kernel spills vector registers
(storm_amd/check_registers.py), on made-up remarks and on those of the build."""
from __future__ import annotations

import importlib.util
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = os.path.join(ROOT, "storm_amd", "check_registers.py")


def remarks(name, spill=0, scratch=0, prefix="/src/kernels.h:7:1: remark: "):
    end = " [-Rpass-analysis=kernel-resource-usage]\n"
    return "".join(prefix + s + end for s in (
        f"Function Name: {name}", "    VGPRs: 90", f"    ScratchSize [bytes/lane]: {scratch}", "    Dynamic Stack: False",
        "    SGPRs Spill: 12", f"    VGPRs Spill: {spill}")) + " 7 | k_transport(\n"


def check(path):
    return subprocess.run([sys.executable, SCRIPT, str(path)], capture_output=True, text=True, timeout=60)


OTHER = remarks("_Z5k_foo", spill=9, scratch=40)


@pytest.mark.parametrize("text,ok", [
    (remarks("_Z11k_transport0") + OTHER, True),
    (remarks("_Z11k_transport0") + remarks("_Z18k_transport_refill1", spill=1), False),
    (remarks("_Z11k_transport0", scratch=4), False),
    (remarks("_Z11k_transport0").replace("VGPRs Spill", "VGPR Spills"), False),  # a compiler that words it another way
    (OTHER, False),
    ("", False)], ids=["clean", "spill", "scratch", "reworded", "no kernel", "nothing"])
def test_check(tmp_path, text, ok):
    (tmp_path / "remarks.txt").write_text(text)
    r = check(tmp_path / "remarks.txt")
    assert (r.returncode == 0) == ok, r.stderr


def test_the_build_has_no_spills():
    path = os.path.join(ROOT, "storm_amd", "_lib", "remarks.txt")
    if not os.path.exists(path):
        pytest.fail("storm_amd/_lib/remarks.txt is not there (run __graft_entry__.build())")
    r = check(path)
    assert r.returncode == 0, r.stderr
    spec = importlib.util.spec_from_file_location("check_registers", SCRIPT)
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    with open(path) as f:
        names = [k for k in m.kernels(f.read()) if "k_transport" in k]
    # two schedules, two precisions, two meshes, four sets of features
    assert len(names) == 32, names
