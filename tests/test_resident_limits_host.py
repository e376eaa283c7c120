"""Host-side check of the chip-resident loop's plans, relaxation mechanisms
included: tests/native/resident_limits.cpp is compiled with g++ against the
library's own dn_resident_plan.cpp and run; no device is involved."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "denise-black-edition_amd", "csrc")
INC = os.path.join(HERE, "..", "include")


def test_resident_limits(tmp_path):
    exe = tmp_path / "resident_limits"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-I", INC,
                    os.path.join(HERE, "native", "resident_limits.cpp"),
                    os.path.join(CSRC, "dn_resident_plan.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr + out.stdout
    assert "resident limits ok" in out.stdout
