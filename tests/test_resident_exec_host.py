"""Host execution of the chip-resident time loop's own kernel source
(dn_resident.inc) with checked memory: tests/native/resident_exec.cpp runs
every thread of every workgroup as a fiber under the address and
undefined-behaviour sanitizers, so an access outside a tile's LDS or outside a
plane, or a misaligned vector, ends it.  Every thread shape has to leave the
same bits.  No device is involved."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "denise-black-edition_amd", "csrc")
INC = os.path.join(HERE, "..", "include")

# what g++ does not know, and where the kernel asks for LDS or spins: {text: (replacement, times)}
REWRITE = {
    'asm volatile("" : "+s"(k));': ("", 1),
    'asm volatile("" : "+v"(v));': ("", 2),
    "float __attribute__((ext_vector_type(VX)))": ("HostVec<VX>", 1),
    "typedef Vec<VX> V __attribute__((aligned(4)));": ("typedef HostVecU<VX> V;", 1),
    "extern __shared__ Vec<4> lds_raw[];": ("void *lds_raw = host_lds;", 1),
    "reinterpret_cast<float *>(lds_raw)": ("static_cast<float *>(lds_raw)", 1),
    "        ++spins;\n": ("        ++spins;\n        host_yield();\n", 1),
}
# half-order, physics (1 P/SV, 2 acoustic, 3 VTI, 4 TTI, 5 SH), relaxation mechanisms, 0 forward / 1 adjoint
CASES = [(4, 1, 0, 0), (4, 1, 0, 1), (6, 1, 2, 0), (5, 1, 3, 1), (2, 2, 0, 0), (1, 4, 0, 1), (3, 5, 0, 1), (6, 3, 0, 0)]


def build_and_run(tmp, case):
    f, ph, l, sw = case
    exe = os.path.join(tmp, "exec_%d_%d_%d_%d" % case)
    subprocess.run(["g++", "-O0", "-std=c++17", "-ffp-contract=off", "-w", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", f"-DCF={f}", f"-DCPH={ph}", f"-DCL={l}", f"-DCSW={sw}",
                    "-I", tmp, "-I", CSRC, "-I", INC, os.path.join(HERE, "native", "resident_exec.cpp"),
                    os.path.join(CSRC, "dn_resident_plan.cpp"), "-o", exe], check=True)
    return subprocess.run([exe], capture_output=True, text=True, timeout=600)


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    tmp = str(tmp_path_factory.mktemp("resident_exec"))
    text = open(os.path.join(CSRC, "dn_resident.inc")).read()
    for old, (new, times) in REWRITE.items():
        assert text.count(old) == times, old
        text = text.replace(old, new)
    with open(os.path.join(tmp, "resident_host.inc"), "w") as f:
        f.write(text)
    os.mkdir(os.path.join(tmp, "hip"))
    with open(os.path.join(tmp, "hip", "hip_runtime.h"), "w") as f:
        f.write("typedef void *hipStream_t;\n")
    with ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
        return dict(zip(CASES, pool.map(lambda c: build_and_run(tmp, c), CASES)))


@pytest.mark.parametrize("case", CASES)
def test_loop_stays_in_bounds_and_shapes_agree(runs, case):
    out = runs[case]
    assert out.returncode == 0, out.stderr[-4000:] + out.stdout[-2000:]
    assert "resident loop ok" in out.stdout
