"""The complex forms of the general line kernel keep their elements in
registers: no scratch memory in the plain lines and the four-step passes, and
in Bluestein lines no more than the few registers a radix of 17 is over.  Reads
the metadata of the objects that the build leaves; skipped where there are none."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "rocket-fft_amd", "_build")
LLVM = "/opt/rocm/llvm/bin"


def spills(obj, tmp):
    """{(type, operation, form): spilled vector registers} of an object's k_lines."""
    fat, code = str(tmp / "fat"), str(tmp / "code")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", obj,
                    str(tmp / "copy.o")], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}"], check=True)
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", code], check=True,
                           capture_output=True, text=True).stdout
    found = re.findall(r"\.name:\s+\S*k_linesI([fd])Li(\d+)ELi(\d+)E.*?\.vgpr_spill_count:\s+(\d+)",
                       notes, re.S)
    return {(t, int(op), int(form)): int(n) for t, op, form, n in found}


@pytest.mark.parametrize("name,most", [("lines_c2c", {"f": 0, "d": 0}),
                                       ("lines_blue", {"f": 48, "d": 128})])
def test_line_kernels_stay_in_registers(name, most, tmp_path):
    obj = os.path.join(BUILD, name + ".o")
    if not os.path.exists(obj) or not os.path.exists(f"{LLVM}/clang-offload-bundler"):
        pytest.skip("no built objects here")
    got = spills(obj, tmp_path)
    assert len(got) >= 4
    for (t, op, form), n in got.items():
        assert n <= most[t], f"{name}: {t} operation {op} form {form} spills {n} registers"
