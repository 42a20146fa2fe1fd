"""What the compiler made of the resident kernels, read from the metadata of the
built objects: their speed rests on the fields and the requested halo staying
in registers, which a few lines of the source steer (empty asm statements, a
never-taken branch) and a compiler may stop honouring without an error."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJ = os.path.join(ROOT, "bh_ringdown_amd", "lib", "obj")
LLVM = "/opt/rocm/llvm/bin"


def kernels(cp, tmp):
    """{(kernel, integrator, built-in rows): scratch bytes a lane} of one object."""
    name = f"teuk_resident_c{cp}.o"
    shutil.copy(os.path.join(OBJ, name), tmp)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", name], cwd=tmp, check=True, capture_output=True)
    device = [f for f in os.listdir(tmp) if f.startswith(name) and "gfx950" in f]
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", device[0]], cwd=tmp, check=True, capture_output=True,
                           text=True).stdout
    out = {}
    for k in notes.split("  - .agpr_count:")[1:]:
        m = re.search(r"\.name:\s+\S*?(k_resident(?:_batch)?)ILi(\d)ELi(\d)ELi(\d+)E", k)
        assert int(m.group(3)) == cp
        out[m.group(1), int(m.group(2)), int(m.group(4))] = int(re.search(r"private_segment_fixed_size:\s+(\d+)", k)[1])
    return out


@pytest.mark.parametrize("cp", [1, 2, 4, 6, 8])
def test_scratch_of_resident_kernels(cp, tmp_path):
    if not os.path.isdir(OBJ) or not os.path.exists(f"{LLVM}/llvm-readelf"):
        pytest.skip("needs the built objects and LLVM's tools")
    found = kernels(cp, str(tmp_path))
    assert len(found) >= 12
    for key, scratch in found.items():
        # (up to 20 spilled registers: rows that are not built in, and RK4's 32-row sweeps of four columns)
        most = 80 if key[2] == 0 or (cp == 8 and key[2] == 32) else 0
        assert scratch <= most, (key, scratch)
