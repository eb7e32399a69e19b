"""No kernel of the library puts registers off to memory, but for the per-point backward kernel with one hit per layer, distortion
and several views, where 28 bytes a lane are faster than the registers of four waves. Read from the notes the compiler leaves in
the library built here."""
import os
import re
import subprocess

import pytest

from vet_amd import build

LLVM = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]


@pytest.mark.skipif(not all(map(os.path.exists, TOOLS)), reason="no LLVM tools")
def test_scratch_memory_of_every_kernel(tmp_path):
    if not os.path.exists(build.LIB_PATH):
        build.build_library(verbose=False)
    objcopy, bundler, readelf = TOOLS
    fat, code = str(tmp_path / "fat.bin"), str(tmp_path / "code.elf")
    subprocess.run([objcopy, "--dump-section", f".hip_fatbin={fat}", build.LIB_PATH, str(tmp_path / "rest.so")], check=True)
    subprocess.run([bundler, "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={fat}", f"--output={code}"], check=True)
    notes = subprocess.run([readelf, "--notes", code], check=True, capture_output=True, text=True).stdout
    found = {}
    for kernel in notes.split("- .agpr_count:")[1:]:
        found[re.search(r"\.name:\s+(\S+)", kernel).group(1)] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1))
    assert len(found) > 50 and any("gather_point_gradients" in k for k in found)
    allowed = re.compile(r"gather_point_gradients_kernelILi\dELi1ELb1ELb1E")  # <channels, one hit, distortion, several views>
    beyond = {k: v for k, v in found.items() if v > (28 if allowed.search(k) else 0)}
    assert not beyond, beyond
