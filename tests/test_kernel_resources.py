"""Kernels that keep their lanes' state in registers: none of those of the solve and the searches has
scratch memory (registers that did not fit the launch's lanes, or arrays with an index known late), in the code
objects that the build left."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = os.environ.get("ROCM_PATH", "/opt/rocm") + "/llvm/bin/"


@pytest.mark.parametrize("source,kernel", [("k_solver", "k_sweeps_blocked"), ("k_solver", "k_pgs"),
                                           ("k_solver", "k_colour_run"), ("k_position", "k_position"),
                                           ("k_ccd", "k_ccd_events"), ("k_broadphase", "k_search")])
def test_no_scratch(tmp_path, source, kernel):
    obj = os.path.join(ROOT, "nphysics_amd", "_build", source + ".o")
    tools = [LLVM + t for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]
    if not all(map(os.path.exists, tools + [obj])):
        pytest.skip("no build objects or no ROCm tools")
    fat, co = str(tmp_path / "fat"), str(tmp_path / "co")
    subprocess.check_call([tools[0], "--dump-section", ".hip_fatbin=" + fat, obj, str(tmp_path / "o")])
    subprocess.check_call([tools[1], "--unbundle", "--type=bc", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                           "--input=" + fat, "--output=" + co])
    notes = subprocess.run([tools[2], "--notes", co], capture_output=True, text=True, check=True).stdout
    found = re.findall(r"\.name:\s+(\S*" + kernel + r"\S*)\n\s+\.private_segment_fixed_size:\s+(\d+)", notes)
    assert found
    assert {n: int(b) for n, b in found if int(b)} == {}
