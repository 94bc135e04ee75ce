"""What the compiler made of the tiled GEMM kernels, read from the metadata of the objects that the library was linked
from (mcw_cppamp_torch_amd/build/, left by build.py)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "mcw_cppamp_torch_amd", "build")
LLVM = "/opt/rocm/llvm/bin"
TILES = ["128x128", "192x128", "64x256", "128x256", "256x128", "64x64", "64x128", "96x128", "32x128", "64x64k4"]


def kernels(obj, tmp_path):
    """{kernel symbol: its metadata} of the gfx950 code in an object."""
    code = str(tmp_path / "code.o")
    fat = str(tmp_path / "fatbin")
    subprocess.check_call([LLVM + "/llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, obj, str(tmp_path / "copy.o")])
    subprocess.check_call([LLVM + "/clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + code,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
    notes = subprocess.check_output([LLVM + "/llvm-readelf", "--notes", code], text=True)
    found = {}
    for part in re.split(r"(?=\n  - \.agpr_count:)", notes)[1:]:
        name = re.search(r"\n +\.name: +(\S+)", part).group(1)
        found[name] = {k: int(v) for k, v in re.findall(r"\n +(?:- )?\.(\w+): +(\d+)(?=\n)", part)}
    return found


@pytest.mark.parametrize("tile", TILES)
def test_tiled_gemm_kernels_keep_their_registers(tile, tmp_path):
    """Accumulators and the operands of a step fill most of the register file: what spills goes through memory once per
    lane, in the loop or around every store.  At most two registers (offsets used once per tile, of the kernels that
    gather single floats along the reduction) may."""
    obj = os.path.join(BUILD, "gemm_fast_%s.o" % tile)
    if not os.path.exists(obj):
        pytest.skip("the library was not built here")
    if not os.path.exists(LLVM + "/clang-offload-bundler"):
        pytest.skip("no ROCm LLVM tools")
    found = kernels(obj, tmp_path)
    assert len(found) >= 6 and all("gemm_fast_kernel" in name or "gemm_pair_kernel" in name for name in found)
    assert any("gemm_pair_kernel" in name for name in found) == (tile == "64x64k4")
    spilled = {name: k["vgpr_spill_count"] for name, k in found.items() if k["vgpr_spill_count"] > 2}
    assert not spilled, spilled
