"""Waves a SIMD holds of the kernels whose launch bounds were measured on both sides: the
compiled library's registers have to allow what the comments at the kernels say."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def waves(built, tmp_path_factory):
    """waves(name, template arguments): from the register counts of the gfx950 code object."""
    tools = {t: os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")}
    if not all(os.path.exists(t) for t in tools.values()):
        pytest.skip("the ROCm LLVM tools are not installed")
    d = tmp_path_factory.mktemp("co")
    subprocess.check_call([tools["llvm-objcopy"], "--dump-section", f".hip_fatbin={d}/fat",
                           f"{ROOT}/cuda-fabipb_amd/lib/libfabipb_hip.so", f"{d}/rest"])
    subprocess.check_call([tools["clang-offload-bundler"], "--unbundle", "--type=o", f"--input={d}/fat",
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={d}/co"])
    notes = subprocess.check_output([tools["llvm-readelf"], "--notes", f"{d}/co"], text=True)
    regs = {}
    for k in notes.split("- .agpr_count:")[1:]:
        name = re.search(r"\.symbol: +(\S+)\.kd", k)
        regs[name[1]] = int(re.search(r"\.vgpr_count: +(\d+)", k)[1])   # accumulation registers included

    def of(name, args):
        hit = [v for s, v in regs.items() if s.startswith(f"_Z{len(name)}{name}{args}")]
        assert len(hit) == 1, (name, args, hit)
        return min(8, 512 // (-(-hit[0] // 8) * 8))
    return of


@pytest.mark.parametrize("name,args,want", [
    ("k_near_apply", "IdE", 5), ("k_near_apply", "IfE", 8),
    ("k_near_mix32", "ILb0E", 5),
    ("k_energy_wave", "ILi8ELi0EfE", 4), ("k_energy_wave", "ILi9ELi0EfE", 4),
    ("k_energy_wave", "ILi8ELi4EdE", 2), ("k_energy_wave", "ILi9ELi4EdE", 2),
])
def test_waves_per_simd(waves, name, args, want):
    assert waves(name, args) == want
