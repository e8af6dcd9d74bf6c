"""The launch rules that count compute units (launch_rules.hpp), compiled with g++: on a whole
MI355X (256 CUs) and on partitions of one."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "diffrax_amd" / "csrc"


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None or not Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers are not available")
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text(
        '#include "launch_rules.hpp"\n'
        'extern "C" int alone(long long b, int c) { return dfx::waves_alone(b, c); }\n'
        'extern "C" int fits(long long w, long long b, int k, int c)'
        ' { return dfx::save_times_fit(w, b, k, c); }\n'
        'extern "C" int waves(int p, long long t, int c) { return dfx::mlp_tile_waves(p, t, c); }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    L, I = ctypes.c_longlong, ctypes.c_int
    lib.alone.argtypes, lib.fits.argtypes, lib.waves.argtypes = [L, I], [L, L, I, I], [I, L, I]
    return lib


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_a_simd_per_wave(rules, cus):
    simds = 4 * cus
    assert rules.alone(1, cus) and rules.alone(64 * simds, cus)
    assert not rules.alone(64 * simds + 1, cus)


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_save_times_in_lds(rules, cus):
    row = 66 * 64 * 8   # 64 save times per instance
    assert rules.fits(row, 64 * 4 * cus, 64, cus)           # four waves on a CU: 132 KB
    assert not rules.fits(row, 64 * 5 * cus, 64, cus)       # five: 165 KB
    assert rules.fits(row, 1, 64, cus) and not rules.fits(row, 1, 128, cus)
    assert rules.fits(66 * 8, 10 ** 9, 256, cus)            # times shared by the batch
    assert rules.fits(64 << 10, 64, 64, cus) and not rules.fits((64 << 10) + 8, 64, 64, cus)


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_waves_of_a_tile(rules, cus):
    assert rules.waves(0, cus, cus) == 8 and rules.waves(0, cus + 1, cus) == 4
    assert rules.waves(1, cus, cus) == 8 and rules.waves(1, 10 * cus, cus) == 8
