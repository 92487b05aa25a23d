"""CPU: the decisions of the schedule build on device memory
(subsweep_amd/csrc/memory_plan.h, compiled here with the host compiler)."""

import ctypes as C
import pathlib
import shutil
import subprocess

import pytest

HEADER = pathlib.Path(__file__).parent.parent / "subsweep_amd" / "csrc" / "memory_plan.h"
SOURCE = f"""
#include "{HEADER}"
extern "C" {{
int64_t state_bytes(int64_t n, int64_t dn, int64_t dp, int64_t rs) {{ return ssw::state_bytes(n, dn, dp, rs); }}
int64_t offset_bytes(int64_t dn, int64_t dp, int64_t rs) {{ return ssw::offset_bytes(dn, dp, rs); }}
int cones_fit(int64_t tiles, int64_t later, int64_t free) {{ return ssw::cones_fit(tiles, later, free); }}
}}
"""
MB = 1 << 20
GB = 1 << 30


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(d / "plan.cpp"), "-o", str(d / "plan.so")],
                   check=True)
    lib = C.CDLL(str(d / "plan.so"))
    for f in (lib.state_bytes, lib.offset_bytes):
        f.restype, f.argtypes = C.c_int64, [C.c_int64] * (4 if f is lib.state_bytes else 3)
    lib.cones_fit.restype, lib.cones_fit.argtypes = C.c_int, [C.c_int64] * 3
    return lib


@pytest.mark.parametrize("tiles,later,free,fits", [
    (4 * MB, 1 * MB, 7 * MB, True),             # a small grid on a nearly full device
    (4 * MB, 1 * MB, 5 * MB, False),
    (0, 0, 1 * MB, True),
    (150 * GB, 20 * GB, 182 * GB, True),        # the largest: 1/16 of what it needs is left
    (150 * GB, 20 * GB, 180 * GB, False),
    (150 * GB, 0, 160 * GB, True),              # its state is there already (a rotation)
    (150 * GB, 0, 0, False),
])
def test_cones_fit(plan, tiles, later, free, fits):
    assert bool(plan.cones_fit(tiles, later, free)) == fits


@pytest.mark.parametrize("rs", [4, 8])
def test_later_allocations(plan, rs):
    n, d, per = 1000, 16, 100
    state = plan.state_bytes(n, n * d, per * d, rs)
    assert state == 2 * n * d * rs + per * d * rs + n * (80 + 2 * rs + 4)
    assert plan.offset_bytes(n * d, per * d, rs) == (n + per) * d * rs
