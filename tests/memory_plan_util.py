"""subsweep_amd/csrc/memory_plan.h through ctypes (not a test module)."""

import ctypes as C
import pathlib
import shutil
import subprocess

import pytest

HEADER = pathlib.Path(__file__).parent.parent / "subsweep_amd" / "csrc" / "memory_plan.h"
GEOMETRIC, PER_LEVEL, GROUPED, DIRECTIONS = range(4)
PROBLEM = "int64_t n, int64_t f, int64_t per, int64_t d, int64_t l, int fp32, int r"
SOURCE = f"""
#include "{HEADER}"
extern "C" {{
int64_t state_bytes(int64_t n, int64_t dn, int64_t dp, int64_t rs) {{ return ssw::state_bytes(n, dn, dp, rs); }}
int64_t offset_bytes(int64_t dn, int64_t dp, int64_t rs) {{ return ssw::offset_bytes(dn, dp, rs); }}
int cones_fit(int64_t tiles, int64_t later, int64_t free) {{ return ssw::cones_fit(tiles, later, free); }}
int64_t replay_bytes({PROBLEM}) {{ return ssw::replay_bytes({{n, f, per, d, l, fp32 != 0}}, (ssw::Replay)r); }}
int64_t handle_bytes({PROBLEM}) {{ return ssw::handle_bytes({{n, f, per, d, l, fp32 != 0}}, (ssw::Replay)r); }}
}}
"""


def build_plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(d / "plan.cpp"), "-o", str(d / "plan.so")],
                   check=True)
    lib = C.CDLL(str(d / "plan.so"))
    for name, args in (("state_bytes", 4), ("offset_bytes", 3), ("cones_fit", 3), ("replay_bytes", 7),
                       ("handle_bytes", 7)):
        f = getattr(lib, name)
        f.restype, f.argtypes = (C.c_int if name == "cones_fit" else C.c_int64), [C.c_int64] * args
    for f in (lib.replay_bytes, lib.handle_bytes):
        f.argtypes = [C.c_int64] * 5 + [C.c_int, C.c_int]
    return lib
