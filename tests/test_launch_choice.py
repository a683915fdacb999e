"""The launch shapes the host picks from sizes alone (CPU: the header is compiled for the host and called)."""

import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pypto_amd" / "csrc"

_SOURCE = """
#include "launch_choice.h"
extern "C" int64_t skinny_workgroups(int64_t slabs, int64_t ks, int64_t most, int64_t min_steps) {
  return pto_hip::skinny_workgroups(slabs, ks, most, min_steps);
}
"""


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    (d / "choice.cpp").write_text(_SOURCE)
    so = d / "choice.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "choice.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.skinny_workgroups.restype = C.c_int64
    lib.skinny_workgroups.argtypes = [C.c_int64] * 4
    return lib


def test_skinny_workgroups_keep_the_cus_busy(choice):
    """Long launches put work on at least five CUs in eight, as far as every wavefront keeps its least number of steps;
    no launch has more workgroups than it may or fewer units than workgroups."""
    most, min_steps = 256, 2
    for ks in (1, 2, 8, 31, 48, 64, 65, 80, 128, 160, 448, 1000):
        for slabs in range(1, 700):
            wgs = choice.skinny_workgroups(slabs, ks, most, min_steps)
            units = slabs * ks
            assert 1 <= wgs <= min(most, units), (slabs, ks)
            if slabs <= most and wgs % slabs == 0 and wgs < most:  # whole workgroups per slab
                assert wgs == slabs or ks // (wgs // slabs) >= 4 * min_steps, (slabs, ks)
            if ks >= 64 and units >= most * 4 * min_steps:
                assert wgs * 8 > most * 5 or (ks + wgs // slabs - 1) // (wgs // slabs) <= 8 * min_steps, (slabs, ks, wgs)
