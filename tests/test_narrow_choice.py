"""When a product takes the small-call form (CPU: the header is compiled for the host and called)."""

import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pypto_amd" / "csrc"
_SOURCE = """
#include "launch_choice.h"
extern "C" int choose_narrow(int m, int n, int k, int dual) {
  int height = 0, splits = 0;
  return pto_hip::choose_narrow(m, n, k, dual != 0, 256, pto_hip::choose_quad(m, n, k, dual != 0, 256, 0, &height, &splits));
}
extern "C" int choose_narrow_splits(int m, int n, int k, int dual) {
  int height = 0, splits = 0;
  const double us = pto_hip::choose_quad(m, n, k, dual != 0, 256, 0, &height, &splits);
  return pto_hip::choose_narrow(m, n, k, dual != 0, 256, us, splits);
}
extern "C" int choose_narrow8(int m, int n, int k, int dual, double tiled_us) { return pto_hip::choose_narrow8(m, n, k, dual != 0, 256, tiled_us); }
extern "C" int beats_skinny(int64_t k, int64_t n, int dual) { return pto_hip::narrow_beats_skinny(k, n, dual != 0); }
"""


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    d = tmp_path_factory.mktemp("narrow")
    (d / "choice.cpp").write_text(_SOURCE)
    so = d / "choice.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "choice.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.choose_narrow8.argtypes = [C.c_int] * 4 + [C.c_double]
    lib.beats_skinny.argtypes = [C.c_int64, C.c_int64, C.c_int]
    return lib


# (m, n, k, pair): tile, the fastest of the measured ones or within 6 % of it
@pytest.mark.parametrize("m,n,k,dual,tiles", [(128, 1024, 512, 1, (1,)), (128, 512, 1024, 0, (1,)), (128, 2048, 1024, 1, (2,)), (512, 512, 1024, 0, (2,)),
                                              (512, 2048, 1024, 1, (4,)), (512, 2048, 2048, 0, (4,)), (40, 512, 512, 0, (1,)), (1024, 512, 512, 0, (3,))])
def test_small_products_take_the_measured_tile(choice, m, n, k, dual, tiles):
    assert choice.choose_narrow(m, n, k, dual) in tiles


def test_large_products_keep_the_tiled_form(choice):
    """Where reading every operand once per tile costs more than the chain it shortens."""
    for m, n, k, dual in ((1024, 2048, 1024, 1), (512, 3584, 1024, 1), (96, 1536, 4096, 0), (256, 2048, 5632, 0), (40, 14336, 4096, 1),
                          (333, 14336, 4096, 1), (2048, 11008, 4096, 1), (2048, 4096, 11008, 0), (1 << 20, 8192, 8192, 0)):
        assert choice.choose_narrow(m, n, k, dual) == 0, (m, n, k, dual)


def test_products_that_measured_slower_in_a_block_keep_the_tiled_form(choice):
    """Ragged channels of a pair, a pair's weights beyond 8 MB, a tiled single product of two or three k splits."""
    for m, n, k, dual in ((65, 4408, 1216, 1), (195, 3680, 1096, 1), (114, 3672, 936, 1), (36, 3928, 1008, 1), (208, 3904, 1216, 1), (232, 4032, 1152, 1),
                          (299, 3264, 1088, 1), (733, 1024, 2176, 0), (894, 768, 1664, 0), (984, 768, 1856, 0)):
        assert choice.choose_narrow_splits(m, n, k, dual) == 0, (m, n, k, dual)
    for m, n, k, dual in ((128, 1024, 512, 1), (128, 512, 1024, 0), (512, 2048, 1024, 1), (931, 832, 1664, 0), (120, 3264, 896, 1), (262, 680, 2408, 0)):
        assert choice.choose_narrow_splits(m, n, k, dual) > 0, (m, n, k, dual)


def test_up_to_32_rows_only_small_weights(choice):
    assert choice.beats_skinny(512, 1536, 1) and choice.beats_skinny(2048, 768, 0) and choice.beats_skinny(1024, 1024, 0)
    assert not choice.beats_skinny(768, 2048, 1) and not choice.beats_skinny(2048, 1024, 0) and not choice.beats_skinny(1 << 29, 1 << 29, 1)


# (m, n, k, pair): the tiled GEMM's measured us and the fastest measured tile of the form (0: none)
@pytest.mark.parametrize("m,n,k,dual,us,tile", [(8, 1024, 512, 1, 7.7, 1), (128, 512, 1024, 0, 11.5, 1), (64, 2816, 768, 1, 8.9, 2), (512, 1024, 512, 1, 8.0, 3),
                                                (192, 768, 2816, 0, 14.0, 2), (512, 2816, 1024, 1, 12.4, 0), (64, 5120, 13824, 0, 25.6, 0),
                                                (8, 11008, 4096, 1, 22.4, 0), (2048, 4096, 11008, 0, 93.0, 0)])
def test_small_e4m3_products_take_the_measured_tile(choice, m, n, k, dual, us, tile):
    assert choice.choose_narrow8(m, n, k, dual, us) == tile
