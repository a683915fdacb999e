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
extern "C" void choose_quad(int m, int n, int k, int dual, int64_t num_cu, int forced, int* height, int* splits) {
  pto_hip::choose_quad(m, n, k, dual != 0, num_cu, forced, height, splits);
}
extern "C" int64_t partition_align(int64_t pairs, int64_t max_ctx, int64_t block, int64_t bytes_per_part, int64_t scratch) {
  return pto_hip::attn_partition_align(pairs, max_ctx, block, 256, bytes_per_part, scratch);
}
extern "C" int64_t partition_align_shape(int64_t pairs, int64_t max_ctx, int64_t block, int64_t rows, int64_t head_dim, int e4m3, int64_t wg_parts) {
  return pto_hip::attn_partition_align(pairs, max_ctx, block, 256, pairs * rows * (head_dim + 2) * 4, 32 << 20, rows, head_dim, e4m3 != 0, wg_parts);
}
extern "C" int64_t e4m3_partition(int64_t pairs, int64_t max_ctx, int64_t bytes_per_part, int64_t scratch, int64_t plain) {
  return pto_hip::attn_e4m3_partition_tokens(pairs, max_ctx, 256, 8, bytes_per_part, scratch, plain);
}
extern "C" int blocked_row(int id, int rows) { return pto_hip::blocked_row(id, rows); }
extern "C" int stream_ahead(int m, int k, int n, int dual, int w16) { return pto_hip::stream_rows_ahead(m, k, n, dual != 0, w16 != 0, 256); }
extern "C" int stream_splits(int k, int n, int dual) { return pto_hip::stream_splits(k, n, dual != 0, 256); }
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
    lib.e4m3_partition.restype = lib.partition_align.restype = C.c_int64
    lib.partition_align.argtypes = [C.c_int64] * 5
    lib.e4m3_partition.argtypes = [C.c_int64] * 5
    lib.partition_align_shape.restype = C.c_int64
    lib.partition_align_shape.argtypes = [C.c_int64] * 5 + [C.c_int, C.c_int64]
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


def _quad(lib, m, n, k, dual, forced=0):
    height, splits = C.c_int(-1), C.c_int(-1)
    lib.choose_quad(m, n, k, int(dual), C.c_int64(256), forced, C.byref(height), C.byref(splits))
    return height.value, splits.value


def test_tile_choice_takes_the_eight_wavefront_form_only_where_its_costs_hold(choice):
    """Height 0 stands for the direct eight-wavefront loop; with k ending in half a 64-row tile that form would stage
    its tiles through registers, at other costs, while the four-wavefront forms take such k as they are."""
    seen = 0
    for m in (65, 130, 257, 300, 400, 643, 900, 1300, 2459, 4000):
        for n in (256, 1024, 3072, 4096, 6144, 6656):
            for k in (32, 96, 512, 544, 1056, 3680, 4096, 4128, 6816, 11008):
                for dual in (False, True):
                    height, splits = _quad(choice, m, n, k, dual)
                    assert 0 <= height <= 4 and 1 <= splits <= 16
                    assert splits == 1 or k >= 4 * 64 * splits
                    if height == 0:
                        seen += 1
                        assert k % 64 == 0 and not dual and m % 256 != 0, (m, n, k)
                    for forced in (1, 2, 3, 4):
                        assert _quad(choice, m, n, k, dual, forced)[0] == forced
    assert seen > 0


def test_tile_choice_on_ragged_columns(choice):
    """Columns or k that end inside a tile are never for the eight-wavefront form, whose loop would stage its tiles through registers."""
    for m in (33, 257, 400, 900, 2459):
        for n, k in ((8, 8), (1000, 1096), (4160, 4096), (2056, 6008), (25952, 7720)):
            for dual in (False, True):
                height, splits = _quad(choice, m, n, k, dual)
                assert 1 <= height <= 4 and 1 <= splits <= 16 and (splits == 1 or k >= 4 * 64 * splits)


@pytest.mark.parametrize("m,n,k", [(1800, 13824, 5120), (3000, 22016, 8192), (2709, 10752, 4096)])
def test_tile_choice_takes_tall_tiles_over_many_rounds(choice, m, n, k):
    """Gate/up passes that measured ahead of every other height on 256-row tiles, by 2 to 9 %."""
    assert _quad(choice, m, n, k, True)[0] == 4


@pytest.mark.parametrize("k", [11008, 14336])
def test_tile_choice_avoids_splits_on_the_same_memory_channels(choice, k):
    """64 rows of a k x 4096 product: splits of 1024 k rows start 8 MiB apart and measured 6 to 18 % behind others."""
    _, splits = _quad(choice, 64, 4096, k, False)
    assert -(-k // (splits * 64)) * 64 % 1024 != 0


def test_e4m3_partitions_cover_the_table_within_the_workgroup_form(choice):
    """Never fewer partitions than a 16-bit cache gets; more only as far as one workgroup's wavefronts and the fixed scratch
    area go; otherwise that rule's own length."""
    scratch = 32 << 20
    for batch in (1, 32, 40, 97, 160, 255, 4000):
        for hkv, group in ((8, 1), (8, 4), (8, 16), (64, 8)):
            pairs = batch * hkv
            if pairs < 256:
                continue
            bytes_per_part = pairs * group * 130 * 4
            for max_ctx in (32, 500, 1024, 1400, 1536, 1537, 2047, 2048, 2049, 2200, 3000, 4096, 6000, 8192, 14000, 32768):
                plain = min(2048, -(-max_ctx // -(-512 // pairs)))
                tokens = choice.e4m3_partition(pairs, max_ctx, bytes_per_part, scratch, plain)
                before, parts = -(-max_ctx // plain), -(-max_ctx // tokens)
                assert parts >= before
                if parts == before:
                    assert tokens == plain
                else:
                    assert parts <= 8 and parts * bytes_per_part <= scratch
                    assert max_ctx > 1536 and 2 * tokens > 512
                    if parts < 8 and (parts + 1) * bytes_per_part <= scratch and max_ctx > 1536:
                        assert tokens <= 1024


def test_partition_alignment_divides_the_block(choice):
    """A divisor of the block in whole 32-token chunks, and halved only while there are too few partitions and their partials fit."""
    scratch = 32 << 20
    for block in (16, 32, 48, 64, 96, 128, 192, 256, 320, 512):
        for pairs in (1, 3, 8, 32, 100, 255, 256, 4000):
            for max_ctx in (block, 3 * block, 1536, 12000, 32768):
                for rows in (1, 16, 64):
                    per_part = pairs * rows * 258 * 4
                    align = choice.partition_align(pairs, max_ctx, block, per_part, scratch)
                    assert block % align == 0
                    if align != block:
                        parts = -(-max_ctx // (2 * align))
                        assert align >= 64 and align % 32 == 0 and pairs * parts < 512 and 2 * parts * per_part <= scratch


@pytest.mark.parametrize("pairs,tokens,block,rows,d,e4m3,want", [
    (8, 1536, 128, 4, 128, False, 64), (8, 1536, 128, 16, 128, False, 64), (8, 768, 128, 4, 128, False, 64),
    (160, 256, 128, 16, 128, False, 64), (128, 256, 128, 32, 128, True, 64), (64, 512, 512, 16, 128, False, 128), (8, 256, 256, 64, 128, False, 64),
    (300, 512, 512, 4, 128, False, 256), (440, 256, 256, 1, 128, True, 128), (300, 512, 512, 1, 256, False, 512), (300, 256, 256, 16, 128, False, 256),
    # a second partial per row costs more than the shorter chain gives
    (8, 128, 128, 16, 128, False, 128), (200, 128, 128, 32, 128, False, 128), (100, 512, 128, 8, 256, False, 128), (96, 512, 128, 32, 128, False, 128),
    (160, 384, 128, 32, 128, False, 128), (160, 384, 128, 16, 256, True, 128), (16, 3072, 128, 16, 256, False, 128), (200, 256, 128, 4, 256, False, 128)])
def test_partitions_are_cut_where_the_partials_cost_less_than_the_chain(choice, pairs, tokens, block, rows, d, e4m3, want):
    """Calls that measured 5 % or more ahead with the partition length given here."""
    assert choice.partition_align_shape(pairs, tokens, block, rows, d, int(e4m3), 0) == want


@pytest.mark.parametrize("d,most", [(128, 8), (256, 4)])
def test_partition_alignment_stays_within_the_workgroup_form(choice, d, most):
    """Asked for, that form is kept wherever whole blocks allow it: no cut takes the count past its wavefronts."""
    for pairs in (1, 8, 100, 255):
        for blocks in range(1, 24):
            for block in (64, 128, 256, 512):
                align = choice.partition_align_shape(pairs, blocks * block, block, 8, d, 0, most)
                assert blocks > most or blocks * block // align <= most


@pytest.mark.parametrize("pairs,tokens,split", [
    (256, 2048, True), (256, 4096, True), (320, 4992, True), (512, 3584, True), (640, 2048, True), (768, 3072, True), (1600, 3584, True),
    (256, 8064, False), (448, 6016, False), (320, 8064, False), (400, 6016, False), (1024, 2688, False), (1096, 2048, False), (1600, 2048, False)])
def test_e4m3_partitions_stay_where_the_cus_are_full(choice, pairs, tokens, split):
    """Pairs and tables that measured ahead with more partitions or not."""
    plain = min(2048, -(-tokens // -(-512 // pairs)))
    assert (choice.e4m3_partition(pairs, tokens, pairs * 4 * 130 * 4, 32 << 20, plain) < plain) == split


@pytest.mark.parametrize("m,n,k,want", [(400, 8128, 8192, (2, 2)), (900, 8128, 8192, (2, 1)), (400, 7232, 8192, (2, 2)), (900, 7232, 8192, (2, 1))])
def test_tile_choice_on_ragged_columns_is_not_the_form_that_spills(choice, m, n, k, want):
    """Single passes that measured 27 to 39 % behind the best pair on 256-row tiles."""
    assert _quad(choice, m, n, k, False) == want


def test_rows_of_one_line_are_written_from_few_xcds(choice):
    """Rows of the blocked layout by workgroup: a permutation, and the eight rows of a line on as few XCDs (id mod 8) as their number allows."""
    for rows in range(33, 200):
        row = [choice.blocked_row(i, rows) for i in range(rows)]
        assert sorted(row) == list(range(rows)), rows
        for base in range(0, rows, 64):
            groups = min(rows - base, 64) // 8
            for g in range(groups):
                lines = {i % 8 for i in range(rows) if base + 8 * g <= row[i] < base + 8 * g + 8}
                assert len(lines) <= -(-8 // groups) + (8 % groups != 0), (rows, base, g)
    assert [choice.blocked_row(i, 0) for i in range(32)] == list(range(32))


# (rows, k, channels, 16-bit): behind the tiled GEMM with 129 to 170 slabs of 128 channels and no k split
@pytest.mark.parametrize("m,k,n,w16", [(36, 4096, 8960, 1), (57, 4992, 9472, 1), (52, 3200, 9216, 1), (96, 3072, 10496, 1), (64, 3456, 8640, 1),
                                       (57, 4288, 9600, 0), (64, 4992, 9728, 0), (80, 4096, 10496, 0), (96, 4992, 8960, 0), (65, 4480, 10880, 0)])
def test_pairs_that_leave_a_third_of_the_cus_idle_do_not_stream(choice, m, k, n, w16):
    assert not choice.stream_ahead(m, k, n, 1, w16)


# two k splits; from 171 slabs on; the down projection streams too; few k; int8 of up to 48 rows; a last slab that is not whole
@pytest.mark.parametrize("m,k,n,w16", [(64, 4992, 8192, 1), (64, 4992, 8192, 0), (96, 4096, 11008, 1), (96, 4096, 11008, 0), (48, 4096, 9984, 1),
                                       (54, 3840, 10624, 1), (45, 2112, 8320, 1), (48, 4992, 8960, 0), (64, 4096, 9984, 0), (96, 4224, 9664, 0)])
def test_pairs_that_stay_streamed(choice, m, k, n, w16):
    assert choice.stream_ahead(m, k, n, 1, w16)


def test_streamed_k_splits_fill_the_cus(choice):
    assert [choice.stream_splits(4992, n, 1) for n in (8192, 8320, 5504, 1024)] == [2, 1, 2, 16] and choice.stream_splits(256, 1024, 0) == 1
