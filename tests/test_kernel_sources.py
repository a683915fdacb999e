"""Rules the kernel sources keep (CPU: they are read and checked by the compiler, nothing runs)."""

import re
import struct
import subprocess
from pathlib import Path

import pytest

from pypto_amd import _lib, build

CSRC = Path(__file__).resolve().parent.parent / "pypto_amd" / "csrc"
_ASM = re.compile(r"asm volatile\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)")


def _instructions(source: str):
    """The instruction lists of a source's asm statements."""
    for m in _ASM.finditer(source):
        text = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m.group(1)))
        yield [i.strip() for i in re.split(r"\\n(?:\\t)?", text) if i.strip()]


def test_a_load_into_lds_never_follows_its_m0_write_directly():
    """A load with its LDS address in m0 needs one wait state after the scalar instruction that writes m0; the compiler
    adds it to its own code and not inside an asm string, so the string has to hold it."""
    seen = 0
    for path in sorted(CSRC.iterdir()):
        if path.suffix not in (".hip", ".h"):
            continue
        for ins in _instructions(path.read_text()):
            for before, after in zip(ins, ins[1:]):
                if re.match(r"s_\w+ m0,", before):
                    seen += 1
                    assert "lds" not in after, f"{path.name}: '{before}' is followed by '{after}'"
    assert seen >= 1


@pytest.mark.parametrize("name", ["rope.hip", "w8a16.hip"])
def test_slab_sums_keep_the_alignment_of_their_sources(name):
    """A caller's qkv may start at any float; a pointer to a 16-byte vector made from it is reported by the compiler
    where it reaches a parameter that expects the vector's own alignment."""
    r = subprocess.run([build.HIPCC, "--offload-arch=gfx950", "--cuda-device-only", "-fsyntax-only", "-std=c++17",
                        "-Werror=align-mismatch", f"-I{build.INCLUDE}", f"-I{CSRC}", str(CSRC / name)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def _registers(pattern: str, tmp_path) -> dict[str, int]:
    """Vector registers of the built kernels whose mangled name matches, from the notes of the library's code objects."""
    data, magic, found = _lib.LIB_PATH.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    at = data.find(magic)
    while at >= 0:
        (entries,), pos = struct.unpack_from("<Q", data, at + len(magic)), at + len(magic) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            target, pos = data[pos + 24:pos + 24 + length], pos + 24 + length
            code = data[at + offset:at + offset + size]
            if b"gfx950" in target and re.search(pattern.encode(), code):
                (tmp_path / "code.elf").write_bytes(code)
                notes = subprocess.run([str(Path(build.HIPCC).parent.parent / "llvm/bin/llvm-readelf"), "--notes", str(tmp_path / "code.elf")],
                                       capture_output=True, text=True, check=True).stdout
                for name, count in re.findall(r"\.name:\s+(\S+)[\s\S]*?\.vgpr_count:\s+(\d+)", notes):
                    if re.search(pattern, name):
                        found[name] = int(count)
        at = data.find(magic, at + 1)
    return found


@pytest.mark.parametrize("head_dim", [128, 256])
def test_the_merge_of_few_partitions_leaves_room_for_eight_wavefronts_per_simd(head_dim, tmp_path):
    """Its launches have thousands of rows; the registers of the path for many partitions must not be charged to it."""
    found = _registers(f"attn_reduce_kernelILi{head_dim}E", tmp_path)
    assert found and min(found.values()) <= 64, found


@pytest.mark.parametrize("head_dim", [128, 256])
def test_the_merge_of_many_rows_leaves_room_for_five_wavefronts_per_simd(head_dim, tmp_path):
    """Thousands of rows of more partitions: a kernel that holds two batches of four partials, not of sixteen (512 registers
    over five wavefronts, in granules of eight)."""
    found = _registers(f"attn_reduce_kernelILi{head_dim}ELi4E", tmp_path)
    assert len(found) == 1 and max(found.values()) <= 96, found
