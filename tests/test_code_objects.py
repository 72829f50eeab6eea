"""Register counts of built kernels, from the code objects' metadata (no GPU).

A kernel that shares an instantiation with a form it does not run pays for that
form's registers; these are the ones where it cost waves in flight."""
from __future__ import annotations

import struct

import pytest

from dflash_mlx import _build

msgpack = pytest.importorskip("msgpack")


def _gfx950_objects(data: bytes):
    """The code objects of the clang offload bundles in a linked library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                yield data[at + off:at + off + size]
            p += 24 + n
        at = data.find(magic, at + 8)


def _kernels(elf: bytes):
    """The AMDGPU metadata note's kernels."""
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        sh = shoff + i * entry
        if struct.unpack_from("<I", elf, sh + 4)[0] != 7:  # SHT_NOTE
            continue
        off, _ = struct.unpack_from("<QQ", elf, sh + 24)
        name, desc, _ = struct.unpack_from("<III", elf, off)
        start = off + 12 + (name + 3 & ~3)
        yield from msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]


@pytest.fixture(scope="module")
def registers():
    if not _build.LIB_PATH.exists():
        pytest.skip("library not built")
    return {k[".name"]: k[".vgpr_count"] for o in _gfx950_objects(_build.LIB_PATH.read_bytes())
            for k in _kernels(o)}


def _scan(registers, dk, ahead):
    tail = f"gdn_scan_kernelILi{dk}ELi1ELi1ELb0ELi0ELb0ELb{int(ahead)}E"
    return [v for name, v in registers.items() if tail in name]


@pytest.mark.parametrize("dk,waves", [(128, 7), (192, 5), (256, 4)])
def test_scan_without_loads_ahead_keeps_its_registers(registers, dk, waves):
    """512 registers a SIMD lane in steps of 8: the waves that fit."""
    (plain,) = _scan(registers, dk, False)
    assert 512 // (-(-plain // 8) * 8) >= waves
    assert all(plain < v for v in _scan(registers, dk, True))
    assert len(_scan(registers, dk, True)) == (1 if dk <= 128 else 0)
