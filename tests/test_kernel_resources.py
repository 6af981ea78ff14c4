"""What the compiler gave the built kernels, read from libcufk_hip.so: registers, spills and scratch.

A register more can cost a wave per SIMD and a spill a round trip through memory in the hottest loop,
and neither shows in a result.  The library's code objects (one offload bundle per translation unit)
carry the figures in their metadata note.
"""

from __future__ import annotations

import functools
import re
import struct

import pytest

import cufk_amd

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
AMDGPU_METADATA = 32  # note type


def _code_objects(blob):
    for m in re.finditer(re.escape(MAGIC), blob):
        at = m.end()
        (count,) = struct.unpack_from("<Q", blob, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<3Q", blob, at)
            triple = blob[at + 24: at + 24 + length]
            at += 24 + length
            if b"amdgcn" in triple and size:
                yield blob[m.start() + offset: m.start() + offset + size]


def _metadata(elf):
    msgpack = pytest.importorskip("msgpack")
    phoff, = struct.unpack_from("<Q", elf, 32)
    entry, count = struct.unpack_from("<2H", elf, 54)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, phoff + i * entry)
        offset, _, _, size = struct.unpack_from("<4Q", elf, phoff + i * entry + 8)
        at, end = offset, offset + size
        while kind == 4 and at < end:  # PT_NOTE
            name, desc, note = struct.unpack_from("<3I", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if note == AMDGPU_METADATA:
                return msgpack.unpackb(elf[at: at + desc])["amdhsa.kernels"]
            at += (desc + 3) // 4 * 4
    return []


@functools.lru_cache
def _kernels():
    with open(cufk_amd._native.HIP_LIBRARY, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for elf in _code_objects(blob) for k in _metadata(elf)}
    assert len(found) > 100
    return found


def _named(pattern):
    got = {n: k for n, k in _kernels().items() if re.search(pattern, n)}
    assert got, pattern
    return got


def test_double_forwards_of_four_steps_run_four_waves():
    """512 registers per lane of a SIMD: four waves up to 128 each."""
    for name, k in _named(r"26reconstruct_forward_kernelIdLi[1-4]ELi4E").items():
        assert k[".vgpr_count"] + k.get(".agpr_count", 0) <= 128, name


def test_double_forwards_do_not_spill():
    for name, k in _named(r"\d(reconstruct(_\w+)?_forward|long_forward_segments)_kernelId").items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name


def test_saved_backwards_do_not_spill():
    """The exact path of a refused chain shares the registers of the position-based one."""
    for name, k in _named(r"reconstruct(_loss)?_backward(_saved)?_kernelI(f|d|DF16)").items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name
