"""Registers and scratch of the built kernels, read from the library's code objects."""
from __future__ import annotations

import functools
import pathlib
import struct

import msgpack

LIB = (pathlib.Path(__file__).resolve().parent.parent / "qwen_3.5_comfy_prompt_enhancer_amd" / "kernels" /
       "libqlin.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _notes(elf):
    """The descriptors of an ELF64 image's AMDGPU metadata notes."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        end = off + size
        while kind == 7 and off + 12 <= end:  # SHT_NOTE
            nlen, dlen, ntype = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (nlen + 3) // 4 * 4
            if ntype == 32 and elf[off + 12:off + 18] == b"AMDGPU":
                yield elf[desc:desc + dlen]
            off = desc + (dlen + 3) // 4 * 4


@functools.cache
def kernels() -> dict:
    """{mangled name: metadata} of every gfx950 kernel in the library."""
    data = LIB.read_bytes()
    out, at = {}, data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name:
                for d in _notes(data[at + off:at + off + size]):
                    out.update({k[".name"]: k for k in msgpack.unpackb(d)["amdhsa.kernels"]})
        at = data.find(MAGIC, at + 24)
    return out


def _find(part):
    found = [k for n, k in kernels().items() if part in n]
    assert found, part
    return found


def test_small_prefill_tiles_leave_room_for_three_waves():
    """The tiled int8 kernel's small tiles: at most 168 registers, so that three workgroups
    of 4 waves fit a CU (template arguments: weight kind, zeros, epilogue, RB, WNW)."""
    for part in ("Li0ELb0ELi0ELi2ELi1E", "Li0ELb0ELi0ELi3ELi1E", "Li0ELb0ELi1ELi2ELi1E", "Li0ELb0ELi2ELi2ELi1E",
                 "Li1ELb0ELi0ELi2ELi1E", "Li1ELb0ELi1ELi2ELi1E", "Li1ELb0ELi2ELi2ELi1E"):
        for k in _find("prefill_i8_kernelI" + part):
            assert k[".vgpr_count"] <= 168, k[".name"]


def test_prefill_tiles_do_not_spill_in_their_loops():
    """A spilled register that the K loop reloads makes every stage wait for its copies in
    flight.  The few that remain (up to three, W4 gate/up with zeros) are stored and read
    outside it."""
    for k in _find("prefill_i8_kernel"):
        assert k[".vgpr_spill_count"] <= 3, (k[".name"], k[".vgpr_spill_count"])


def test_polling_w4_calls_use_no_scratch():
    """ecall_kernel<W4, polling, jobs, late>: the form of calls without a producer, and of
    three jobs (a single call behind a producer loads its descriptor early, and spills)."""
    for part in ("Lb1ELb1ELi1ELb1E", "Lb1ELb1ELi3ELb0E"):
        for k in _find("ecall_kernelI" + part):
            assert k[".private_segment_fixed_size"] == 0 and k[".sgpr_spill_count"] == 0, k[".name"]
