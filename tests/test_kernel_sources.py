"""What no run of a built kernel shows: properties of the kernels' sources and of the code that was built from them."""

import os
import re
import struct
import zlib

import msgpack
import pytest

from kllm_amd import kernels
from kllm_amd.csrc import build

SOURCES = [f for f in sorted(os.listdir(build.HERE)) if f.endswith((".hip", ".hpp")) and "global_load_lds" in open(os.path.join(build.HERE, f)).read()]


@pytest.mark.parametrize("name", SOURCES)
def test_loads_into_lds_are_waited_for_in_front_of_a_barrier(name):
    """A barrier waits for no load from memory, and what another wave reads behind it has to be in LDS: between a load that goes there by itself
    and the next barrier in the text there is a wait for it, written out (where the barrier is a function's or a loop's, in that text)."""
    text = open(os.path.join(build.HERE, name)).read()
    for load in re.finditer(r"__builtin_amdgcn_global_load_lds", text):
        rest = text[load.end():]
        barrier = re.search(r"__syncthreads\(\)|_barrier\(\)", rest)
        assert barrier is None or not barrier.group().startswith("__sync") or "s_waitcnt" in rest[:barrier.start()], \
            text[:load.start()].count("\n") + 1


def kernels_of(library):
    """What the compiler wrote about the kernels in the library (code objects in offload bundles, their notes): by mangled name."""
    data, at, found = open(library, "rb").read(), -1, {}
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)) >= 0:
        place, (count,) = at + 32, struct.unpack_from("<Q", data, at + 24)
        for _ in range(count if count < 8 else 0):               # (more: the name itself, in host code)
            offset, size, length = struct.unpack_from("<QQQ", data, place)
            target, place = data[place + 24:place + 24 + length], place + 24 + length
            if b"gfx950" not in target:
                continue
            elf = data[at + offset:at + offset + size]
            (sections,), (step, number) = struct.unpack_from("<Q", elf, 0x28), struct.unpack_from("<HH", elf, 0x3A)
            for i in range(number):
                kind, = struct.unpack_from("<I", elf, sections + i * step + 4)
                note, end = struct.unpack_from("<QQ", elf, sections + i * step + 0x18)
                end += note
                while kind == 7 and note < end:                  # notes
                    name, text, type_ = struct.unpack_from("<III", elf, note)
                    note += 12 + (name + 3) // 4 * 4
                    if type_ == 32:
                        found.update((k[".name"], k) for k in msgpack.unpackb(elf[note:note + text])["amdhsa.kernels"])
                    note += (text + 3) // 4 * 4
    return found


@pytest.mark.parametrize("kernel,instances", [("attn_latent_mfma_kernel", 7), ("attn_f32_decode_kernel", 4), ("attn_decode_mfma_kernel", 60)])
def test_kernels_whose_registers_all_fit(kernel, instances):
    """Instances that hold a round's operands in registers, up to all 512 of a lane: none of them goes by way of memory."""
    own = [k for name, k in kernels_of(build.ensure_built()).items() if kernel in name]
    assert len(own) >= instances
    assert not [(k[".name"], k[".vgpr_spill_count"]) for k in own if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]


def test_the_interface_and_its_version_move_together():
    """A library of another interface is refused by its version and not by a missing symbol or a wrong argument: who changes a declaration raises the
    version (kernels.ABI_VERSION and kllm_abi_version) and writes both down here."""
    text = re.sub(r"/\*.*?\*/|//[^\n]*", "", open(os.path.join(build.HERE, "kllm_kernels.h")).read(), flags=re.S)
    declared = sorted(" ".join(d.split()) for d in re.findall(r"^[a-z]\w*[\w \*]*\bkllm_\w+\([^;{]*\);", text, re.S | re.M))
    assert (kernels.ABI_VERSION, len(declared), zlib.crc32("\n".join(declared).encode())) == (24, 103, 1960918298)
