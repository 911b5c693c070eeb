"""Scratch memory of the tile kernels, as the built library's own kernel descriptors state it.

The 128-wide kernels use every register there is.  A value the compiler spills inside their tile loops comes back behind a wait
for all tile loads in flight; the few bytes allowed here are written and read outside those loops (once per work item or
walked head).  What exceeds them is listed, with what it is."""
import struct
import subprocess

import pytest


def _code_objects(path):
    """The gfx950 ELF images inside the library's offload bundles."""
    data = open(path, "rb").read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + name_len]
            entry += 24 + name_len
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _metadata(elf):
    msgpack = pytest.importorskip("msgpack")
    section_at, = struct.unpack_from("<Q", elf, 40)
    section_size, sections = struct.unpack_from("<HH", elf, 58)
    for n in range(sections):
        kind, = struct.unpack_from("<I", elf, section_at + n * section_size + 4)
        offset, size = struct.unpack_from("<QQ", elf, section_at + n * section_size + 24)
        at = offset
        while kind == 7 and at < offset + size:                      # SHT_NOTE
            name_len, length, note = struct.unpack_from("<III", elf, at)
            start = at + 12 + (name_len + 3) // 4 * 4
            if note == 32 and elf[at + 12:at + 18] == b"AMDGPU":      # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[start:start + length])["amdhsa.kernels"]
            at = start + (length + 3) // 4 * 4


@pytest.fixture(scope="module")
def scratch(fa):
    kernels = {}
    for elf in _code_objects(fa.LIB_PATH):
        for k in _metadata(elf):
            kernels[k[".name"]] = k[".private_segment_fixed_size"]
    names = subprocess.run(["c++filt"], input="\n".join(kernels), capture_output=True, text=True, check=True).stdout.split("\n")
    table = {}
    for name, size in zip(names, kernels.values()):
        name = name.replace("(anonymous namespace)::", "").replace("void ", "").split("(")[0]
        kind, _, args = name.partition("<")
        table[(kind, tuple(args.rstrip("> ").split(", ")))] = size
    return table


# bytes that any instantiation may have
LIMIT = {"fa_fwd_pipelined": 0, "fa_fwd_decode": 0, "fa_fwd_small": 0}
# (kernel, head dimension, masked, layout, ALiBi, dropout) -> bytes
MORE = {
    ("fa_bwd_dkdv", "128", "true", "1", "false", "true"): 84,          # read once per walked head
    ("fa_bwd_dkdv", "128", "true", "2", "true", "true"): 80,
    # (masked, ALiBi, general, dropout: once per work item)
    ("fa_fwd_pipelined", "128", "true", "false", "true", "false"): 16,
    ("fa_fwd_pipelined", "128", "true", "true", "true", "false"): 20,
    ("fa_fwd_pipelined", "128", "false", "false", "true", "true"): 16,
    ("fa_fwd_pipelined", "128", "false", "true", "true", "true"): 24,
    ("fa_fwd_pipelined", "128", "true", "true", "true", "true"): 16,
    # (row blocks, waves, ALiBi, streaming)
    ("fa_fwd_decode", "128", "1", "4", "true", "false"): 8,
    ("fa_fwd_decode", "128", "1", "4", "true", "true"): 8,
}


@pytest.mark.parametrize("kernel", ["fa_fwd_pipelined", "fa_fwd_decode", "fa_fwd_small", "fa_bwd_dq", "fa_bwd_dkdv", "fa_bwd_dq_from_ds"])
def test_tile_loops_do_not_spill(scratch, kernel):
    seen = {args: size for (kind, args), size in scratch.items() if kind == kernel}
    assert seen
    over = {args: size for args, size in seen.items() if size > max(LIMIT.get(kernel, 24), MORE.get((kernel,) + args[1:6], 0))}
    assert not over, over
