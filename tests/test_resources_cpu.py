"""What the built kernels take of a CU, read from the library's own code objects: kernels that are laid out for a number of workgroups
a CU have to keep within the registers that leaves them, and a compiler that spills to do so undoes what it was for."""
import os
import re
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")


def _notes(elf):
    at, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3A)
    for s in range(count):
        kind, = struct.unpack_from("<I", elf, at + s * size + 4)
        if kind != 7:
            continue
        p, length = struct.unpack_from("<QQ", elf, at + s * size + 0x18)
        end = p + length
        while p < end:
            name, desc, note = struct.unpack_from("<III", elf, p)
            p += 12 + (name + 3 & ~3)
            if note == 32:
                yield msgpack.unpackb(elf[p:p + desc], strict_map_key=False)
            p += desc + 3 & ~3


@pytest.fixture(scope="module")
def kernels():
    """{name with template arguments: (registers, bytes of scratch a lane)}"""
    from dest3d_amd import _lib as L
    if not os.path.exists(L.LIB_PATH):
        from dest3d_amd.build import build
        build(verbose=False)
    lib, magic, found = open(L.LIB_PATH, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    for m in re.finditer(magic, lib):
        o = m.start() + len(magic)
        entries, = struct.unpack_from("<Q", lib, o)
        o += 8
        for _ in range(entries if entries < 8 else 0):
            at, size, n = struct.unpack_from("<QQQ", lib, o)
            target, o = lib[o + 24:o + 24 + n], o + 24 + n
            if b"gfx950" in target and lib[m.start() + at:m.start() + at + 4] == b"\x7fELF":
                for note in _notes(lib[m.start() + at:m.start() + at + size]):
                    for k in note["amdhsa.kernels"]:
                        found[k[".name"]] = (k[".vgpr_count"], k[".private_segment_fixed_size"])
    plain = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.split("\n")
    return {re.sub(r"^void |issm::|\(.*", "", p): found[n] for n, p in zip(found, plain)}


@pytest.mark.parametrize("name,variants,registers,spilled", [
    # rows' gradient, one set a workgroup of 16 waves: two workgroups a CU
    (r"k_interp_rows_grad<[124], (true|false), false>", 4, 64, 0),
    # chunk backward in tile-base form, incomplete tiles: two of four waves
    (r"k_bwd_tile<[234], true, false, (true|false), (true|false), false, (true|false)>", 24, 256, 0),
    (r"k_bwd_tile<[234], false, false, (true|false), false, false, (true|false)>", 12, 256, 0),
    # both directions, and two heads side by side: one workgroup of eight waves
    (r"k_bwd_tile<1[012], (true|false), (true|false), false, false, true, false>", 7, 256, 0),
    (r"k_bwd_tile<(18|19|20), (true|false), (true|false), false, false, (true|false), false>", 18, 256, 0),
    # two groups of four waves: with up to two head tiles two workgroups a CU
    (r"(k_chunk_scan|k_bwd_dx)<2, (true|false), (true|false), (true|false), 2>", 16, 128, 0),
    (r"(k_chunk_scan|k_bwd_dx)<[34], (true|false), (true|false), (true|false), 2>", 32, 256, 0),
    # workgroups of sixteen waves
    (r"(k_layer_end<.*>|k_three_nn_grid<1024, .*>|k_box_dist_fwd<.*>)", 11, 128, 0),
    # generation's backward by whole steps: four workgroups a CU, one form with an address in scratch outside its loops
    (r"k_pgen_bwd<(true|false), true, (true|false), (true|false)>", 8, 128, 12),
    # sums of the distance table's gradient: three, which cost scratch (40 bytes fp32, 12 bf16) and are faster than two without
    (r"k_bds_accum<(true|false)>", 2, 168, 52),
    # two of them a CU, and four of eight
    (r"k_three_nn_grid<(1024, [24]|512, 3)>", 3, 64, 0),
])
def test_registers_leave_room_for_the_workgroups(kernels, name, variants, registers, spilled):
    hit = {k: v for k, v in kernels.items() if re.fullmatch(name, k)}
    assert len(hit) == variants
    for k, (r, scratch) in hit.items():
        assert r <= registers and scratch <= spilled, (k, r, scratch)
    assert sum(scratch for _, scratch in hit.values()) == spilled
