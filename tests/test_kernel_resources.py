"""What the compiler gave the kernels of the built library: the send side's select may not go through scratch memory.

Untransformed gradients often hold more candidates than the select has slots for (rows of zeros, a large k), and the exact search
that then runs over a chunk's 64 registers a lane makes up to thirty passes: with some of them spilled it took 1.1 to 1.6 times
as long."""
import struct
import subprocess

import pytest

import bench_profiles

from templar_amd import _lib


def _kernels():
    """{symbol: metadata} of every code object in the library."""
    import msgpack

    data = open(_lib.LIB_PATH, "rb").read()
    out, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, len_id = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24: pos + 24 + len_id].decode()
            pos += 24 + len_id
            if "gfx950" in target and size:
                out.update(_metadata(data[at + off: at + off + size], msgpack))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return out


def _metadata(elf, msgpack):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, _, _, off, size = struct.unpack_from("<IQQQQ", elf, shoff + i * shentsize + 4)
        if kind != 7:  # notes
            continue
        while size > 12:
            len_name, len_desc, note = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (len_name + 3) // 4 * 4
            if note == 32 and elf[off + 12: off + 18] == b"AMDGPU":
                meta = msgpack.unpackb(elf[desc: desc + len_desc], strict_map_key=False)
                return {k[".name"]: k for k in meta["amdhsa.kernels"]}
            step = desc + (len_desc + 3) // 4 * 4 - off
            off, size = off + step, size - step
    return {}


@pytest.mark.parametrize("kernel,count", [("k_encode_topk_pack", 2), ("k_encode_chunk", 8), ("k_topk_rows", 5)])
def test_selects_keep_their_chunk_in_registers(kernel, count):
    found = {name: k for name, k in _kernels().items() if kernel in name}
    assert len(found) >= count, sorted(found)
    for name, k in found.items():
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, (name, k)


def test_profiled_kernels_are_in_the_library():
    names = subprocess.run(["c++filt"], input="\n".join(_kernels()), capture_output=True, text=True, check=True).stdout.splitlines()
    asked = [bench_profiles.kernel_of(S, phase) for S in bench_profiles.SETS.values() for phase in S["phases"]]
    asked += [m[0] for m in bench_profiles.MINER]
    for kernel in set(asked):
        assert any(f"tplr::{kernel}" in n for n in names), kernel
