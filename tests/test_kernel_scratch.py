"""What the built library's kernels need of scratch memory, from their code object's metadata: a tile
keeps its cells in registers on every path, the integer one for large values included.  (A path that
saves or spills them moves 85 KB a tile: the products and closures of large values took up to 2.2
times as long.)"""

import os
import struct

import pytest

import fastapsp_amd as fa

msgpack = pytest.importorskip("msgpack")


def kernel_metadata():
    """The metadata of every gfx950 kernel of the library, by symbol."""
    if not os.path.exists(fa.LIB_PATH):
        pytest.skip("library not built")
    blob = open(fa.LIB_PATH, "rb").read()
    out, at = {}, blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (count,), p = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, p)
            triple, p = blob[p + 24:p + 24 + n], p + 24 + n
            if b"gfx950" in triple and size:
                out.update(elf_kernels(blob[at + off:at + off + size]))
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return out


def elf_kernels(elf):
    (shoff,), (shentsize, shnum) = struct.unpack_from("<Q", elf, 0x28), struct.unpack_from("<HH", elf, 0x3A)
    out = {}
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if note == 32 and elf[off + 12:off + 18] == b"AMDGPU":
                for k in msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]:
                    out[k[".name"]] = k
            off = desc + (descsz + 3) // 4 * 4
    return out


# bytes a lane: a few words beside the loops at most (fw_rest's 128 x 128 form is left out where it also
# closes the next diagonal block, in a function of its own)
@pytest.mark.parametrize("kernel", ["minplus_gemm_kernel", "minplus_parts_kernel", "hidx_cross_kernel",
                                    "fw_pair128_kernel", "fw_rest_kernelILi8ELb0E",
                                    "fw_rest_kernelILi4E", "fw_panel_kernel", "bidx_expand_kernel",
                                    "bidx_block_kernelILi4ELi4E"])
def test_tiles_stay_in_registers(kernel):
    found = {n: k[".private_segment_fixed_size"] for n, k in kernel_metadata().items() if kernel in n}
    assert found
    assert all(size <= 48 for size in found.values()), found
