"""Registers that the dense wide kernels spill, from the metadata of the code objects in the built library.

A visit keeps its whole proposal in registers.  With five label sets loaded at once the float modes spilled 111 vector
registers (G = 4 and 8), and 512 chains of a 3-regular graph of 2000 vertices took up to twice as long as with 70."""
import struct

import msgpack

from treesa_gpu_amd import capi


def kernels(path):
    """{mangled name: metadata} of every gfx950 kernel in a shared library."""
    with open(path, "rb") as f:
        data = f.read()
    out, at = {}, data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, at + 40)
            shentsize, shnum = struct.unpack_from("<HH", data, at + 58)
            for i in range(shnum):
                sec = at + shoff + i * shentsize
                kind, = struct.unpack_from("<I", data, sec + 4)
                off, = struct.unpack_from("<Q", data, sec + 24)
                if kind != 7:  # SHT_NOTE
                    continue
                namesz, descsz, _ = struct.unpack_from("<III", data, at + off)
                desc = at + off + 12 + (namesz + 3 & ~3)
                for k in msgpack.unpackb(data[desc:desc + descsz])["amdhsa.kernels"]:
                    out[k[".name"]] = k
        at = data.find(b"\x7fELF", at + 1)
    return out


def test_dense_wide_kernels_keep_a_visit_in_registers():
    all_k = kernels(capi.LIB_PATH)
    # k_wide<G, MODE, COOP, SUMS = false, SLICE = false>
    dense = {n: k for n, k in all_k.items() if "k_wideILi" in n and n.split("k_wideILi")[1].split("E")[3:5] == ["Lb0", "Lb0"]}
    assert len(dense) == 30, sorted(dense)  # G = 4 .. 64, three modes, one and several workgroups per chain
    worst = {n: k[".vgpr_spill_count"] for n, k in dense.items() if k[".vgpr_spill_count"] > 16}
    assert not worst, worst
