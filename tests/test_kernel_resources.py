"""CPU checks of what the compiler reports for the built kernels (the AMDGPU
metadata notes of the code objects inside the library)."""
import struct

import msgpack
import pytest

NT_AMDGPU_METADATA = 32


def _kernels(path):
    """name -> metadata of every kernel in the ELF code objects of a library."""
    data = open(path, "rb").read()
    out = {}
    at = data.find(b"\x7fELF", 4)   # (the library itself starts with one)
    while at >= 0:
        e_machine, = struct.unpack_from("<H", data, at + 18)
        if e_machine == 224:        # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, at + 40)
            shentsize, shnum = struct.unpack_from("<HH", data, at + 58)
            for i in range(shnum):
                sh = at + shoff + i * shentsize
                sh_type, = struct.unpack_from("<I", data, sh + 4)
                off, size = struct.unpack_from("<QQ", data, sh + 24)
                if sh_type != 7:    # SHT_NOTE
                    continue
                p, end = at + off, at + off + size
                while p + 12 <= end:
                    nlen, dlen, kind = struct.unpack_from("<III", data, p)
                    desc = p + 12 + (nlen + 3) // 4 * 4
                    if kind == NT_AMDGPU_METADATA and data[p + 12:p + 12 + nlen] == b"AMDGPU\0":
                        md = msgpack.unpackb(data[desc:desc + dlen])
                        out.update({k[".name"]: k for k in md["amdhsa.kernels"]})
                    p = desc + (dlen + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)
    return out


@pytest.fixture(scope="module")
def kernels(yl):
    return _kernels(yl.LIB_PATH)


def test_gemm_kernels_keep_their_registers(kernels):
    # every tile configuration, epilogue and format of the many-token matmul
    # runs its K loop without spilled vector registers
    gemm = {n: k for n, k in kernels.items() if "k_gemm" in n and "k_gemv" not in n}
    assert len(gemm) >= 100
    spilled = {n: k[".vgpr_spill_count"] for n, k in gemm.items() if k[".vgpr_spill_count"]}
    assert not spilled, spilled
