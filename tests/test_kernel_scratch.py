"""No kernel of the library keeps private arrays in scratch memory: a lambda
that the compiler does not inline, or an array it cannot keep in registers,
turns a kernel's operand fragments into memory traffic without any error (the
few-rows kernel over FP8 weights and f32 rows ran 4 times slower that way).
Read from the metadata of the code objects built here."""

import struct

import msgpack

import lightx2v_hip as H

NT_AMDGPU_METADATA = 32


def _kernels():
    data = open(H.LIB_PATH, "rb").read()
    at = data.find(b"\x7fELF", 4)  # (the first is the library itself)
    while at >= 0:
        phoff, = struct.unpack_from("<Q", data, at + 0x20)
        phentsize, phnum = struct.unpack_from("<HH", data, at + 0x36)
        for i in range(phnum):
            ptype, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + i * phentsize)
            if ptype != 4:  # PT_NOTE
                continue
            p, end = at + off, at + off + size
            while p < end:
                nlen, dlen, kind = struct.unpack_from("<III", data, p)
                desc = p + 12 + (nlen + 3) // 4 * 4
                if kind == NT_AMDGPU_METADATA:
                    yield from msgpack.unpackb(data[desc:desc + dlen])["amdhsa.kernels"]
                p = desc + (dlen + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)


def test_no_kernel_uses_scratch_memory():
    size = {k[".name"]: k[".private_segment_fixed_size"] for k in _kernels()}
    assert len(size) > 100 and any("k_gemm_rows_w16" in n for n in size)
    assert not {n: s for n, s in size.items() if s}
