"""What the compiler gave the built kernels, read from the metadata notes of libparas_hip.so's own code objects."""
import struct

import msgpack

import capi


def kernels():
    """The kernel records of every AMDGPU ELF embedded in the library (NT_AMDGPU_METADATA notes, msgpack)."""
    data = capi.LIB_PATH.read_bytes()
    at = 0
    while (at := data.find(b"\x7fELF\x02\x01\x01\x40", at + 1)) > 0:
        phoff, = struct.unpack_from("<Q", data, at + 0x20)
        phentsize, phnum = struct.unpack_from("<HH", data, at + 0x36)
        for i in range(phnum):
            kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + i * phentsize)
            p, end = at + off, at + off + size
            while kind == 4 and p + 12 <= end:                       # PT_NOTE
                name, desc, tag = struct.unpack_from("<III", data, p)
                body = p + 12 + (name + 3) // 4 * 4
                if tag == 32:
                    yield from msgpack.unpackb(data[body:body + desc])["amdhsa.kernels"]
                p = body + (desc + 3) // 4 * 4


def test_fp32_attention_keeps_its_operands_in_registers():
    """The key loop of the one-pass fp32 kernel runs out of registers at large head sizes if operands are requested
    ahead of time there, or if turns that a mask closes are handled inside it: no form may spill vector registers."""
    forms = {k[".name"]: k[".vgpr_spill_count"] for k in kernels() if "sdpa_f32_kernel" in k[".name"]}
    assert len(forms) == 39
    assert not any(forms.values()), {n: s for n, s in forms.items() if s}
