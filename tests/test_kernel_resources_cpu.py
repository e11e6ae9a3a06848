"""What the compiler gave the built kernels, read from libparas_hip.so's own code objects (metadata notes, instructions)."""
import re
import struct
import subprocess

import msgpack
import pytest

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


OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def instructions(kernel, tmp_path):
    """{address: (mnemonic, branch target or None)} of the kernel whose name holds this text, in the order of the addresses."""
    data = capi.LIB_PATH.read_bytes()
    at = 0
    while (at := data.find(b"\x7fELF\x02\x01\x01\x40", at + 1)) > 0:
        sections, = struct.unpack_from("<Q", data, at + 0x28)
        entsize, count = struct.unpack_from("<HH", data, at + 0x3A)
        elf = data[at:at + sections + entsize * count]
        if kernel.encode() in elf:
            name = re.search(rb"_Z\w*" + kernel.encode() + rb"\w*", elf)[0].decode()
            (tmp_path / "k").write_bytes(elf)
            text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={name}", str(tmp_path / "k")], capture_output=True, text=True, check=True).stdout
            first = int(re.search(r"^([0-9a-f]+) <", text, re.M)[1], 16)
            found = re.findall(r"^\s+(\w+).*// ([0-9A-F]+):[ 0-9A-F]*(?:<\w+\+0x([0-9a-f]+)>)?", text, re.M)
            return {int(where, 16): (op, first + int(to, 16) if to else None) for op, where, to in found}
    raise KeyError(kernel)


@pytest.mark.parametrize("dtype", ["INS_6bf16_tELi1E", "INS_5f16_tELi1E"])
def test_swiglu_forms_no_fp64_value_that_it_does_not_need(dtype, tmp_path):
    """From the first load of a vector to its store, with no element to be evaluated again: the compiler may not move the fp64 formula
    in front of its branch (it did for half of the elements, 8.3 -> 13.6 us over 474 x 14336 in bf16)."""
    code = instructions("swiglu_fwd_vec" + dtype, tmp_path)
    following = dict(zip(code, list(code)[1:]))
    at = next(a for a, (op, _) in code.items() if op == "global_load_dwordx4")
    seen = []
    while code[at][0] != "global_store_dwordx4" and len(seen) < 5000:
        op, to = code[at]
        seen.append(op)
        at = to if op in ("s_branch", "s_cbranch_execz") else following[at]          # (no lane takes the way to the formula)
    assert code[at][0] == "global_store_dwordx4" and seen.count("v_exp_f32_e32") == 8, seen
    assert not [op for op in seen if "f64" in op]
