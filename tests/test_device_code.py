"""What the compiler cannot keep by itself in the device code of librwkv_hip.so, read from its disassembly (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
REGISTERS = re.compile(r"v(?:\[(\d+):(\d+)\]|(\d+))")


def registers(operand):
    m = REGISTERS.match(operand.strip().lstrip("-|"))
    if not m:
        return set()
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}


def early_matrix_reads(lines):
    """Matrix instructions with fewer than two wait states between a vector instruction and the product that reads its result."""
    found, products = [], 0
    kernel, written = None, []  # written: (wait states since, registers, instruction)
    for line in lines:
        if line.endswith(">:"):
            kernel, written = line.split("<")[1][:-2], []
            continue
        text = line.split("//")[0].strip()
        if not text or not line.startswith("\t"):
            continue
        name, _, rest = text.partition(" ")
        operands = re.split(r",\s*(?![^\[]*\])", rest)
        states, result = 1, set()
        if name.startswith(("v_mfma", "v_smfmac")):
            products += 1
            read = set().union(*[registers(o) for o in operands[1:4]])
            found += [(kernel, w, text) for since, r, w in written if since < 2 and r & read]
        elif name == "s_nop":
            states = int(operands[0], 0) + 1
        elif name.startswith("v_"):
            result = registers(operands[0]) | (registers(operands[1]) if "swap" in name else set())
        written = [(since + states, r, w) for since, r, w in written if since + states < 2]
        if result:
            written.append((0, result, text))
    return found, products


def test_the_check_sees_a_product_that_reads_too_early():
    product = "\tv_mfma_f32_32x32x16_f16 v[2:17], v[54:57], v[34:37], v[2:17]"
    write = "\tv_cvt_f16_i16_sdwa v57, sext(v31) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3"
    for between, early in (([], 1), (["\ts_nop 0"], 1), (["\ts_waitcnt lgkmcnt(0)"], 1), (["\ts_nop 1"], 0), (["\ts_nop 0", "\ts_nop 0"], 0)):
        found, products = early_matrix_reads(["0 <k>:", write, *between, product])
        assert len(found) == early and products == 1


def test_products_wait_for_the_vector_instructions_they_read(tmp_path):
    """gfx950 asks for two wait states between a vector instruction and a matrix instruction that reads its result.  The compiler keeps
    them for its own instructions and does not see those inside an asm block."""
    from rwkv_lightning_cuda_amd import hip
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    library = shutil.copy(hip.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", library], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(f for f in os.listdir(tmp_path) if "gfx950" in f)
    assert objects
    products = 0
    for name in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        found, n = early_matrix_reads(text.splitlines())
        products += n
        assert not found, "%d, the first: %s" % (len(found), found[0])
    assert products > 1000
