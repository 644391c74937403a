"""What the kernels' inline assembly relies on and the compiler does not look after: declared
clobbers (source), and, in the code the compiler made of it, the wait states of matrix products
written as assembly and of their results read by assembly. No device call is made here."""

import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "hack-fe30cb28-opus-5-5-ultracode_amd")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _asm_statements():
    for path in sorted(glob.glob(os.path.join(PKG, "csrc", "*"))):
        text = open(path).read()
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\(((?:[^;\"]|\"[^\"]*\")*)\)\s*;", text):
            yield os.path.basename(path), m.group(1)


def test_assembly_declares_what_it_changes():
    """M0 and memory are in the clobbers of every statement that writes them (LDS DMA does both)."""
    seen = 0
    for name, body in _asm_statements():
        code, *operands = body.split(":")
        clobbers = operands[2] if len(operands) > 2 else ""
        if re.search(r"\bm0\b", code):
            assert '"m0"' in clobbers, (name, body)
        if re.search(r"\blds\b|\bds_write|_store_", code):
            seen += 1
            assert '"memory"' in clobbers, (name, body)
    assert seen >= 2


def _regs(text):
    """Registers an operand list names: {("v", 3), ("a", 7), ..}."""
    out = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))\b", text):
        out |= {(kind, r) for r in range(int(lo or one), int(hi or one) + 1)}
    return out


def _kernels(tmp_path, want):
    """{kernel: [(mnemonic, [operand, ..]), ..]} of the library's device code."""
    lib = os.path.join(PKG, "libqlora_amd.so")
    copy = tmp_path / "lib.so"
    copy.write_bytes(open(lib, "rb").read())
    subprocess.run([OBJDUMP, "--offloading", copy.name], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    kernels, body = {}, None
    for obj in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", str(obj)], check=True, capture_output=True,
                              text=True).stdout
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if m:
                body = kernels.setdefault(m.group(1), []) if want in m.group(1) else None
            elif body is not None and line.startswith("\t"):
                op, _, args = line.split("//")[0].strip().partition(" ")
                body.append((op, [a.strip() for a in re.split(r",\s+(?![^\[]*\])", args)]))
    assert kernels
    return kernels


needs_objdump = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")


@needs_objdump
def test_products_written_as_assembly_find_their_operands(tmp_path):
    """hgemm256_kernel's v_mfma_f32_16x16x32_f16: no VALU instruction writes an operand in the two
    before it, and nothing else reads or writes its accumulators within 11 wait states (8 passes and
    3) after it."""
    for name, code in _kernels(tmp_path, "hgemm256_kernel").items():
        products = [i for i, (op, _) in enumerate(code) if op.startswith("v_mfma_f32_16x16x32")]
        assert len(products) >= 128, name
        for i in products:
            reads = _regs(" ".join(code[i][1][1:]))
            for op, args in code[max(0, i - 2):i]:
                if op.startswith("v_") and not op.startswith("v_mfma"):
                    assert not _regs(args[0]) & reads, (name, i, op, args)
            acc, states = _regs(code[i][1][0]), 0
            for op, args in code[i + 1:i + 12]:
                if states >= 11 or op in ("s_endpgm", "s_branch"):
                    break
                if not op.startswith("v_mfma"):
                    assert not _regs(" ".join(args)) & acc, (name, i, op, args)
                states += 1 + int(args[0]) if op == "s_nop" else 1


@needs_objdump
def test_maxima_written_as_assembly_find_their_products(tmp_path):
    """attn_fwd_kernel's v_max3_f32: behind the last product that wrote an operand lie two others
    (16 passes each) or 18 wait states."""
    for name, code in _kernels(tmp_path, "attn_fwd_kernel").items():
        assert any(op == "v_max3_f32" for op, _ in code), name
        for i, (op, args) in enumerate(code):
            if op != "v_max3_f32":
                continue
            reads, products, states = _regs(" ".join(args[1:])), 0, 0
            for before, bargs in reversed(code[max(0, i - 18):i]):
                if before.startswith("v_mfma"):
                    if _regs(bargs[0]) & reads:
                        raise AssertionError((name, i, args, before, bargs))
                    products += 1
                states += 1 + int(bargs[0]) if before == "s_nop" else 1
                if products >= 2 or states >= 18 or before in ("s_endpgm", "s_branch"):
                    break
