"""Checks of the device sources and of the built code object that need no GPU."""
import os
import re
import subprocess

import pytest

import mxfa

PKG = os.path.dirname(os.path.abspath(mxfa.__file__))
CSRC = os.path.join(PKG, "csrc")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def test_inline_assembly_that_writes_m0_declares_it():
    """The compiler keeps its own value in m0 (LDS DMA builtins, indexed registers) across a statement
    that does not name m0 among its clobbers."""
    found = 0
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            for stmt in re.findall(r"__asm__[^;]*;", f.read()):
                if re.search(r"s_mov_b32 m0\b", stmt):
                    found += 1
                    assert '"m0"' in stmt.split("\\n\\t")[-1], f"{name}: {stmt}"
    assert found > 0


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_no_matrix_instruction_in_a_saturation_window(tmp_path):
    """Between sat_begin and sat_end (MODE.FP16_OVFL set) no MFMA may issue: it would make infinite and
    NaN results finite.  Every prefill kernel of rule R1, split and block-packed ones included, is
    straight-line code there."""
    with open(os.path.join(PKG, "mxfa_kernels.hsaco"), "rb") as f:
        bundle = f.read()
    elf = tmp_path / "kernels.elf"
    elf.write_bytes(bundle[bundle.index(b"\x7fELF"):])
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(elf)], check=True, capture_output=True, text=True).stdout
    kernel, window, windows = None, None, {}
    for line in text.splitlines():
        label = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if label:
            assert window is None, f"{kernel}: the window is open at its end"
            kernel = label.group(1)
            continue
        ins = line.split("//")[0].strip()
        if ins.startswith("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1)"):
            value = int(ins.split(",")[-1], 0)
            assert (window is None) == (value == 1), f"{kernel}: unpaired {ins}"
            if value == 1:
                window = []
            else:
                assert any("v_cvt" in i for i in window), kernel
                bad = [i for i in window if "mfma" in i or i.startswith(("s_cbranch", "s_branch"))]
                assert not bad, f"{kernel}: {bad[0]}"
                windows[kernel] = windows.get(kernel, 0) + 1
                window = None
        elif window is not None:
            window.append(ins)
    r1 = [k for k in windows if k.startswith("mxfa_prefill3")]
    for form in ("mxfa_prefill3_d", "mxfa_prefill3n_d", "mxfa_prefill3s_d"):
        for suffix in ("64", "128", "256", "128_softcap", "128_blk"):
            assert form + suffix in windows, form + suffix
    assert not [k for k in r1 if "_r2" in k]
