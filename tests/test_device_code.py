"""Checks of the device sources that need no GPU."""
import os
import re

import mxfa

PKG = os.path.dirname(os.path.abspath(mxfa.__file__))
CSRC = os.path.join(PKG, "csrc")


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
