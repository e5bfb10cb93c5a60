"""LDS-direct copies are written as inline assembly, where the compiler inserts no wait states: every such load must have the one that
the hardware needs behind the write of M0 (its LDS base) in the same statement."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "densecore_amd", "csrc")


def test_every_lds_direct_load_waits_behind_its_write_of_m0():
    loads = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        for text in re.findall(r'asm volatile\("([^"]*)"', open(path).read()):
            if "_lds_dword" not in text:
                continue
            loads += 1
            assert re.fullmatch(r"s_mov_b32 m0, %\d\\n\\ts_nop 0\\n\\tglobal_load_lds_dword(x4)? %0, (%1|off)", text), (path, text)
    assert loads > 0
