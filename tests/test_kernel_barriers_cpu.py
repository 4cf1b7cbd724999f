"""Workgroup barriers in the compiled kernels, read from the built library's
gfx950 code.  A kernel whose waves fill an LDS table together and then read it
each on their own needs a barrier between the two: without it a wave can read
entries that another has not written, which runs show only by chance."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "fx-corr_amd", "libfxcorr.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def kernels(tmp_path, name):
    """{symbol: [instruction mnemonics]} of the library's kernels whose symbol holds `name`."""
    lib = shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)   # code objects beside it
    out = {}
    for f in sorted(os.listdir(tmp_path)):
        if "gfx950" not in f:
            continue
        syms = subprocess.run([OBJDUMP, "-t", tmp_path / f], check=True, capture_output=True, text=True).stdout
        names = [w for w in re.findall(r"\.text\s.*\s(\S+)$", syms, re.M) if name in w and not w.endswith(".kd")]
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names),
                               tmp_path / f], check=True, capture_output=True, text=True).stdout
        for sym, body in re.findall(r"^\S+ <(\S+)>:\n(.*?)(?=^\S+ <|\Z)", text, re.M | re.S):
            out[sym] = [m for m in re.findall(r"^\s+([a-z]\w+)", body, re.M)]
    return out


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not installed")
def test_wave_kernel_orders_its_tables(tmp_path):
    """Every instance of the wave kernel: the table fill's LDS writes, then a
    barrier, then the first LDS read (the first round's decode)."""
    ks = kernels(tmp_path, "k_sector_wave")
    assert len(ks) >= 40   # six sizes, four with an MFMA form; band shift or not; products or phased sum
    for sym, ins in ks.items():
        write = next(i for i, m in enumerate(ins) if m.startswith("ds_write"))
        read = next(i for i, m in enumerate(ins) if m.startswith("ds_read"))
        barrier = ins.index("s_barrier")
        assert write < barrier < read, (sym, write, barrier, read)
