"""Waits of the kernels that stage rows by LDS DMA beside loads into registers, read off their gfx950
assembly (compiled here; no GPU).  Per unit of their main loop, from barrier to barrier:

* no wait for all loads (vmcnt(0)): two units of weights stay in flight.  The compiler puts one in where
  a DMA counts as a flat access, where it tracks the DMAs into one of several LDS variables, or
  where a half rate's words are shifted right behind their loads;
* at least as many loads as the wait for the rows counts on: it holds back until only those of the
  later units are in flight, so fewer of them would let a unit start before its rows have landed."""
import os
import re
import shutil
import subprocess

import pytest

from ampstein_amd import build


def units(src, defines, kernel, tmp_path):
    """Instructions from each barrier of `kernel`'s instances to the next, where they hold MFMAs."""
    if shutil.which(build.HIPCC) is None:
        pytest.skip("no hipcc")
    out = os.path.join(tmp_path, "k.s")
    subprocess.run([build.HIPCC, *build.COMMON, *defines, "-x", "hip", "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, src), "-o", out], check=True, capture_output=True)
    found, fn, cur = [], None, []
    for line in open(out):
        line = line.strip()
        m = re.match(r"(_Z\w+):", line)
        if m:
            fn, cur = m.group(1), []
        elif line.startswith("s_barrier"):
            if fn and kernel in fn and any(i.startswith("v_mfma") for i in cur):
                found.append(cur)
            cur = []
        elif re.match(r"[a-z]+_", line):
            cur.append(line)
    return found


@pytest.mark.parametrize("src,defines,kernel,ahead", [
    ("exl3_moeg.hip", ["-DEXL3_MOEG_CB=2", "-DEXL3_MOEG_R=2"], "moeg_kernel", (2, 2)),
    ("exl3_moeg.hip", ["-DEXL3_MOEG_CB=1", "-DEXL3_MOEG_R=6"], "moeg_kernel", (2, 2)),
    ("exl3_rows.hip", ["-DEXL3_INST_K=5"], "rows_kernel", (2, 3)), ("exl3_rows.hip", ["-DEXL3_INST_K=18"], "rows_kernel", (2, 3))])
def test_unit_waits(src, defines, kernel, ahead, tmp_path):
    """ahead: units whose row DMAs and whose weight loads the row wait leaves in flight."""
    found = units(src, defines, kernel, tmp_path)
    assert len(found) >= 16
    checked = 0
    for ins in found:
        dma = [i for i in ins if re.match(r"(global|buffer)_load", i) and " lds" in i]
        loads = [i for i in ins if i.startswith("global_load") and " lds" not in i]
        waits = [i for i in ins if i.startswith("s_waitcnt")]
        assert dma and all(i.startswith("buffer_load") for i in dma)
        assert not any(re.search(r"vmcnt\(0\)", w) for w in waits[:-1]), waits
        m = re.search(r"vmcnt\((\d+)\)", waits[-1])
        if m and int(m.group(1)):                     # (the wait behind an item's last unit is for everything)
            assert ahead[0] * len(dma) + ahead[1] * len(loads) >= int(m.group(1)), (dma, loads, waits)
            checked += 1
    assert checked >= 12
