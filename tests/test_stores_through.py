"""A kernel that tells recorded passes that its results need no release has none that do.

Between two launches of a pass the release at the end of the first is left out where its code object holds
<kernel>_through (reef_amd/csrc/hal/aql.cpp).  Then every store to memory has to carry the scope that takes it past the L2
(sc1), and has to be acknowledged before the wavefront ends.
"""
import os
import re
import shutil
import subprocess

import pytest

from reef_amd.paths import code_object

LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.parametrize("flavour", ["raw", "be", "trans"])
def test_marked_kernels_write_through(flavour, tmp_path):
    if not shutil.which(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no disassembler")
    elf = str(tmp_path / "kernels.elf")
    subprocess.check_call([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o",
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + code_object(flavour), "--output=" + elf])
    names = subprocess.check_output([os.path.join(LLVM, "llvm-readelf"), "-sW", elf], text=True)
    marked = set(re.findall(r" (\w+)_through$", names, re.M))
    assert len(marked) > 80 and "reef_conv2d_p1_v_16x16k4" in marked and "reef_softmax" in marked
    name, stores, plain, unwaited = None, 0, set(), set()
    waited = True
    for line in subprocess.Popen([os.path.join(LLVM, "llvm-objdump"), "-d", elf], stdout=subprocess.PIPE, text=True).stdout:
        m = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if m:
            name = m.group(1)
        elif re.search(r"\b(global|buffer|flat)_store", line):
            stores += 1
            waited = False
            if name in marked and " sc1" not in line:
                plain.add(name)
        elif re.search(r"\bs_waitcnt\b", line) and "vmcnt(0)" in line:
            waited = True
        elif "s_endpgm" in line:
            if name in marked and not waited:
                unwaited.add(name)
            waited = True
    assert stores > 500
    assert not plain and not unwaited
