"""What the compiler is told of the workspace of the norms' backward by columns: a caller's, at any float (the stores of
floats in the compiled device code, built here; the rows' own stores are of 16-bit elements)."""
import os
import re
import subprocess

import pytest

from megalodon_amd import _build


def test_declared_alignment_of_partial_sums(tmp_path):
    if not os.path.exists(_build.HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path / "norms.ll"
    flags = [f if f != "-O3" else "-O1" for f in _build.FLAGS]
    r = subprocess.run([_build.HIPCC, *flags, "--cuda-device-only", "-S", "-emit-llvm", str(_build.CSRC / "norms.hip"), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    kernels = re.findall(r"define[^\n]*@\S*norm_bwd_columns_kernel\S*\(.*?\n}", out.read_text(), re.S)
    assert kernels
    for body in kernels:
        puts = re.findall(r"store (?:<\d x float>|float) [^\n]*addrspace\(1\)[^\n]*align (\d+)", body)
        assert puts and all(int(m) <= 4 for m in puts)
