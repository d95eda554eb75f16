"""What the compiler is told of the convolution operator's accesses at any element: float32 pairs are multiples of 4 bytes, 16-bit
pairs of 2 (the loads and stores of the compiled device code, built here)."""
import os
import re
import subprocess

import pytest

from megalodon_amd import _build

SNIPPET = """
#include <hip/hip_runtime.h>
#include "{csrc}/fftconv_rows.hpp"
using namespace mega;
template <int DT>
__device__ void move(const void* from, void* to) {{
  const unsigned off = 6u * threadIdx.x;
  float a, b;
  Pair<DT>::unpack(Pair<DT>::load_any(from, off), a, b);
  Pair<DT>::store_any(to, off, Pair<DT>::pack(b, a));
}}
extern "C" __global__ void pairs_f32(const void* from, void* to) {{ move<MEGA_F32>(from, to); }}
extern "C" __global__ void pairs_bf16(const void* from, void* to) {{ move<MEGA_BF16>(from, to); }}
extern "C" __global__ void pairs_f16(const void* from, void* to) {{ move<MEGA_F16>(from, to); }}
"""


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    if not os.path.exists(_build.HIPCC):
        pytest.skip("no hipcc")
    tmp = tmp_path_factory.mktemp("align")
    src, out = tmp / "pairs.hip", tmp / "pairs.ll"
    src.write_text(SNIPPET.format(csrc=_build.CSRC))
    r = subprocess.run([_build.HIPCC, *_build.FLAGS, "--cuda-device-only", "-S", "-emit-llvm", str(src), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out.read_text()


@pytest.mark.parametrize("name,align", [("pairs_f32", 4), ("pairs_bf16", 2), ("pairs_f16", 2)])
def test_declared_alignment(code, name, align):
    body = re.search(r"define[^\n]*@%s\(.*?\n}" % name, code, re.S)[0]
    moves = re.findall(r"(?:load|store) [^\n]*addrspace\(1\)[^\n]*align (\d+)", body)
    assert len(moves) == 2 and all(int(m) <= align for m in moves), body
