"""The wait for copies to LDS orders the reads behind it in the source: the copies are
issued by inline assembly, so without that the compiler may read what they write before
the wait.  Shown on the compiler's IR of a probe that reads an LDS value on both sides of
the wait (no GPU needed): a value read before the wait may not stand for the one after."""
import os
import re
import subprocess

import pytest

from sod2d_amd import build

PROBE = """
#include "pipe.hpp"
using namespace sodhip;
extern "C" __global__ void probe(const int *in, int *out)
{
    __shared__ int s[64];
    const int i = threadIdx.x;
    dma_lds<4>(in + i, lds_addr(s));
    const int before = s[i];
    wait_vm<0>();
    out[i] = s[i] - before;
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_reads_stay_behind_the_wait(tmp_path):
    src = tmp_path / "probe.hip"
    src.write_text(PROBE)
    r = subprocess.run([build.HIPCC, "-O3", "-std=c++17", "-x", "hip", *build.HIP_FLAGS,
                        f"-I{build.CSRC}", "--offload-device-only", "-S", "-emit-llvm", str(src),
                        "-o", "-"], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    body = re.search(r"define[^\n]*@probe\(.*?\n}", r.stdout, re.S).group(0)
    wait = body.index("@llvm.amdgcn.s.waitcnt")
    reads = [m.start() for m in re.finditer(r"load i32, ptr addrspace\(3\)", body)]
    assert len(reads) == 2 and reads[0] < wait < reads[1], body
