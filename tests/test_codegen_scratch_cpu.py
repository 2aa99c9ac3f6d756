"""Register spills of the LU path's kernels (CPU only): the scratch that the
compiler gives each kernel, where hipcc is present.  Two FP64 forms of the
batched factorization spill 25 registers, and the batched solve in 16 waves
keeps a return address for its rare second solve; nothing else has any."""
import concurrent.futures as cf
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lapack_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "--offload-device-only", "-S", "-o", "-"]
# bytes a lane, by a part of the kernel's name
ALLOWED = {"batched_leaf.hip": {"leaf_kernelIdLi512E": 108, "leaf_kernelIdLi256E": 104},
           "batched_solve.hip": {"Li1024ELi8E": 8}, "swap_trsm.hip": {}, "tri_line.hip": {}, "panel.hip": {}}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_scratch():
    def sizes(src):
        r = subprocess.run([HIPCC] + FLAGS + [os.path.join(CSRC, src)], capture_output=True, text=True, cwd=CSRC)
        assert r.returncode == 0, r.stderr[-2000:]
        return re.findall(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", r.stdout)
    with cf.ThreadPoolExecutor(max_workers=len(ALLOWED)) as ex:
        found = dict(zip(ALLOWED, ex.map(sizes, ALLOWED)))
    for src, kernels in found.items():
        assert kernels, src
        for name, size in kernels:
            limit = max([v for k, v in ALLOWED[src].items() if k in name], default=0)
            assert int(size) <= limit, (src, name, size)
