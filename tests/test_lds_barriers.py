"""Every kernel's workgroup barrier is sync_lds (gf_sync.hpp), which waits for
the wave's LDS accesses itself: the compiler leaves that wait out before some
barriers."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "parallelpopgen_amd", "csrc")


def test_barriers_wait_for_lds():
    bare, waited = [], 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        code = re.sub(r"/\*.*?\*/|//[^\n]*", "", open(path).read(), flags=re.S)
        waited += code.count("sync_lds()")
        if os.path.basename(path) == "gf_sync.hpp":
            assert re.search(r's_waitcnt lgkmcnt\(0\)".*?__syncthreads\(\)', code, re.S)
            continue
        bare += [os.path.basename(path)] * len(re.findall(r"__syncthreads|builtin_amdgcn_s_barrier", code))
    assert not bare and waited > 40
