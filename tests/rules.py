"""The library's rules on sizes (``csrc/tms_rules.h``), built with g++ and bound with ctypes, so
that tests can say which form of a kernel a call takes."""
import ctypes
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def lib():
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    with tempfile.TemporaryDirectory() as tmp:
        so = os.path.join(tmp, "rules.so")
        build = subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                                os.path.join(REPO, "tilemaxsim_amd", "csrc"), os.path.join(REPO, "tests", "rules_c.cpp"),
                                "-o", so], capture_output=True, text=True)
        assert build.returncode == 0, build.stderr
        out = ctypes.CDLL(so)
    i64, integer = ctypes.c_int64, ctypes.c_int
    out.dense_split_waves.argtypes = [i64, i64, ctypes.c_size_t, integer, integer]
    out.topk_group_lanes.argtypes = [i64, i64, integer]
    out.topk_workspace.argtypes = [i64, i64, integer]
    out.topk_workspace.restype = i64
    out.pq_per_query.argtypes = [i64] * 6
    return out


def dense_split(qdt: str, ddt: str, d: int, nq: int, B: int, nd: int) -> int:
    """Waves per document of a dense call of the general kernel (``tms_dense_kernel.h``: its
    blocks per launch, LDS and tile; aligned operands). 1 where the launch has no split form."""
    split = "float32" in (qdt, ddt)
    steps = -(-d // 32)

    def lds(nqb):
        return nqb * steps * 2 * 64 * 16 * (2 if split else 1)

    reg = d % 32 == 0 and 0 < d <= 128
    nqb = 2 if nq > 32 and (reg or lds(2) <= 64 * 1024) else 1
    if not reg and lds(nqb) > 80 * 1024:  # eight-wave workgroups
        return 1
    tile = 16 if ddt == "float32" and reg else 32
    return lib().dense_split_waves(B, -(-nd // tile), 0 if reg else lds(nqb), nqb, steps if reg else 0)
