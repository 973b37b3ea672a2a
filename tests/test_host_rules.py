"""Rules that size launches and place boundaries, from the headers the kernels include, compiled for
the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "common.hpp"
using namespace dplus;
extern "C" void patch_sets(long long nchunks, int *D, int *nset) { mc_patch_sets(nchunks, *D, *nset); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, out = str(d / "rules.cpp"), str(d / "librules.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "dplus-dev_amd", "csrc"), src, "-o", out], check=True)
    return ctypes.CDLL(out)


def test_mc_patch_sets_fit_the_partial_sums(rules):
    """Every count of chunks: the sets cover the chunks, no set is empty, and the workgroups write
    no more blocks than the partial sums' buffer holds (chunk / 256 a chunk)."""
    D, nset = ctypes.c_int(), ctypes.c_int()
    for n in list(range(4, 5000)) + [10 ** 6, 10 ** 6 + 1]:
        rules.patch_sets(ctypes.c_longlong(n), ctypes.byref(D), ctypes.byref(nset))
        per = 4 * D.value
        assert D.value in (1, 2, 4) and (nset.value - 1) * per < n <= nset.value * per
        for chunk in (256, 512, 768, 8192):
            assert chunk // 64 * nset.value <= n * chunk // 256, (n, chunk)
