"""The launchers' rules of sizes (csrc/spmla_rules.h), compiled for the host, against measured points on both sides."""
import ctypes
import os
import shutil
import subprocess

import pytest

from arcagi2_flashnext_dots3_amd import build


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text('#include "spmla_rules.h"\n'
                             'extern "C" int wide(int T, int H, int K, int S) { return spmla::rules::attn_wide(T, H, K, S); }\n'
                             'extern "C" double cost(long long n, int K, int s, bool r) { return spmla::rules::split_cost(n, K, s, r); }\n'
                             'extern "C" int splits(int T, int H, int K, int S, bool r) { return spmla::rules::merged_splits(T, H, K, S, r); }\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", build.CSRC, str(d / "r.cpp"), "-o",
                    str(d / "r.so")], check=True, capture_output=True)
    L = ctypes.CDLL(str(d / "r.so"))
    L.cost.restype, L.cost.argtypes = ctypes.c_double, [ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_bool]
    return L


@pytest.mark.parametrize("T,H,K,hg,fwd", [                          # us of the head-group kernel and of fwd_kernel
    (129, 128, 2048, 142, 169), (224, 128, 2048, 195, 172), (300, 128, 2048, 253, 319), (400, 128, 2048, 345, 325),
    (2048, 128, 2048, 1618, 1406), (1500, 32, 2048, 384, 874), (512, 160, 2048, 523, 645), (129, 128, 1024, 86, 94),
    (300, 128, 512, 100, 108), (400, 128, 1024, 209, 187), (128, 128, 96, 29, 33),
    (129, 128, 128, 39, 31), (129, 128, 40, 34, 22), (300, 128, 128, 65, 54), (2000, 64, 128, 233, 184),
    (512, 64, 32, 45, 34), (512, 160, 256, 160, 144), (1000, 160, 40, 228, 160)])
def test_attention_kernel_choice(lib, T, H, K, hg, fwd):
    assert bool(lib.wide(T, H, K, 1)) == (fwd < hg)


def test_lists_beyond_the_prefill_kernel(lib):
    assert lib.wide(4096, 128, 2048, 1) and not lib.wide(4096, 128, 2049, 1) and lib.wide(4096, 128, 4096, 2)
    assert not lib.wide(0, 128, 2048, 1)


def test_split_cost_is_the_callers(lib):
    from arcagi2_flashnext_dots3_amd import kernels
    for n in (1, 4, 33, 100, 128):
        for K in (0, 40, 512, 2048, 12000):
            for i in range(1, 9):
                for rb in (kernels.ROW656, kernels.ROW576):
                    assert lib.cost(n, K, i, rb == 576) == pytest.approx(kernels._split_cost(n, K, i, 256, rb), abs=1e-9)


@pytest.mark.parametrize("T,H,K,S,chosen", [
    (5, 160, 1536, 5, 5), (8, 128, 2048, 8, 8), (32, 16, 512, 8, 8), (1, 128, 64, 8, 8),         # one round: as asked
    (32, 128, 2048, 8, 2), (64, 128, 256, 4, 1), (200, 128, 2048, 8, 1), (129, 32, 2048, 2, 1), (23, 128, 12000, 8, 5)])
def test_merged_splits_beyond_one_round(lib, T, H, K, S, chosen):
    """A merged launch of more than one round of workgroups takes the cheapest of up to S splits, which is what auto_split
    takes too."""
    from arcagi2_flashnext_dots3_amd import kernels
    for r576 in (False, True):
        assert lib.splits(T, H, K, S, r576) == chosen
    if T * ((H + 31) // 32) * S > 256:
        assert lib.splits(T, H, K, 8, True) == kernels.auto_split576(T, H, K)
