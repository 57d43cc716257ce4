"""The table lookup of the paged attention kernels, compiled for the host from the header that they include: rows as the
oracle's rule gives them, and no read of the table for a position that has no entry in it."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from arcagi2_flashnext_dots3_amd import _lib, build, kernels

SRC = r"""
#include "spmla_common.h"
extern "C" void rows(const int* btrow, int cols, int sh, long long stride, const int* x, int n, int* out) {
  const spmla::Pages g{nullptr, btrow, 0, cols, sh, stride};
  for (int i = 0; i < n; ++i) out[i] = spmla::page_row(g, x[i], spmla::page_entry(g, btrow, x[i], x));
}
"""
CHILD = r"""
import ctypes, mmap, sys
import numpy as np
f = ctypes.CDLL(sys.argv[1]).rows
f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
libc = ctypes.CDLL(None)
libc.mmap.restype = ctypes.c_void_p
libc.mmap.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
wall = libc.mmap(None, 1 << 16, 0, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS, -1, 0)       # any access faults
x = np.array([-1, -7, -2 ** 31, 640, 641, 2 ** 31 - 1], np.int32)
out = np.zeros_like(x)
f(wall + (1 << 15), 10, 6, 64, x.ctypes.data, x.size, out.ctypes.data)
assert (out == -1).all(), out
print("no access")
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("pages")
    (d / "rows.hip").write_text(SRC)
    out = d / "rows.so"
    subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", build.CSRC,
                    str(d / "rows.hip"), "-o", str(out)], check=True, capture_output=True)
    return str(out)


def test_positions_without_an_entry_read_nothing(lib):
    r = subprocess.run([sys.executable, "-c", CHILD, lib], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "no access" in r.stdout, (r.returncode, r.stderr[-500:])


@pytest.mark.parametrize("sh,cols,stride", [(0, 7, 1), (6, 10, 64), (6, 10, 67), (11, 3, 2048)])
def test_rows_of_positions(lib, sh, cols, stride):
    import ctypes
    f = ctypes.CDLL(lib).rows
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int,
                  ctypes.c_void_p]
    rng = np.random.default_rng(sh)
    bt = rng.integers(0, 1000, cols).astype(np.int32)
    bt[cols // 2] = -3
    x = np.arange(-5, (cols << sh) + 5, dtype=np.int32)
    out = np.zeros_like(x)
    f(bt.ctypes.data, cols, sh, stride, x.ctypes.data, x.size, out.ctypes.data)
    blk = x >> sh
    entry = np.where((x >= 0) & (blk < cols), bt[np.clip(blk, 0, cols - 1)], -1)
    assert np.array_equal(out, np.where(entry >= 0, entry * stride + (x & ((1 << sh) - 1)), -1))


@pytest.mark.parametrize("nreq,npos,taken", [(4, 4, True), (6, 5, True), (3, 4, False), (4, 3, False), (0, 4, False)])
def test_fewer_request_ids_or_positions_than_tokens(monkeypatch, nreq, npos, taken):
    """The kernel reads a request id and a list of positions for every token: attend_paged leaves calls with fewer to
    the separate conversion, which looks up only what a position needs."""
    calls = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(kernels, "_stream", lambda t: None)
    monkeypatch.setattr(kernels, "auto_split", lambda T, H, K: 1)
    q = torch.zeros(4, 16, 576, dtype=torch.bfloat16)
    i32 = dict(dtype=torch.int32)
    out = kernels.attend_paged(q, torch.zeros(64, 656, dtype=torch.uint8), torch.zeros(npos, 64, **i32),
                               torch.zeros(nreq, **i32), torch.zeros(2, 1, **i32), 64, 64, 0.1)
    assert (out is not None) == taken and calls == (["spmla_attn_paged"] if taken else [])
