"""The loader's native callables (csrc/py_call.cpp) against the ctypes functions they stand for."""
import ctypes
import os

import pytest
import torch

from arcagi2_flashnext_dots3_amd import _lib, build

pytestmark = pytest.mark.skipif(not os.path.exists(build.NATIVE), reason="built without Python's headers")


def test_every_entry_point_takes_the_declared_arguments():
    _lib.lib()
    for name, args in _lib.SIGNATURES.items():
        if name in ("spmla_version", "spmla_host_e4m3_encode"):
            continue
        with pytest.raises(TypeError, match=f"{len(args)} arguments expected"):
            _lib._FN[name](*range(len(args) + 1))


@pytest.mark.parametrize("name,args", [
    ("spmla_attn576", (264, 576, 576, 256, 100, 256, 8, 8, None, 1, 1, 1.0, 1, 1, 256, 512, 512, 256, 1, None, None, None)),
    ("spmla_cache_write", (None, -5, None, 0, None, -1, None, 0, 1, 0, 0, 1.0, None)),
    ("spmla_attn_ws_bytes", (7, 128, 8)),
    ("spmla_attn_ws_bytes", (-1, 128, 8)),
    ("spmla_topk_ws_bytes", (64, 1 << 20, 2048)),
    ("spmla_topk_ws_bytes", ((1 << 32) + 64, 4096, True)),     # integers wrap to their C type, booleans count
    ("spmla_topk_scratch_bytes", ()),
])
def test_same_result_as_ctypes(name, args):
    L = _lib.lib()
    assert _lib._FN[name] is not getattr(L, name)
    assert _lib._FN[name](*args) == getattr(L, name)(*args)


def test_other_argument_types_go_through_ctypes():
    _lib.lib()
    with pytest.raises(TypeError):
        _lib._FN["spmla_attn_ws_bytes"](1.5, 128, 8)
    with pytest.raises(ctypes.ArgumentError):
        _lib.call("spmla_attn_ws_bytes", 1.5, 128, 8)
    with pytest.raises(RuntimeError, match="-2"):              # a ctypes pointer is an address too
        _lib.call("spmla_cache_write", ctypes.c_void_p(256), 0, None, 0, None, -1, None, 0, 1, 0, 0, 1.0, None)


def test_logits_hist_takes_numpy_integers(monkeypatch):
    import numpy as np
    from arcagi2_flashnext_dots3_amd import kernels
    monkeypatch.setattr(kernels, "_stream", lambda t: 0)
    f32, i32, K, Lc, bs = dict(dtype=torch.float32), dict(dtype=torch.int32), *map(np.int64, (16, 1000, 64))
    args = (torch.zeros(0, 64, 128, dtype=torch.bfloat16), torch.zeros(0, 64, **f32), torch.zeros(64, 132), 64, 64, 8448,
            torch.zeros(1, 16, **i32), bs, torch.zeros(0, **i32), torch.zeros(0, **i32), Lc, K, torch.zeros(0, 1000, **f32),
            torch.zeros(64, dtype=torch.uint8))
    assert kernels.logits_hist(*args)                          # no rows: nothing is launched
    with pytest.raises(RuntimeError, match="-2"):
        kernels.logits_hist(*args[:11], np.int64(0), *args[12:])


@pytest.mark.gpu
def test_stream_handle(dev):
    from arcagi2_flashnext_dots3_amd import kernels
    t = torch.empty(1, device=dev)
    s = torch.cuda.Stream()
    assert kernels._stream(t) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(s):
        assert kernels._stream(t) == kernels._device_stream(t.device) == s.cuda_stream
