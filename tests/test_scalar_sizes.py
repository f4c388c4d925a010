"""Checkpoint and workspace sizes of a scalar-gate call: what its own kernels need, no more and no
less, where the shape's sizes cover every dtype and layout."""
import ctypes
import os

import pytest

from delta_kernels import _lib

SMALL, F32, BF16 = 4, 0, 1


@pytest.fixture(scope="module")
def L():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libgdn2_amd.so not built")
    return _lib.lib()


def _shape(B, T, H, K, V=None):
    return _lib.Gdn2Shape(B, T, H, K, V or K)


def _view(shape, dtype, width, data=0x1000, stride=1):
    t = (shape.time * shape.heads * width, shape.heads * width, width, stride)
    return _lib.Gdn2View(data, dtype, 0, (ctypes.c_int64 * 4)(*t))


def _sizes(L, shape, chunk, views):
    r = ctypes.byref
    a = (r(shape), chunk)
    qkv = [r(x) for x in views]
    return (L.gdn_scalar_call_checkpoint_bytes(*a, *qkv), L.gdn_scalar_call_workspace_bytes(*a, *qkv),
            L.gdn_scalar_checkpoint_bytes(*a), L.gdn_scalar_workspace_bytes(*a))


# What these kernels keep for 64 tokens of a head, in bytes: the layouts in gdn2_chunk.h.
@pytest.mark.parametrize("B,T,H,D,ck,ws", [(16, 512, 8, 64, 91136, 32768),
                                           (4, 8192, 16, 128, 174592, 131072)])
def test_chunk_calls_pay_for_their_own_kernels(L, B, T, H, D, ck, ws):
    s = _shape(B, T, H, D)
    n = B * H * T // 64
    got = _sizes(L, s, 64, [_view(s, BF16, D)] * 3)
    assert got[:2] == (n * ck, n * ws)
    assert got[2] >= got[0] and got[3] >= got[1]


@pytest.mark.parametrize("change", ["f32", "offset", "strided", "chunk"])
def test_other_calls_pay_for_the_f32_kernels(L, change):
    s = _shape(2, 100, 3, 64)
    dtype = F32 if change == "f32" else BF16
    v = [_view(s, dtype, 64, 0x1002 if change == "offset" else 0x1000, 2 if change == "strided" else 1),
         _view(s, dtype, 64), _view(s, dtype, 64)]
    chunk = 16 if change == "chunk" else 64
    got = _sizes(L, s, chunk, v)
    assert got[0] == got[2] and got[0] > _sizes(L, s, 64, [_view(s, BF16, 64)] * 3)[0]


def _scan(L, shape, views, size):
    gate, mask = _view(shape, F32, 1), _lib.Gdn2View(0x2000, F32)
    r = ctypes.byref
    return L.gdn_scalar_scan(r(shape), 64, *[r(x) for x in views], r(gate), r(gate), r(mask),
                             r(mask), r(_lib.Gdn2View(None, F32)), ctypes.c_void_p(0x3000),
                             views[0].dtype, ctypes.c_void_p(0x4000), ctypes.c_void_p(0x5000),
                             ctypes.c_void_p(0x6000), size, None)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("T", [9, 100])
def test_smaller_checkpoints_are_refused(L, dtype, T):
    s = _shape(2, T, 3, 64)
    v = [_view(s, dtype, 64)] * 3
    assert _scan(L, s, v, _sizes(L, s, 64, v)[0] - 1) == SMALL


def test_bad_arguments_have_no_size(L):
    s = _shape(2, 100, 3, 64)
    v = [_view(s, F32, 64)] * 3
    assert _sizes(L, s, 65, v) == (0, 0, 0, 0)
    assert _sizes(L, s, 64, [v[0], _view(s, BF16, 64), v[2]])[:2] == (0, 0)
    assert _sizes(L, _shape(2, 0, 3, 64), 64, v) == (0, 0, 0, 0)
