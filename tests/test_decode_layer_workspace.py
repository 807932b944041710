"""Scratch of a token through the layer: never more than the 4096 + 2 Hkv partial rows of a group that callers size it by."""
import ctypes as C

import pytest

from fsa_hip import _lib


class Args(C.Structure):
    """fsa_decode_layer_args"""
    _fields_ = [(n, C.c_void_p) for n in ("x", "w_q", "w_k", "w_v", "w_gate", "w_o", "k_cache", "v_cache", "ck_cache", "cv_cache")] + \
               [(n, C.c_int64) for n in ("k_sn", "k_sh", "v_sn", "v_sh", "ck_sn", "ck_sh", "cv_sn", "cv_sh")] + \
               [(n, C.c_void_p) for n in ("ck_new", "cv_new", "inv_freq")] + [("cache_len", C.c_int64), ("ck_len", C.c_int64)] + \
               [(n, C.c_int32) for n in ("dtype", "hidden", "hq", "hkv", "d", "kernel_size", "kernel_stride", "block_size", "topk",
                                         "init_blocks", "local_blocks", "window")] + \
               [("softmax_scale", C.c_float), ("rope_scale", C.c_float)] + \
               [(n, C.c_void_p) for n in ("k_new", "v_new", "y", "workspace")] + [("workspace_bytes", C.c_size_t)]


@pytest.mark.parametrize("hkv", [1, 3, 8, 32, 33, 64, 100, 255, 256, 257, 1024])
@pytest.mark.parametrize("g,d,n", [(1, 64, 50), (4, 128, 3000), (16, 256, 65000)])
def test_partial_rows(hkv, g, d, n):
    a = Args(hidden=1024, hq=g * hkv, hkv=hkv, d=d, kernel_size=32, kernel_stride=16, block_size=64, topk=16, init_blocks=1,
             local_blocks=2, window=512, cache_len=n, ck_len=(n - 32) // 16 + 1)
    up = lambda x: (x + 255) // 256 * 256   # noqa: E731
    row, blocks = up(g * hkv * d * 2), (n + 64) // 64
    others = 4 * row + 256 + up(hkv * min(16, blocks) * 4) + up(hkv * ((a.ck_len + 1 + 3) // 4 * 4) * 4)
    total = _lib.load().fsa_decode_layer_workspace_bytes(C.addressof(a))
    assert others < total <= others + up((4096 + 2 * hkv) * g * (4 + d) * 4)
