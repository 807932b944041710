"""Memory that the fused layer asks for (host arithmetic of the C entry points, no device needed)."""
import ctypes as C

import pytest

from fsa_hip import _lib


class LayerArgs(C.Structure):
    _fields_ = ([(n, C.c_int32) for n in ("dtype", "hidden", "num_q_heads", "num_kv_heads", "head_dim", "kernel_size",
                                          "kernel_stride", "block_size", "topk", "init_blocks", "local_blocks", "window",
                                          "batch", "inference")]
                + [(n, C.c_int64) for n in ("total_tokens", "total_ck", "max_len", "max_ck")]
                + [(n, C.c_float) for n in ("softmax_scale", "rope_scale")]
                + [(n, C.c_void_p) for n in ("x", "w_gate", "q", "k", "v", "w_ck", "w_cv", "pe", "cu_seqlens", "inv_freq",
                                             "saved", "workspace")]
                + [(n, C.c_size_t) for n in ("saved_bytes", "workspace_bytes")])


def args(n, hq=32, hkv=8, d=128, hidden=4096, batch=1, inference=0, window=512):
    ck = (n - 32) // 16 + 1
    return LayerArgs(dtype=0, hidden=hidden, num_q_heads=hq, num_kv_heads=hkv, head_dim=d, kernel_size=32, kernel_stride=16,
                     block_size=64, topk=16, init_blocks=1, local_blocks=2, window=window, batch=batch, inference=inference,
                     total_tokens=n, total_ck=ck, max_len=n, max_ck=ck, softmax_scale=0.1, rope_scale=1.0)


@pytest.mark.parametrize("n", [200, 5003, 32768])
def test_inference_reserves_nothing_for_a_backward(n):
    lib = _lib.load()
    train, infer = args(n), args(n, inference=1)
    less = lib.fsa_layer_saved_bytes(C.byref(train)) - lib.fsa_layer_saved_bytes(C.byref(infer))
    o, lse = n * 32 * 128 * 2, n * 32 * 4            # output and lse of the selected branch
    tiles = lib.fsa_selattn_tiles_bytes(1, n, 32, 8, 128, min(16, (n + 63) // 64), 64, (n + 63) // 64 + 1)
    assert less >= o + lse + tiles


def test_backward_after_inference_is_refused():
    lib = _lib.load()
    a = args(200, inference=1)
    for f, _ in LayerArgs._fields_[20:32]:
        setattr(a, f, 0x10000)
    a.saved_bytes = a.workspace_bytes = 1 << 40
    grads = (C.c_void_p * 9)(*[0x10000] * 9)
    assert lib.fsa_layer_backward(C.byref(a), C.byref(grads), None) == -1
    assert b"inference" in lib.fsa_last_error()
