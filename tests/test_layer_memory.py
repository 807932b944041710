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


def _tile_rows(rows_total, g, d):
    """Rows per work-group of the key-major kernel (64-key tiles), as the library chooses them."""
    cap = min(1024 + 2048 * g, 8192)
    rows = -(-(rows_total // (2 * 256 * (2 if d <= 128 else 1))) // 128) * 128
    return max(128, min(rows, cap))


def _partial_bytes(n, blocks, rows_of_block, tile_rows, batch, hq, hkv, d):
    """Workspace up to the partials, and the partials of the tiles that the kernel will really deal."""
    def up(x):
        return (x + 255) // 256 * 256
    tiles = sum(-(-r // tile_rows) for r in rows_of_block)
    head = up(n * hq * 4) + up((batch + 1) * 4) + up(hkv * blocks * 4) + up(hkv * (blocks + 1) * 4)
    return head, hkv * tiles * 2 * 64 * d * 4


@pytest.mark.parametrize("lens", [[1], [64], [65], [5003], [300, 77, 511], [32768], [1, 2, 3000, 64, 129], [700] * 9])
@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (4, 4, 64), (6, 2, 256), (8, 1, 128)])
@pytest.mark.parametrize("window", [0, 33, 512, 4096])
def test_dense_backward_partials_fit(lens, hq, hkv, d, window):
    """The room for fp32 dK / dV partials: enough for every tile, and without a spare one for every 64 keys."""
    lib = _lib.load()
    n, g, batch, longest = sum(lens), hq // hkv, len(lens), max(lens)
    blocks = (n + 63) // 64 + batch
    rows = [min(s - f, 64 + window) * g for s in lens for f in range(0, s, 64)]
    tr = _tile_rows(blocks * (64 + window) * hq, g, d)
    head, parts = _partial_bytes(n, blocks, rows, tr, batch, hq, hkv, d)
    got = lib.fsa_winattn_bwd_workspace_bytes(n, longest, window, batch, hq, hkv, d)
    assert got >= head + parts
    assert got <= head + hkv * blocks * -(-(64 + window) * g // tr) * 2 * 64 * d * 4 + 256
    nc = [(s - 32) // 16 + 1 if s >= 32 else 0 for s in lens]
    if sum(nc):
        blocks = (sum(nc) + 63) // 64 + batch
        rows = [max(0, s - (f * 16 + 31)) * g for s, c in zip(lens, nc) for f in range(0, c, 64)]
        tr = _tile_rows(blocks * longest * hq // 2, g, d)
        head, parts = _partial_bytes(n, blocks, rows, tr, batch, hq, hkv, d)
        assert lib.fsa_cmpattn_bwd_workspace_bytes(n, sum(nc), longest, batch, hq, hkv, d) >= head + parts
