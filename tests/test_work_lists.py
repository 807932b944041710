"""Where the selected forward runs from the block lists, nothing is kept or built for the kernels that it stands in for: no work
list of the forward in training, no index where no backward follows."""
import ctypes as C

import pytest
import torch

from fsa_hip import _lib
from test_layer_memory import args


def _saved_bytes(n, hq, hkv, d, topk, block, lists):
    """What a layer in training has to keep: `lists` of the two work lists (0: forward, 1: backward)."""
    ck, nb = (n - 32) // 16 + 1, (n + block - 1) // block + 1
    t = min(topk, (n + block - 1) // block)
    kv, q = n * hkv * d * 2, n * hq * d * 2
    parts = [2 * 4, n * d * 2, n * 3 * 2, q, kv, ck * hkv * d * 2, ck * hkv * d * 2, q, q, q, *[n * hq * 4] * 3,
             2 * 4, hkv * nb * 4, hkv * (nb + 1) * 4, hkv * n * t * 4, hkv * n * t * 4]
    parts += [_lib.load().fsa_selattn_tiles_bytes(i, n, hq, hkv, d, t, block, nb) for i in lists]
    return sum((p + 255) // 256 * 256 for p in parts)


@pytest.mark.parametrize("n,lists", [(200, [1]), (2000, [1]), (32768, [0, 1])])
def test_layer_keeps_no_forward_list_for_the_direct_forward(n, lists):
    lib = _lib.load()
    assert lib.fsa_selattn_direct_preferred(n, n, 8, 128, min(16, (n + 63) // 64), 64, 1) == (0 if 0 in lists else 1)
    a = args(n, hq=8, hkv=2)
    assert lib.fsa_layer_saved_bytes(C.byref(a)) == _saved_bytes(n, 8, 2, 128, 16, 64, lists)


def test_one_work_list_is_enough():
    """Neither list: an argument error, as with fake pointers and sizes that are refused behind that check."""
    lib, f = _lib.load(), 0x1000
    for fwd, bwd, word in ((None, None, b"null pointer"), (None, f, b"bad sizes"), (f, None, b"bad sizes")):
        rc = lib.fsa_build_index_tiles(f, 16, 16, f, 1, 64, 2, 16, 64, 2, f, f, f, f, f, 3, 128, fwd, bwd, f, 0, None)
        assert rc == -1 and word in lib.fsa_last_error(), lib.fsa_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("n,direct", [(500, True), (9000, False)])
def test_functional_forward_builds_an_index_where_it_is_read(dev, n, direct):
    from fsa.ops import FSA_topk_sparse_attention
    from nsa_ref.ops.topk_sparse_attention import _topk_sparse_attention_fwd
    from synth_inputs import make_qkv, make_topk_idx

    hq, hkv, d, block, topk = 4, 2, 128, 64, 8
    q, k, v, do = (x.to(dev) for x in make_qkv(n, hq, hkv, d, torch.bfloat16, seed=1))
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    idx = make_topk_idx([0, n], hkv, block, topk, seed=2).to(dev)
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    _lib.profile_enable(True)
    o, lse = _topk_sparse_attention_fwd(q, k, v, idx, block, cu, cu, n, n, d ** -0.5)
    torch.cuda.synchronize()
    functional = [name for name, _ in _lib.profile_records()]
    _lib.profile_enable(True)
    y = FSA_topk_sparse_attention(*x, idx, block, cu)
    grads = torch.autograd.grad(y, x, do)
    torch.cuda.synchronize()
    operator = [name for name, _ in _lib.profile_records()]
    _lib.profile_enable(False)
    assert ("selattn_direct_fwd" in functional) == ("selattn_direct_fwd" in operator) == direct
    assert ("index_build" in functional) == (not direct) and "index_build" in operator
    assert torch.equal(o, y) and all(torch.isfinite(t).all() for t in grads)
