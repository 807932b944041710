"""GPU: block selection from scores that are NaN with every bit set (the largest value that a score can have as a number):
as many ids as asked for, distinct, in range, and nothing stored outside the list."""
import math

import pytest
import torch

from fsa_hip import _lib, ops

pytestmark = pytest.mark.gpu

NAN = 0x7FFFFFFF


@pytest.mark.parametrize("n,topk,bf16", [
    (640, 4, 1), (5000, 4, 1), (10000, 4, 1), (20000, 4, 1), (60000, 4, 1),   # two to sixteen scores per lane
    (640, 4, 0), (5000, 64, 0), (70000, 4, 1), (6000, 70, 0), (6000, 70, 1),  # scores in LDS
])
def test_prefill_selection(dev, n, topk, bf16):
    h, d, ks, st, bs = 1, 64, 32, 16, 64
    print(f"case n={n} topk={topk} bf16={bf16}", flush=True)
    q = torch.randn(n, h, d, device=dev, dtype=torch.bfloat16)
    nc, nblk = (n - ks) // st + 1, (n + bs - 1) // bs
    ck = torch.randn(nc, h, d, device=dev, dtype=torch.bfloat16)
    lse = torch.full((h, n), NAN, device=dev, dtype=torch.int32).view(torch.float32)
    cu_q, cu_k = (torch.tensor([0, m], dtype=torch.int32, device=dev) for m in (n, nc))
    lib = _lib.load()
    guard = 4096
    out = torch.full((guard + h * n * topk + guard,), 7777, device=dev, dtype=torch.int32)
    score = torch.zeros(h, n, nblk, device=dev)
    ws = torch.empty(lib.fsa_cmp_topk_workspace_bytes(n, h, nc // 4 + 1), dtype=torch.uint8, device=dev)
    rc = lib.fsa_cmp_topk(q.data_ptr(), ck.data_ptr(), lse.data_ptr(), 0, h * d, d, h * d, d, cu_q.data_ptr(), cu_k.data_ptr(),
                          1, n, n, nc, h, h, d, ks, st, bs, topk, 1, 2, bf16, 0, 1 / math.sqrt(d), out.data_ptr() + guard * 4,
                          score.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "fsa_cmp_topk")
    torch.cuda.synchronize()
    last = score[0, -1].view(torch.int32) >> 16 & 0x7FFF
    assert (last == 0x7FFF).sum() > topk                    # the case is the one that is meant
    assert (out[:guard] == 7777).all() and (out[-guard:] == 7777).all()
    idx = out[guard:-guard].view(n, topk)
    blocks = torch.arange(n, device=dev) // bs
    taken = torch.minimum(blocks + 1, torch.tensor(topk, device=dev))
    assert ((idx >= 0).sum(1) == taken).all() and (idx <= blocks[:, None]).all()
    ids = idx.masked_fill(idx < 0, nblk).sort(1).values     # distinct but for the padding
    assert ((ids[:, 1:] > ids[:, :-1]) | (ids[:, 1:] == nblk)).all()


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("L", [1000, 20000, 100000, 140000])   # blocks: one, four and eight per lane, and in LDS
def test_decode_selection(dev, L, bf16):
    ks, st, bs, topk, h, b = 32, 16, 64, 5, 2, 3
    print(f"case L={L} bf16={bf16}", flush=True)
    nc, nblk = (L - ks) // st + 1, (L + bs - 1) // bs
    raw = torch.full((h, b, (nc + 3) // 4 * 4), NAN, device=dev, dtype=torch.int32).view(torch.float32)
    i32 = dict(dtype=torch.int32, device=dev)
    idx, score = ops.decode_topk(raw, torch.zeros(h, b, device=dev), torch.arange(b + 1, **i32) * nc, torch.full((b,), L - 1, **i32),
                                 torch.full((b,), L, **i32), h, ks, st, bs, topk, nblk, return_block_score=True,
                                 scores_to_bf16=bf16)
    torch.cuda.synchronize()
    assert ((score.view(torch.int32) & 0x7FFFFFFF) == NAN).sum() > topk * h * b
    s = idx.sort(-1).values
    assert (s >= 0).all() and (s < nblk).all() and (s[..., 1:] > s[..., :-1]).all()
