"""Tokens that belong to no sequence (cu_seqlens covers a part of the buffer, as where a fixed-size buffer is filled to a length
that only the device knows): both forms of the selected forward write their rows alike, and the gradients are written whole."""
import math

import pytest
import torch

from fsa.ops import FSA_topk_sparse_attention
from fsa_hip import _lib, ops
from synth_inputs import make_qkv, make_topk_idx

pytestmark = pytest.mark.gpu

# rounding of the probabilities and of the result to the type, as in the tests of the forward; gradients: one unit of the type
# (2^-8, 2^-11 of the value, either side) on top, since dK and dV add up many rows
O_TOL = {torch.bfloat16: 2e-2, torch.float16: 5e-3}
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}
LSE_TOL = 1e-3

CASES = [
    # cu_seqlens, tokens in all, Hq, Hkv, D, block, T, dtype
    ([0, 250, 500], 600, 4, 2, 128, 64, 4, torch.bfloat16),      # behind the end, which is inside a block
    ([40, 300, 600], 600, 8, 2, 64, 32, 6, torch.float16),       # in front of the first sequence
    ([7, 135, 135], 300, 3, 1, 128, 128, 2, torch.bfloat16),     # both, and nothing but an empty sequence at the end
    ([0, 65, 640], 1000, 2, 2, 256, 64, 8, torch.bfloat16),      # the end is at the edge of a block
    ([0, 10], 500, 2, 1, 64, 128, 3, torch.bfloat16),            # positions behind the end that see the whole last block
    ([33, 33], 90, 2, 1, 128, 64, 2, torch.bfloat16),            # no token in a sequence
    ([3 + 5 * i for i in range(101)], 520, 2, 2, 64, 32, 2, torch.float16),   # more sequences than a wave has lanes
]


def _close(a, b, tol, ulp=0.0):
    a, b = a.float(), b.float()
    assert not torch.isnan(a).any() and not torch.isnan(b).any()
    same = a == b    # (-inf in the log-sum-exp)
    assert (torch.where(same, 0.0, (a - b).abs()) <= tol + ulp * torch.where(same, 0.0, b.abs())).all()


@pytest.mark.parametrize("lists", ["none", "blocks"])
@pytest.mark.parametrize("cu,n,hq,hkv,d,block,topk,dtype", CASES)
def test_rows_of_no_sequence(dev, cu, n, hq, hkv, d, block, topk, dtype, lists):
    print(f"case {cu} {n} {hq} {hkv} {d} {block} {topk} {dtype} {lists}", flush=True)
    q, k, v, do = (x.to(dev) for x in make_qkv(n, hq, hkv, d, dtype, seed=1))
    outside = torch.ones(n, dtype=torch.bool)
    outside[cu[0]:cu[-1]] = False
    idx = torch.full((hkv, n, topk), -1, dtype=torch.int32)
    inner = make_topk_idx([c - cu[0] for c in cu], hkv, block, topk, seed=2)
    idx[:, cu[0]:cu[-1]] = inner
    if lists == "blocks":   # ids of the first and the last blocks of a sequence, and one that is none
        idx[:, outside] = torch.tensor([t // 2 if t % 2 else (cu[-1] - cu[-2] - 1) // block - t // 2 for t in range(topk)],
                                       dtype=torch.int32).clamp(min=-1)
        idx[:, outside, -1] = n
    idx, cut, outside = idx.to(dev), torch.tensor(cu, dtype=torch.int32, device=dev), outside.to(dev)
    do[outside] = 0

    index = ops.build_index(idx, cut, block)
    o, lse = ops.selattn_fwd(q, k, v, index)                                # block-major
    o_direct, lse_direct = torch.full_like(o, math.nan), torch.full_like(lse, math.nan)
    longest = max(1, max(b - a for a, b in zip(cu, cu[1:])))
    _lib.check(_lib.load().fsa_selattn_direct_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), 0 if dtype == torch.bfloat16 else 1, q.stride(0), q.stride(1), k.stride(0),
        k.stride(1), v.stride(0), v.stride(1), idx.data_ptr(), idx.stride(0), idx.stride(1), cut.data_ptr(), len(cu) - 1, n,
        longest, hq, hkv, d, topk, block, 1.0 / math.sqrt(d), o_direct.data_ptr(), o_direct.stride(0), o_direct.stride(1),
        lse_direct.data_ptr(), torch.cuda.current_stream().cuda_stream), "direct")
    _close(o_direct, o, O_TOL[dtype])
    _close(lse_direct, lse, LSE_TOL)
    if lists == "none":
        assert (o_direct[outside] == 0).all() and (lse_direct[:, outside] == -math.inf).all()

    # the operator, forward and backward, on memory that held NaN before
    assert _lib.load().fsa_selattn_direct_preferred(n, n, hq, d, topk, block, 1) == 1
    want = ops.selattn_bwd(q, k, v, o, do, lse, index)
    used = [torch.full_like(o, math.nan) for _ in range(4)] + [torch.full_like(lse, math.nan) for _ in range(4)]
    del used
    x = [t.detach().requires_grad_() for t in (q, k, v)]
    y = FSA_topk_sparse_attention(*x, idx, block, cut)
    got = torch.autograd.grad(y, x, do)
    _close(y, o, O_TOL[dtype])
    for a, b in zip(got, want):
        _close(a, b, O_TOL[dtype], ULP[dtype])
    assert all((t[outside] == 0).all() for t in got[1:])


def test_recorded_step_with_lengths_on_the_device(dev):
    """A step recorded for the whole buffer and replayed on shorter sequences, which only the device knows: every replay equals
    the eager step on those lengths, whatever the outputs held before."""
    n, hq, hkv, d, block, topk, dtype = 600, 4, 2, 128, 64, 4, torch.bfloat16
    q, k, v, do = (x.to(dev) for x in make_qkv(n, hq, hkv, d, dtype, seed=3))
    cut = torch.tensor([0, 250, n], dtype=torch.int32, device=dev)
    idx = make_topk_idx([0, 250, n], hkv, block, topk, seed=4).to(dev)

    def step():
        index = ops.build_index(idx, cut, block)
        o, lse = ops.selattn_fwd(q, k, v, index, None, idx)
        return o, lse, *ops.selattn_bwd(q, k, v, o, do, lse, index)

    assert _lib.load().fsa_selattn_direct_preferred(n, n, hq, d, topk, block, 1) == 1
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = step()
    for rep, cu in enumerate(([0, 100, 500], [0, 33, 64], [40, 300, 590], [0, 250, n])):
        print(f"replay {rep} {cu}", flush=True)
        cut.copy_(torch.tensor(cu, dtype=torch.int32))
        idx.fill_(-1)
        idx[:, cu[0]:cu[-1]] = make_topk_idx([c - cu[0] for c in cu], hkv, block, topk, seed=5 + rep).to(dev)
        for t in out:
            t.fill_(math.nan)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        want = step()
        torch.cuda.synchronize()
        for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), got, want):
            assert torch.equal(a, b) and not torch.isnan(a).any(), f"replay {rep}: {name}"
