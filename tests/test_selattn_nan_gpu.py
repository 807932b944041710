"""A NaN or an infinite value in q, k or v: both forms of the selected forward give NaN for the rows that it reaches, in o and in
the log-sum-exp, and for no others; the gradients that follow are the same."""
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


def _alike(a, b, tol, ulp=0.0):
    a, b = a.float(), b.float()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    same = torch.isnan(b) | (a == b)
    assert (torch.where(same, 0.0, (a - b).abs()) <= tol + ulp * torch.where(same, 0.0, b.abs())).all()


@pytest.mark.parametrize("d,block,dtype", [(128, 64, torch.bfloat16), (64, 32, torch.float16), (256, 128, torch.bfloat16)])
@pytest.mark.parametrize("which,value", [("q", math.nan), ("k", math.nan), ("k", math.inf), ("v", math.nan)])
def test_nan_reaches_the_same_rows_in_both_forms(dev, which, value, d, block, dtype):
    print(f"case {which} {value} {d} {block} {dtype}", flush=True)
    n, hq, hkv, topk, first, last = 640, 4, 2, 3, 260, 266       # tokens first .. last - 1 of head 1 are set
    q, k, v, do = (x.to(dev) for x in make_qkv(n, hq, hkv, d, dtype, seed=1))
    {"q": q, "k": k, "v": v}[which][first:last, 1] = value       # (q head 1 belongs to kv head 0)
    idx = make_topk_idx([0, n], hkv, block, topk, seed=2)
    idx[:, 500] = -1                                             # a query without a block
    idx[1, 520:530] = first // block                             # queries of nothing but the block with the value
    cut = torch.tensor([0, n], dtype=torch.int32, device=dev)

    pos = torch.arange(n)
    rows = torch.zeros(n, hq, dtype=torch.bool)                  # the rows that the value reaches
    near = rows.clone()                                          # ... and those of the block where 0 * NaN does
    if which == "q":
        rows[first:last, 1] = True
        near = rows
    else:
        chosen = (idx[1] == first // block).any(-1)              # (a key is a whole row of the value: q . k is NaN)
        near[chosen, hq // hkv:] = True
        rows = near if which == "v" else near & (pos >= first)[:, None]   # a score of a later key is masked, its v is multiplied by 0
    assert rows.any() and not rows.all()
    idx, rows, near = idx.to(dev), rows.to(dev), near.to(dev)

    index = ops.build_index(idx, cut, block)
    forms = [ops.selattn_fwd(q, k, v, index), ops.selattn_fwd(q, k, v, index, None, idx)]   # block-major, direct
    assert _lib.load().fsa_selattn_direct_preferred(n, n, hq, d, topk, block, 1) == 1
    for o, lse in forms:
        assert torch.equal(torch.isnan(o).all(-1), rows) and torch.equal(torch.isnan(o).any(-1), rows)
        assert torch.equal(torch.isnan(lse), rows.T if which != "v" else torch.zeros_like(rows.T))
        assert (lse[:, 500] == -math.inf).all() and (o[500] == 0).all()
    _alike(forms[1][0], forms[0][0], O_TOL[dtype])
    _alike(forms[1][1], forms[0][1], LSE_TOL)

    want = ops.selattn_bwd(q, k, v, forms[0][0], do, forms[0][1], index)
    x = [t.detach().requires_grad_() for t in (q, k, v)]
    y = FSA_topk_sparse_attention(*x, idx, block, cut)
    _alike(y, forms[0][0], O_TOL[dtype])
    got = torch.autograd.grad(y, x, do)
    for a, b in zip(got, want):
        _alike(a, b, O_TOL[dtype], ULP[dtype])
    # nothing reaches the other kv head, the rows that the value does not reach, or the keys that none of those selected
    other = 0 if which != "q" else 1
    assert all(torch.isfinite(t[:, other]).all() for t in got[1:])
    assert torch.isfinite(got[0][~near]).all()
