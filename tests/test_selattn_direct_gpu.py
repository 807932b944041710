"""The query-major forward of short sequences (fsa_selattn_direct_fwd) against attention written out in float64 and against
the block-major kernels, over the forms of block lists that both take."""
import math

import pytest
import torch

from fsa.ops import FSA_topk_sparse_attention
from fsa_hip import _lib, ops
from synth_inputs import make_qkv, make_topk_idx

pytestmark = pytest.mark.gpu

# bounds of the forward's tests: rounding of the probabilities (2^-9, 2^-12) and of the result to the type
O_TOL = {torch.bfloat16: 2e-2, torch.float16: 5e-3}
LSE_TOL = 1e-3


def _direct(q, k, v, idx, cu, block, max_len=None):
    n, hq, d = q.shape
    o, lse = torch.empty(n, hq, d, dtype=q.dtype, device=q.device), torch.empty(hq, n, device=q.device)
    _lib.check(_lib.load().fsa_selattn_direct_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), 0 if q.dtype == torch.bfloat16 else 1, q.stride(0), q.stride(1), k.stride(0),
        k.stride(1), v.stride(0), v.stride(1), idx.data_ptr(), idx.stride(0), idx.stride(1), cu.data_ptr(), cu.numel() - 1, n,
        max_len or n, hq, k.shape[1], d, idx.shape[2], block, 1.0 / math.sqrt(d), o.data_ptr(), o.stride(0), o.stride(1),
        lse.data_ptr(), torch.cuda.current_stream().cuda_stream), "direct")
    torch.cuda.synchronize()
    return o, lse


def _reference(q, k, v, idx, cu, block):
    """float64, a block that a list names m times weighted m times; NaN and infinite values only reach who selected them."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    o, lse = torch.zeros(n, hq, d, dtype=torch.float64), torch.full((hq, n), -math.inf, dtype=torch.float64)
    q, k, v = (x.double().cpu() for x in (q, k, v))
    idx, cu = idx.cpu(), cu.tolist()
    for s0, s1 in zip(cu, cu[1:]):
        m = s1 - s0
        if m == 0:
            continue
        nb = (m + block - 1) // block
        for h in range(hkv):
            ids = idx[h, s0:s1].long()
            times = torch.zeros(m, nb + 1).scatter_add_(1, torch.where((ids < 0) | (ids >= nb), nb, ids), torch.ones(ids.shape))
            w = times[:, :nb].repeat_interleave(block, 1)[:, :m].double()
            w = w * (torch.arange(m)[:, None] >= torch.arange(m)[None, :])
            for j in range(hq // hkv):
                hh = h * (hq // hkv) + j
                s = q[s0:s1, hh] @ k[s0:s1, h].nan_to_num(0, 0, 0).T / math.sqrt(d)
                bad = ~torch.isfinite(k[s0:s1, h]).all(1)
                s = torch.where(bad[None, :], math.nan, s)
                s = torch.where(w > 0, s + torch.log(w), -math.inf)
                l_ = torch.logsumexp(s, 1)
                p = torch.where(w > 0, torch.exp(s - l_[:, None]), 0.0)
                bad = ~torch.isfinite(v[s0:s1, h]).all(1)
                r = p @ v[s0:s1, h].nan_to_num(0, 0, 0)
                r[(w[:, bad] > 0).any(1)] = math.nan
                seen = (w > 0).any(1)
                o[s0:s1, hh] = torch.where(seen[:, None], r, 0.0)
                lse[hh, s0:s1] = torch.where(seen, l_ / math.log(2.0), -math.inf)
    return o, lse


def _check(got, ref, dtype):
    for x, y, tol in ((got[0].double().cpu(), ref[0], O_TOL[dtype]), (got[1].double().cpu(), ref[1], LSE_TOL)):
        assert torch.equal(torch.isnan(x), torch.isnan(y))
        same = torch.isnan(y) | (x == y)    # (infinite values)
        assert torch.where(same, 0.0, (x - y).abs()).max().item() <= tol


CASES = [
    # cu_seqlens, Hq, Hkv, D, block, T, dtype
    ([0, 1], 1, 1, 128, 64, 1, torch.bfloat16),                       # a single key
    ([0, 31, 63, 96], 2, 2, 128, 64, 4, torch.bfloat16),              # around one row tile
    ([0, 33, 161], 4, 1, 64, 32, 3, torch.float16),                   # an odd number of steps of 32 keys
    ([0, 127, 256, 385], 2, 1, 256, 128, 2, torch.bfloat16),
    ([0, 300], 6, 2, 128, 32, 5, torch.float16),                      # group of 3: queries across row tiles
    ([0, 200], 80, 1, 64, 64, 3, torch.bfloat16),                     # group larger than a row tile
    ([0, 0, 450, 450, 513], 16, 1, 128, 128, 3, torch.bfloat16),      # empty sequences
    ([0, 700], 4, 4, 64, 128, 4, torch.bfloat16),
    ([0, 420], 4, 2, 256, 64, 4, torch.float16),
    ([0, 390], 2, 2, 256, 32, 8, torch.bfloat16),
    ([0, 640], 80, 80, 128, 64, 6, torch.bfloat16),                   # two waves per work-group (more than 1536 row tiles)
]


@pytest.mark.parametrize("cu,hq,hkv,d,block,topk,dtype", CASES)
def test_matches_reference(dev, cu, hq, hkv, d, block, topk, dtype):
    print(f"case {cu} {hq} {hkv} {d} {block} {topk} {dtype}", flush=True)
    q, k, v = (x.to(dev) for x in make_qkv(cu[-1], hq, hkv, d, dtype, seed=1, with_do=False))
    cut = torch.tensor(cu, dtype=torch.int32, device=dev)
    idx = make_topk_idx(cu, hkv, block, topk, seed=2).to(dev)
    longest = max(b - a for a, b in zip(cu, cu[1:]))
    _check(_direct(q, k, v, idx, cut, block, longest), _reference(q, k, v, idx, cut, block), dtype)


# Sizes that the rule gives to the kernels of many row tiles: two row tiles and two key groups, four row tiles and one group (at
# least 3e7 rows x keys).  Row tiles that are not full, whose queries lie in two of them, without keys, of several sequences.
MANY_ROWS = [
    # cu_seqlens, Hq, Hkv, D, block, T, dtype, kv heads looked at
    ([0, 1501], 32, 32, 128, 64, 16, torch.bfloat16, [0, 31]),             # 2 x 2
    ([0, 1990], 12, 12, 256, 128, 4, torch.float16, [0, 11]),              # (one row tile still, of head_dim 256)
    ([0, 2301], 20, 20, 256, 128, 4, torch.float16, [0, 19]),              # 2 x 2
    ([0, 3100], 24, 8, 64, 32, 8, torch.bfloat16, [3]),                    # 2 x 2, a query in two row tiles
    ([0, 33, 33, 240], 1536, 512, 128, 32, 5, torch.float16, [0, 511]),    # 1 x 4, the same, an empty sequence
    ([0, 129, 260], 1024, 1024, 128, 64, 3, torch.bfloat16, [0, 1023]),    # 1 x 4, a row tile of one row
    ([0, 310], 1200, 20, 64, 64, 4, torch.bfloat16, [0, 19]),              # 1 x 4, group larger than a row tile
    ([0, 190, 383], 384, 384, 256, 128, 2, torch.bfloat16, [0, 383]),      # 1 x 4
]


@pytest.mark.parametrize("cu,hq,hkv,d,block,topk,dtype,heads", MANY_ROWS)
@pytest.mark.parametrize("kind", ["plain", "twice", "nan"])
def test_many_row_tiles(dev, cu, hq, hkv, d, block, topk, dtype, heads, kind):
    print(f"case {cu} {hq} {hkv} {d} {block} {topk} {dtype} {kind}", flush=True)
    q, k, v = (x.to(dev) for x in make_qkv(cu[-1], hq, hkv, d, dtype, seed=1, with_do=False))
    cut = torch.tensor(cu, dtype=torch.int32, device=dev)
    idx = make_topk_idx(cu, hkv, block, topk, seed=2).to(dev)
    if kind == "twice":
        idx[:, ::5, -1] = idx[:, ::5, 0]
    if kind == "nan":
        s0 = cu[-2]   # first key of a block: every query that selected the block sees it
        v[s0 + (cu[-1] - s0) // block // 2 * block] = math.nan
    o, lse = _direct(q, k, v, idx, cut, block, max(b - a for a, b in zip(cu, cu[1:])))
    g = hq // hkv
    for h in heads:
        mine = slice(h * g, h * g + g)
        _check((o[:, mine], lse[mine]), _reference(q[:, mine], k[:, h:h + 1], v[:, h:h + 1], idx[h:h + 1], cut, block), dtype)


def _odd_lists(n, hkv, block, topk, kind):
    g = torch.Generator().manual_seed(3)
    nb = (n + block - 1) // block
    own = torch.arange(n) // block
    idx = make_topk_idx([0, n], hkv, block, topk, seed=4)
    if kind == "shuffled":      # any order, padding in front and between
        perm = torch.rand(idx.shape, generator=g).argsort(-1)
        return idx.gather(-1, perm)
    if kind == "twice":         # the first id again in the last place
        idx[..., -1] = idx[..., 0]
    if kind == "later":         # blocks behind the query's own, and ids that are no block
        idx[..., -1] = torch.minimum(own + 1, torch.tensor(nb - 1))
        idx[:, ::3, -2] = nb + 5
    if kind == "nothing":       # queries without a block, and with nothing they may see
        idx[:, 5::7] = -1
        idx[:, 6::7] = torch.where(own[6::7] + 1 < nb, own[6::7] + 1, -1)[None, :, None]
    return idx.to(torch.int32)


@pytest.mark.parametrize("kind", ["shuffled", "twice", "later", "nothing"])
@pytest.mark.parametrize("d,block", [(128, 64), (64, 32), (128, 128)])
def test_forms_of_lists(dev, d, block, kind):
    n, hq, hkv, topk = 500, 4, 2, 4
    q, k, v = (x.to(dev) for x in make_qkv(n, hq, hkv, d, torch.float16, seed=5, with_do=False))
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    idx = _odd_lists(n, hkv, block, topk, kind).to(dev)
    got = _direct(q, k, v, idx, cu, block)
    _check(got, _reference(q, k, v, idx, cu, block), torch.float16)
    o, lse = ops.selattn_fwd(q, k, v, ops.build_index(idx, cu, block))   # the block-major kernels on the same lists
    _check(got, (o.double().cpu(), lse.double().cpu()), torch.float16)


@pytest.mark.parametrize("value", [math.inf, math.nan])
@pytest.mark.parametrize("which", ["k", "v"])
def test_infinite_values_reach_only_who_selected_them(dev, which, value):
    n, hq, hkv, d, block, topk = 512, 2, 1, 128, 64, 3
    q, k, v = (x.to(dev) for x in make_qkv(n, hq, hkv, d, torch.bfloat16, seed=6, with_do=False))
    (k if which == "k" else v)[130:140] = value
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    idx = make_topk_idx([0, n], hkv, block, topk, seed=7)
    idx[:, 192:] = torch.where(idx[:, 192:] == 2, 1, idx[:, 192:])       # block 2: its own queries only ...
    idx[:, 300, 0] = 2                                                   # ... and one more
    idx = idx.to(dev)
    o, lse = _direct(q, k, v, idx, cu, block)
    hit = (idx[0] == 2).any(-1)
    clean = torch.isfinite(o).all(-1).all(-1)
    assert not clean[hit][-1] and clean[~hit].all()
    ref = _reference(q, k, v, idx, cu, block)[0]
    assert (o.double().cpu() - ref)[~hit.cpu()].abs().max().item() <= O_TOL[torch.bfloat16]


def test_strides_and_operator(dev):
    """Rows of a fused projection, a strided list, a block of 256 keys, and the operator's own choice of this path."""
    n, hq, hkv, d = 600, 8, 2, 128
    g = torch.Generator().manual_seed(8)
    qkv = torch.randn(n, (hq + 2 * hkv) * d, generator=g).to(torch.bfloat16).to(dev)
    q, k, v = (x.view(n, -1, d) for x in qkv.split([hq * d, hkv * d, hkv * d], 1))
    cu = torch.tensor([0, 250, n], dtype=torch.int32, device=dev)
    wide = torch.full((hkv, n, 9), 7, dtype=torch.int32, device=dev)
    wide[..., :6] = make_topk_idx([0, 250, n], hkv, 64, 6, seed=9).to(dev)
    idx = wide[..., :6]
    ref = _reference(q, k, v, idx, cu, 64)
    _check(_direct(q, k, v, idx, cu, 64), ref, torch.bfloat16)
    assert _lib.load().fsa_selattn_direct_preferred(n, n, hq, d, 6, 64, 1) == 1
    assert (FSA_topk_sparse_attention(q, k, v, idx, 64, cu).double().cpu() - ref[0]).abs().max().item() <= O_TOL[torch.bfloat16]
    idx = make_topk_idx([0, 250, n], hkv, 256, 2, seed=10).to(dev)
    ref = _reference(q, k, v, idx, cu, 256)[0]
    assert (FSA_topk_sparse_attention(q, k, v, idx, 256, cu).double().cpu() - ref).abs().max().item() <= O_TOL[torch.bfloat16]


def test_refuses(dev):
    q, k, v = (x.to(dev) for x in make_qkv(256, 2, 2, 128, torch.bfloat16, seed=11, with_do=False))
    cu = torch.tensor([0, 256], dtype=torch.int32, device=dev)
    idx = make_topk_idx([0, 256], 2, 64, 2, seed=12).to(dev)
    with pytest.raises(ValueError):
        _direct(q, k[:1].expand(256, 2, 128), v, idx, cu, 64)            # rows of k overlap
    with pytest.raises(ValueError):
        _direct(q, k, v, idx, cu, 64, 257)
    with pytest.raises(ValueError):
        _direct(q, k, v, idx, cu, 48)


@pytest.mark.parametrize("hq,hkv,d,block,topk", [(2, 1, 128, 64, 3), (4, 4, 64, 32, 20), (1, 1, 256, 128, 3), (80, 80, 128, 64, 6)])
@pytest.mark.parametrize("kind", ["own", "none", "late"])
def test_first_blocks_that_nobody_selected(dev, hq, hkv, d, block, topk, kind):
    """What is requested ahead is not visited: lists of the own block only, of nothing for whole row tiles, of late blocks with
    more entries than are requested at once."""
    print(f"case {hq} {hkv} {d} {block} {topk} {kind}", flush=True)
    n, cu = 641, [0, 641]
    q, k, v = (x.to(dev) for x in make_qkv(n, hq, hkv, d, torch.bfloat16, seed=5, with_do=False))
    k[:2 * block], v[:2 * block] = math.nan, math.nan
    own = torch.arange(n) // block
    idx = torch.full((hkv, n, topk), -1, dtype=torch.int32)
    if kind != "none":
        for t in range(topk if kind == "late" else 1):
            idx[..., t] = torch.where((own - t >= 2) & (torch.arange(n) % 160 > 70), own - t, -1).int()
    idx, cut = idx.to(dev), torch.tensor(cu, dtype=torch.int32, device=dev)
    _check(_direct(q, k, v, idx, cut, block), _reference(q, k, v, idx, cut, block), torch.bfloat16)


def test_line_between_the_forms(dev):
    """Where an index is built anyway the line lies lower; the two forms agree in between."""
    lib = _lib.load()
    sides = [[lib.fsa_selattn_direct_preferred(n, n, 4, 128, 16, 64, needed) for n in range(500, 9000, 500)] for needed in (0, 1)]
    assert all(x == sorted(x, reverse=True) and x[0] == 1 and x[-1] == 0 for x in sides) and sum(sides[0]) > sum(sides[1])
    n = 6000
    assert [lib.fsa_selattn_direct_preferred(n, n, 4, 128, 16, 64, needed) for needed in (0, 1)] == [1, 0]
    q, k, v = (x.to(dev) for x in make_qkv(n, 4, 4, 128, torch.bfloat16, seed=11, with_do=False))
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    idx = make_topk_idx([0, n], 4, 64, 16, seed=12).to(dev)
    alone = FSA_topk_sparse_attention(q, k, v, idx, 64, cu)
    trained = FSA_topk_sparse_attention(q.requires_grad_(), k, v, idx, 64, cu)
    assert (alone.float() - trained.float()).abs().max().item() <= O_TOL[torch.bfloat16]


def _kernels(run):
    run()
    torch.cuda.synchronize()
    _lib.profile_enable(True)
    out = run()
    torch.cuda.synchronize()
    names = {name for name, _ in _lib.profile_records()}
    _lib.profile_enable(False)
    return out, names


def test_packed_batch_is_not_priced_as_one_sequence(dev):
    """Where one sequence of all the tokens would take the block-major kernels, a batch of documents does not."""
    n, hq, d = 3000, 4, 256
    lib = _lib.load()
    assert [lib.fsa_selattn_direct_preferred(n, m, hq, d, 6, 64, 1) for m in (n, n - n // 4)] == [0, 1]
    cu = [0, 800, 1500, 2300, n]
    q, k, v = (x.to(dev) for x in make_qkv(n, hq, hq, d, torch.bfloat16, seed=13, with_do=False))
    cut, idx = torch.tensor(cu, dtype=torch.int32, device=dev), make_topk_idx(cu, hq, 64, 6, seed=14).to(dev)
    o, names = _kernels(lambda: FSA_topk_sparse_attention(q, k, v, idx, 64, cut))
    assert names == {"selattn_direct_fwd"}
    ref = _reference(q, k, v, idx, cut, 64)[0]
    assert (o.double().cpu() - ref).abs().max().item() <= O_TOL[torch.bfloat16]
    q.requires_grad_()
    _, names = _kernels(lambda: FSA_topk_sparse_attention(q, k, v, idx, 64, cut))
    assert "selattn_direct_fwd" in names and "selattn_fwd_main" not in names


def test_packed_batch_beyond_the_tables(dev):
    """A batch with more blocks than the direct kernels have tables for, long lists that would make them the cheaper ones."""
    n, block, topk = 33000, 32, 512
    assert _lib.load().fsa_selattn_direct_preferred(n, n - n // 4, 1, 64, topk, block, 0) == 1 and n > 1024 * block
    q, k, v = (x.to(dev) for x in make_qkv(n, 1, 1, 64, torch.bfloat16, seed=15, with_do=False))
    cu, cut = [0, 200, n], torch.tensor([0, 200, n], dtype=torch.int32, device=dev)
    own = torch.cat([torch.arange(b - a) // block for a, b in zip(cu, cu[1:])])
    idx = (own[None, :, None] - torch.arange(topk)).clamp_(min=-1).int().to(dev)     # the last 512 blocks
    o, names = _kernels(lambda: FSA_topk_sparse_attention(q, k, v, idx, block, cut))
    assert "selattn_direct_fwd" not in names and torch.isfinite(o.float()).all()
    for row in (0, 199, 200, 17000, n - 1):
        s0 = 0 if row < 200 else 200
        lo = max(s0, s0 + ((row - s0) // block - topk + 1) * block)
        p = torch.softmax((k[lo:row + 1, 0].double() @ q[row, 0].double()) / 8, 0)
        assert (o[row, 0].double() - p @ v[lo:row + 1, 0].double()).abs().max().item() <= O_TOL[torch.bfloat16]
