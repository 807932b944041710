"""GPU: dQ, dK and dV of window and compressed attention where q and dO go straight to LDS, against the kernel that takes any rows (the same
tensors one element off their alignment): GQA groups that fill a pass of 64 rows in different ways, key tiles and passes that end early,
tiles of one work-group and of several, rows of a head far apart or not.  (Statistics as two arrays; a layer hands over pairs.)"""
import pytest
import torch

from fsa_hip import ops

pytestmark = pytest.mark.gpu


def _off(x):
    """the same values, one element off the alignment"""
    flat = torch.empty(x.numel() + 8, device=x.device, dtype=x.dtype)[1:1 + x.numel()].view(x.shape)
    assert flat.data_ptr() % 16 != 0
    return flat.copy_(x)


def _heads_first(x):
    return x.transpose(0, 1).contiguous().transpose(0, 1)


@pytest.mark.parametrize("lens,hq,hkv,d,window,dtype", [
    ([1, 63, 64, 65], 4, 4, 128, 512, torch.bfloat16),     # one key, a tile less one, a tile, a tile and one
    ([700, 31, 129], 4, 2, 64, 100, torch.float16),
    ([1000], 8, 2, 128, 1, torch.bfloat16),                # a query sees two keys
    ([2100, 40], 16, 2, 128, 127, torch.float16),          # the window ends inside a wave's keys
    ([515], 64, 4, 64, 200, torch.bfloat16),               # four queries to a pass
    ([300, 77], 64, 1, 128, 64, torch.bfloat16),           # one query to a pass
    ([5000], 32, 8, 128, 512, torch.bfloat16),             # key tiles of one work-group
    ([300], 128, 1, 64, 64, torch.float16),                # (no whole query in a pass: as gathered rows)
    ([900, 20], 6, 2, 128, 128, torch.bfloat16),           # (three heads to a group: the same)
    ([900, 33], 8, 2, 256, 200, torch.bfloat16),           # (head_dim 256: the same; dQ of keys off their alignment keeps dO in LDS)
    ([40, 31, 515], 4, 4, 256, 64, torch.float16),
])
@pytest.mark.parametrize("heads_first", [False, True])
def test_forms(dev, lens, hq, hkv, d, window, dtype, heads_first):
    print(f"case lens={lens} hq={hq} hkv={hkv} d={d} window={window} {dtype} heads_first={heads_first}", flush=True)
    gen = torch.Generator().manual_seed(sum(lens) + hq)
    n = sum(lens)
    rand = lambda *s: torch.randn(*s, generator=gen).to(dev, dtype)   # noqa: E731
    q, k, v, do = rand(n, hq, d), rand(n, hkv, d), rand(n, hkv, d), rand(n, hq, d)
    n_ck = [max(0, (x - 32) // 16 + 1) for x in lens]
    ck, cv = rand(max(1, sum(n_ck)), hkv, d)[:sum(n_ck)], rand(max(1, sum(n_ck)), hkv, d)[:sum(n_ck)]
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    cu_ck = torch.tensor([0] + torch.tensor(n_ck).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    if heads_first:
        q, do = _heads_first(q), _heads_first(do)
    # one rounding of the result on either side, and probabilities that are rounded the other way: fp32 sums of another order
    tol = 4e-3 if dtype == torch.bfloat16 else 6e-4
    o, lse = ops.winattn_fwd(q, k, v, cu, max(lens), window)
    oc, lsec = ops.cmpattn_fwd(q, ck, cv, 32, 16, cu, cu_ck, max(lens))
    for name, k_, v_, run in (
            ("window", k, v, lambda q, k, v, do: ops.winattn_bwd(q, k, v, o, do, lse, cu, max(lens), window)),
            ("compressed", ck, cv, lambda q, k, v, do: ops.cmpattn_bwd(q, k, v, oc, do, lsec, 32, 16, cu, cu_ck, max(lens)))):
        got, want = run(q, k_, v_, do), run(_off(q.contiguous()), k_, v_, _off(do.contiguous()))
        # keys and values that cannot go straight to LDS take the same steps through the registers
        assert all(torch.equal(x, y) for x, y in zip(got, run(q, _off(k_), _off(v_), do))), name
        for part, x, y in zip(("dq", "dk", "dv"), got, want):
            assert torch.isfinite(x.float()).all(), (name, part)
            if y.numel():
                err = ((x.float() - y.float()).norm() / y.float().norm().clamp_min(1e-20)).item()
                assert err < tol, (name, part, err)


def test_rows_that_are_not_visible(dev):
    """A query whose q and log-sum-exp are NaN reaches dK and dV of no tile without a key that it sees, and in the other tiles dV of
    no key that it does not see."""
    n, window, dtype = 400, 50, torch.bfloat16
    gen = torch.Generator().manual_seed(5)
    q, k, v, do = (torch.randn(n, 4, 128, generator=gen).to(dev, dtype) for _ in range(4))
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    o, lse = ops.winattn_fwd(q, k, v, cu, n, window)
    _, dk, dv = ops.winattn_bwd(q, k, v, o, do, lse, cu, n, window)
    q2, lse2 = q.clone(), lse.clone()
    q2[200] = float("nan")           # keys 150 .. 200 see it
    lse2[:, 200] = float("nan")
    _, dk2, dv2 = ops.winattn_bwd(q2, k, v, o, do, lse2, cu, n, window)
    for keys in (slice(0, 128), slice(256, 400)):    # tiles of 64 keys without one of them
        assert torch.equal(dk[keys], dk2[keys]) and torch.equal(dv[keys], dv2[keys])
    assert torch.isfinite(dv2[128:150].float()).all() and torch.isnan(dv2[150:201].float()).all()
