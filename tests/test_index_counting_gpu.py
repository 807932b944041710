"""GPU: counting kernels of the index at the edges of their variants (bits of a bucket, copies of a counter, lists that lie apart
in memory, repeated ids): every array bit-exact against the oracle, work lists against the block counts."""
import numpy as np
import pytest
import torch

from fsa_hip import _lib
from oracle import selattn as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("lens,hkv,bk,t", [
    ([9000], 2, 128, 16),              # 73 buckets: seven bits
    ([8300], 1, 64, 16),               # 132 buckets: the most with a copy of every counter per lane
    ([8300, 30], 1, 64, 16),           # 134
    ([20000], 2, 32, 8),               # 627
    ([40000], 1, 32, 4),               # 1252
    ([131008], 1, 32, 1),              # 4096 buckets, the most that there are
    ([30001], 1, 64, 5),               # tiles that are no whole number of rounds
])
def test_counting_kernels(dev, lens, hkv, bk, t, apart):
    print(f"case lens={lens} hkv={hkv} bk={bk} t={t} apart={apart}", flush=True)
    lib = _lib.load()
    rng = np.random.default_rng(t)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, batch = int(cu[-1]), len(lens)
    own = np.concatenate([np.arange(x) for x in lens]) // bk
    # any ids up to the own block, some padding, some out of range, some twice in a list
    topk = (rng.integers(0, 1 << 30, (hkv, n, t)) % (own[None, :, None] + 1)).astype(np.int32)
    topk[..., 0] = 0
    topk[rng.random(topk.shape) < 0.1] = -1
    topk[rng.random(topk.shape) < 0.01] = 1 << 20
    topk[:, ::97, -1] = topk[:, ::97, 0]
    mb = (n + bk - 1) // bk + batch
    i32 = dict(dtype=torch.int32, device=dev)
    idx = torch.full((hkv, n, t + 3), 1, **i32)[..., :t] if apart else torch.empty((hkv, n, t), **i32)
    idx.copy_(torch.from_numpy(topk))
    cu_t = torch.from_numpy(cu).to(dev)
    out = [torch.full(s, -7, **i32) for s in ((batch + 1,), (hkv, mb), (hkv, mb + 1), (hkv, n * t), (hkv, n, t))]
    tiles = [torch.full((lib.fsa_selattn_tiles_bytes(b, n, hkv, hkv, 128, t, bk, mb) // 4,), -7, **i32) for b in (0, 1)]
    nbytes = lib.fsa_index_workspace_bytes(n, t, hkv, mb)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    _lib.check(lib.fsa_build_index_tiles(idx.data_ptr(), idx.stride(0), idx.stride(1), cu_t.data_ptr(), batch, n, hkv, t,
                                         bk, mb, *[x.data_ptr() for x in out], hkv, 128, tiles[0].data_ptr(),
                                         tiles[1].data_ptr(), ws.data_ptr(), nbytes, None), "fsa_build_index_tiles")
    torch.cuda.synchronize()
    ref = orc.build_index_ref(torch.from_numpy(topk), cu.tolist(), bk)
    nb = int(ref[0][-1])
    assert np.array_equal(out[0].cpu().numpy(), ref[0])
    assert np.array_equal(out[1].cpu().numpy()[:, :nb], ref[1])
    assert np.array_equal(out[2].cpu().numpy()[:, :nb + 1], ref[2])
    assert np.array_equal(out[3].cpu().numpy(), ref[3]) and np.array_equal(out[4].cpu().numpy(), ref[4])
    for mem in tiles:
        prefix = mem[:hkv * (mb + 1)].view(hkv, mb + 1).cpu().numpy()
        block = mem[hkv * (mb + 1):].view(hkv, -1).cpu().numpy()
        per_block = np.diff(prefix, axis=1)
        assert ((per_block > 0) == (out[1].cpu().numpy() > 0)).all()
        for h in range(hkv):
            want = np.repeat(np.arange(mb), per_block[h])
            assert prefix[h, 0] == 0 and np.array_equal(block[h, :len(want)], want)
