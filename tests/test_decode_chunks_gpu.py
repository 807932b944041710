"""GPU: decode attention whose (request, kv head) pairs have several work-groups, the last of which merges: edges of the sizes it
is chosen for, recorded calls, a workspace that holds anything."""
import math

import pytest
import torch

from fsa_hip import _lib, ops
from test_decode_one_gpu import _reference

pytestmark = pytest.mark.gpu


def _case(dev, n_keys, hq, hkv, d, dtype, seed=0):
    torch.manual_seed(seed)
    total = sum(n_keys) + 1
    q = torch.randn(len(n_keys), hq, d, device=dev, dtype=dtype)
    k, v = (torch.randn(total, hkv, d, device=dev, dtype=dtype) for _ in range(2))
    cu = torch.tensor([0] + torch.tensor(n_keys).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    pos = torch.tensor([31 + 16 * max(n - 1, 0) if n else 5 for n in n_keys], dtype=torch.int32, device=dev)
    return q, k, v, cu, pos


@pytest.mark.parametrize("n_keys,hq,hkv,d,dtype", [
    ([513], 4, 1, 128, torch.bfloat16),               # 17 tiles for 20 waves
    ([2049, 0, 33], 8, 2, 128, torch.float16),        # requests with fewer tiles than work-groups, and with none
    ([8192, 1], 4, 1, 64, torch.bfloat16),            # 64 work-groups per pair
    ([32768], 2, 1, 64, torch.float16),               # ... of four tiles per wave
    ([32769], 2, 1, 64, torch.float16),               # one key more: shares of the persistent grid
    ([1025, 700], 34, 2, 256, torch.bfloat16),        # two launches per group
    ([1030] * 16, 16, 16, 128, torch.bfloat16),       # 256 pairs, a tile more than two work-groups of each would take: shares
    ([1030] * 20, 8, 8, 128, torch.float16),          # 160 pairs of three work-groups
    ([1000] * 12, 16, 8, 128, torch.bfloat16),        # 96 pairs of five, four tiles for a wave of a single one
    ([700] * 12, 16, 8, 128, torch.float16),          # ... three tiles: a single one
    ([1000] * 16, 16, 8, 64, torch.bfloat16),         # head_dim 64: a single one, too
    ([700, 520] * 8, 12, 6, 64, torch.float16),       # 96 pairs of it
    ([700] * 19, 10, 5, 64, torch.bfloat16),          # 95: five work-groups
    ([530] * 24, 8, 4, 256, torch.bfloat16),          # head_dim 256, half as many in all: two for each of 96 pairs
    ([1000, 600] * 16, 8, 4, 256, torch.float16),     # ... of 128
    ([530] * 43, 6, 3, 256, torch.float16),           # 129 pairs: one would be left
])
def test_compressed(dev, n_keys, hq, hkv, d, dtype):
    print(f"case n_keys={n_keys[:3]} x{len(n_keys)} hq={hq} hkv={hkv} d={d} {dtype}", flush=True)
    q, k, v, cu, pos = _case(dev, n_keys, hq, hkv, d, dtype)
    o, lse, raw = ops.decode_cmpattn(q, k, v, cu, pos, 32, 16, max(n_keys))
    for i, n in enumerate(n_keys):
        at = int(cu[i])
        ref = _reference(q[i], k, v, [range(at, at + n)] * hkv)
        assert (o[i].float() - ref).abs().max().item() < (2e-2 if dtype == torch.bfloat16 else 3e-3)
        assert n > 0 or torch.isinf(lse[:, i]).all()
        for h in range(hkv if n else 0):
            s = k[at:at + n, h].float() @ q[i, h * (hq // hkv)].float()
            assert (raw[h, i, :n] - s).abs().max().item() < 1e-2


def test_replays(dev):
    """A recorded call finds its own numbers nowhere, however often it runs, and eager calls in between change nothing."""
    q, k, v, cu, pos = _case(dev, [3000, 200], 8, 2, 128, torch.bfloat16)
    idx = torch.arange(20, dtype=torch.int32, device=dev).expand(2, 2, 20).contiguous()

    def step():
        return (*ops.decode_cmpattn(q, k, v, cu, pos, 32, 16, 3000), *ops.decode_selattn(q, k, v, cu, idx, 64))

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for i in range(5):
        q.copy_(torch.randn(q.shape, device=dev))
        want = step()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(out, want):
            x, y = (t[..., :200] if t.dim() == 3 and t.shape[-1] > 200 else t for t in (x, y))   # (scores of keys that exist)
            assert torch.equal(x, y)


def test_any_workspace(dev):
    lib = _lib.load()
    q, k, v, cu, pos = _case(dev, [4000, 2500], 8, 2, 128, torch.float16)
    want, want_lse, _ = ops.decode_cmpattn(q, k, v, cu, pos, 32, 16, 4000)
    n = lib.fsa_decode_workspace_bytes(2, 8, 2, 128, 4000)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    o, lse = torch.empty_like(want), torch.empty_like(want_lse)
    for fill in (255, 0, None, None):   # None: what the call before has left
        if fill is not None:
            ws.fill_(fill)
        o.fill_(math.nan)
        _lib.check(lib.fsa_decode_cmpattn(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0),
            v.stride(1), cu.data_ptr(), pos.data_ptr(), 2, 8, 2, 128, 32, 16, 1.0 / math.sqrt(128), 0, 4000, o.data_ptr(),
            lse.data_ptr(), None, 0, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream), "decode_cmpattn")
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(lse, want_lse)
