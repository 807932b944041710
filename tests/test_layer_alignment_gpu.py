"""The attention core of the layer through the C ABI with `v` (and `saved`, where the rotated keys go) at addresses that are
aligned to 8 bytes only: the same bits as with aligned ones, in training and in inference, where short sequences take the kernel
that loads K and V by 16 bytes."""
import ctypes as C
import math

import pytest
import torch

from fsa_hip import _lib
from test_layer_memory import LayerArgs

pytestmark = pytest.mark.gpu


def _shifted(t, shift):
    """A copy of `t` whose first element lies `shift` bytes behind an aligned address."""
    flat = torch.empty(t.numel() * t.element_size() + 256, dtype=torch.uint8, device=t.device)
    out = flat[shift:shift + t.numel() * t.element_size()].view(torch.uint8)
    out.copy_(t.reshape(-1).view(torch.uint8))
    assert out.data_ptr() % 16 == shift
    return out


@pytest.mark.parametrize("inference", [0, 1])
@pytest.mark.parametrize("n,hq,hkv,d,block,dtype", [(333, 4, 2, 128, 64, torch.bfloat16), (97, 2, 1, 64, 32, torch.float16)])
def test_addresses_aligned_to_eight_bytes(dev, n, hq, hkv, d, block, dtype, inference):
    print(f"case {n} {hq} {hkv} {d} {block} {dtype} {inference}", flush=True)
    lib, hidden, topk = _lib.load(), 128, 4
    g = torch.Generator().manual_seed(1)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(dtype).to(dev)

    x, q, k, v = rand(n, hidden), rand(n, hq, d), rand(n, hkv, d), rand(n, hkv, d)
    w_gate, pe = rand(3, hidden, std=0.1), rand(hkv, 32, d)
    w_ck, w_cv = rand(hkv, 32 * d, d, std=0.02), rand(hkv, 32 * d, d, std=0.02)
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    inv_freq = (10000.0 ** (-torch.arange(0, d, 2).float() / d)).to(dev)
    ck = (n - 32) // 16 + 1
    assert lib.fsa_selattn_direct_preferred(n, n, hq, d, min(topk, (n + block - 1) // block), block, 1 - inference) == 1

    def run(shift):
        a = LayerArgs(dtype=0 if dtype == torch.bfloat16 else 1, hidden=hidden, num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
                      kernel_size=32, kernel_stride=16, block_size=block, topk=topk, init_blocks=1, local_blocks=2, window=50,
                      batch=1, inference=inference, total_tokens=n, total_ck=ck, max_len=n, max_ck=ck,
                      softmax_scale=1.0 / math.sqrt(d), rope_scale=1.0)
        a.saved_bytes, a.workspace_bytes = (lib.fsa_layer_saved_bytes(C.byref(a)), lib.fsa_layer_workspace_bytes(C.byref(a), 0))
        # (zeros: padding between the parts is not written)
        saved = _shifted(torch.zeros(a.saved_bytes, dtype=torch.uint8, device=dev), shift)
        ws = _shifted(torch.zeros(a.workspace_bytes, dtype=torch.uint8, device=dev), shift)
        v_ = _shifted(v, shift)
        for name, t in dict(x=x, w_gate=w_gate, q=q, k=k, v=v_, w_ck=w_ck, w_cv=w_cv, pe=pe, cu_seqlens=cu, inv_freq=inv_freq,
                            saved=saved, workspace=ws).items():
            setattr(a, name, t.data_ptr())
        out = torch.full((n, hq * d), math.nan, dtype=dtype, device=dev)
        idx = torch.full((hkv, n, min(topk, (n + block - 1) // block)), -9, dtype=torch.int32, device=dev)
        rc = lib.fsa_layer_forward(C.byref(a), out.data_ptr(), idx.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        _lib.check(rc, "fsa_layer_forward")
        return out, idx

    want, got = run(0), run(8)
    assert torch.isfinite(want[0]).all()
    assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0])
