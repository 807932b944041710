"""GPU: the fused decode step rotates a cached key by the angles that prefill rotates it by, also at far positions, where
the fp32 rounding of position times frequency decides the 16-bit cosine and sine.

One head, one active pair of dims and one-hot value rows make every probability of the window branch visible in the output,
and the softmax scale of the scores makes one step of a cosine's 16-bit form a change of three per cent."""
import pytest
import torch

from fsa.module.fsa import RopeConfig
from fsa_preview.module import FlashSparseAttentionDecode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pair", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("L", [70000, 131000])
def test_angles_of_far_keys(dev, L, pair):
    d, hidden, n = 64, 64, 64                       # the window holds as many keys as a value row has dims
    mod = FlashSparseAttentionDecode(hidden, 1, 1, d, 32, 16, 64, 16, 1, 2, n - 1, RopeConfig(head_dim=d))
    with torch.no_grad():
        for p in mod.parameters():
            p.zero_()
        mod.proj_q.weight[pair, 0] = 64.0           # scores of up to 64 / sqrt(64) = 8
        mod.proj_k.weight[pair, 0] = 1.0
        mod.proj_v.weight[d - 1, 0] = 1.0
        mod.proj_o.weight.copy_(torch.eye(d))
        mod.gate[0].weight[:, 0] = torch.tensor([-80.0, -80.0, 80.0])
    mod = mod.to(dev).to(torch.bfloat16)
    k = torch.zeros(L, 1, d, device=dev, dtype=torch.bfloat16)
    k[:, 0, pair] = 1
    v = torch.zeros_like(k)
    v[torch.arange(L - n + 1, L, device=dev), 0, torch.arange(n - 1, device=dev)] = 1
    nc = (L - 32) // 16 + 1
    ck = torch.zeros(nc, 1, d, device=dev, dtype=torch.bfloat16)
    x = torch.zeros(1, hidden, device=dev, dtype=torch.bfloat16)
    x[0, 0] = 1
    cu_q, cu_k = (torch.tensor(c, dtype=torch.int32, device=dev) for c in ([0, 1], [0, L + 1]))
    assert mod._fused_step(x, k, v, ck, ck) is not None
    got = mod(x, cu_q, cu_k, k, v, ck, ck).float()[0]
    mod._fused_step = lambda *a: None               # rotates the caches by the kernel that prefill uses
    ref = mod(x, cu_q, cu_k, k, v, ck, ck).float()[0]
    assert (ref > 0).all() and abs(ref.sum().item() - 1) < 0.02
    ratio = (got / ref).log()
    off = ((ratio - ratio.median()).abs() > 0.015).sum().item()   # two bf16 roundings of the output are below 0.008
    print(f"  L={L} pair={pair}: {off} of {n} keys", flush=True)
    # the hardware's sine and cosine are good to about 1e-6: one entry in some thousands rounds the other way
    assert off <= 1
