"""GPU: the layer's backward where a gate rounds to zero.  The fused backward folds the gate into the log-sum-exp of its
branch; a token without a compressed key has no log-sum-exp either (-inf), and the two must not meet as -inf - -inf."""
import pytest
import torch

from fsa.module.fsa import FlashSparseAttention, RopeConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("closed", [0, 1, 2])
def test_closed_gate(dev, closed, dtype):
    print(f"case closed={closed} {dtype}", flush=True)
    torch.manual_seed(closed)
    layer = FlashSparseAttention(256, 4, 2, 64, 32, 16, 64, 4, 1, 2, 64, RopeConfig(head_dim=64)).to(dev).to(dtype)
    lens = [100, 20, 60]                         # the second sequence has no compressed key at all
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    x = torch.randn(sum(lens), 256, device=dev, dtype=dtype)
    x[:, 0] = 1
    with torch.no_grad():
        layer.gate[0].weight[closed, 0] = -200   # sigmoid(-200) is zero in either type
    x.requires_grad_(True)
    dy = torch.randn(sum(lens), 256, device=dev, dtype=dtype)

    def run():
        layer.zero_grad(set_to_none=True)
        x.grad = None
        layer(x, cu).backward(dy)
        return {"x": x.grad, **{n: p.grad for n, p in layer.named_parameters()}}

    got = run()
    layer._fused_core = lambda *a: None
    ref = run()
    tol = 1.5e-2 if dtype == torch.bfloat16 else 3e-3   # as in the comparison of the two forms with open gates
    for name, b in ref.items():
        a = got[name]
        assert torch.isfinite(a.float()).all(), name
        assert ((a.float() - b.float()).norm() / b.float().norm().clamp(min=1e-20)).item() < tol, name
