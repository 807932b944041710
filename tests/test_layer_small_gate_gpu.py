"""GPU: precision of the fp16 layer's value gradients where the gates are small.  dV is a product of probabilities times
gate with the output gradient; gate times probability is far below fp16's normal range there."""
import math

import pytest
import torch

from fsa.module.fsa import FlashSparseAttention, RopeConfig
from oracle.module import fsa_layer_ref

pytestmark = pytest.mark.gpu


def _errors(dev, gate):
    """Relative errors against the fp32 oracle of the gradients that come from dV, every block selected."""
    torch.manual_seed(0)
    n, hidden, hq, hkv, d = 1024, 64, 2, 1, 64
    layer = FlashSparseAttention(hidden, hq, hkv, d, 32, 16, 64, 16, 1, 2, n, RopeConfig(head_dim=d)).to(dev).half()
    x = torch.randn(n, hidden, device=dev, dtype=torch.float16)
    x[:, 0] = 1
    with torch.no_grad():
        layer.gate[0].weight.zero_()
        layer.gate[0].weight[:, 0] = math.log(gate / (1 - gate))
    # the size of the gradients grows as the gates shrink: dV itself stays in the normal range
    dy = (torch.randn(n, hidden, device=dev) / gate).half()
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    y, idx = layer(x, cu, return_topk_idx=True)
    y.backward(dy)
    names = ["proj_v.weight", "compress_value"]
    params = {k: p.detach().cpu().float().requires_grad_(k in names) for k, p in layer.named_parameters()}
    cfg = dict(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, kernel_size=32, kernel_stride=16, block_size=64, topk=16,
               init_blocks=1, local_blocks=2, window_size=n, inv_freq=layer.rope.table(torch.device("cpu")))
    ref, _, _ = fsa_layer_ref(params, x.cpu(), [0, n], cfg, topk_idx=idx.cpu(), table_dtype=torch.float16)
    grads = torch.autograd.grad(ref, [params[k] for k in names], dy.cpu().float())
    got = dict(layer.named_parameters())
    return {k: ((got[k].grad.cpu().float() - g).norm() / g.norm()).item() for k, g in zip(names, grads)}


@pytest.mark.parametrize("gate", [0.02, 0.002, 0.0002])
def test_value_gradients_with_small_gates(dev, gate):
    usual, small = _errors(dev, 0.5), _errors(dev, gate)
    for name in usual:
        print(f"  {name}: error {usual[name]:.1e} at gate 0.5, {small[name]:.1e} at {gate}", flush=True)
        # the same arithmetic on the same values but for the gate: no more than the scatter of the errors
        assert small[name] < 1.5 * usual[name], name
