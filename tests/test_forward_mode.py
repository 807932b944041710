"""Forward-mode differentiation is not implemented: a tangent must be refused, not dropped.  (The refusal comes before
any look at the device.)"""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from fsa.module.fsa import FlashSparseAttention, RopeConfig
from fsa.ops import FSA_topk_sparse_attention
from fsa_hip import ops
from fsa_preview.module import FlashSparseAttentionDecode


def _dual(t):
    return fwAD.make_dual(t, torch.ones_like(t))


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("grad", [True, False])
def test_operator(which, grad):
    qkv = [torch.randn(64, 2, 64, dtype=torch.bfloat16) for _ in range(3)]
    idx = torch.zeros(2, 64, 1, dtype=torch.int32)
    cu = torch.tensor([0, 64], dtype=torch.int32)
    with fwAD.dual_level(), torch.set_grad_enabled(grad):
        qkv[which] = _dual(qkv[which])
        with pytest.raises(NotImplementedError):
            FSA_topk_sparse_attention(*qkv, idx, 64, cu)


CONFIG = (128, 2, 1, 64, 32, 16, 64, 4, 1, 2, 64, RopeConfig(head_dim=64))


@pytest.mark.parametrize("which", ["x", "proj_q.weight", "proj_o.weight", "gate.0.weight", "compress_key", "compress_value",
                                   "intra_block_pe"])
@pytest.mark.parametrize("grad", [True, False])
def test_layer(which, grad):
    layer = FlashSparseAttention(*CONFIG).to(torch.bfloat16)
    x = torch.randn(64, 128, dtype=torch.bfloat16)
    t = {"x": x, **dict(layer.named_parameters())}
    with fwAD.dual_level(), torch.set_grad_enabled(grad):
        t[which] = _dual(t[which].detach())
        with pytest.raises(NotImplementedError):
            ops.layer_core(t["x"], torch.tensor([0, 64], dtype=torch.int32),
                           tuple(t[f"proj_{n}.weight"] for n in "qkvo"), t["gate.0.weight"], t["compress_key"],
                           t["compress_value"], t["intra_block_pe"], layer.rope.table(x.device), 1.0,
                           (2, 1, 64, 32, 16, 64, 4, 1, 2, 64, 128), False)


def test_decode_step():
    layer = FlashSparseAttentionDecode(*CONFIG).to(torch.bfloat16)
    k, ck = torch.randn(100, 1, 64, dtype=torch.bfloat16), torch.randn(5, 1, 64, dtype=torch.bfloat16)
    x = torch.randn(1, 128, dtype=torch.bfloat16)
    with fwAD.dual_level():
        for args in ((_dual(x), k, k, ck, ck), (x, _dual(k), k, ck, ck), (x, k, k, ck, _dual(ck))):
            with pytest.raises(NotImplementedError):
                layer._fused_step(*args)
