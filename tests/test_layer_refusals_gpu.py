"""GPU: a layer whose weights do not have the sizes of its configuration, or do not live where its input lives, is refused
(as by the composition of the single operators), not run over the end of its weights.  Nothing here reaches a kernel with
sizes that do not fit: the fused calls decline, and the composed layer raises."""
import pytest
import torch

from fsa.module.fsa import FlashSparseAttention, RopeConfig
from fsa_preview.module import FlashSparseAttentionDecode

pytestmark = pytest.mark.gpu

HIDDEN, HQ, HKV, D, KS = 256, 4, 2, 64, 32
N = 200


def _config(ks=KS, d=D, rope_d=D):
    return (HIDDEN, HQ, HKV, d, ks, 16, 64, 4, 1, 2, 64, RopeConfig(head_dim=rope_d))


def _weight(*shape):
    return torch.nn.Parameter(torch.randn(*shape, device="cuda:0", dtype=torch.bfloat16) * 0.02)


def _set(layer, name, value):
    owner, _, attr = name.rpartition(".")
    setattr(layer.get_submodule(owner), attr, value)


WRONG = {   # parameter -> shape that its Linear or LinearCompress does not have
    "proj_q.weight": (HQ * D - 64, HIDDEN), "proj_k.weight": (HKV * D - 64, HIDDEN), "proj_v.weight": (HKV * D // 2, HIDDEN),
    "proj_o.weight": (HIDDEN, HQ * D - 64), "gate.0.weight": (2, HIDDEN), "compress_key": (HKV, KS * D // 2, D),
    "compress_value": (HKV - 1, KS * D, D), "intra_block_pe": (HKV, KS // 2, D),
}
REFUSED = (AssertionError, RuntimeError, ValueError)


def _prefill(layer, x):
    cu = torch.tensor([0, x.shape[0]], dtype=torch.int32, device=x.device)
    return layer._fused_core(x, cu, False), lambda: layer(x, cu)


def _decode(layer, x):
    k = torch.randn(N, HKV, layer.head_dim, device=x.device, dtype=x.dtype)
    ck = torch.randn((N - layer.kernel_size) // 16 + 1, HKV, layer.head_dim, device=x.device, dtype=x.dtype)
    cu = [torch.tensor(c, dtype=torch.int32, device=x.device) for c in ([0, 1], [0, N + 1])]
    return layer._fused_step(x[:1], k, k, ck, ck), lambda: layer(x[:1], *cu, k, k, ck, ck)


@pytest.mark.parametrize("cls,call", [(FlashSparseAttention, _prefill), (FlashSparseAttentionDecode, _decode)])
@pytest.mark.parametrize("name", WRONG)
def test_wrong_sizes(dev, cls, call, name):
    layer = cls(*_config()).to(dev).to(torch.bfloat16)
    x = torch.randn(N, HIDDEN, device=dev, dtype=torch.bfloat16)
    assert call(layer, x)[0] is not None                 # as configured: the fused call runs
    _set(layer, name, _weight(*WRONG[name]))
    fused, run = call(layer, x)
    assert fused is None
    if cls is FlashSparseAttentionDecode and name in ("compress_key", "compress_value", "intra_block_pe"):
        return                                           # this token completes no window: the weights are not used
    with pytest.raises(REFUSED):
        run()


@pytest.mark.parametrize("cls,call", [(FlashSparseAttention, _prefill), (FlashSparseAttentionDecode, _decode)])
@pytest.mark.parametrize("name", ["proj_q.weight", "proj_o.weight", "gate.0.weight", "compress_key", "intra_block_pe"])
def test_weight_on_another_device(dev, cls, call, name):
    layer = cls(*_config()).to(dev).to(torch.bfloat16)
    x = torch.randn(N, HIDDEN, device=dev, dtype=torch.bfloat16)
    _set(layer, name, torch.nn.Parameter(dict(layer.named_parameters())[name].detach().cpu()))
    fused, run = call(layer, x)
    assert fused is None
    if cls is FlashSparseAttentionDecode and name in ("compress_key", "intra_block_pe"):
        return
    with pytest.raises(REFUSED):
        run()


@pytest.mark.parametrize("ks", [48, 80])
def test_window_sizes_that_the_compression_does_not_take(dev, ks):
    layer = FlashSparseAttention(*_config(ks=ks)).to(dev).to(torch.bfloat16)
    x = torch.randn(N, HIDDEN, device=dev, dtype=torch.bfloat16)
    fused, run = _prefill(layer, x)
    assert fused is None
    with pytest.raises(AssertionError):
        run()


@pytest.mark.parametrize("cls,call", [(FlashSparseAttention, _prefill), (FlashSparseAttentionDecode, _decode)])
def test_frequencies_of_another_head_dim(dev, cls, call):
    layer = cls(*_config(rope_d=32)).to(dev).to(torch.bfloat16)
    x = torch.randn(N, HIDDEN, device=dev, dtype=torch.bfloat16)
    fused, run = call(layer, x)
    assert fused is None
    with pytest.raises(AssertionError):
        run()
