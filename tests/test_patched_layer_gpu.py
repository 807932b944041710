"""GPU: a layer with a submodule that was patched (activation capture, adapters, quantised weights) runs the patch."""
import pytest
import torch

from fsa.module.fsa import FlashSparseAttention, RopeConfig
from fsa_preview.module import FlashSparseAttentionDecode

pytestmark = pytest.mark.gpu

CONFIG = (256, 4, 2, 64, 32, 16, 64, 4, 1, 2, 64, RopeConfig(head_dim=64))


def _call(layer, dev):
    gen = torch.Generator(device=dev).manual_seed(0)

    def rows(*shape):
        return torch.randn(*shape, device=dev, dtype=torch.bfloat16, generator=gen)

    with torch.no_grad():
        if isinstance(layer, FlashSparseAttention):
            return layer(rows(200, 256), torch.tensor([0, 200], dtype=torch.int32, device=dev))
        cu = [torch.tensor(c, dtype=torch.int32, device=dev) for c in ([0, 1], [0, 201])]
        return layer(rows(1, 256), *cu, rows(200, 2, 64), rows(200, 2, 64), rows(11, 2, 64), rows(11, 2, 64))


@pytest.mark.parametrize("cls,name", [(FlashSparseAttention, "proj_v"), (FlashSparseAttention, "proj_o"),
                                      (FlashSparseAttention, "gate.1"), (FlashSparseAttentionDecode, "proj_o"),
                                      (FlashSparseAttentionDecode, "gate.1")])
def test_instance_forward(dev, cls, name):
    torch.manual_seed(0)
    layer = cls(*CONFIG).to(dev)
    for p in layer.parameters():
        torch.nn.init.xavier_uniform_(p)
    layer = layer.to(torch.bfloat16)
    usual = _call(layer, dev)
    m, seen = layer.get_submodule(name), []
    plain = m.forward
    m.forward = lambda x: seen.append(1) or 2 * plain(x)
    patched = _call(layer, dev)
    assert seen
    # the output is linear in what the patch doubles, and the selection does not depend on it; the two routes round apart
    err = ((patched.float() - 2 * usual.float()).norm() / usual.float().norm()).item()
    assert err < 5e-2


def test_global_hook(dev):
    layer = FlashSparseAttention(*CONFIG).to(dev).to(torch.bfloat16)
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, y: seen.append(type(m).__name__) and None)
    try:
        _call(layer, dev)
    finally:
        handle.remove()
    assert seen.count("Linear") == 5 and "RotaryEmbedding" in seen
