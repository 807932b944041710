"""GPU: `fsa_matmul` on both sides of the lines between its tiles, with contractions that end inside a step, against fp32 products;
a result that keeps the order of its sum is the same bits whatever tile computes it."""
import ctypes as C

import pytest
import torch

from fsa_hip import _lib
from test_matmul_gpu import NN, NT, TN, Out, Part

pytestmark = pytest.mark.gpu
IN_ORDER = 4


def _run(results, form, dtype):
    outs = (Out * len(results))()
    for o, (c, parts, add) in zip(outs, results):
        for i, (a, b, k) in enumerate(parts):
            o.part[i] = Part(a.data_ptr(), b.data_ptr(), a.stride(0), b.stride(0), k)
        o.parts, o.m, o.n, o.c, o.ldc = len(parts), c.shape[0], c.shape[1], c.data_ptr(), c.stride(0)
        o.add = add.data_ptr() if add is not None else None
    _lib.check(_lib.load().fsa_matmul(C.addressof(outs), len(results), form, 0 if dtype == torch.bfloat16 else 1,
                                      torch.cuda.current_stream().cuda_stream), "fsa_matmul")
    torch.cuda.synchronize()


@pytest.mark.parametrize("form", [NT, NN, TN])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,ks", [
    (8, 8, [8]),                # less than a tile and a step
    (520, 520, [520]),          # 64 x 64, split: nine steps for two groups
    (1024, 1024, [448, 72]),    # the last that is split, two pairs of operands
    (1032, 1024, [520]),        # 64 x 64, whole
    (1544, 1416, [200]),        # short contraction
    (2048, 1024, [1032]),       # 128 x 64, split
    (2048, 1024, [520, 512]),
    (2056, 1032, [1032]),       # 128 x 128, split
    (2056, 2048, [200]),        # 128 x 128, whole
])
def test_tiles(dev, form, dtype, m, n, ks):
    print(f"case form={form} {m}x{n} {ks} {dtype}", flush=True)
    torch.manual_seed(m + n)
    if form != TN:
        m -= 3 if m > 8 else 7
    parts, ref = [], 0
    for k in ks:
        if form == TN:
            k -= 3
        a = torch.randn(*((k, m) if form == TN else (m, k)), device=dev, dtype=dtype)
        b = torch.randn(*((n, k) if form == NT else (k, n)), device=dev, dtype=dtype)
        parts.append((a, b, k))
        ref = ref + (a.t() if form == TN else a).float() @ (b.t() if form == NT else b).float()
    c = torch.full((m, n + 8), 7.0, device=dev, dtype=dtype)
    _run([(c[:, :n], parts, None)], form, dtype)
    # one rounding of the result (2^-9, 2^-12), fp32 sums
    err = ((c[:, :n].float() - ref).norm() / ref.norm()).item()
    assert err < (3e-3 if dtype == torch.bfloat16 else 5e-4), err
    assert (c[:, n:] == 7.0).all()


@pytest.mark.parametrize("k", [264, 2056])
def test_order_of_the_sum(dev, k):
    torch.manual_seed(k)
    a, b = torch.randn(4100, k, device=dev, dtype=torch.bfloat16), torch.randn(1032, k, device=dev, dtype=torch.bfloat16)
    many, few = (torch.empty(rows, 1032, device=dev, dtype=torch.bfloat16) for rows in (4100, 300))
    _run([(many, [(a, b, k)], None)], NT | IN_ORDER, a.dtype)   # 128 x 128
    _run([(few, [(a[:300], b, k)], None)], NT | IN_ORDER, a.dtype)   # 64 x 64
    assert torch.equal(many[:300], few)
