"""GPU: `fsa_matmul` with FSA_MM_IN_ORDER: a sum is one chain in the order of the contraction, so a result has the same bits
whatever tile the size of the problem leads to."""
import ctypes as C

import pytest
import torch

from fsa_hip import _lib
from test_matmul_gpu import NN, NT, TN, Out, Part

pytestmark = pytest.mark.gpu

IN_ORDER = 4


def _product(form, a, b, m, n, k, flags):
    """c = a b for m rows of the result"""
    c = torch.empty(m, n, device=a.device, dtype=a.dtype)
    o = (Out * 1)()
    o[0].part[0] = Part(a.data_ptr(), b.data_ptr(), a.stride(0), b.stride(0), k)
    o[0].parts, o[0].m, o[0].n, o[0].c, o[0].ldc, o[0].add = 1, m, n, c.data_ptr(), n, None
    code = 0 if a.dtype == torch.bfloat16 else 1
    _lib.check(_lib.load().fsa_matmul(C.addressof(o), 1, form | flags, code, torch.cuda.current_stream().cuda_stream), "fsa_matmul")
    return c


@pytest.mark.parametrize("form", [NT, NN, TN])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [64, 520, 2048])
def test_bits_do_not_depend_on_the_tile(dev, form, dtype, k):
    torch.manual_seed(k)
    m, n = 2176, 2048                                       # 128 x 128 tiles for more than every CU
    a = torch.randn(*((k, m) if form == TN else (m, k)), device=dev, dtype=dtype)
    b = torch.randn(*((n, k) if form == NT else (k, n)), device=dev, dtype=dtype)
    big = _product(form, a, b, m, n, k, IN_ORDER)
    ref = (a.t() if form == TN else a).float() @ (b.t() if form == NT else b).float()
    torch.cuda.synchronize()
    assert ((big.float() - ref).norm() / ref.norm()).item() < (3e-3 if dtype == torch.bfloat16 else 5e-4)
    for rows in (8, 72, 1000, 1544):                        # 64 x 64 tiles, and those that would split the contraction
        assert torch.equal(_product(form, a, b, rows, n, k, IN_ORDER), big[:rows]), rows
