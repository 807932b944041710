"""Grids of the largest problems: every dimension of every launch stays below 2^32 work-items, and LDS below what its kernel
is allowed.  Runs on the stand-in for the runtime of test_lds_per_device.py: nothing is launched, no GPU is involved."""
import os
import subprocess
import sys

import pytest

from test_lds_per_device import stub  # noqa: F401  (fixture)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import ctypes as C, os, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2] + "/flash-sparse-attention_amd", sys.argv[2] + "/tests"]
from fsa_hip import _lib
from test_layer_memory import LayerArgs
lib = _lib.load()
f, big = 0x10000, 1 << 60

def dense(batch, longest, others=200, hq=32, hkv=8, d=128):
    n = longest + batch * others
    nc = n // 16
    s = [hq * d, d]
    k = [hkv * d, d]
    return [
        lib.fsa_cmpattn_fwd(f, f, f, 0, *s, *k, *k, f, f, batch, n, longest, hq, hkv, d, 32, 16, .1, f, *s, f, None),
        lib.fsa_winattn_fwd(f, f, f, 0, *s, *k, *k, f, batch, n, longest, hq, hkv, d, 512, .1, f, *s, f, None),
        lib.fsa_cmpattn_bwd(f, f, f, f, f, f, 0, *s, *k, *k, *s, *s, f, f, batch, n, nc, longest, hq, hkv, d, 32, 16, .1, f, f, f,
                            f, big, None),
        lib.fsa_winattn_bwd(f, f, f, f, f, f, 0, *s, *k, *k, *s, *s, f, batch, n, longest, hq, hkv, d, 512, .1, f, f, f, f, big,
                            None),
        lib.fsa_cmp_topk(f, f, f, 0, *s, *k, f, f, batch, n, longest, longest // 16, hq, hkv, d, 32, 16, 64, 16, 1, 2, 1, 0, .1, f,
                         None, f, big, None)]

def layer(batch, longest, n, hq=32, hkv=8, d=128, hidden=4096):
    ck = longest // 16
    a = LayerArgs(dtype=1, hidden=hidden, num_q_heads=hq, num_kv_heads=hkv, head_dim=d, kernel_size=32, kernel_stride=16,
                  block_size=64, topk=16, init_blocks=1, local_blocks=2, window=512, batch=batch, total_tokens=n,
                  total_ck=n // 16, max_len=longest, max_ck=ck, softmax_scale=.1, rope_scale=1.)
    for name, t in LayerArgs._fields_:
        if t is C.c_void_p:
            setattr(a, name, f)
    a.saved_bytes = a.workspace_bytes = big
    grads = (C.c_void_p * 9)(*[f] * 9)
    return [lib.fsa_layer_forward(C.byref(a), f, f, None), lib.fsa_layer_backward(C.byref(a), C.byref(grads), None)]

cases = {
  "dense_one_long_of_600": lambda: dense(600, 131072),
  "dense_100000_short": lambda: dense(100000, 100, 20),
  "dense_one": lambda: dense(1, 1 << 20),
  "layer_one_long_of_600": lambda: layer(600, 131072, 131072 + 600 * 200),
  "layer_one": lambda: layer(1, 1 << 19, 1 << 19),
  "layer_wide": lambda: layer(1, 800000, 800000, hq=8, hkv=2, hidden=8192),   # chunks of the gate's pass over x
  "layer_d256": lambda: layer(3, 4000, 5000, hq=4, hkv=2, d=256),
}
stub.stub_set(0, 0)
rc = cases[sys.argv[3]]()
assert not any(rc), (rc, lib.fsa_last_error())
print("launches", stub.stub_launches(), "oversized", stub.stub_oversized(), "lds", stub.stub_refused())
assert stub.stub_launches() > 3 and stub.stub_oversized() == 0 and stub.stub_refused() == 0, (stub.stub_oversized(), stub.stub_refused())
os._exit(0)
"""


@pytest.mark.parametrize("name", ["dense_one_long_of_600", "dense_100000_short", "dense_one", "layer_one_long_of_600",
                                  "layer_one", "layer_wide", "layer_d256"])
def test_grids_of_large_problems(stub, name):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", CHILD, stub, ROOT, name], capture_output=True, text=True, timeout=120,
                       env={**os.environ, "HIP_VISIBLE_DEVICES": ""})
    assert r.returncode == 0, (r.stdout + r.stderr)[-600:]
