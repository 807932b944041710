"""Kernels with much dynamic LDS need an attribute set on every device that runs them, by whichever call comes first there,
and a call that could not set it must not spoil the next.  The library runs here on a runtime of its own making (a shared
object loaded in front of the real one, in a child process) that has several devices, launches nothing and notes every
launch beyond 64 KB whose kernel has no attribute on the current device.  No GPU is involved."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r"""
#include <cstddef>
#include <cstdint>
#include <map>
#include <utility>
struct dim3 { uint32_t x, y, z; };
static int device = 0, failing = 0, large = 0, refused = 0, launches = 0, oversized = 0;
static std::map<std::pair<const void*, int>, int> limit;
extern "C" {
void stub_set(int d, int f) { device = d; failing = f; }
int stub_large() { return large; }       // launches beyond 64 KB
int stub_refused() { return refused; }   // of those, without an attribute that allows them
int stub_launches() { return launches; }
int stub_oversized() { return oversized; }   // launches with 2^32 or more work-items, or no work-group, in a dimension
int hipGetDevice(int* d) { *d = device; return 0; }
int hipFuncSetAttribute(const void* f, int, int v) {
  if (failing) return 2;
  limit[{f, device}] = v;
  return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t lds, void*) {
  ++launches;
  auto bad = [](uint32_t n, uint32_t t) { return n == 0 || (uint64_t)n * t >= (1ull << 32); };
  if (bad(g.x, b.x) || bad(g.y, b.y) || bad(g.z, b.z)) ++oversized;
  if (lds > 65536) {
    ++large;
    auto it = limit.find({f, device});
    if (it == limit.end() || (size_t)it->second < lds) ++refused;
  }
  return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stub error"; }
static size_t cfg_lds;
static dim3 cfg_grid, cfg_block;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void*) { cfg_grid = g; cfg_block = b; cfg_lds = lds; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
  *g = cfg_grid; *b = cfg_block; *lds = cfg_lds; *s = nullptr; return 0;
}
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* v, const void*, int, size_t) { *v = 8; return 0; }
}
"""

CHILD = r"""
import ctypes as C, os, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from fsa_hip import _lib
lib = _lib.load()
f, big = 0x10000, 1 << 60
calls = {
  "selattn_fwd": lambda: lib.fsa_selattn_fwd(f, f, f, 0, 1024, 256, 1024, 256, 1024, 256, f, 1, 1024, 4, 4, 256, 8, 128, 9, .1,
                                             f, f, f, f, f, f, 1024, 256, f, f, big, None),
  "selattn_bwd": lambda: lib.fsa_selattn_bwd(f, f, f, f, f, f, 0, *[1024, 256] * 5, f, 1, 1024, 4, 4, 256, 8, 128, 9, .1,
                                             f, f, f, f, f, f, f, f, f, big, None),
  "index_once": lambda: lib.fsa_build_index(f, 65536, 16, f, 1, 4096, 4, 16, 64, 1900, f, f, f, f, f, f, big, None),
  "index_place": lambda: lib.fsa_build_index(f, 1 << 20, 16, f, 1, 65536, 4, 16, 16, 4094, f, f, f, f, f, f, big, None),
  "cmpattn_fwd": lambda: lib.fsa_cmpattn_fwd(f, f, f, 0, *[1024, 256] * 3, f, f, 1, 1024, 1024, 4, 4, 256, 32, 16, .1, f, 1024,
                                             256, f, None),
  "cmpattn_bwd": lambda: lib.fsa_cmpattn_bwd(f, f, f, f, f, f, 0, *[1024, 256] * 5, f, f, 1, 1024, 63, 1024, 4, 4, 256, 32, 16,
                                             .1, f, f, f, f, big, None),
  "winattn_fwd": lambda: lib.fsa_winattn_fwd(f, f, f, 0, *[1024, 256] * 3, f, 1, 1024, 1024, 4, 4, 256, 64, .1, f, 1024, 256, f,
                                             None),
  "winattn_bwd": lambda: lib.fsa_winattn_bwd(f, f, f, f, f, f, 0, *[1024, 256] * 5, f, 1, 1024, 1024, 4, 4, 256, 64, .1, f, f, f,
                                             f, big, None),
  "compress_fwd": lambda: lib.fsa_linear_compress_fwd(f, f, f, 0, 16384, 256, f, f, 1, 63, 64, 256, 32, 16, f, None, None),
  "compress_bwd": lambda: lib.fsa_linear_compress_bwd(f, f, f, f, 0, 1024, 256, f, f, 1, 1024, 63, 4, 256, 32, 16, f, f, f, f,
                                                      None),
  "decode_one": lambda: lib.fsa_decode_selattn(f, f, f, 0, 512, 128, 512, 128, 512, 128, f, None, f, 1, 4, 4, 128, 4, 64, .1, f,
                                               f, f, big, None),
  "topk_lds": lambda: lib.fsa_cmp_topk(f, f, f, 0, 256, 64, 256, 64, f, f, 1, 1 << 21, 1 << 21, 131071, 4, 4, 64, 32, 16, 64, 70,
                                       1, 2, 1, 0, .1, f, None, f, big, None),
}
call = calls[sys.argv[3]]
stub.stub_set(0, 1)
rc = call()
assert rc == 2 and b"stub error" in lib.fsa_last_error(), ("a failure is reported", rc, lib.fsa_last_error())
for device in (0, 1, 0, 3, 70):
    stub.stub_set(device, 0)
    before = stub.stub_large()
    rc = call()
    assert rc == 0, ("a failure does not stick", device, rc, lib.fsa_last_error())
    assert stub.stub_large() > before, "the case launches a kernel with much LDS"
    assert stub.stub_refused() == 0, ("attribute missing on device", device)
os._exit(0)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    path = tmp_path_factory.mktemp("stub")
    src, so = path / "stub.cpp", path / "libstub.so"
    src.write_text(STUB)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    return str(so)


@pytest.mark.parametrize("name", ["selattn_fwd", "selattn_bwd", "index_once", "index_place", "cmpattn_fwd", "cmpattn_bwd",
                                  "winattn_fwd", "winattn_bwd", "compress_fwd", "compress_bwd", "decode_one", "topk_lds"])
def test_attribute_is_set_on_every_device(stub, name):
    r = subprocess.run([sys.executable, "-c", CHILD, stub, os.path.join(ROOT, "flash-sparse-attention_amd"), name],
                       capture_output=True, text=True, timeout=120, env={**os.environ, "HIP_VISIBLE_DEVICES": ""})
    assert r.returncode == 0, (r.stdout + r.stderr)[-800:]
