"""The pinned chunks of a large domain's read-back are a help, not a need.

The library runs in a child process over a stand-in for the HIP runtime whose
device memory is host memory and whose kernels do nothing, but for the one that
copies a chunk, so that a pinned allocation, an event or a device switch can be
refused at will.  A field set
and read back then goes through the staging buffer and back: the bytes that
come out are those that went in, whichever way they were copied.
"""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "weldformgpu_amd", "libwfhip.so")

SHIM = r"""
#include <atomic>
#include <cstdlib>
#include <cstring>
static std::atomic<int> events{0}, live{0}, pinned_copies{0};
static thread_local int sticky = 0;
static char *pin_lo = nullptr, *pin_hi = nullptr;
static int num(const char* k) { const char* v = getenv(k); return v ? atoi(v) : 0; }
static int refuse() { sticky = 2; return 2; }
static int grab(void** p, size_t n) { *p = calloc(1, n ? n : 1); live++; return 0; }
static int drop(void* p) { if (p) live--; free(p); return 0; }
extern "C" {
int wf_test_live() { return live; }
int wf_test_pinned_copies() { return pinned_copies; }
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
static const void* copy_chunk = nullptr;
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  if (strstr(name, "k_copy_chunk")) copy_chunk = f;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
struct Dim3 { unsigned x, y, z; };
static thread_local Dim3 grid_, block_;
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t, void*) { grid_ = g; block_ = b; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** s) {
  *g = grid_; *b = block_; *lds = 0; *s = nullptr;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t, void*) {
  if (f != copy_chunk) return 0;
  const char* src = *(const char**)args[0];
  char* dst = *(char**)args[1];
  const int bytes = *(int*)args[2];
  if (dst < pin_lo || dst + bytes > pin_hi || 16ull * grid.x * block.x < (unsigned)bytes) abort();
  pinned_copies++;
  memcpy(dst, src, bytes);
  return 0;
}
int hipExtLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*, void*, void*, int) { return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return num("REFUSE_SET_DEVICE") ? refuse() : 0; }
int hipGetLastError() { int e = sticky; sticky = 0; return e; }
const char* hipGetErrorString(int) { return "refused"; }
int hipMalloc(void** p, size_t n) { return grab(p, n); }
int hipFree(void* p) { return drop(p); }
int hipHostMalloc(void** p, size_t n, unsigned) {
  if (n >= (1u << 20)) {
    if (num("REFUSE_PINNED")) return refuse();
    grab(p, n);
    pin_lo = (char*)*p;
    pin_hi = pin_lo + n;
    return 0;
  }
  return grab(p, n);
}
int hipHostFree(void* p) { return drop(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  memcpy(d, s, n);
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) {
  return ++events == num("REFUSE_EVENT") ? refuse() : grab(e, 1);
}
int hipEventCreate(void** e) { return grab(e, 1); }
int hipEventDestroy(void* e) { return drop(e); }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* f, void*, void*) { *f = 0.f; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return grab(s, 1); }
int hipStreamDestroy(void* s) { return drop(s); }
int hipStreamSynchronize(void*) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return 0; }
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from weldformgpu_amd import _abi
from weldformgpu_amd.domain import Domain
n = 300000
cfg = _abi.default_config()
cfg.n_particles = cfg.solid_count = n
cfg.h_glob = cfg.dt = 1.0
a = np.random.default_rng(1).standard_normal((n, 6))
for _ in range(2):
    with Domain(cfg) as d:
        for k, v in (("sigma", a), ("T", a[:, 0])):
            d.set(k, v)
            assert np.array_equal(d.get(k), v), k
    assert shim.wf_test_live() == 0, shim.wf_test_live()
print("pinned copies", shim.wf_test_pinned_copies())
"""


@pytest.mark.parametrize("refused", ["", "REFUSE_PINNED=1", "REFUSE_EVENT=1", "REFUSE_EVENT=5",
                                     "REFUSE_SET_DEVICE=1"])
def test_read_back_without_pinned_chunks(tmp_path, refused):
    if not os.path.exists(LIB):
        pytest.fail("libwfhip.so is not built")
    src, shim = tmp_path / "shim.cpp", tmp_path / "libshim.so"
    src.write_text(SHIM)
    subprocess.run([shutil.which("g++"), "-O1", "-shared", "-fPIC", str(src), "-o", str(shim)],
                   check=True)
    env = dict(os.environ, PYTHONPATH=ROOT)
    if refused:
        env.update([refused.split("=")])
    r = subprocess.run([sys.executable, "-c", CHILD, str(shim)], env=env, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    copies = int(r.stdout.split()[-1])
    if refused in ("", "REFUSE_SET_DEVICE=1"):
        assert copies == 2 * 14  # a 14.4 MB field twice, in chunks of 1 MiB
    elif refused == "REFUSE_PINNED=1":
        assert copies == 0
