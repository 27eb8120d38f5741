"""A stand-in for the HIP runtime, for tests of the library's host code
without a GPU: device memory is host memory, copies are done at once, kernels
are counted and not run.  `run` starts a Python process in which the stub's
functions come before the runtime's; `script` sees `lib` (the package's
bindings), `stub` (the functions below) and numpy as np."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>
#include <map>
#include <mutex>
#include <vector>
namespace {
std::mutex mu;
struct Copy { const void *dst, *src; size_t bytes; int kind; };
struct Limit { const void *f; int value; };
std::vector<Copy> copies;
std::vector<Limit> limits;
std::map<const char *, size_t> pinned, device;
int fail_pinned, fail_malloc, mallocs, launches, syncs;
float event_ms;
dim3 cfg_grid, cfg_block;
size_t cfg_lds;
hipStream_t cfg_stream;
void *take(std::map<const char *, size_t> &m, size_t n) {
    char *p = static_cast<char *>(calloc(n ? n : 1, 1));
    std::lock_guard<std::mutex> lk(mu);
    m[p] = n;
    return p;
}
void drop(std::map<const char *, size_t> &m, void *p) {
    std::lock_guard<std::mutex> lk(mu);
    m.erase(static_cast<char *>(p));
    free(p);
}
bool inside(const std::map<const char *, size_t> &m, const void *p) {
    auto it = m.upper_bound(static_cast<const char *>(p));
    return it != m.begin() && (--it, static_cast<const char *>(p) < it->first + it->second);
}
hipError_t copy(void *d, const void *s, size_t n, int kind) {
    memcpy(d, s, n);
    std::lock_guard<std::mutex> lk(mu);
    copies.push_back({d, s, n, kind});
    return hipSuccess;
}
}  // namespace
extern "C" {
void stub_fail_pinned(int on) { fail_pinned = on; }
void stub_fail_malloc(int k) { fail_malloc = k; mallocs = 0; }  // the k-th hipMalloc from here fails
int stub_mallocs() { return mallocs; }
void stub_clear() { std::lock_guard<std::mutex> lk(mu); copies.clear(); limits.clear(); launches = syncs = 0; }
int stub_syncs() { return syncs; }
int stub_copies() { return (int)copies.size(); }
const void *stub_copy_dst(int i) { return copies[i].dst; }
const void *stub_copy_src(int i) { return copies[i].src; }
long stub_copy_bytes(int i) { return (long)copies[i].bytes; }
int stub_limits() { return (int)limits.size(); }
const void *stub_limit_kernel(int i) { return limits[i].f; }
int stub_limit_value(int i) { return limits[i].value; }
int stub_launches() { return launches; }
long stub_pinned() { return (long)pinned.size(); }
void *stub_pin(long n) { return take(pinned, n); }
void *stub_device(long n) { return take(device, n); }

hipError_t hipMalloc(void **p, size_t n) {
    if (++mallocs == fail_malloc) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = take(device, n);
    return hipSuccess;
}
hipError_t hipFree(void *p) { drop(device, p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (fail_pinned) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = take(pinned, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { drop(pinned, p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::lock_guard<std::mutex> lk(mu);
    memset(a, 0, sizeof *a);
    a->type = inside(pinned, p) ? hipMemoryTypeHost : inside(device, p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v) {
    std::lock_guard<std::mutex> lk(mu);
    limits.push_back({f, v});
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *m = take(device, (size_t)128 << 20);
    *p = m;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { launches++; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    cfg_grid = g; cfg_block = b; cfg_lds = l; cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) {
    *g = cfg_grid; *b = cfg_block; *l = cfg_lds; *s = cfg_stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(malloc(1)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = event_ms += 1.0f; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(malloc(1)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { syncs++; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { *d = 0; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub error"; }
}
"""

PRELUDE = r"""
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for f, r, a in (("stub_copy_dst", C.c_void_p, [C.c_int]), ("stub_copy_src", C.c_void_p, [C.c_int]),
                ("stub_copy_bytes", C.c_long, [C.c_int]), ("stub_limit_kernel", C.c_void_p, [C.c_int]),
                ("stub_pinned", C.c_long, []), ("stub_pin", C.c_void_p, [C.c_long]),
                ("stub_device", C.c_void_p, [C.c_long])):
    getattr(stub, f).restype, getattr(stub, f).argtypes = r, a
sys.path.insert(0, sys.argv[2])
import numpy as np
import mms_gpu as mg
lib = mg.lib()
F = np.float32
def copies():
    return [(stub.stub_copy_dst(i), stub.stub_copy_src(i), stub.stub_copy_bytes(i)) for i in range(stub.stub_copies())]
def limits():
    return [(stub.stub_limit_kernel(i), stub.stub_limit_value(i)) for i in range(stub.stub_limits())]
"""


def run(tmp_path, script):
    src, so = tmp_path / "stub.cpp", tmp_path / "stub.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-w", "-std=c++17", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", str(so), str(src)],
                   check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, str(so), os.path.join(ROOT, "mms-gpu_amd")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
