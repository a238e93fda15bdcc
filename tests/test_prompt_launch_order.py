"""Two host threads on one stream, on the CPU: the library's calls into HIP end in a shim that only writes down who launched what, so the order in which launches reach a stream can be read off
without a device."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = r"""
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <unistd.h>
#include <mutex>
#include <vector>
struct Launch { int thread; const void * kernel; };
static std::mutex mu;
static std::vector<Launch> seen;
static thread_local int me = -1;
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t st; } cfg;
extern "C" {
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) { cfg = {grid, block, lds, st}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 * grid, dim3 * block, size_t * lds, hipStream_t * st) { *grid = cfg.grid; *block = cfg.block; *lds = cfg.lds; *st = cfg.st; return hipSuccess; }
hipError_t hipLaunchKernel(const void * f, dim3, dim3, void **, size_t, hipStream_t) {
    { std::lock_guard<std::mutex> lk(mu); seen.push_back({me, f}); }
    usleep(300);                                   // (the other thread's turn)
    return hipSuccess;
}
hipError_t hipMalloc(void ** p, size_t) { *p = malloc(64); return hipSuccess; }
hipError_t hipFree(void * p) { free(p); return hipSuccess; }
hipError_t hipGetDevice(int * d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
void shim_thread(int id) { me = id; }
long shim_seen(int * thread, unsigned long * kernel, long n) {
    std::lock_guard<std::mutex> lk(mu);
    for (long i = 0; i < (long) seen.size() && i < n; ++i) { thread[i] = seen[i].thread; kernel[i] = (unsigned long) seen[i].kernel; }
    return (long) seen.size();
}
}
"""
PROGRAM = r"""
import ctypes as C, sys, threading
shim, lib = C.CDLL(sys.argv[1]), C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_q_wide
f.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p] * 6 + [C.c_int64, C.c_int64, C.c_int, C.c_void_p, C.c_void_p]
shim.shim_seen.restype = C.c_long
K, N, T, CALLS = 8192, 256, 40, 20                     # 32 super-blocks over two row tiles: split along K
buf = C.create_string_buffer(256)
at = C.addressof(buf)
bad = []
def work(i):
    shim.shim_thread(i)
    ty, W, y, n = (C.c_int * 1)(12), (C.c_void_p * 1)(at), (C.c_void_p * 1)(at), (C.c_int64 * 1)(N)
    for _ in range(CALLS):
        rc = f(ty, 1, W, n, y, None, None, at, K, T, 0, at, 1)
        if rc: bad.append(rc)
ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
[t.start() for t in ts]; [t.join() for t in ts]
assert not bad, bad
th, ke = (C.c_int * 4096)(), (C.c_ulong * 4096)()
n = shim.shim_seen(th, ke, 4096)
log = [(th[i], ke[i]) for i in range(n)]
assert n == 2 * CALLS * 3, n                           # quantizer, product, its slices added up
names = [k for t, k in log if t == 0][:3]
assert len(set(names)) == 3, names
both = [e for e in log if e[1] != names[0]]            # (the quantizer writes memory of the call's own)
for i in range(0, len(both), 2):
    t = both[i][0]
    assert both[i:i + 2] == [(t, names[1]), (t, names[2])], (i, both[max(i - 2, 0):i + 4])
switches = sum(log[i][0] != log[i + 1][0] for i in range(n - 1))
assert switches > 4, switches                          # (the threads did meet)
print("ok", n, switches)
"""


def test_slices_of_a_product_are_added_up_before_another_product_of_the_stream(tmp_path):
    """The slices of a product that is split along K wait in scratch memory of the (device, stream) for the launch that adds them up: no other thread's launch of the same kind comes between."""
    lib = os.path.join(ROOT, "prima_cpp_amd", "libprima_mi355.so")
    if not os.path.exists(lib):
        pytest.skip("library not built")
    src, shim = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(src), "-o", str(shim), "-lpthread"], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(shim), lib], env=dict(os.environ, LD_PRELOAD=str(shim)), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
