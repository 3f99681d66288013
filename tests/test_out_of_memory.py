"""Calls that keep workspaces, with every one of their device allocations failing in turn: the failed
call reports it, and a second call either has all of its workspaces or reports it again, so that no
kernel is launched on a buffer that is not there. Runs on the CPU: the HIP runtime's entry points are
a small stand-in whose allocations are host memory, whose copies are memcpy and whose launches do
nothing, loaded ahead of the library in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STAND_IN = r"""
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
#include <map>
static long countdown = -1;
static std::map<void*, size_t> live;
extern "C" {
void stand_in_fail_at(long n) { countdown = n; }
long stand_in_failed() { return countdown < -1; }
long stand_in_live(long* sizes, long cap) {
    long k = 0;
    for (auto& a : live) if (k < cap) sizes[k++] = (long)a.second;
    return (long)live.size();
}
hipError_t hipMalloc(void** p, size_t n) {
    if (countdown >= 0 && countdown-- == 0) { countdown = -2; *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::calloc(n + 1, 1);
    live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) { if (p) { live.erase(p); std::free(p); } return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(n + 1, 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (n && (!d || !s)) return hipErrorInvalidValue;
    if (n) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    if (n && !d) return hipErrorInvalidValue;
    if (n) std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->warpSize = 64; p->multiProcessorCount = 256; p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 64; return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char s[1 << 16]; *p = s; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)0x10; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)0x20; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.01f; return hipSuccess; }
}
"""

PROGRAM = r"""
import ctypes, sys
stand_in = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/muscade.jl_amd"]
import numpy as np
import muscade_amd as mc
from muscade_amd import _lib
from muscade_amd._lib import dptr, i64ptr, lib
from muscade_amd.workloads import base_section

def live():
    sizes = (ctypes.c_long * 4096)()
    n = stand_in.stand_in_live(sizes, 4096)
    return sorted(sizes[:n])

def context(OX):
    m = mc.Model("beams")
    mc.addnode(m, np.array([[0., 0., 0.], [1., 0., 0.], [2., 0., 0.], [9., 9., 9.]]))
    mc.addelement(m, mc.EulerBeam3D, np.array([[1, 2]]), mat=base_section(), orient2=np.array([0., 1., 0.]))
    mc.addelement(m, mc.EulerBeam3DAU, np.array([[2, 3, 4, 4]]), mat=base_section(), orient2=np.array([0., 1., 0.]),
                  scaled=("EA",), afield="k")
    st = mc.initialize(m, nXder=3)
    return mc.AssemblySweepX(OX, m, st.dis)

def vjp(a, OX):
    err = _lib.mh_err()
    lib.mh_vjp_lagrangian(a.ctx.h, OX, ctypes.byref(err))    # (no kernel runs: the flag word is not looked at)
    return lib.mh_last_error(a.ctx.h).decode()

def chained(a):
    pos = np.arange(1, a.nX + 1, dtype=np.int64)
    a.ctx.check(lib.mh_chain_prepare(a.ctx.h, 6, a.nX // 6, i64ptr(pos), 0, None, 0, None), "chain")

idx, val = np.arange(1, 4, dtype=np.int64), np.ones(3)
def sparse(a):
    lib.mh_adjoint_solve_sparse(a.ctx.h, 3, i64ptr(idx), dptr(val), 1.)
    return lib.mh_last_error(a.ctx.h).decode()
def newton(a):
    r = lib.mh_newton_prepare(a.ctx.h, dptr(np.ones(a.nX)))
    if r:
        norms = np.zeros(2)
        assert lib.mh_newton_update(a.ctx.h, 0, 1, None, dptr(norms)) == _lib.MH_ERR_ARG, "update without its workspaces"
    return lib.mh_last_error(a.ctx.h).decode()

def with_lambda(a):
    a.ctx.check(lib.mh_set_lambda(a.ctx.h, dptr(np.zeros(a.nX))), "lambda")
def with_newton(a):
    chained(a)
    newton(a)

if sys.argv[3] == "records":   # 64 to a tile, 69 and 137 numbers a record at first and second order, 57 without derivatives
    def records(numbers):
        return 2 * 64 * numbers * 8      # the two groups' tiles
    a = context(1)
    with_lambda(a)
    assert records(69) in live() and records(137) not in live(), live()
    vjp(a, 1)
    assert records(69) in live(), live()
    vjp(a, 2)
    assert records(137) in live() and records(69) not in live(), live()
    vjp(a, 1)
    assert records(137) in live(), live()
    del a
    a = context(1)                       # no room for the larger ones: the smaller ones stay
    with_lambda(a)
    vjp(a, 1)
    stand_in.stand_in_fail_at(0)
    assert "out of memory" in vjp(a, 2)
    assert records(69) in live()
    vjp(a, 2)
    assert records(137) in live() and records(69) not in live(), live()
    del a
    a = context(0)
    assert not {records(57), records(69), records(137)} & set(live()), live()
    d = mc.AssemblyDirect(0, 0, 0, a.model, a.dis, nA=a.model.ndof["A"])
    assert records(57) in live(), live()
    print("checked")
    sys.exit()

cases = {"adjoint of a static preparation": (0, with_lambda, lambda a: vjp(a, 2)),
         "adjoint": (2, with_lambda, lambda a: vjp(a, 2)),
         "sparse adjoint solve": (0, with_newton, sparse),
         "decrement": (0, chained, newton)}
OX, before, call = cases[sys.argv[3]]
a = context(OX)
before(a)
base = len(live())
call(a)
whole = live()
assert len(whole) > base, "the call allocates nothing"
del a
failures = 0
for n in range(100):
    a = context(OX)
    before(a)
    stand_in.stand_in_fail_at(n)
    said = call(a)
    failed = stand_in.stand_in_failed()
    stand_in.stand_in_fail_at(-1)
    if failed:
        failures += 1
        assert "out of memory" in said, (n, said)
    call(a)
    assert live() == whole, (n, len(live()), len(whole))
    del a
    if not failed:
        break
assert failures > 1, failures
print("checked", failures, "failures")
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    d = tmp_path_factory.mktemp("stand_in")
    src, so = d / "stand_in.cpp", d / "stand_in.so"
    src.write_text(STAND_IN)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(src), "-o", str(so)],
                   check=True)
    return so


@pytest.mark.parametrize("call", ["adjoint of a static preparation", "adjoint", "sparse adjoint solve", "decrement"])
def test_failed_allocation_leaves_nothing_half_made(stand_in, call):
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(stand_in), ROOT, call], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "checked" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


def test_records_take_the_order_in_use(stand_in):
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(stand_in), ROOT, "records"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "checked" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]
