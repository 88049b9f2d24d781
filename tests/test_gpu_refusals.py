"""Launch options that are refused, or accepted, whatever kernel the lattice runs on."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT


def _load(kq, lat):
    fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3, seed_fat=21, seed_long=22)
    kq.kuqcd_gauge_free()
    kq.load_gauge_pair(fat, lng, lat)


# split kernels at every size of the first lattice; one thread per site for FP64 on the second
@pytest.mark.gpu
@pytest.mark.parametrize("lat", [(6, 5, 4, 3), (20, 20, 20, 14)])
def test_blocking_options_that_no_kernel_has(gpu, lat):
    """Threads per block other than 64, 128 and 256 and blocks other than 1, 2, 3, 4 and 8 vectors are
    refused by the timing entry point and the solvers, also where the kernel that runs has a block
    size of its own; the library works on afterwards."""
    kq = gpu
    _load(kq, lat)
    b = [kq.gen_source(lat, 0, seed=3)]
    p = kq.InvertParam(shifts=np.array([[0.5, 0.2]]), tol=1.0, max_iter=50, num_shift=2)
    for mode in (1, 2, 3, 4):
        for nr, nt in ((1, 32), (1, 100), (2, 512), (5, 64), (6, 256)):
            print("case", lat, mode, nr, nt, flush=True)
            assert kq.bench_dslash(mode, 1, nr, nt, 1)[0] != 0, "timing"
            x = [np.zeros_like(b[0]) for _ in range(2)]
            opt = kq.default_options(mode=mode, rel_tol=1e-6, nr=nr, nt=nt, verbose=0)
            assert kq.solve_batched(x, b, p, opt)[0] != 0, "solve"
            assert "unsupported" in kq.last_error()
        x = [np.zeros_like(b[0]) for _ in range(2)]
        opt = kq.default_options(mode=mode, rel_tol=1e-6, nr=1, nt=128, verbose=0)
        assert kq.solve_batched(x, b, p, opt)[0] == 0, kq.last_error()
        assert kq.bench_dslash(mode, 1, 1, 128, 1)[0] == 0, kq.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("lat", [(6, 5, 4, 3), (16, 16, 16, 16)])
def test_autotuning_for_any_number_of_vectors(gpu, lat):
    """The blocking is timed on blocks, not on the caller's number of vectors: none, and more than the
    card holds or a launch has blocks for, get an answer on any lattice."""
    kq = gpu
    _load(kq, lat)
    for mode in (1, 2):
        for nrhs in (0, 1, 1000000):
            print("case", lat, mode, nrhs, flush=True)
            nr, nt = C.c_int(), C.c_int()
            assert kq.L.lib().kq_autotune_dslash(mode, nrhs, C.byref(nr), C.byref(nt)) == 0, kq.last_error()
            assert nr.value in ((1, 2) if mode == 1 else (1, 2, 3, 4, 8)) and nt.value in (64, 128, 256)


_SHIM = """
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
int moved = 0;
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    static hipError_t (*real)(hipPointerAttribute_t *, const void *);
    if (!real)
        real = dlsym(dlopen("/opt/rocm/lib/libamdhip64.so.7", RTLD_LAZY), "hipPointerGetAttributes");
    if (!real)
        return hipErrorNotFound;
    hipError_t e = real(a, p);
    if (e == hipSuccess && a->type == hipMemoryTypeDevice) {
        ++a->device;
        ++moved;
    }
    return e;
}
"""

_PEER = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
shim = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
import numpy as np
import kuqcd_amd.api as kq
kq.set_verbosity(0)
assert kq.kuqcd_init() == kq.KUQCD_SUCCESS
lat = (8, 4, 4, 8)
fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3)
kq.load_gauge_pair(fat, lng, lat)
L, src = kq.L.lib(), kq.gen_source(lat, 0, seed=9)
want, out, host = np.empty_like(src), np.empty_like(src), np.empty_like(src)
assert kq.mdaggm(src, want, 0, 0.1, 0) == 0
d = [L.kq_device_alloc(src.nbytes) for _ in range(2)]
assert L.kq_memcpy(d[0], src.ctypes.data, src.nbytes) == 0
for call in (lambda: L.kq_mdaggm_noalloc(C.c_void_p(d[0]), C.c_void_p(d[1]), 0, 0.1),
             lambda: L.kq_mdaggm(C.c_void_p(d[0]), C.c_void_p(d[1]), 0, 0.1, 0)):
    before = C.c_int.in_dll(shim, "moved").value
    assert call() == 0, kq.last_error()
    assert C.c_int.in_dll(shim, "moved").value > before
    assert L.kq_synchronize() == 0
    assert L.kq_memcpy(out.ctypes.data, d[1], out.nbytes) == 0
    assert np.array_equal(out, want)
    out[:] = 0
assert L.kq_mdaggm_noalloc(C.c_void_p(src.ctypes.data), C.c_void_p(host.ctypes.data), 0, 0.1) == kq.KUQCD_ERR_INVALID_PARAM
kq.kuqcd_gauge_free()
kq.kuqcd_end()
"""


@pytest.mark.gpu
def test_arrays_on_another_gpu_are_accepted(gpu, tmp_path):
    """Device memory that belongs to another GPU: the operator entry points take it, the one without
    allocations as well, which refuses only what is not device memory. One GPU stands for two: a shim
    in front of the HIP runtime reports another device for every array."""
    src, shim = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(_SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-D_GNU_SOURCE", "-I/opt/rocm/include", str(src), "-o", str(shim),
                    "-ldl"], check=True, timeout=60)
    r = subprocess.run([sys.executable, "-c", _PEER.format(root=str(ROOT), shim=str(shim))], env=dict(os.environ),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


_FAILING_COPY = """
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
int armed = 0, failed = 0;
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    static hipError_t (*real)(void *, const void *, size_t, hipMemcpyKind, hipStream_t);
    if (!real)
        real = dlsym(dlopen("/opt/rocm/lib/libamdhip64.so.7", RTLD_LAZY), "hipMemcpyAsync");
    if (!real)
        return hipErrorNotFound;
    if (armed && k == hipMemcpyDeviceToHost && n >= (1u << 20) && --armed == 0) {
        ++failed;
        return hipErrorOutOfMemory;
    }
    return real(d, s, n, k, st);
}
"""

_AFTER_ERROR = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
shim = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
import numpy as np
import kuqcd_amd.api as kq
hip = C.CDLL("/opt/rocm/lib/libamdhip64.so.7")
kq.set_verbosity(0)
assert kq.kuqcd_init() == kq.KUQCD_SUCCESS
lat, ns = (32, 32, 32, 32), 32
fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3)
kq.load_gauge_pair(fat, lng, lat)
L, b = kq.L.lib(), kq.gen_source(lat, 0, seed=9)
bd, xd = L.kq_device_alloc(b.nbytes), [L.kq_device_alloc(b.nbytes) for _ in range(ns - 2)]
assert L.kq_memcpy(bd, b.ctypes.data, b.nbytes) == 0
first, last, got, want = (np.zeros_like(b) for _ in range(4))
xp, bp = (C.c_void_p * ns)(first.ctypes.data, *xd, last.ctypes.data), (C.c_void_p * 1)(bd)
p = kq.InvertParam(shifts=np.array([[0.1] * ns]), tol=1.0, max_iter=2, num_shift=ns)
opt = kq.default_options(mode=1, rel_tol=1e-9, refine=0, verbose=0)
def solve():
    return L.kq_solve_multishift_batched(1, xp, bp, C.byref(p.struct()), C.byref(opt), None)
assert solve() == 0, kq.last_error()
assert L.kq_memcpy(want.ctypes.data, xd[-1], want.nbytes) == 0 and np.any(want)
zero = np.zeros_like(b)
for x in xd:
    assert L.kq_memcpy(x, zero.ctypes.data, zero.nbytes) == 0
# the first solution goes to the host in chunks of 8 MiB; the last one's first chunk fails
C.c_int.in_dll(shim, "armed").value = -(-b.nbytes // (8 << 20)) + 1
last_kib = C.c_void_p(got.ctypes.data), C.c_void_p(xd[-1] + b.nbytes - 1024), C.c_size_t(1024), 2
st = solve()
# on the null stream, which does not wait for the library's
err = hip.hipMemcpy(*last_kib)
assert err == 0 and st != 0 and C.c_int.in_dll(shim, "failed").value == 1
assert np.array_equal(got.reshape(-1)[:128], want.reshape(-1)[-128:])
assert solve() == 0, kq.last_error()
kq.kuqcd_gauge_free()
kq.kuqcd_end()
"""


@pytest.mark.gpu
def test_nothing_runs_on_after_an_error(gpu, tmp_path):
    """A solve whose last solution cannot be copied to the host (a shim fails that copy) has returned with
    the device arrays of the others written: no kernel on the caller's memory is left running."""
    src, shim = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(_FAILING_COPY)
    subprocess.run(["gcc", "-shared", "-fPIC", "-D_GNU_SOURCE", "-I/opt/rocm/include", str(src), "-o", str(shim), "-ldl"],
                   check=True, timeout=60)
    r = subprocess.run([sys.executable, "-c", _AFTER_ERROR.format(root=str(ROOT), shim=str(shim))], env=dict(os.environ),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
