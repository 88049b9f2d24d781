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
