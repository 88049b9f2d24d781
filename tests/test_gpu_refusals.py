"""Launch options that are refused, or accepted, whatever kernel the lattice runs on."""
import ctypes as C

import numpy as np
import pytest


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
