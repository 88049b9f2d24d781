"""Which kernel a hopping term runs on, and that what may not depend on that choice does not."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from conftest import ROOT, rel_err


def _load(kq, lat, u3=False, general=False, prec=8):
    """A weak-field pair; long links as multiples of SU(3), U(3), or (general) neither."""
    fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3, seed_fat=21, seed_long=22)
    if u3:
        ph = np.exp(1j * np.random.default_rng(5).normal(size=lng.shape[:2]))[:, :, None]
        lng = np.ascontiguousarray(((lng[..., 0] + 1j * lng[..., 1]) * ph).view(np.float64).reshape(lng.shape))
    if general:
        lng = lng * (1.0 + 0.05 * np.random.default_rng(8).normal(size=lng.shape))
    kq.kuqcd_gauge_free()
    kq.load_gauge_pair(fat, lng, lat, prec=prec)
    return fat, lng


def _solve(kq, b, mode, nr, shifts=(0.05, 0.3, 1.0), **opt):
    ns = len(shifts)
    given = np.concatenate([shifts[:1], np.array(shifts[1:]) - shifts[0]])
    x = [np.zeros_like(b[0]) for _ in range(len(b) * ns)]
    p = kq.InvertParam(shifts=np.array([given] * len(b)), tol=1.0, max_iter=400, num_shift=ns)
    st, rep = kq.solve_batched(x, b, p, kq.default_options(mode=mode, rel_tol=1e-10, nr=nr, verbose=0, **opt))
    assert st == 0, kq.last_error()
    return x, rep


# 16^4 and 22x18x15x13: two systems are one pair of 32768 or 38610 sites (the split kernel) or two
# single ones (which would fill the chip in one-thread form); 16^3x8: four systems likewise; 32x16^3:
# pairs staged in LDS against single ones in one-thread form
@pytest.mark.gpu
@pytest.mark.parametrize("lat,n", [((16, 16, 16, 16), 2), ((22, 18, 15, 13), 2), ((16, 16, 16, 8), 4), ((16, 16, 16, 8), 3),
                                   ((32, 16, 16, 16), 2)])
def test_fp64_results_do_not_depend_on_the_blocking(gpu, lat, n):
    """The FP64 solve of several systems and its verification give the same bits in every process,
    although the autotuner picks their blocking by timing: blocks of 1 and 2 add in the same order."""
    kq = gpu
    _load(kq, lat)
    b = [kq.gen_source(lat, 0, seed=50 + r) for r in range(n)]
    out = {}
    for nr in (1, 2, 0):
        print("case", lat, n, nr, flush=True)
        out[nr] = _solve(kq, b, 1, nr)
    for nr in (2, 0):
        for r in range(n):
            assert out[nr][1][r].iter == out[1][1][r].iter
            assert list(out[nr][1][r].true_rel_res) == list(out[1][1][r].true_rel_res)
        assert all(np.array_equal(u, v) for u, v in zip(out[nr][0], out[1][0])), nr


@pytest.mark.gpu
@pytest.mark.parametrize("links", ["su3", "u3"])
@pytest.mark.parametrize("mode", [3, 4])
def test_split_term_with_two_waves_in_solves(gpu, mode, links):
    """Blocks of 8 with 16-bit long links on more than 49152 sites of one parity run with 2 waves per
    64 sites, in both terms of an iteration: solves whose every shift reaches an FP64 residual that
    the oracle confirms, in about the iterations of the FP64 solve (a wrong term would not converge,
    or only after many more; the 16-bit fat links of mode 3 leave the base system some)."""
    kq = gpu
    lat, shifts = (24, 16, 16, 18), (0.05, 0.1, 0.3, 1.0)
    print("case", mode, links, flush=True)
    fat, lng = _load(kq, lat, u3=links == "u3")
    assert kq.hop_kernel(lat, 8, 8, 256, fp64=False, small_long=True) == 2
    b = [kq.gen_source(lat, 0, seed=70 + r) for r in range(2)]
    _, rep1 = _solve(kq, b, 1, 2, shifts)
    x, rep = _solve(kq, b, mode, 8, shifts)
    for r in range(2):
        for k, s in enumerate(shifts):
            v = x[r * len(shifts) + k]
            res = b[r] - (s * v - oracle.mdaggm(fat, lng, v, lat, 0))
            assert np.linalg.norm(res) <= 1.01e-10 * np.linalg.norm(b[r]), (r, k)
        assert rep[r].iter <= (2 if mode == 3 else 1.2) * rep1[r].iter + 5


@pytest.mark.gpu
@pytest.mark.parametrize("prec,links", [(8, "general"), (4, "general"), (4, "u3")])
@pytest.mark.parametrize("lat", [(6, 5, 4, 3), (10, 6, 6, 6)])
def test_host_layout_in_every_link_format(gpu, lat, prec, links):
    """The operator and every blocking of the hopping term on the caller's arrays, in the long-link
    formats that the other tests of these kernels do not load: 18 reals, and FP32 in 12 reals with a
    complex scale. Bounds of the path: 1e-13 (FP64), 1e-5 (FP32)."""
    kq = gpu
    dt, tol = (np.float64, 1e-13) if prec == 8 else (np.float32, 1e-5)
    fat, lng = _load(kq, lat, u3=links == "u3", general=links == "general", prec=prec)
    fat, lng = (a.astype(dt).astype(np.float64) for a in (fat, lng))
    src = np.stack([kq.gen_source(lat, 0, seed=80 + r) for r in range(9)]).astype(dt)
    want = np.stack([oracle.dslash(fat, lng, v.astype(np.float64), lat, 1) for v in src])
    for nr in (1, 2, 3, 4, 8):
        print("case", lat, prec, links, nr, flush=True)
        out = np.full_like(src, np.nan)
        assert kq.dslash_batched(src, out, 1, 0, nr, 256) == 0, kq.last_error()
        for r in range(len(src)):
            assert rel_err(out[r], want[r]) <= tol, r
    v, out = np.ascontiguousarray(src[0]), np.empty_like(src[0])
    assert kq.mdaggm(v, out, 0, 0.07, 0) == 0, kq.last_error()
    assert rel_err(out, 0.07 * v.astype(np.float64) - oracle.mdaggm(fat, lng, v.astype(np.float64), lat, 0)) <= tol


# Lx = 32 and more than 98304 sites of one parity: blocks of any size are staged. One workgroup per (x, y) plane
# with more staged rows than the plane has (the y wrap repeats rows), and two per plane.
STAGED = [(32, 16, 16, 32), (32, 32, 16, 16)]
MIXED_NRS = (2, 3, 4, 8)


def test_the_staged_kernel_is_the_one_tested(kq):
    for lat in STAGED:
        for nr in MIXED_NRS:
            for small in (False, True):
                assert kq.hop_kernel(lat, 5, nr, 256, fp64=False, small_long=small) == 1
        assert kq.hop_kernel(lat, 5, 1, 256, fp64=False) == 0
        assert kq.hop_kernel(lat, 2, 2, 256, fp64=True) == 1 and kq.hop_kernel(lat, 2, 1, 256, fp64=True) == 0


@pytest.mark.parametrize("lat", [(2, 1, 1, 1), (6, 5, 4, 3), (8, 8, 8, 8), (32, 32, 16, 2), (16, 16, 16, 8)])
def test_lattices_of_the_direction_update_take_eight_waves(kq, lat):
    """Up to 16384 sites of one parity the solvers of one system update its direction inside the hopping
    term, whose kernel has 8 waves per 64 sites."""
    for fp64 in (False, True):
        for nt in (64, 256):
            assert kq.hop_kernel(lat, 1, 1, nt, fp64=fp64) == 8


@pytest.mark.gpu
@pytest.mark.parametrize("lat", STAGED)
@pytest.mark.parametrize("mode,tol", [(2, 1e-5), (3, 3e-3), (4, 5e-4)])
def test_staged_rows_of_the_mixed_terms(gpu, lat, mode, tol):
    """Blocks with their rows in LDS against single vectors (one thread per site, the same arithmetic to
    rounding) and the oracle, with a padded last block."""
    kq = gpu
    fat, lng = _load(kq, lat)
    src = np.stack([kq.gen_source(lat, 0, seed=200 + r) for r in range(5)])
    single = np.empty_like(src)
    for r in range(5):
        assert kq.dslash(np.ascontiguousarray(src[r]), single[r], 1, mode) == 0
    for r in (0, 4):
        assert rel_err(single[r], oracle.dslash(fat, lng, src[r], lat, 1)) <= tol
    for nr in MIXED_NRS:
        print("case", lat, mode, nr, flush=True)
        out = np.full_like(src, np.nan)
        assert kq.dslash_batched(src, out, 1, mode, nr, 256) == 0, kq.last_error()
        assert rel_err(out, single) <= 1e-6, nr


_UNSTAGED = """
import sys
sys.path[:0] = [{root!r}, {tests!r}]
import numpy as np
import kuqcd_amd.api as kq
import test_gpu_kernel_choice as T
kq.set_verbosity(0)
assert kq.kuqcd_init() == kq.KUQCD_SUCCESS
np.save({path!r}, T.staged_results(kq, {lat!r}))
kq.kuqcd_gauge_free()
kq.kuqcd_end()
"""


def staged_results(kq, lat):
    """Everything that the staged kernel computes on this lattice: the mixed terms in blocks, and an FP64
    solve of two systems as pairs in workgroups of 256."""
    _load(kq, lat)
    src = np.stack([kq.gen_source(lat, 0, seed=300 + r) for r in range(5)])
    res = []
    for mode in (2, 3, 4):
        for nr in MIXED_NRS:
            print("case", lat, mode, nr, flush=True)
            out = np.empty_like(src)
            assert kq.dslash_batched(src, out, 1, mode, nr, 256) == 0, kq.last_error()
            res.append(out)
    x, rep = _solve(kq, [src[0], src[1]], 1, 2, nt=256)
    res.append(np.stack(x))
    return np.concatenate([v.reshape(-1) for v in res] + [np.array(rep[r].true_rel_res) for r in range(2)])


@pytest.mark.gpu
@pytest.mark.parametrize("lat", STAGED)
def test_staged_rows_bitwise_equal_to_unstaged(gpu, tmp_path, lat):
    """The staged kernel (with its link prefetch for 4 or more FP32 vectors) adds in the unstaged one's
    order: the bits are those of a process with the staging switched off."""
    out = staged_results(gpu, lat)
    path = str(tmp_path / "unstaged.npy")
    code = _UNSTAGED.format(root=str(ROOT), tests=str(ROOT / "tests"), path=path, lat=lat)
    r = subprocess.run([sys.executable, "-c", code], env={**os.environ, "KQ_STAGE": "0"}, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert np.array_equal(out, np.load(path))


@pytest.mark.gpu
@pytest.mark.parametrize("links", ["su3", "u3", "general"])
def test_fp64_blocks_on_large_lattices(gpu, links):
    """FP64 vectors in blocks of 3, 4 and 8 above the sizes of the split term run on colour planes of the
    source, one thread per site, and write the caller's layout: whole, padded and single blocks against the
    oracle (1e-13) and blocks of 2, from device arrays aligned to one real, host arrays, and a source that
    overlaps the destination."""
    kq, L, lat = gpu, gpu.L.lib(), (18, 18, 18, 18)
    fat, lng = _load(kq, lat, u3=links == "u3", general=links == "general")
    src = np.stack([kq.gen_source(lat, 0, seed=90 + r) for r in range(9)])
    want = np.stack([oracle.dslash(fat, lng, v, lat, 1) for v in src])
    base = L.kq_device_alloc(2 * src.nbytes + 64)
    s, d = base + 8, base + 8 + src.nbytes
    out = np.empty_like(src)
    try:
        for n in (1, 2, 3, 4, 5, 9):
            for nr in (2, 3, 4, 8):
                print("case", links, n, nr, flush=True)
                assert L.kq_memcpy(s, src.ctypes.data, src.nbytes) == 0
                size = n * src[0].nbytes
                assert L.kq_dslash_batched(n, C.c_void_p(s), C.c_void_p(d), 1, 0, nr, 256) == 0, kq.last_error()
                assert L.kq_memcpy(out.ctypes.data, d, size) == 0
                assert all(rel_err(out[r], want[r]) <= 1e-13 for r in range(n))
                host = np.full_like(src[:n], np.nan)
                assert kq.dslash_batched(np.ascontiguousarray(src[:n]), host, 1, 0, nr, 256) == 0, kq.last_error()
                assert np.array_equal(host, out[:n])
                # over the source's second half (which is no longer its own afterwards)
                at = s + size // 2
                assert L.kq_dslash_batched(n, C.c_void_p(s), C.c_void_p(at), 1, 0, nr, 256) == 0, kq.last_error()
                assert L.kq_memcpy(host.ctypes.data, at, size) == 0
                assert np.array_equal(host, out[:n])
    finally:
        L.kq_device_free(base)
