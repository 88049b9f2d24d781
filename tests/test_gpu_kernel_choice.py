"""Which kernel a hopping term runs on, and that what may not depend on that choice does not."""
import numpy as np
import pytest


def _load(kq, lat, u3=False, general=False):
    """A weak-field double pair; long links as multiples of SU(3), U(3), or (general) neither."""
    fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3, seed_fat=21, seed_long=22)
    if u3:
        ph = np.exp(1j * np.random.default_rng(5).normal(size=lng.shape[:2]))[:, :, None]
        lng = np.ascontiguousarray(((lng[..., 0] + 1j * lng[..., 1]) * ph).view(np.float64).reshape(lng.shape))
    if general:
        lng = lng * (1.0 + 0.05 * np.random.default_rng(8).normal(size=lng.shape))
    kq.kuqcd_gauge_free()
    kq.load_gauge_pair(fat, lng, lat)
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
