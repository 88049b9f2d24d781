"""The operator entry points on the caller's own device arrays (host layout): hopping term and
A = sigma - D D against the oracle on lattices with remainders of every tile (64 sites, 8 XCDs, 256
sites), on both sides of the sizes at which the split and the one-thread kernels change over, for
every right-hand-side blocking and with a padded last block; addresses aligned to one real only; and
sources that overlap the destination."""
import ctypes as C

import numpy as np
import pytest

import oracle
from conftest import rel_err

TOL = {8: 1e-13, 4: 1e-5}  # the path's parity bounds (FP64, FP32)


def _load(kq, lat, prec, u3=False):
    fat, lng = kq.gen_gauge(lat, kind=kq.KQ_GEN_WEAK, eps=0.3, seed_fat=21, seed_long=22)
    if u3:  # a phase on every long link: the complex-scale forms
        ph = np.exp(1j * np.random.default_rng(5).normal(size=lng.shape[:2]))[:, :, None]
        lng = np.ascontiguousarray(((lng[..., 0] + 1j * lng[..., 1]) * ph).view(np.float64).reshape(lng.shape))
    kq.kuqcd_gauge_free()
    kq.load_gauge_pair(fat, lng, lat, prec=prec)
    return fat, lng


class _Dev:
    """A device array of `nbytes` bytes starting `shift` bytes after an allocation's start."""

    def __init__(self, kq, nbytes, shift=0):
        self.kq, self.n = kq, nbytes
        self.base = kq.L.lib().kq_device_alloc(nbytes + 64)
        self.p = self.base + shift

    def put(self, a):
        assert self.kq.L.lib().kq_memcpy(self.p, a.ctypes.data, a.nbytes) == 0

    def get(self, like):
        out = np.empty_like(like)
        assert self.kq.L.lib().kq_memcpy(out.ctypes.data, self.p, out.nbytes) == 0
        return out

    def free(self):
        self.kq.L.lib().kq_device_free(self.base)


# Vh = 180 (less than the 8 tiles), 2048, 38610 (ragged), 56000 (FP64 one-thread kernel in workgroups
# of 64), 131072 (FP32 likewise), 262144 (workgroups of 256)
LATS = [(6, 5, 4, 3), (8, 8, 8, 8), (22, 18, 15, 13), (20, 20, 20, 14), (32, 16, 16, 32), (32, 32, 32, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("lat", LATS)
def test_operator_on_device_arrays(gpu, lat, prec):
    kq, L = gpu, gpu.L.lib()
    dt = np.float64 if prec == 8 else np.float32
    fat, lng = _load(kq, lat, prec, u3=lat[1] % 2 == 1)
    fat, lng = (a.astype(dt).astype(np.float64) for a in (fat, lng))
    sigma = 0.07
    for parity in (0, 1):
        print("case", lat, prec, parity, flush=True)
        src = kq.gen_source(lat, parity, seed=31).astype(dt)
        want = sigma * src.astype(np.float64) - oracle.mdaggm(fat, lng, src.astype(np.float64), lat, parity)
        hop = oracle.dslash(fat, lng, src.astype(np.float64), lat, 1 - parity)
        for shift in (0, prec):  # aligned, and to one real only
            s, d = _Dev(kq, src.nbytes, shift), _Dev(kq, src.nbytes, shift)
            try:
                s.put(src)
                assert L.kq_mdaggm(C.c_void_p(s.p), C.c_void_p(d.p), parity, sigma, 0) == 0, kq.last_error()
                out = d.get(src)
                assert rel_err(out, want) <= TOL[prec]
                assert np.array_equal(s.get(src), src)
                host = np.empty_like(src)
                assert kq.mdaggm(src, host, parity, sigma, 0) == 0
                assert np.array_equal(host, out)
                assert L.kq_dslash(C.c_void_p(s.p), C.c_void_p(d.p), 1 - parity, 0) == 0, kq.last_error()
                assert rel_err(d.get(src), hop) <= TOL[prec]
                # in place
                assert L.kq_mdaggm(C.c_void_p(s.p), C.c_void_p(s.p), parity, sigma, 0) == 0
                assert np.array_equal(s.get(src), out)
            finally:
                s.free()
                d.free()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,nrs", [(8, (1, 2, 4, 8)), (4, (1, 2, 3, 4, 8))])
@pytest.mark.parametrize("lat", [(6, 5, 4, 3), (16, 12, 8, 8), (22, 18, 15, 13)])
def test_block_of_vectors_on_device_arrays(gpu, lat, prec, nrs):
    kq, L = gpu, gpu.L.lib()
    dt = np.float64 if prec == 8 else np.float32
    fat, lng = _load(kq, lat, prec)
    fat, lng = (a.astype(dt).astype(np.float64) for a in (fat, lng))
    for nrhs in (1, 5, 9):  # whole and padded blocks
        src = np.stack([kq.gen_source(lat, 1, seed=40 + r) for r in range(nrhs)]).astype(dt)
        want = np.stack([oracle.dslash(fat, lng, v.astype(np.float64), lat, 0) for v in src])
        both = _Dev(kq, 2 * src.nbytes)
        try:
            for nr in nrs:
                print("case", lat, prec, nrhs, nr, flush=True)
                for at in (src.nbytes, src.nbytes // 2):  # apart; destination over the source's second half
                    both.put(src)
                    assert L.kq_dslash_batched(nrhs, C.c_void_p(both.p), C.c_void_p(both.p + at), 0, 0, nr, 256) == 0
                    out = np.empty_like(src)
                    assert L.kq_memcpy(out.ctypes.data, both.p + at, out.nbytes) == 0
                    assert rel_err(out, want) <= TOL[prec]
        finally:
            both.free()


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nrhs", [((6, 5, 4, 3), 5), ((22, 18, 15, 13), 9), ((24, 24, 24, 16), 8), ((24, 24, 24, 24), 8)])
@pytest.mark.parametrize("mode", [2, 3, 4])
def test_blocks_of_the_mixed_terms(gpu, lat, nrhs, mode):
    """Every blocking of the 32-bit terms on colour planes, split (small lattices, and blocks of 8 on
    any) and one thread per site (24^4 in blocks up to 4), with padded last blocks. Bounds as for the
    formats elsewhere: FP32 1e-5, 16-bit links 3e-3, 16-bit long links 5e-4."""
    kq = gpu
    fat, lng = _load(kq, lat, 8, u3=mode == 4)
    src = np.stack([kq.gen_source(lat, 0, seed=60 + r % 3) for r in range(nrhs)])
    want = [oracle.dslash(fat, lng, src[r], lat, 1) for r in range(3)]
    for nr in (1, 2, 3, 4, 8):
        print("case", lat, mode, nr, flush=True)
        out = np.full_like(src, np.nan)
        assert kq.dslash_batched(src, out, 1, mode, nr, 64) == 0, kq.last_error()
        for r in range(nrhs):
            assert rel_err(out[r], want[r % 3]) <= {2: 1e-5, 3: 3e-3, 4: 5e-4}[mode], r


@pytest.mark.gpu
@pytest.mark.parametrize("links", ["su3", "u3", "general"])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
def test_split_terms_in_solves(gpu, links, mode):
    """The split terms with the fused epilogue, as the solvers run them, in every link format (SU(3)
    products, U(3) products and general long links) and blocking: solves on a lattice with a partial
    last workgroup, every shift to an FP64 residual that the oracle confirms. A wrong term would not
    converge, or only after many more iterations than the FP64 solve."""
    kq = gpu
    lat = (10, 6, 6, 6)
    fat, lng = _load(kq, lat, 8, u3=links == "u3")
    if links == "general":
        rng = np.random.default_rng(8)
        lng = lng * (1.0 + 0.05 * rng.normal(size=lng.shape))
        kq.kuqcd_gauge_free()
        kq.load_gauge_pair(fat, lng, lat)
    shifts = np.array([0.05, 0.1, 0.3, 0.6, 1.0, 2.0, 3.0, 4.0])
    given = np.concatenate([shifts[:1], shifts[1:] - shifts[0]])
    nrhs = 2
    b = [kq.gen_source(lat, 0, seed=70 + r) for r in range(nrhs)]
    iters = {}
    for m, nr in [(1, 1)] + [(mode, n) for n in ([2] if mode == 1 else [1, 2, 3, 4, 8])]:
        print("case", links, m, nr, flush=True)
        x = [np.zeros_like(b[0]) for _ in range(nrhs * len(shifts))]
        p = kq.InvertParam(shifts=np.array([given] * nrhs), tol=1.0, max_iter=400, num_shift=len(shifts))
        st, rep = kq.solve_batched(x, b, p, kq.default_options(mode=m, rel_tol=1e-10, nr=nr, verbose=0))
        assert st == 0, kq.last_error()
        iters[m, nr] = rep[0].iter
        for r in range(nrhs):
            for k in range(len(shifts)):
                v = x[r * len(shifts) + k]
                res = b[r] - (shifts[k] * v - oracle.mdaggm(fat, lng, v, lat, 0))
                assert np.linalg.norm(res) <= 1.01e-10 * np.linalg.norm(b[r]), (m, nr, r, k)
        # the 16-bit fat links leave the base system some more iterations (its refinement does the rest)
        assert rep[0].iter <= (2 if m == 3 else 1.2) * iters[1, 1] + 5


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [8, 4])
def test_solves_and_gradients_on_device_arrays(gpu, prec):
    """Sources and solutions on the device, aligned and one real off, and in host arrays: the same numbers."""
    kq, L = gpu, gpu.L.lib()
    lat, ns = (10, 6, 6, 6), 4
    dt = np.float64 if prec == 8 else np.float32
    _load(kq, lat, prec)
    b = kq.gen_source(lat, 0, seed=81).astype(dt)

    def par():
        return kq.InvertParam(shifts=[0.05, 0.1, 0.5, 1.0], tol=1e-8, max_iter=400, num_shift=ns, prec=prec)

    want = [np.zeros_like(b) for _ in range(ns)]
    assert kq.kuqcd_solve_multishift(want, b, par()) == 0, kq.last_error()
    for shift in (0, prec):
        bd, xd = _Dev(kq, b.nbytes, shift), [_Dev(kq, b.nbytes, shift) for _ in range(ns)]
        try:
            bd.put(b)
            xp = (C.c_void_p * ns)(*[x.p for x in xd])
            assert L.kq_solve_multishift(xp, C.c_void_p(bd.p), C.byref(par().struct())) == 0, kq.last_error()
            for k in range(ns):
                assert np.array_equal(xd[k].get(b), want[k])
        finally:
            for a in [bd] + xd:
                a.free()
    if prec == 4:
        return
    w = kq.ptnet_init_weights(3, 0.2)
    e = kq.gen_source(lat, 0, seed=82)
    res = []
    for shift in (None, 0, 8):
        dev = [] if shift is None else [_Dev(kq, b.nbytes, shift) for _ in range(2)]
        try:
            for a, v in zip(dev, (b, e)):
                a.put(v)
            at = [a.p for a in dev] or [b.ctypes.data, e.ctypes.data]
            loss, only, g = C.c_double(), C.c_double(), np.empty(2 * kq.KQ_PT_PARAMS)
            assert L.kq_ptnet_loss_grad(C.byref(w), 0, 0.05, C.c_void_p(at[0]), C.c_void_p(at[1]), C.byref(loss),
                                        g.ctypes.data_as(C.POINTER(C.c_double))) == 0, kq.last_error()
            assert L.kq_ptnet_loss_grad(C.byref(w), 0, 0.05, C.c_void_p(at[0]), C.c_void_p(at[1]), C.byref(only),
                                        None) == 0, kq.last_error()
            assert only.value == loss.value > 0.0
            res.append(np.append(g, loss.value))
        finally:
            for a in dev:
                a.free()
    assert np.array_equal(res[0], res[1]) and np.array_equal(res[0], res[2])
    # a zero pair: loss and gradient are 0
    z = np.zeros_like(b)
    assert L.kq_ptnet_loss_grad(C.byref(w), 0, 0.05, z.ctypes.data_as(C.c_void_p), z.ctypes.data_as(C.c_void_p),
                                C.byref(loss), g.ctypes.data_as(C.POINTER(C.c_double))) == 0
    assert loss.value == 0.0 and not g.any()


@pytest.mark.gpu
@pytest.mark.parametrize("lat", [(6, 5, 4, 3), (32, 32, 32, 18), (32, 32, 32, 34)])
def test_refinement_over_its_partial_sums(gpu, lat):
    """The flexible CG with fewer sites than a workgroup, and where the network layer's partials
    (above 262144 half-lattice sites) and the operator's (above 524288) are summed in slices first:
    plain CG and the network's iteration reach the residual, which the operator confirms."""
    kq, L = gpu, gpu.L.lib()
    _load(kq, lat, 8)
    b = kq.gen_source(lat, 0, seed=91)
    # channel 0 is D r, the output 8/b r - c A r = (8/b - c sigma) r + c D D r: positive up to A = b
    nu, sigma, bound = kq.ptnet_norms(), 0.5, 5.0
    c = 0.9 * 8.0 / bound**2
    hop = np.array([(-1.0 if t & 2 else 1.0) * nu[t & 1] for t in range(16)])
    W1, W2 = np.zeros((4, 16), complex), np.zeros((4, 16), complex)
    W1[0], W2[0] = hop, c * hop
    assert kq.ptnet_set_weights(kq.weights_from_array(W1, W2, 8.0 / bound - c * sigma)) == 0
    for learned in (0, 1):
        print("case", lat, learned, flush=True)
        x = np.zeros_like(b)
        st, rep = kq.fcg_refine(b, x, sigma, 0, kq.refine_options(rel_tol=1e-9, learned=learned, max_iter=300))
        assert st == 0, kq.last_error()
        assert rep.converged and not rep.fallback and rep.iter < 100
        ax = np.empty_like(b)
        assert kq.mdaggm(x, ax, 0, sigma, 1) == 0
        assert np.linalg.norm(b - ax) <= 1.01e-9 * np.linalg.norm(b)


@pytest.mark.gpu
@pytest.mark.parametrize("links", ["su3", "u3", "general"])
@pytest.mark.parametrize("prec", [8, 4])
def test_direction_update_in_the_hopping_term(gpu, prec, links):
    """The reference solve on small lattices, where the hopping term updates the direction (and on the smallest
    one where it no longer does): stopped after
    every kind of place in its chunks of 15 iterations (first, second, last, first of the next, within
    the phase of one live shift) it has the oracle's iterate, with one shift and with several, on
    ragged and odd extents. Bounds: rounding of at most 34 iterations of a system of condition
    below 100, 1e-12 in FP64 and 1e-4 in FP32."""
    kq = gpu
    dt = np.float64 if prec == 8 else np.float32
    for lat in ((6, 5, 4, 3), (10, 6, 6, 6), (16, 16, 16, 8), (18, 16, 16, 8)):
        fat, lng = _load(kq, lat, prec, u3=links == "u3")
        if links == "general":
            lng = (lng * (1.0 + 0.05 * np.random.default_rng(8).normal(size=lng.shape))).astype(dt)
            kq.kuqcd_gauge_free()
            kq.load_gauge_pair(fat, lng, lat, prec=prec)
        b = kq.gen_source(lat, 0, seed=95).astype(dt)
        for given in ([0.5], [0.5, 0.2, 3.0]):
            for max_iter in (1, 2, 15, 16, 17, 34):
                print("case", prec, links, lat, given, max_iter, flush=True)
                sh = np.array(given, dt)
                x = [np.zeros_like(b) for _ in sh]
                p = kq.InvertParam(shifts=np.array(given), tol=1e-6 if prec == 4 else 1e-18, max_iter=max_iter,
                                   num_shift=len(given), prec=prec)
                assert kq.kuqcd_solve_multishift(x, b, p) == 0, kq.last_error()
                want, it = oracle.cgm(fat.astype(dt), lng.astype(dt), lat, 0, sh, b, p.tol, max_iter)
                assert abs(p.iter - it) <= (0 if prec == 8 else 1)
                if p.iter == it:
                    for k in range(len(given)):
                        assert rel_err(x[k], want[k]) <= (1e-12 if prec == 8 else 1e-4), k
