"""Timed cases of the library's main path: the HISQ operator, its multishift solvers and the learned preconditioner.

Every case goes through the public entry points (the C ABI of include/kuqcd_hip.h, or its Python mirror kuqcd_amd.api).
A program loads one gauge configuration and then applies the operator to, or solves for, many sources: so the gauge
pair belongs to the case (its "gauge" is the seed of the links, loaded once), and the sources belong to the seed of
prepare(). Lattices run from 8^4, where latency and launches count, over 16^4 and 24^4 to 32^4 and, for the operator,
48^3x96.

Links are synthetic, as the library's own generator makes them: fat = 0.9 eta_mu G plus a little noise (smeared links
are not unitary), long = -1/24 eta_mu W, with G and W near the identity and the staggered phases eta folded in; with
"u3" the long links carry a U(3) phase, as reunitarised smeared links do.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import kuqcd_amd.api as A

DEV = "cuda"
#: lowest and highest eigenvalue of -DD that the iteration counts of work() assume (weak links of the kind above)
EIG_LOW, EIG_HIGH = 4e-3, 4.2


def listed():
    return [
        # one operator application on the smallest lattice by a caller that must not allocate: pure latency
        dict(name="apply_8", kind="apply", lat="8,8,8,8", prec="double", entry="noalloc", parity=0, sigma=0.02, u3=False, gauge=1),
        # ragged extents, odd sites: remainders of every tile and wrap, a correlator's odd-site application
        dict(name="apply_ragged", kind="apply", lat="22,18,15,13", prec="double", entry="mdaggm", parity=1, sigma=0.02, u3=True, gauge=2),
        # the operator on the headline lattice: residual checks, eigenvector projections
        dict(name="apply_32", kind="apply", lat="32,32,32,32", prec="double", entry="mdaggm", parity=0, sigma=1e-4, u3=False, gauge=3),
        # the same on the largest lattice the library is run on
        dict(name="apply_48", kind="apply", lat="48,48,48,96", prec="double", entry="mdaggm", parity=0, sigma=2.5e-5, u3=True, gauge=4),
        # hopping term on a block of single-precision vectors: deflation, stochastic traces
        dict(name="hop_block_24", kind="hop", lat="24,24,24,24", prec="float", nrhs=8, nr=4, parity=0, u3=False, gauge=5),
        # drop-in multishift solve on the smallest lattice, source and solutions in host memory
        dict(name="solve_8", kind="solve", lat="8,8,8,8", prec="double", where="host", parity=0, nshift=4, lo=1e-2, hi=1.0, rel=1e-10, u3=False, gauge=6),
        # single-precision force solve of a rational approximation
        dict(name="solve_16_float", kind="solve", lat="16,16,16,16", prec="float", where="host", parity=0, nshift=9, lo=1e-2, hi=3.0, rel=1e-6, u3=True, gauge=7),
        # the drop-in solve of the headline problem: 12 shifts, double, host arrays
        dict(name="solve_32", kind="solve", lat="32,32,32,32", prec="double", where="host", parity=0, nshift=12, lo=2e-4, hi=1.0, rel=1e-10, u3=False, gauge=3),
        # the headline: mixed precision with FP64 reliable updates, everything resident
        dict(name="mixed_32", kind="mixed", lat="32,32,32,32", mode="fp32", nrhs=1, parity=0, nshift=12, lo=2e-4, hi=1.0, rel=1e-11, u3=False, gauge=3),
        # several sources of a middle-sized configuration in one batched solve, 16-bit long links
        dict(name="mixed_16_batch", kind="mixed", lat="16,16,16,32", mode="fp32_l16", nrhs=4, parity=0, nshift=6, lo=1e-3, hi=1.0, rel=1e-11, u3=True, gauge=8),
        # flexible CG with the parallel-transport network on one light shift
        dict(name="refine_24", kind="refine", lat="24,24,24,24", parity=0, sigma=1e-3, rel=1e-11, u3=False, gauge=9),
        # loss and weight gradient of the network: one sample of a training step
        dict(name="grad_16", kind="grad", lat="16,16,16,16", parity=0, sigma=1e-2, u3=False, gauge=10),
    ]


def _draw_lattice(rng, top, odd):
    """Extents with x even and 8^4 <= V <= top (or a little less, for ragged ones), V log-uniform."""
    vol = math.exp(rng.uniform(math.log(8 ** 4), math.log(top)))
    while True:
        side = vol ** 0.25
        ext = [max(6, round(side * math.exp(rng.uniform(-0.3, 0.3)))) for _ in range(3)]
        ext.append(max(6, round(vol / (ext[0] * ext[1] * ext[2]))))
        lat = [2 * ((e + 1) // 2) for e in ext]
        if odd:
            lat[1:] = ext[1:]
        v = lat[0] * lat[1] * lat[2] * lat[3]
        if 8 ** 4 * 0.8 <= v <= top:
            return ",".join(map(str, lat))


def draw(rng):
    kind = rng.choice(["apply", "apply", "hop", "solve", "solve", "mixed", "mixed", "refine", "grad"])
    case = dict(kind=kind, parity=rng.randrange(2), u3=rng.random() < 0.5, gauge=rng.randrange(100, 1 << 20))
    if kind == "apply":
        case.update(lat=_draw_lattice(rng, 32 ** 4, rng.random() < 0.5), prec=rng.choice(["double", "double", "float"]),
                    entry=rng.choice(["mdaggm", "mdaggm", "noalloc"]), sigma=10 ** rng.uniform(-4, 0))
    elif kind == "hop":
        case.update(lat=_draw_lattice(rng, 32 ** 4, rng.random() < 0.5), prec=rng.choice(["float", "double"]))
        case.update(nrhs=rng.randint(1, 12), nr=rng.choice([1, 2, 4, 8] if case["prec"] == "float" else [1, 2]))
    elif kind == "solve":
        case.update(lat=_draw_lattice(rng, 32 ** 4, False), prec=rng.choice(["double", "double", "float"]),
                    where=rng.choice(["host", "device"]), nshift=rng.randint(1, 12))
        low = 1e-2 if case["prec"] == "float" else 10 ** rng.uniform(-3, -1)
        case.update(lo=low, hi=10 ** rng.uniform(-0.5, 0.5), rel=1e-6 if case["prec"] == "float" else 1e-10)
    elif kind == "mixed":
        case.update(lat=_draw_lattice(rng, 24 ** 4, False), mode=rng.choice(["fp32", "fp32_l16"]), nrhs=rng.randint(1, 4),
                    nshift=rng.randint(2, 8), lo=10 ** rng.uniform(-3, -1), hi=1.0, rel=1e-11)
    elif kind == "refine":
        case.update(lat=_draw_lattice(rng, 24 ** 4, False), sigma=10 ** rng.uniform(-3, -1), rel=1e-11)
    else:
        case.update(lat=_draw_lattice(rng, 24 ** 4, False), sigma=10 ** rng.uniform(-3, -1))
    return case


# ------------------------------------------------------------------------------------------------ inputs
def _lat(case):
    return tuple(int(v) for v in case["lat"].split(","))


def _half(case):
    return math.prod(_lat(case)) // 2


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _coords(lat, q):
    """Full coordinates of the sites of parity q, x fastest (checkerboard order)."""
    s = torch.arange(math.prod(lat) // 2, device=DEV)
    xh = lat[0] // 2
    xcb, r = s % xh, s // xh
    y, r = r % lat[1], r // lat[1]
    z, t = r % lat[2], r // lat[2]
    return [2 * xcb + ((y + z + t + q) & 1), y, z, t]


def _near_unitary(n, eps, u3, gen):
    """(3, 3, n) complex128: 1 + i eps H with its rows made orthonormal, times a phase where u3."""
    a = torch.randn((3, 3, n, 2), dtype=torch.float64, device=DEV, generator=gen)
    a = torch.view_as_complex(a) * (eps / math.sqrt(2.0))
    m = 1j * (a + a.transpose(0, 1).conj()) / math.sqrt(2.0) + torch.eye(3, dtype=torch.complex128, device=DEV)[:, :, None]
    for _ in range(2):  # twice: orthonormal to rounding
        r0 = m[0] / m[0].abs().square().sum(0).sqrt()
        r1 = m[1] - r0 * (r0.conj() * m[1]).sum(0)
        r1 = r1 / r1.abs().square().sum(0).sqrt()
        r2 = torch.stack([r0[1] * r1[2] - r0[2] * r1[1], r0[2] * r1[0] - r0[0] * r1[2], r0[0] * r1[1] - r0[1] * r1[0]]).conj()
        m = torch.stack([r0, r1, r2])
    if u3:
        ph = torch.randn((n,), dtype=torch.float64, device=DEV, generator=gen) * eps
        m = m * torch.complex(ph.cos(), ph.sin())
    return m


def _links(case):
    """Fat and long links as a program loads them: (2, 4, 3, 3, Vh) complex128 each (parity, direction, row, column, site)."""
    lat, gen, n = _lat(case), _gen(1000003 * case["gauge"] + 17), _half(case)
    fat = torch.empty((2, 4, 3, 3, n), dtype=torch.complex128, device=DEV)
    lng = torch.empty_like(fat)
    for q in range(2):
        x, y, z, _ = _coords(lat, q)
        for mu in range(4):
            eta = (1 - 2 * ((0, x, x + y, x + y + z)[mu] & 1)) if mu else torch.ones(n, device=DEV)
            noise = torch.view_as_complex(torch.randn((3, 3, n, 2), dtype=torch.float64, device=DEV, generator=gen))
            fat[q, mu] = (0.9 * _near_unitary(n, 0.3, False, gen) + 0.02 * noise) * eta
            del noise
            lng[q, mu] = _near_unitary(n, 0.5, case["u3"], gen) * (-eta / 24.0)
    return fat, lng


def _source(case, seed, count, dtype):
    """`count` Gaussian sources on one parity in the host layout (count, Vh, 3, 2), E|z|^2 = 1."""
    v = torch.randn((count, _half(case), 3, 2), dtype=torch.float64, device=DEV, generator=_gen(7919 * seed + 5))
    return (v * math.sqrt(0.5)).to(dtype).contiguous()


def _is_float(case):
    return case.get("prec") == "float"


_loaded = None  # what the library's gauge slots hold now


def _load(case):
    """Loads the case's gauge pair, as a program does once per configuration."""
    global _loaded
    key = (case["lat"], case["gauge"], case["u3"], _is_float(case))
    if _loaded == key:
        return
    if _loaded is None:
        A.set_verbosity(0)
        if A.kuqcd_init() != A.KUQCD_SUCCESS:
            raise RuntimeError(A.L.last_error())
    _loaded = ()
    A.kuqcd_gauge_free()
    prec, dt = (A.KUQCD_SINGLE, torch.float32) if _is_float(case) else (A.KUQCD_DOUBLE, torch.float64)
    for links, kind in zip(_links(case), (A.KUQCD_FAT_LINK, A.KUQCD_LONG_LINK)):
        n = links.shape[-1]
        host = torch.empty((2, n, 4, 9, 2), dtype=dt, device=DEV)
        host.copy_(torch.view_as_real(links.reshape(2, 4, 9, n)).permute(0, 3, 1, 2, 4))
        torch.cuda.synchronize()
        par = A.gauge_param(_lat(case), prec=prec, link_type=kind)
        _ok(A.L.lib().kq_load_gaugefield(C.c_void_p(host.data_ptr()), C.byref(par)))
        del links, host
    torch.cuda.empty_cache()
    _loaded = key


def _ok(status):
    if status != A.KUQCD_SUCCESS:
        raise RuntimeError("status %d: %s" % (status, A.L.last_error()))


def _shifts(case):
    """Absolute shifts of one source, logarithmic from lo to hi."""
    n = case["nshift"]
    return [case["lo"] * (case["hi"] / case["lo"]) ** (k / max(1, n - 1)) for k in range(n)]


def _given(case):
    """The shifts in the solver's convention: all after the first relative to it."""
    s = _shifts(case)
    return [s[0]] + [v - s[0] for v in s[1:]]


MODES = {"fp32": A.KQ_MODE_MIXED_FP32, "fp32_l16": A.KQ_MODE_MIXED_FP32_L16}


def _weights(case):
    """Network weights of a trained shape: channel 0 the degree-1 polynomial 8/b - 0.9 (8/b^2) A, the others small; and for
    the gradient a start with noise on every weight. Complex (4, 16), (4, 16), scalar, in float32."""
    g = torch.Generator().manual_seed(31 * case["gauge"] + 3)
    w1, w2 = (0.01 * torch.view_as_complex(torch.randn((4, 16, 2), dtype=torch.float64, generator=g)).numpy() for _ in range(2))
    beta = 1.02 * (EIG_HIGH + case["sigma"])
    c = 0.9 * 8 / beta ** 2
    sign = np.array([1, 1, -1, -1] * 4)  # taps: direction by direction, hops +1 +3 -1 -3
    # root-mean-square row norms of the folded links: 0.5 * 0.9 (and the noise), 1/48 * 1/24
    nu = np.array([0.5 * math.sqrt(0.81 + 3 * 2 * 0.02 ** 2), 1.0 / 1152.0] * 8)
    w1[0], w2[0] = sign * nu, c * sign * nu
    return w1.astype(np.complex64), w2.astype(np.complex64), np.complex64(8 / beta - c * case["sigma"])


def prepare(case, seed):
    _load(case)
    kind, n = case["kind"], _half(case)
    dt = torch.float32 if _is_float(case) else torch.float64
    st = dict(case=case, kind=kind)
    if kind in ("apply", "hop"):
        st["src"] = _source(case, seed, case.get("nrhs", 1), dt)
        st["dst"] = torch.empty_like(st["src"])
    elif kind in ("solve", "mixed"):
        nrhs, ns = case.get("nrhs", 1), case["nshift"]
        b = _source(case, seed, nrhs, dt)
        norm2 = [float(v) for v in b.double().square().sum((1, 2, 3))]
        st["par"] = A.InvertParam(shifts=np.array([_given(case)] * nrhs), tol=case["rel"] ** 2 * norm2[0], max_iter=20000, num_shift=ns,
                                  prec=A.KUQCD_SINGLE if _is_float(case) else A.KUQCD_DOUBLE,
                                  matpc_type=A.KUQCD_ODD_ODD if case["parity"] else A.KUQCD_EVEN_EVEN)
        if case.get("where") == "host":
            st["b"], st["x"] = b[0].cpu().numpy(), np.zeros((ns, n, 3, 2), b[0].cpu().numpy().dtype)
        else:
            st["b"], st["x"] = b, torch.zeros((nrhs * ns, n, 3, 2), dtype=dt, device=DEV)
            st["bp"] = (C.c_void_p * nrhs)(*[v.data_ptr() for v in b])
            st["xp"] = (C.c_void_p * (nrhs * ns))(*[v.data_ptr() for v in st["x"]])
        if kind == "mixed":
            st["opt"] = A.default_options(mode=MODES[case["mode"]], rel_tol=case["rel"], verbose=0)
            st["rep"] = (A.KqSolveReport * nrhs)()
    elif kind == "refine":
        A.ptnet_set_weights(A.weights_from_array(*_weights(case)))
        st["b"] = _source(case, seed, 1, dt)
        st["x"] = torch.empty_like(st["b"])
        st["opt"] = A.refine_options(rel_tol=case["rel"], learned=1)
        st["rep"] = A.KqRefineReport()
    else:
        st["w"] = A.weights_from_array(*_weights(case))
        # a pair as training takes it: a residual and a smooth guess of its error
        st["r"], st["e"] = _source(case, seed, 2, dt) / math.sqrt(3.0 * n)
        st["loss"], st["grad"] = C.c_double(), np.empty(2 * A.KQ_PT_PARAMS)
    return st


def run(st):
    case, kind, lib = st["case"], st["kind"], A.L.lib()
    if kind == "apply":
        src, dst = C.c_void_p(st["src"].data_ptr()), C.c_void_p(st["dst"].data_ptr())
        if case["entry"] == "noalloc":
            _ok(lib.kq_mdaggm_noalloc(src, dst, case["parity"], case["sigma"]))
        else:
            _ok(lib.kq_mdaggm(src, dst, case["parity"], case["sigma"], A.KQ_MODE_REFERENCE))
        return st["dst"]
    if kind == "hop":
        _ok(lib.kq_dslash_batched(case["nrhs"], C.c_void_p(st["src"].data_ptr()), C.c_void_p(st["dst"].data_ptr()), case["parity"],
                                  A.KQ_MODE_REFERENCE, case["nr"], 256))
        return st["dst"]
    if kind == "solve":
        if case["where"] == "host":
            _ok(A.kuqcd_solve_multishift(list(st["x"]), st["b"], st["par"]))
        else:
            _ok(lib.kq_solve_multishift(st["xp"], st["bp"][0], C.byref(st["par"].struct())))
        return st["x"]
    if kind == "mixed":
        _ok(lib.kq_solve_multishift_batched(case["nrhs"], st["xp"], st["bp"], C.byref(st["par"].struct()), C.byref(st["opt"]), st["rep"]))
        return st["x"]
    if kind == "refine":
        st["x"].zero_()
        torch.cuda.current_stream().synchronize()  # the library works on a stream of its own
        _ok(lib.kq_fcg_refine(case["parity"], case["sigma"], C.c_void_p(st["b"].data_ptr()), C.c_void_p(st["x"].data_ptr()),
                              C.byref(st["opt"]), C.byref(st["rep"])))
        return st["x"]
    _ok(lib.kq_ptnet_loss_grad(C.byref(st["w"]), case["parity"], case["sigma"], C.c_void_p(st["r"].data_ptr()), C.c_void_p(st["e"].data_ptr()),
                               C.byref(st["loss"]), st["grad"].ctypes.data_as(C.POINTER(C.c_double))))
    # both are formed from FP32 fields and go to FP32 master weights
    return np.float32(st["loss"].value), st["grad"].astype(np.float32)


# ------------------------------------------------------------------------------------------------ work
def _iterations(sigma, rel):
    """Conjugate-gradient iterations from 0 to the relative residual `rel` by the Chebyshev bound."""
    return 0.5 * math.sqrt((EIG_HIGH + sigma) / (EIG_LOW + sigma)) * math.log(2.0 / rel)


def work(case):
    """Bytes and operations of one pass. A hopping term reads every link (fat 18 reals, long 14: the smallest exact forms)
    and cannot start before the one that made its source has ended, so each counts its own pass over the links."""
    n, kind, ns = _half(case), case["kind"], case.get("nshift", 1)
    real = 4 if _is_float(case) or kind in ("mixed", "refine", "grad") else 8
    links, vec, flops = 8 * (18 + 14) * real * n, 6 * real * n, 1146.0 * n
    if kind == "apply":
        return dict(bytes=2 * links + 2 * vec, flops=2 * flops)
    if kind == "hop":
        return dict(bytes=links + 2 * case["nrhs"] * vec, flops=case["nrhs"] * flops)
    if kind in ("solve", "mixed"):
        it, nrhs = _iterations(case["lo"], case["rel"]), case.get("nrhs", 1)
        return dict(bytes=it * (2 * links + nrhs * 8 * vec) + nrhs * (1 + ns) * 6 * 8 * n, flops=nrhs * it * 2 * flops)
    if kind == "refine":  # half of plain CG's iterations, each with two hopping terms and two network layers
        it = 0.5 * _iterations(case["sigma"], case["rel"])
        return dict(bytes=it * (4 * links + 10 * vec), flops=it * (2 * flops + 8e3 * n))
    # forward (2), A twice (4), backward layer, two weight-gradient contractions and A e (2)
    return dict(bytes=11 * links + 24 * vec, flops=11 * flops + 2e4 * n)


# ------------------------------------------------------------------------------------------------ exact
class _Op:
    """The operator in plain torch, complex128, vectors (3, Vh)."""

    def __init__(self, case):
        lat = _lat(case)
        fat, lng = _links(case)
        if _is_float(case):  # what was loaded
            fat, lng = fat.to(torch.complex64).to(torch.complex128), lng.to(torch.complex64).to(torch.complex128)
        self.links = {1: fat * 0.5, 3: lng * (-1.0 / 48.0)}
        self.nbr = []
        stride = [0, lat[0] // 2, lat[0] // 2 * lat[1], lat[0] // 2 * lat[1] * lat[2]]
        s = torch.arange(math.prod(lat) // 2, device=DEV)
        for q in range(2):
            c = _coords(lat, q)
            tab = {}
            for mu in range(4):
                for h in (1, 3, -1, -3):
                    v = (c[mu] + h) % lat[mu]
                    tab[mu, h] = s + ((v >> 1) - (c[0] >> 1)) if mu == 0 else s + (v - c[mu]) * stride[mu]
            self.nbr.append(tab)

    def tap(self, q, mu, h, v):
        """Transport of v (parity 1 - q) by hop h along mu to the sites of parity q."""
        if h > 0:
            return (self.links[h][q, mu] * v[:, self.nbr[q][mu, h]][None]).sum(1)
        u = self.links[-h][1 - q, mu]
        return (u.conj() * v[:, None]).sum(0)[:, self.nbr[q][mu, h]]

    def hop(self, q, v):
        out = 0
        for mu in range(4):
            for h in (1, 3):
                out = out + self.tap(q, mu, h, v) - self.tap(q, mu, -h, v)
        return out

    def apply(self, q, sigma, v):
        return sigma * v - self.hop(q, self.hop(1 - q, v))


def _inner(src):
    return torch.view_as_complex(src.double().contiguous()).T.contiguous()  # (Vh, 3, 2) -> (3, Vh)


def _outer(v):
    return torch.view_as_real(v.T.contiguous())


def _solve(op, q, shifts, b):
    """Multishift conjugate gradients, all shifts to a residual of 1e-14."""
    zeta, zeta_old = [1.0] * len(shifts), [1.0] * len(shifts)
    x, p, r = [torch.zeros_like(b) for _ in shifts], [b.clone() for _ in shifts], b.clone()
    rr, beta_old, alpha = float(r.abs().square().sum()), 1.0, 0.0
    stop = 1e-28 * rr
    live = len(shifts)
    while live:
        s = op.apply(q, shifts[0], p[0])
        beta = -rr / float((p[0].conj() * s).sum().real)
        r = r + beta * s
        new = float(r.abs().square().sum())
        a, old = new / rr, list(zip(zeta, zeta_old))
        for k in range(live):
            z, zo = old[k]
            zn = z if k == 0 else z * zo * beta_old / (beta * alpha * (zo - z) + zo * beta_old * (1 - (shifts[k] - shifts[0]) * beta))
            bk = beta if k == 0 else beta * zn / z
            x[k] -= bk * p[k]
            ak = a if k == 0 else a * zn * bk / (z * beta)
            p[k] = zn * r + ak * p[k]
            zeta[k], zeta_old[k] = zn, z
        while live and zeta[live - 1] ** 2 * new < stop:
            live -= 1
        rr, beta_old, alpha = new, beta, a
    return x


def exact(case, seed):
    kind, q, n = case["kind"], case["parity"], _half(case)
    dt = torch.float32 if _is_float(case) else torch.float64
    if kind in ("apply", "hop"):
        op, src = _Op(case), _source(case, seed, case.get("nrhs", 1), dt)
        return torch.stack([_outer(op.apply(q, case["sigma"], _inner(v)) if kind == "apply" else op.hop(q, _inner(v))) for v in src])
    if kind in ("solve", "mixed", "refine"):
        shifts = [case["sigma"]] if kind == "refine" else _shifts(case)
        if _iterations(shifts[0], 1e-14) * n * (16 + len(shifts)) * case.get("nrhs", 1) > 1.2e10:
            return None  # well over 20 seconds
        op = _Op(case)
        return torch.stack([_outer(x) for b in _source(case, seed, case.get("nrhs", 1), dt) for x in _solve(op, q, shifts, _inner(b))])
    op = _Op(case)
    r, e = (_inner(v) for v in _source(case, seed, 2, dt) / math.sqrt(3.0 * n))
    nu = torch.tensor([math.sqrt(float(op.links[h].abs().square().sum()) / (24 * n)) for h in (1, 3)] * 8, device=DEV)

    def rounded(w, scale):  # the kernels' weights: bfloat16 of w / nu
        w = torch.view_as_real(torch.from_numpy(np.asarray(w)).to(DEV)).double() / (scale[None, :, None] if scale is not None else 1.0)
        return torch.view_as_complex(w.float().bfloat16().double()).requires_grad_(True)

    w1, w2, w0 = _weights(case)
    w1, w2, w0 = rounded(w1, nu), rounded(w2, nu), rounded(w0.reshape(1), None)
    taps = [(mu, h) for mu in range(4) for h in (1, 3, -1, -3)]
    tr = [op.tap(1 - q, mu, h, r) for mu, h in taps]
    hid = [sum(w1[c, t] * tr[t] for t in range(16)) for c in range(4)]
    z = w0 * r + sum(op.tap(q, mu, h, sum(w2[c, t] * hid[c] for c in range(4))) for t, (mu, h) in enumerate(taps))
    loss = op.apply(q, case["sigma"], z - e).abs().square().sum() / op.apply(q, case["sigma"], e).abs().square().sum()
    # the derivative by conj(w) is half of what torch returns for a complex leaf
    g1, g2, g0 = (g / 2 for g in torch.autograd.grad(loss, (w1, w2, w0)))
    grad = torch.cat([(g1 / nu).reshape(-1), (g2 / nu).reshape(-1), g0])
    return loss.detach().float(), torch.view_as_real(grad).reshape(-1).float()
