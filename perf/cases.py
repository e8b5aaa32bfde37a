"""The calls whose speed this package is kept by: one list of cases over the range it is used in.

A case is one pass of the work a spherical-shell time step (or a batch job) asks of the
library, through the package's public names:

  legendre  StP and PtS of one plan (all m, FP64 or a split-precision form)
  batch     the grouped StP and PtS of many independent problems
  step      spectral -> physical, a product of fields on the grid, physical -> spectral
  radial    the Chebyshev side: radial derivatives, synthesis, analysis, de-aliasing
  space     the passes between the radial and the spectral layout: Transpose_1a2a,
            rlm_spacea's and rlm_spaceb's passes, Transpose_2b1b
  dense     the implicit solve, dense path: factor one matrix per l, solve its columns
  band      the implicit solve, band path

Sizes follow the benchmark configurations (l_max 63 / 255 / 511 / 1023) and the grids in
between that users of a pseudo-spectral shell code choose: N_theta any smooth even
number, N_phi = 2 N_theta, l_max = 2 N_theta / 3 - 1.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import rayleigh_amd as ra

RMIN, RMAX = 0.35, 1.0
DEV = "cuda"


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the headline benchmark: every m at l_max = 511, N_r = 192, 8 fields
        dict(name="legendre_l511", kind="legendre", nt=768, lmax=511, nr=192, nf=8, precision="fp64"),
        # the same contraction in the split form that holds 1e-12, a mid-sized run
        dict(name="legendre_int8x6_l383", kind="legendre", nt=576, lmax=383, nr=64, nf=5, precision="int8x6"),
        # an ensemble: twelve independent transforms of ragged sizes in one grouped launch
        dict(name="batch_12", kind="batch",
             problems="31:32:2 47:96:1 63:48:4 84:32:5 127:64:3 131:32:8 170:64:2 191:96:1 239:32:4 255:64:2 319:32:3 383:32:2"),
        # the smallest run (a laptop-sized benchmark, many short calls)
        dict(name="step_l31", kind="step", nt=48, lmax=31, nr=32, nf=2),
        # the small benchmark configuration
        dict(name="step_l63", kind="step", nt=96, lmax=63, nr=48, nf=4),
        # an ordinary production run: N_theta = 256, N_phi = 512, l_max not a round number
        dict(name="step_l169", kind="step", nt=256, lmax=169, nr=96, nf=6),
        # the transform-stack benchmark configuration
        dict(name="step_l255", kind="step", nt=384, lmax=255, nr=128, nf=8),
        # the largest grid, on the share of the radii one of eight GPUs holds
        dict(name="step_l1023", kind="step", nt=1536, lmax=1023, nr=32, nf=5),
        # Chebyshev stages of the l_max = 169 run above: N_r = 96 is not a power of two
        dict(name="radial_n96", kind="radial", lmax=169, nr=96, nf=4),
        # spectral-space passes of a magnetic run at l_max = 255 (16 fields)
        dict(name="space_l191", kind="space", nt=288, lmax=191, nr=64),
        # the implicit solve of every l of the l_max = 255 run: coupled W-P system of 2 N_r
        dict(name="dense_n256", kind="dense", lmax=255, n=256),
        # the band solve of a four-domain run with N_r = 96
        dict(name="band_n192", kind="band", lmax=169, n=192, kl=72),
    ]


def _smooth(lo, hi):
    """Even numbers in [lo, hi] with no prime factor above 7: the N_theta (= N_phi / 2) users pick."""
    out = []
    for n in range(lo + (lo & 1), hi + 1, 2):
        k = n
        for p in (2, 3, 5, 7):
            while k % p == 0:
                k //= p
        if k == 1:
            out.append(n)
    return out


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(values, x):
    return min(values, key=lambda v: abs(math.log(v / x)))


def _cost(case):
    w = work(case)
    return w["bytes"] / 3e12 + w["flops"] / 3e13


def draw(rng):
    limit = max(_cost(c) for c in listed())
    kind = rng.choice(["legendre", "legendre", "batch", "step", "step", "step", "radial", "radial", "space", "dense",
                       "band"])
    while True:
        nt = _near(_smooth(24, 1536), math.exp(rng.uniform(math.log(40), math.log(1200))))
        lmax = 2 * nt // 3 - 1
        nr, nf = _log_int(rng, 12, 200), rng.randint(1, 8)
        if kind == "legendre":
            case = dict(kind=kind, nt=nt, lmax=lmax, nr=nr, nf=nf,
                        precision=rng.choice(["fp64", "fp64", "fp64", "int8x6", "bf16x6", "int8x3"]))
        elif kind == "batch":
            case = dict(kind=kind, problems=" ".join(
                "%d:%d:%d" % (2 * _log_int(rng, 12, 192) - 1, _log_int(rng, 16, 96), rng.randint(1, 4))
                for _ in range(rng.randint(3, 16))))
        elif kind == "step":
            case = dict(kind=kind, nt=nt, lmax=lmax, nr=nr, nf=nf)
        elif kind == "radial":
            case = dict(kind=kind, lmax=min(lmax, 255), nr=rng.choice([32, 48, 64, 72, 96, 128, 144, 192, 256, nr + 12]),
                        nf=rng.randint(1, 5))
        elif kind == "space":
            case = dict(kind=kind, nt=nt, lmax=min(lmax, 383), nr=nr)
        elif kind == "dense":
            case = dict(kind=kind, lmax=min(lmax, 255), n=_log_int(rng, 24, 512))
        else:
            n = _log_int(rng, 48, 512)
            case = dict(kind=kind, lmax=min(lmax, 255), n=n, kl=max(2, min(n - 1, 192, int(n * rng.uniform(0.1, 0.45)))))
        if case["kind"] == "batch" or case.get("lmax", 15) >= 15:
            if _cost(case) <= limit:
                return case


def _problems(case):
    """(n_theta, l_max, n_r, n_fields) of each problem of a batch: N_theta even, 3 (l_max + 1) / 2 or the next."""
    out = []
    for p in case["problems"].split():
        lmax, nr, nf = (int(v) for v in p.split(":"))
        nt = (3 * (lmax + 1) + 1) // 2
        out.append((nt + (nt & 1), lmax, nr, nf))
    return out


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, dtype=torch.float64, device=DEV, generator=g)


def _offsets(lmax, mv, cols):
    return np.concatenate([[0], np.cumsum((lmax - mv.astype(np.int64) + 1) * cols)])


def _spectral(g, lmax, mv, nr, nf):
    """Coefficients (N(0,1) + i N(0,1)) (l+1)^-2 sin(pi r / (N_r + 1)), m = 0 real: a resolved run's spectrum."""
    off = _offsets(lmax, mv, 2 * nr * nf)
    s = _randn(g, int(off[-1]))
    lf = (torch.arange(lmax + 1, dtype=torch.float64, device=DEV) + 1.0) ** -2
    rf = torch.sin(math.pi * torch.arange(1, nr + 1, dtype=torch.float64, device=DEV) / (nr + 1)).view(1, 1, nr, 1)
    for mp, m in enumerate(mv):
        b = s[int(off[mp]): int(off[mp + 1])].view(nf, 2, nr, lmax - int(m) + 1)
        b.mul_(lf[int(m):]).mul_(rf)
        if m == 0:
            b[:, 1] = 0.0
    return s


def _hybrid(g, nt, mv, nr, nf):
    """What PtS meets after r2c: modes of grid-space products, falling with m, rough in theta."""
    p = _randn(g, len(mv), 2 * nr * nf * nt)
    p.mul_((torch.as_tensor(mv.astype(np.float64), device=DEV) + 1.0).pow(-1.0).view(-1, 1))
    return p.view(-1)


def _empty(n):
    return torch.empty(int(n), dtype=torch.float64, device=DEV)


def _grid_ops(n):
    """T, dT/dr, d2T/dr2 (n x n: radius by coefficient) on the zeros grid of [RMIN, RMAX], and the radii."""
    th = (np.arange(n) + 0.5) * np.pi / n
    x, k = np.cos(th), np.arange(n)
    T = np.cos(np.outer(th, k))
    T[:, 0] *= 0.5
    s = np.sin(th)[:, None]
    c = np.cos(th)[:, None]
    D = k * np.sin(np.outer(th, k)) / s
    D2 = (-k * k * np.cos(np.outer(th, k)) + c / s * k * np.sin(np.outer(th, k))) / s ** 2
    half = (RMAX - RMIN) / (x[0] - x[-1])
    return T, D / half, D2 / half ** 2, RMIN + (x - x[-1]) * half


def _implicit_matrices(n, nl, g):
    """One two-variable implicit system per l: rows (1 - dt (d2/dr2 + 2/r d/dr - l(l+1)/r^2)) of each
    variable, coupled through first derivatives, with boundary rows; column-major."""
    h = n // 2
    sizes = (h, n - h)
    A = torch.zeros((nl, n, n), dtype=torch.float64, device=DEV)
    ell = torch.arange(nl, dtype=torch.float64, device=DEV)
    jit = 1.0 + 0.1 * torch.rand((4,), dtype=torch.float64, device=DEV, generator=g)
    at = 0
    for v, k in enumerate(sizes):
        T, D, D2, r = (torch.from_numpy(np.ascontiguousarray(q)).to(DEV) for q in _grid_ops(k))
        dt = 2e-5 * jit[v]
        blk = T - dt * (D2 + (2.0 / r)[:, None] * D) + (dt * (ell * (ell + 1.0))).view(-1, 1, 1) * (T / (r * r)[:, None])
        blk[:, 0], blk[:, -1] = T[0], T[-1]
        A[:, at: at + k, at: at + k] = blk
        q = min(sizes)
        o = 0 if v else h
        C = 0.01 * jit[2 + v] * D[:q, :q]
        C[0], C[-1] = 0.0, 0.0
        A[:, at: at + q, o: o + q] += C
        at += k
    return A.transpose(1, 2).contiguous().view(-1)


def _columns(lmax, n, g):
    """2 (l + 1) right-hand sides per l (re and im of every m <= l), packed; offsets and counts."""
    nc = [2 * (l + 1) for l in range(lmax + 1)]
    off = np.concatenate([[0], np.cumsum([c * n for c in nc])]).astype(np.int64)
    return (_randn(g, int(off[-1])), torch.from_numpy(off[:-1]).to(DEV), torch.tensor(nc, dtype=torch.int32, device=DEV),
            max(nc))


class State:
    pass


def prepare(case, seed):
    st, g, kind = State(), _gen(seed), case["kind"]
    st.kind = kind
    if kind in ("legendre", "step"):
        mv = ra.m_values_balanced(case["lmax"])
        st.plan = ra.LegendrePlan(case["nt"], case["lmax"], mv, case["nr"], case["nf"],
                                  precision=case.get("precision", "fp64"))
        st.s = _spectral(g, case["lmax"], mv, case["nr"], case["nf"])
        st.s_out = torch.empty_like(st.s)
        st.p2 = _empty(st.plan.hybrid_size)
        if kind == "legendre":
            st.p2_in = _hybrid(g, case["nt"], mv, case["nr"], case["nf"])
        else:
            st.nphi = 2 * case["nt"]
            st.u, st.uu = (_empty((st.nphi + 2) * case["nr"] * case["nt"] * case["nf"]) for _ in range(2))
    elif kind == "batch":
        st.plans, st.s, st.p2_in = [], [], []
        for nt, lmax, nr, nf in _problems(case):
            mv = ra.m_values_balanced(lmax)
            st.plans.append(ra.LegendrePlan(nt, lmax, mv, nr, nf))
            st.s.append(_spectral(g, lmax, mv, nr, nf))
            st.p2_in.append(_hybrid(g, nt, mv, nr, nf))
        st.batch = ra.LegendreBatch(st.plans)
        st.p2 = [torch.empty_like(p) for p in st.p2_in]
        st.s_out = [torch.empty_like(s) for s in st.s]
    elif kind == "radial":
        n, nlm = case["nr"], (case["lmax"] + 1) * (case["lmax"] + 2) // 2
        st.cheb = ra.ChebyGrid(n, RMIN, RMAX)
        fall = (torch.arange(n, dtype=torch.float64, device=DEV) + 1.0) ** -3
        # variables: the solution's coefficients, its first and its second derivative
        st.buf = torch.zeros((3, case["nf"] * nlm * 2 * n), dtype=torch.float64, device=DEV)
        st.buf[0] = (_randn(g, case["nf"] * nlm * 2, n) * fall).view(-1)
        st.out = torch.empty_like(st.buf)
        st.rhs = _randn(g, case["nf"] * nlm * 2 * n)  # the nonlinear terms on the grid, after Transpose_2b1b
        st.c_rhs = torch.empty_like(st.rhs)
    elif kind == "space":
        mv = ra.m_values_balanced(case["lmax"])
        st.plan = ra.LegendrePlan(case["nt"], case["lmax"], mv, case["nr"], 16)
        st.p1 = _randn(g, st.plan.spectral_size)
        st.buf = torch.empty_like(st.p1)
        st.p1_out = torch.empty_like(st.p1)
        st.prof = {k: torch.rand(case["nr"], dtype=torch.float64, device=DEV, generator=g) + 0.5
                   for k in ("over_rhor", "over_rhorsq", "drho_term", "two_over_r", "dlnrho", "one_over_rsq")}
    elif kind == "dense":
        n, nl = case["n"], case["lmax"] + 1
        st.n = n
        st.mats0 = _implicit_matrices(n, nl, g)
        st.mats = torch.empty_like(st.mats0)
        st.piv = torch.empty(nl * n, dtype=torch.int32, device=DEV)
        st.info = torch.empty(nl, dtype=torch.int32, device=DEV)
        st.rhs0, st.off, st.nc, st.most = _columns(case["lmax"], n, g)
        st.rhs = torch.empty_like(st.rhs0)
    elif kind == "band":
        n, kl, nl = case["n"], case["kl"], case["lmax"] + 1
        ldab = 3 * kl + 1
        st.n, st.kl = n, kl
        ab = torch.zeros((nl, n, ldab), dtype=torch.float64, device=DEV)
        ab[:, :, kl:] = _randn(g, nl, n, 2 * kl + 1)
        ab[:, :, 2 * kl].add_(2.0 * math.sqrt(2.0 * kl))  # a diagonal that is often, not always, the pivot
        j = torch.arange(n, device=DEV).view(n, 1)
        i = j + torch.arange(ldab, device=DEV).view(1, ldab) - 2 * kl
        ab[:, ~((i >= 0) & (i < n))] = 0.0
        st.mats0 = ab.view(-1)
        st.mats = torch.empty_like(st.mats0)
        st.piv = torch.empty(nl * n, dtype=torch.int32, device=DEV)
        st.info = torch.empty(nl, dtype=torch.int32, device=DEV)
        st.rhs0, st.off, st.nc, st.most = _columns(case["lmax"], n, g)
        st.rhs = torch.empty_like(st.rhs0)
    else:
        raise ValueError(kind)
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    kind = st.kind
    if kind == "legendre":
        st.plan.stp(st.s, st.p2)
        st.plan.pts(st.p2_in, st.s_out)
        return st.p2, st.s_out
    if kind == "batch":
        st.batch.stp(st.s, st.p2)
        st.batch.pts(st.p2_in, st.s_out)
        return st.p2, st.s_out
    if kind == "step":
        st.plan.spectral_to_physical(st.s, st.p2, st.u, st.nphi)
        torch.mul(st.u, st.u, out=st.uu)  # the nonlinear term on the grid
        st.plan.physical_to_spectral(st.uu, st.p2, st.s_out, st.nphi)
        return st.u, st.s_out
    if kind == "radial":
        st.cheb.d_by_dr_cp(1, 2, st.buf, 1)
        st.cheb.d_by_dr_cp(1, 3, st.buf, 2)
        st.cheb.from_spectral(st.buf, st.out)
        st.cheb.to_spectral(st.rhs, st.c_rhs)
        st.cheb.dealias_buffer(st.c_rhs)
        return st.buf, st.out, st.c_rhs
    if kind == "space":
        st.plan.transpose_1a2a(st.p1, st.buf)
        st.plan.rlm_spacea_hydro(st.buf, list(range(10)), st.prof)
        st.plan.compute_bandcurlb(st.buf, list(range(10, 16)), st.prof["one_over_rsq"])
        st.plan.adjust_emf(st.buf, 10, 11)
        st.plan.rlm_spaceb_hydro(st.buf, 0, 1, 3)
        st.plan.transpose_2b1b(st.buf, st.p1_out)
        return st.buf, st.p1_out
    st.mats.copy_(st.mats0)  # the loaded matrices and right-hand sides: both are overwritten
    st.rhs.copy_(st.rhs0)
    if kind == "dense":
        ra.lu_decompose_full(st.mats, st.piv, st.info, st.n)
        ra.lu_solve_full(st.mats, st.piv, st.rhs, st.off, st.nc, st.n, st.most)
    else:
        ra.lu_decompose_band(st.mats, st.piv, st.info, st.n, st.kl)
        ra.lu_solve_band(st.mats, st.piv, st.rhs, st.off, st.nc, st.n, st.kl, st.most)
    return st.mats, st.piv, st.info, st.rhs


# ---------------------------------------------------------------- what a pass cannot do without
def _legendre_work(nt, lmax, nr, nf):
    nrhs, nlm = 2 * nr * nf, (lmax + 1) * (lmax + 2) // 2
    return (8.0 * (nlm * nrhs + (lmax + 1) * nrhs * nt + nlm * nt / 2), 1.0 * nt * nrhs * nlm)


def work(case):
    kind = case["kind"]
    if kind == "legendre":
        b, f = _legendre_work(case["nt"], case["lmax"], case["nr"], case["nf"])
        return dict(bytes=2 * b, flops=2 * f)
    if kind == "batch":
        w = [_legendre_work(*p) for p in _problems(case)]
        return dict(bytes=2 * sum(b for b, _ in w), flops=2 * sum(f for _, f in w))
    if kind == "step":
        nt, lmax, nr, nf = case["nt"], case["lmax"], case["nr"], case["nf"]
        nlm, lines, nphi = (lmax + 1) * (lmax + 2) // 2, nt * nr * nf, 2 * nt
        _, f = _legendre_work(nt, lmax, nr, nf)
        # the spectra in and out, the tables, the grid written by each of the two grid-space
        # calls and read by the next
        return dict(bytes=8.0 * (2 * nlm * 2 * nr * nf + nlm * nt + 4 * lines * (nphi + 2)),
                    flops=2 * f + lines * (2 * 2.5 * nphi * math.log2(nphi) + nphi))
    if kind == "radial":
        vals = case["nf"] * (case["lmax"] + 1) * (case["lmax"] + 2) * case["nr"]
        # one variable read and its two derivatives written, three synthesised, one analysed
        return dict(bytes=8.0 * vals * (3 + 3 + 2), flops=vals * (4 * 2.5 * math.log2(case["nr"]) + 9))
    if kind == "space":
        per = 2 * case["nr"] * (case["lmax"] + 1) * (case["lmax"] + 2) // 2
        return dict(bytes=8.0 * per * 16 * 3, flops=1.0 * per * 110)
    n, nl = case["n"], case["lmax"] + 1
    cols = nl * (nl + 1)
    if kind == "dense":
        return dict(bytes=8.0 * (2 * nl * n * n + 2 * cols * n), flops=nl * 2.0 * n ** 3 / 3 + 2.0 * n * n * cols)
    kl = case["kl"]
    return dict(bytes=8.0 * (2 * nl * n * (3 * kl + 1) + 2 * cols * n), flops=nl * 4.0 * n * kl * kl + 6.0 * n * kl * cols)


# ---------------------------------------------------------------- the same in plain 64-bit torch / numpy
def _m_order(lmax):
    """The one-rank m order: 0, l_max, 1, l_max - 1, ..."""
    n = lmax + 1
    return np.array([v for i in range(n // 2) for v in (i, n - 1 - i)] + ([n // 2] if n % 2 else []), dtype=np.int32)


def _nodes(nt):
    """Gauss-Legendre nodes, ascending, and weights (Newton from the asymptotic guess, long double)."""
    x = np.cos(np.pi * (np.arange(nt, 0, -1, dtype=np.longdouble) - 0.25) / (nt + 0.5))
    for _ in range(6):
        p0, p1 = np.ones_like(x), x.copy()
        for l in range(2, nt + 1):
            p0, p1 = p1, ((2 * l - 1) * x * p1 - (l - 1) * p0) / l
        d = nt * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / d
    return x.astype(np.float64), (2 / ((1 - x * x) * d * d)).astype(np.float64)


def _plm(nt, lmax):
    """[m][l][theta] orthonormal P_lm with the Condon-Shortley sign; values carry a power of two until
    they are stored, since sin^m falls far below the smallest double. Also the weights."""
    xh, wh = _nodes(nt)
    x, w = torch.from_numpy(xh).to(DEV), torch.from_numpy(wh).to(DEV)
    m = torch.arange(lmax + 1, dtype=torch.float64, device=DEV).view(-1, 1)
    k = np.arange(1, lmax + 1)
    amp = np.concatenate([[0.0], np.cumsum(0.5 * np.log2((2 * k + 1) / (2.0 * k)))]) - 0.5 * math.log2(4 * math.pi)
    lg = torch.from_numpy(amp).to(DEV).view(-1, 1) + m * (0.5 * torch.log2((1 - x) * (1 + x))).view(1, -1)
    e = torch.floor(lg)
    prev = torch.exp2(lg - e) * torch.where(m % 2 == 0, 1.0, -1.0)  # P_mm
    out = torch.zeros((lmax + 1, lmax + 1, nt), dtype=torch.float64, device=DEV)
    cur = torch.zeros_like(prev)  # P_{l-1} and P_l of every m at the loop's l
    last = torch.zeros_like(prev)
    two = torch.tensor(2.0, dtype=torch.float64, device=DEV)
    for l in range(lmax + 1):
        if l > 0:
            a = torch.sqrt(((4.0 * l * l - 1.0) / (l * l - m * m).clamp_min(1.0)))
            b = torch.sqrt((((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1.0) ** 2 - 1.0)).clamp_min(0.0))
            nxt = a * (x * cur - b * last)
            nxt[l:] = 0.0
            last, cur = cur, nxt
        cur[l] = prev[l]
        big = 498.0 * (cur.abs() > 1e150).to(torch.float64)
        f = torch.exp2(-big)
        cur, last, e = cur * f, last * f, e + big
        # 2^e in two halves: neither overflows, the product underflows to zero where the value does
        e1 = torch.clamp(torch.floor(e * 0.5), -1000.0, 1000.0)
        out[: l + 1, l] = (cur * torch.pow(two, e1) * torch.pow(two, torch.clamp(e - e1, -1000.0, 1000.0)))[: l + 1]
    return out, w


def _stp(P, lmax, mv, cols, s):
    off = _offsets(lmax, mv, cols)
    return torch.stack([(s[int(off[i]): int(off[i + 1])].view(cols, lmax - int(m) + 1) @ P[int(m), int(m):].contiguous())
                        * (1.0 if m == 0 else 0.5) for i, m in enumerate(mv)])


def _pts(P, w, lmax, mv, cols, p2):
    nt = w.numel()
    p2 = p2.view(len(mv), cols, nt)
    return torch.cat([((p2[i] * (w * (2 * math.pi / nt * (0.5 if m == 0 else 1.0)))) @ P[int(m), int(m):].t().contiguous())
                      .reshape(-1) for i, m in enumerate(mv)])


def _legendre_exact(nt, lmax, nr, nf, s, p2_in):
    mv, cols = _m_order(lmax), 2 * nr * nf
    P, w = _plm(nt, lmax)
    return _stp(P, lmax, mv, cols, s).view(-1), _pts(P, w, lmax, mv, cols, p2_in)


def _step_exact(nt, lmax, nr, nf, s):
    mv, cols, nphi = _m_order(lmax), 2 * nr * nf, 2 * nt
    P, w = _plm(nt, lmax)
    p2 = _stp(P, lmax, mv, cols, s).view(len(mv), nf, 2, nr, nt)
    at = torch.as_tensor(mv.astype(np.int64), device=DEV)
    u = torch.zeros((nf, nt, nr, nphi + 2), dtype=torch.float64, device=DEV)
    back = torch.empty_like(p2)
    for f in range(nf):
        X = torch.zeros((nt, nr, nt + 1), dtype=torch.complex128, device=DEV)
        X[:, :, at] = torch.complex(p2[:, f, 0], p2[:, f, 1]).permute(2, 1, 0)
        u[f, :, :, :nphi] = torch.fft.irfft(X, n=nphi, norm="forward")
        Y = torch.fft.rfft(u[f, :, :, :nphi] ** 2)[:, :, at].permute(2, 1, 0)
        back[:, f, 0], back[:, f, 1] = Y.real, Y.imag
    return u.view(-1), _pts(P, w, lmax, mv, cols, back.view(-1))


def _radial_exact(case, st):
    n = case["nr"]
    th = (np.arange(n) + 0.5) * np.pi / n
    T = torch.from_numpy(np.cos(np.outer(np.arange(n), th))).to(DEV)  # [k][i]
    scale = (math.cos(th[0]) - math.cos(th[-1])) / (RMAX - RMIN)
    c = st.buf[0].view(-1, n)

    def deriv(a):
        d = torch.zeros((n + 2, a.shape[0]), dtype=torch.float64, device=DEV)
        at = a.t().contiguous()
        for i in range(n - 2, -1, -1):
            d[i] = d[i + 2] + 2.0 * (i + 1) * at[i + 1]
        return (d[:n] * scale).t().contiguous()

    d1 = deriv(c)
    buf = torch.stack([c, d1, deriv(d1)])
    out = buf @ T - 0.5 * buf[:, :, :1]
    rhs = (st.rhs.view(-1, n) @ T.t().contiguous()) * (2.0 / n)
    rhs[:, (2 * n) // 3:] = 0.0
    return buf.view(3, -1), out.view(3, -1), rhs.view(-1)


def _space_exact(case, st):
    lmax, nr, nf = case["lmax"], case["nr"], 16
    mv = _m_order(lmax)
    lm = [(l, i) for l in range(lmax + 1) for i in range(len(mv)) if mv[i] <= l]
    where = {}
    for k, (l, i) in enumerate(lm):
        where.setdefault(i, []).append(k)
    p1 = st.p1.view(nf, len(lm), 2, nr)
    out1 = torch.empty_like(p1)
    pr = {k: v.view(1, nr, 1) for k, v in st.prof.items()}
    blocks = []
    for i, m in enumerate(int(v) for v in mv):
        k = torch.tensor(where[i], device=DEV)
        a = p1[:, k].permute(0, 2, 3, 1).contiguous()  # [f][imi][r][l]
        l = torch.arange(m, lmax + 1, dtype=torch.float64, device=DEV)
        ll = l * (l + 1)
        ol = torch.where(l == 0, 1.0, 1.0 / ll.clamp_min(1.0))
        q = torch.sqrt((l + m) * (l - m) / ((2 * l + 1) * (2 * l - 1)).abs())
        q1 = torch.sqrt((l + 1 + m) * (l + 1 - m) / ((2 * l + 1) * (2 * l + 3)))

        def theta(x, lo, hi):
            y = torch.zeros_like(x)
            y[..., 1:] += x[..., :-1] * (lo * q)[1:]
            y[..., :-1] -= x[..., 1:] * (hi * q1)[:-1]
            return y

        def dt(x):
            return theta(x, l - 1, l + 2)

        def sdt(x):
            return theta(x, l + 1, l)

        def dp(x):
            return torch.stack([-m * x[1], m * x[0]])

        W, dW, d2W, Z, dZ, T = (a[v].clone() for v in range(6))
        vr = ll * W * pr["over_rhorsq"]
        vt, vp = (dt(dW) + dp(Z)) * pr["over_rhor"], (dp(dW) - dt(Z)) * pr["over_rhor"]
        a[8] = (dt(d2W) + dp(dZ)) * pr["over_rhor"] - vt * pr["drho_term"]
        a[9] = (dp(d2W) - dt(dZ)) * pr["over_rhor"] - vp * pr["drho_term"]
        a[0], a[6], a[7] = vr, vt, vp
        a[1] = ll * dW * pr["over_rhorsq"] - vr * pr["two_over_r"] - vr * pr["dlnrho"]
        a[4], a[3], a[2] = dt(vr), ll * Z * pr["over_rhorsq"], dt(T)
        C, A, dC, dA, d2C = (a[10 + v].clone() for v in range(5))
        br = ll * C * pr["one_over_rsq"]
        e = d2C - br
        a[10], a[15] = br, ll * A * pr["one_over_rsq"]
        a[13], a[14] = dp(dA) + dt(e), dt(dA) - dp(e)
        a[11], a[12] = dp(A) + dt(dC), dp(dC) - dt(A)
        et, ep = a[10].clone(), a[11].clone()
        a[10], a[11] = (sdt(ep) - dp(et)) * ol, (dp(ep) + sdt(et)) * ol
        P, Z = a[1].clone(), a[3].clone()
        a[0], a[3], a[1] = a[0] * ol, (dp(P) - sdt(Z)) * ol, (sdt(P) + dp(Z)) * ol
        if m == 0:
            for v in (0, 1, 3):
                a[v][..., 0] = 0.0
        a[..., -1] = 0.0
        blocks.append(a.reshape(-1))
        out1[:, k] = a.permute(0, 3, 1, 2)
    return torch.cat(blocks), out1.view(-1)


def _solve_exact(full, n, lmax, rhs0):
    """The solutions, matrix by matrix (numpy, LAPACK)."""
    full, b, out, at = full.cpu().numpy(), rhs0.cpu().numpy(), [], 0
    for l in range(lmax + 1):
        k = 2 * (l + 1)
        out.append(np.linalg.solve(full[l], b[at: at + k * n].reshape(k, n).T).T.ravel())
        at += k * n
    return None, None, None, np.concatenate(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        g, s, p = _gen(seed), [], []
        for nt, lmax, nr, nf in _problems(case):
            mv = _m_order(lmax)
            s.append(_spectral(g, lmax, mv, nr, nf))
            p.append(_hybrid(g, nt, mv, nr, nf))
        pairs = [_legendre_exact(*q, a, b) for q, a, b in zip(_problems(case), s, p)]
        return [a for a, _ in pairs], [b for _, b in pairs]
    st = prepare(case, seed)
    if kind == "legendre":
        return _legendre_exact(case["nt"], case["lmax"], case["nr"], case["nf"], st.s, st.p2_in)
    if kind == "step":
        return _step_exact(case["nt"], case["lmax"], case["nr"], case["nf"], st.s)
    if kind == "radial":
        return _radial_exact(case, st)
    if kind == "space":
        return _space_exact(case, st)
    n, nl = case["n"], case["lmax"] + 1
    if kind == "dense":
        return _solve_exact(st.mats0.view(nl, n, n).transpose(1, 2), n, case["lmax"], st.rhs0)
    kl = case["kl"]
    ab = st.mats0.view(nl, n, 3 * kl + 1)
    full = torch.zeros((nl, n, n), dtype=torch.float64, device=DEV)
    for d in range(-kl, kl + 1):  # a(j + d, j) sits at row 2 kl + d of column j
        j = torch.arange(max(0, -d), min(n, n - d), device=DEV)
        full[:, j + d, j] = ab[:, j, 2 * kl + d]
    return _solve_exact(full, n, case["lmax"], st.rhs0)
