"""The work that users of this framework have it do, as cases that can be timed.

Every case goes through the public Python entry points (mini_mdft_amd.mdft),
over the sizes of the benchmark configurations, the tests and the served mixes:

* energy: one c-proj evaluation (F_exc and its gradient array) of a density
  field that is already on the GPU, alone or as a same-shape batch;
* chain: the same evaluation by the five calls of the reference's class API
  (get_delta_rho, angl2proj, Convolution.execute, proj2angl, get_delta_f);
* vext: the external potential of a solute and the start point taken from it;
* solve: one solute from its sites to the converged density;
* serve: several solutes submitted to a server and run to the end.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mini_mdft_amd import FP32, FP64, MIXED_X6, MIXED_X6F, luc, solute
from mini_mdft_amd import mdft as M

FORMS = {"fp64": FP64, "fp32": FP32, "x6": MIXED_X6, "x6f": MIXED_X6F}
TEMP, N0 = 298.15, M.SOLVENTS["spce"]["n0"]
C_SEED, XI_AMP = 2024, 0.1  # the benchmark's c(q) draw and the spread of its xi
WATER = solute.SOLVENT_SITES["tip3p"]
VMAX_KT, QSCALE = 100.0, 0.1  # cap of V_ext and charge scale of the solve configurations
GTOL, MAX_ITER = 1e-5, 400
SPACING = 0.47  # A per grid side of the large and served grids


def _case(kind, n, mmax, form, mrso=2, box=None, **more):
    n = (n,) * 3 if isinstance(n, int) else n
    box = box or [SPACING * v for v in n]
    return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], lx=box[0], ly=box[1], lz=box[2], mmax=mmax, mrso=mrso,
                form=form, **more)


def listed():
    b30 = (30.0,) * 3
    cases = {
        # the benchmark's evaluation in its fastest mixed form: 64^3, 30 A, mmax 5
        "energy_x6f_64": _case("energy", 64, 5, "x6f", box=b30, batch=1),
        # the same in plain FP64, the form the reference's users know
        "energy_fp64_64": _case("energy", 64, 5, "fp64", box=b30, batch=1),
        # FP64 fields with mixed arithmetic on a large-solute grid
        "energy_x6_80": _case("energy", 80, 5, "x6", batch=1),
        # the largest grid of the configurations
        "energy_x6f_96": _case("energy", 96, 5, "x6f", batch=1),
        # the single-ion configuration: 32^3, 20 A, mmax 3, FP64
        "energy_fp64_32": _case("energy", 32, 3, "fp64", box=(20.0,) * 3, batch=1),
        # the smallest calls (unit-test sized systems): launches and latency
        "energy_x6f_8": _case("energy", 8, 3, "x6f", box=(10.0,) * 3, batch=1),
        # the reference's ScalarType = float on a ragged, non-cubic grid
        "energy_fp32_45x36x50": _case("energy", (45, 36, 50), 4, "fp32", batch=1),
        # one tick of a server's evaluation: four same-shape fields together
        "batch_x6f_4x48": _case("energy", 48, 5, "x6f", batch=4),
        # a caller that keeps the reference's own sequence of calls, a
        # molecule without a symmetry axis, an odd grid
        "chain_fp64_30x42x27": _case("chain", (30, 42, 27), 3, "fp64", mrso=1),
        # per solute: V_ext of a 20-site solute and the start point
        "vext_64": _case("vext", 64, 5, "fp64", box=b30, sites=20),
        # the time to a converged density of a 20-site solute
        "solve_x6f_64": _case("solve", 64, 5, "x6f", box=b30, sites=20),
        # a small served batch: four solutes of one shape
        "serve_x6f_4x32": _case("serve", 32, 3, "x6f", sites=10, batch=4),
    }
    return [dict(c, name=k) for k, c in cases.items()]


def _smooth(lo, hi, primes=(2, 3, 5, 7, 11, 13)):
    out = []
    for v in range(lo, hi + 1):
        r = v
        for p in primes:
            while r % p == 0:
                r //= p
        if r == 1:
            out.append(v)
    return out


_SIDES = _smooth(8, 96)
_MOST = 96**3 * 330  # field values of the largest listed evaluation


def _side(rng):
    """A grid side of 8 .. 96, uniform in its logarithm."""
    v = math.exp(rng.uniform(math.log(8), math.log(96.99)))
    return min(_SIDES, key=lambda s: abs(s - v))


def _no(mmax, mrso):
    return (mmax + 1) * (2 * mmax + 1) * (2 * (mmax // mrso) + 1)


def draw(rng):
    kind = rng.choice(["energy"] * 6 + ["chain"] * 2 + ["vext", "solve", "serve"])
    if kind in ("solve", "serve"):
        # the served grids: cubic, sides of a multiple of 4, mmax 3 or 5
        side, mmax = 4 * rng.randint(5, 16 if kind == "solve" else 12), rng.choice([3, 5])
        more = dict(batch=rng.randint(2, 4)) if kind == "serve" else {}
        return _case(kind, side, mmax, rng.choice(["x6f", "x6f", "fp64"]), sites=rng.randint(5, 40), **more)
    while True:
        mmax = rng.choice([2, 3, 4, 5, 5, 5])
        mrso = 1 if mmax <= 3 and rng.random() < 0.25 else 2
        n = [_side(rng)] * 3 if rng.random() < 0.5 else [_side(rng) for _ in range(3)]
        if kind == "vext":
            c = _case(kind, n, mmax, "fp64", mrso, sites=rng.randint(5, 40))
            cost = n[0] * n[1] * n[2] * _no(mmax, mrso) * 2
        elif kind == "chain":
            c = _case(kind, n, mmax, rng.choice(["fp64", "fp32"]), mrso)
            cost = n[0] * n[1] * n[2] * _no(mmax, mrso) * 3
        else:
            batch = rng.choice([1, 1, 1, 2, 3, 4])
            if (n[0] * n[1] * n[2]) % 64:
                batch = 1
            form = rng.choice(["x6f", "x6f", "fp64", "x6", "fp32"])
            c = _case(kind, n, mmax, form, mrso, batch=batch)
            cost = n[0] * n[1] * n[2] * _no(mmax, mrso) * batch * (2 if form in ("fp64", "x6") else 1)
        if cost <= _MOST:
            return c


# ---------------------------------------------------------------------------
def _grid(c):
    return (c["nx"], c["ny"], c["nz"]), (c["lx"], c["ly"], c["lz"])


def _table(c):
    """The c(q) of a case: the benchmark's synthetic draw for evaluations, the
    exchange-symmetric model for minimisations."""
    n, L = _grid(c)
    nq = luc.nq_for(luc.qmax_of_grid(n, L), luc.DQ_TIP3P) + 2
    make = luc.model_c_symmetric if c["kind"] in ("solve", "serve") else luc.synthetic_c
    return make(c["mmax"], c["mrso"], nq, seed=C_SEED)


def _solvent(c):
    return M.rho0_of(N0, c["mrso"]), M.prefactor_of(TEMP, c["mrso"], N0)


def _solute(c, seed):
    radius = min(5.0, 0.3 * min(_grid(c)[1]))
    sep = 1.2 if radius > 4 else 0.25 * radius
    return solute.synthetic_solute(c["sites"], seed % 100003 + 1, _grid(c)[1], radius=radius, min_sep=sep,
                                   charge_scale=QSCALE)


def prepare(c, seed):
    n, L = _grid(c)
    prec = FORMS[c["form"]]
    g, ag = M.SpatialGrid(n, L), M.AngularGrid(c["mmax"], c["mrso"])
    mp = M.OrientationProjectionMap(ag)
    rho0, pref = _solvent(c)
    kT = M.kT(TEMP)
    s = dict(case=c, g=g, ag=ag, rho0=rho0, pref=pref, kT=kT)
    if c["kind"] == "vext":
        s.update(solute=_solute(c, seed), V=torch.empty((g.N, ag.m_no), dtype=torch.float64, device="cuda"))
        s["xi"] = torch.empty_like(s["V"])
        return s
    if c["kind"] == "serve":
        srv = M.Server(_table(c), c["mrso"], N0, TEMP, prec, capacity=4, m=1, max_iter=MAX_ITER, gtol=GTOL,
                       budget_bytes=60e9)
        srv.start_from_vext(True)
        s.update(server=srv, solutes=[_solute(c, seed + 1000 * j) for j in range(c["batch"])],
                 xi=[torch.empty((g.N, ag.m_no), dtype=torch.float64, device="cuda") for _ in range(c["batch"])])
        return s
    conv = M.Convolution.from_table(_table(c), g, ag, mp, prec)
    if c["kind"] == "solve":
        solver = M.Solver(conv, rho0, pref, prec)
        V = torch.empty((g.N, ag.m_no), dtype=torch.float64, device="cuda")
        s.update(V=V, xi=torch.empty_like(V), functional=M.Functional(solver, V, kT), solute=_solute(c, seed))
        return s
    dt = torch.float64 if c["form"] in ("fp64", "x6") else torch.float32
    shape = (c.get("batch", 1), g.N, ag.m_no) if c["kind"] == "energy" else (g.N, ag.m_ntheta, ag.m_nphi, ag.m_npsi)
    xi = torch.empty(shape, dtype=dt, device="cuda")
    M.fill_uniform(xi, seed, 1.0 - XI_AMP, 1.0 + XI_AMP)
    s.update(xi=xi, df=torch.empty_like(xi))
    if c["kind"] == "energy":
        s["solver"] = M.Solver(conv, rho0, pref, prec, capacity=c["batch"])
        return s
    s.update(conv=conv, opt=M.OrientationProjectionTransform(g, ag, mp, prec), field=torch.empty_like(xi),
             p=torch.empty((ag.m_np,) + n, dtype=torch.complex128 if c["form"] == "fp64" else torch.complex64,
                           device="cuda"),
             w=torch.from_numpy(ag.m_w).to("cuda"))
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "energy":
        if c["batch"] == 1:
            return dict(ff=s["solver"].energy_cproj(s["xi"], s["df"]), df=s["df"])
        return dict(ff=s["solver"].energy_cproj_batch(s["xi"], s["df"]), df=s["df"])
    if kind == "chain":
        xi, field, p, df = s["xi"], s["field"], s["p"], s["df"]
        M.get_delta_rho(xi, field, s["rho0"])
        s["opt"].angl2proj(field, p)
        s["conv"].execute(p)
        s["opt"].proj2angl(p, field)
        n, no = s["g"].m_n_nodes, s["ag"].m_no
        v = [t.view(*n, no) for t in (xi, field, df)]
        ff = M.get_delta_f(v[0], v[1], s["w"], v[2], s["rho0"], s["pref"])
        return dict(ff=ff, df=df, vexc=field, p=p)
    if kind == "vext":
        M.vext(s["g"], s["ag"], s["solute"], WATER, VMAX_KT * s["kT"], out=s["V"])
        M.xi_from_vext(s["V"], s["kT"], out=s["xi"])
        return dict(V=s["V"], xi=s["xi"])
    if kind == "solve":
        M.vext(s["g"], s["ag"], s["solute"], WATER, VMAX_KT * s["kT"], out=s["V"])
        M.xi_from_vext(s["V"], s["kT"], out=s["xi"])
        r = s["functional"].minimize(s["xi"], m=1, max_iter=MAX_ITER, gtol=GTOL)
        return dict(F=list(r["F"]), iterations=r["iterations"], status=r["status"], xi=s["xi"])
    n, L = _grid(c)
    srv = s["server"]
    ids = [srv.submit(n, L, c["mmax"], sol, WATER, VMAX_KT * s["kT"], out=x)
           for sol, x in zip(s["solutes"], s["xi"])]
    got = srv.run()
    return dict(F=[list(got[i]["F"]) for i in ids], status=[got[i]["status"] for i in ids],
                iterations=[got[i]["iterations"] for i in ids], xi=s["xi"])


# ---------------------------------------------------------------------------
def work(c):
    """One read of every input and one write of every output, and the
    operations of the factorised transforms, 3D FFTs and the OZ pass."""
    N = c["nx"] * c["ny"] * c["nz"]
    mmax, mrso = c["mmax"], c["mrso"]
    no, kphi, kmu = _no(mmax, mrso), 2 * mmax + 1, mmax // mrso + 1
    np_ = sum((2 * m + 1) * (m // mrso + 1) for m in range(mmax + 1))
    e = 8 if c["form"] in ("fp64", "x6") else 4
    O = N * no
    # per point and direction: psi sums, phi sums, theta sums
    proj = 4 * no * kmu + 8 * (mmax + 1) * kphi * kphi * kmu + 4 * (mmax + 1) * np_
    oz = 0  # per point: two rotations and the product over the terms
    for m in range(mmax + 1):
        oz += 2 * (m // mrso + 1) * (2 * m + 1) ** 2 * 4
        for chi in range(-m, m + 1):
            oz += 8 * (m // mrso + 1) * sum(2 * (k // mrso) + 1 for k in range(abs(chi), mmax + 1))
    flops = N * (2 * proj + oz + 2 * np_ * 5 * math.log2(max(2, N)))
    if c["kind"] == "energy":
        return dict(bytes=2 * O * e * c["batch"], flops=flops * c["batch"])
    if c["kind"] == "chain":
        # the calls' own arrays: drho, p, vexc are the caller's
        P = N * np_ * 2 * e
        return dict(bytes=7 * O * e + 4 * P, flops=flops)
    pairs = 3 * c["sites"]
    vext = dict(bytes=16 * O, flops=O * pairs * 20)
    if c["kind"] == "vext":
        return vext
    # a solve from the V_ext start point takes about 14 evaluations, each
    # with the iterate, V, the gradient and one pair read, x and a pair written
    per = dict(bytes=(2 * e + 6 * 8) * O, flops=flops + 40 * O)
    nsol = c.get("batch", 1)
    return dict(bytes=nsol * (vext["bytes"] + 14 * per["bytes"]), flops=nsol * (vext["flops"] + 14 * per["flops"]))


# ---------------------------------------------------------------------------
# The same results in 64 bits, by the formulas of the path in plain torch.
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _small_d(l, a, b, ch, sh):
    """Wigner's d^l_{ab} from cos(theta/2) and sin(theta/2) (explicit sum)."""
    f = math.factorial
    acc = torch.zeros_like(ch)
    for s in range(max(0, a - b), min(l + a, l - b) + 1):
        w = (-1.0) ** s / (f(l + a - s) * f(l - b - s) * f(s) * f(s - a + b))
        acc = acc + w * ch ** (2 * l + a - b - 2 * s) * sh ** (2 * s - a + b)
    return math.sqrt(f(l + a) * f(l - a) * f(l + b) * f(l - b)) * acc


def _projections(mmax, mrso):
    return [(m, mup, k) for m in range(mmax + 1) for mup in range(-m, m + 1) for k in range(m // mrso + 1)]


def _angular(mmax, mrso, dev):
    """Quadrature weights (no,) and the two dense maps (2 np, no): projections
    of a field, and a field from projections (rows: real, imaginary part)."""
    x, w = np.polynomial.legendre.leggauss(mmax + 1)
    th = torch.tensor(np.arccos(x[::-1].copy()), dtype=torch.float64)
    wt = torch.tensor(w[::-1].copy() / 2, dtype=torch.float64)
    nphi, npsi = 2 * mmax + 1, 2 * (mmax // mrso) + 1
    j = torch.arange(nphi, dtype=torch.float64)[:, None]
    k = torch.arange(npsi, dtype=torch.float64)[None, :]
    wq = (wt[:, None, None] * torch.ones(nphi, npsi, dtype=torch.float64)) * (8 * math.pi**2 / (nphi * npsi * mrso))
    fwd, bwd = [], []
    for m, mup, mu2 in _projections(mmax, mrso):
        d = _small_d(m, mup, mu2 * mrso, torch.cos(th / 2), torch.sin(th / 2)) * math.sqrt(2 * m + 1)
        a = 2 * math.pi * (mup * j / nphi + mu2 * k / npsi)
        for t in (torch.cos(a), torch.sin(a)):
            fwd.append(((wt * d)[:, None, None] * t / (nphi * npsi)).reshape(-1))
            bwd.append((d[:, None, None] * t * (1.0 if mu2 == 0 else 2.0)).reshape(-1))
    return wq.reshape(-1).to(dev), torch.stack(fwd).to(dev), torch.stack(bwd).to(dev)


def _k(n, L):
    return np.array([(i if i <= n // 2 else i - n) for i in range(n)]) * (2 * math.pi / L)


def _convolve(p, c, eps):
    """FFT, rotation to the q frame, OZ product with c(q), back, inverse FFT of
    p (np, nx, ny, nz) complex."""
    dev = p.device
    n, L = _grid(c)
    mmax, mrso = c["mmax"], c["mrso"]
    N = n[0] * n[1] * n[2]
    tab = _table(c)
    h = mmax // mrso
    proj = _projections(mmax, mrso)
    ip = {t: i for i, t in enumerate(proj)}
    row = {(int(a), int(b), int(u) // mrso, int(v) // mrso, int(x)): i for i, (a, b, u, v, x) in enumerate(tab.tuples)}
    cq = torch.tensor(tab.c, dtype=torch.complex128, device=dev)
    pq = torch.fft.fftn(p, dim=(1, 2, 3)).reshape(len(proj), N)
    out = torch.zeros_like(pq)
    # the designated member of each (q, -q)
    ii = np.meshgrid(*(np.arange(v) for v in n), indexing="ij")
    mm = [np.where(a == 0, 0, v - a) for a, v in zip(ii, n)]
    inplane = mm[2] == ii[2]
    first = (ii[1] < mm[1]) | ((ii[1] == mm[1]) & (ii[0] <= mm[0]))
    des = (ii[2] <= n[2] // 2) & (~inplane | first)
    own = (mm[0] == ii[0]) & (mm[1] == ii[1]) & (mm[2] == ii[2])
    sing = own & ((ii[0] == n[0] // 2) | (ii[1] == n[1] // 2) | (ii[2] == n[2] // 2))
    lin = lambda a: ((a[0] * n[1] + a[1]) * n[2] + a[2])[des]  # noqa: E731
    to = lambda a, t: torch.tensor(a, dtype=t, device=dev)  # noqa: E731
    at, am, sg = to(lin(ii), torch.long), to(lin(mm), torch.long), to(sing[des], torch.bool)
    q = [to(_k(v, l)[a[des]], torch.float64) for v, l, a in zip(n, L, ii)]
    for i0 in range(0, at.numel(), 1 << 15):
        sl = slice(i0, i0 + (1 << 15))
        a, b, qx, qy, qz = at[sl], am[sl], q[0][sl], q[1][sl], q[2][sl]
        qn, qt = torch.sqrt(qx * qx + qy * qy + qz * qz), torch.sqrt(qx * qx + qy * qy)
        half = torch.atan2(qt, qz) / 2  # theta_q / 2 (0 at q = 0)
        ch, sh = torch.cos(half), torch.sin(half)
        phi = torch.where(qt > 0, torch.atan2(qy, qx), torch.zeros_like(qt))
        R = {}
        for m in range(mmax + 1):
            d = torch.stack([torch.stack([_small_d(m, u, x, ch, sh) for x in range(-m, m + 1)], 1)
                             for u in range(-m, m + 1)], 1)
            u = torch.arange(-m, m + 1, device=dev, dtype=torch.float64)
            R[m] = torch.polar(torch.ones_like(phi)[:, None] * torch.ones_like(u), -phi[:, None] * u)[:, :, None] * d
        gq, gm = pq[:, a].T, pq[:, b].T
        dq, dm = {}, {}
        for m in range(mmax + 1):
            for k in range(m // mrso + 1):
                src = [ip[(m, u, k)] for u in range(-m, m + 1)]
                vq = (gq[:, src].unsqueeze(2) * R[m]).sum(1)
                vm = (gm[:, src].unsqueeze(2) * R[m].flip(2)).sum(1) * (-1) ** m
                for x in range(-m, m + 1):
                    dq[(m, x, k)], dm[(m, x, k)] = vq[:, x + m], vm[:, x + m]
        eff = qn / tab.dq
        iq = torch.clamp(eff.long(), max=tab.nq - 2)
        al = (eff - iq)[:, None]
        sq, sm = {}, {}
        for x in range(-mmax, mmax + 1):
            ins = [(k, v) for k in range(abs(x), mmax + 1) for v in range(-(k // mrso), k // mrso + 1)]
            xq = torch.stack([dq[(k, x, -v)] if v < 0 else dm[(k, x, v)].conj() for k, v in ins], 1)
            xm = torch.stack([dm[(k, x, -v)] if v < 0 else dq[(k, x, v)].conj() for k, v in ins], 1)
            sign = torch.tensor([(-1.0) ** (x + v * mrso) if v < 0 else (-1.0) ** k for k, v in ins],
                                dtype=torch.float64, device=dev)
            for m in range(abs(x), mmax + 1):
                for k in range(m // mrso + 1):
                    r = cq[[row[(m, j, k, v, x)] for j, v in ins]]
                    cc = (r[:, iq].T * (1 - al) + r[:, iq + 1].T * al) * sign
                    for dst, v in ((sq, xq), (sm, xm)):
                        t = torch.view_as_real((cc * v).sum(1))
                        dst[(m, x, k)] = torch.view_as_complex(torch.where(t.abs() < eps, torch.zeros_like(t), t))
        for m in range(mmax + 1):
            for k in range(m // mrso + 1):
                vq = torch.stack([sq[(m, x, k)] for x in range(-m, m + 1)], 1)
                vm = torch.stack([sm[(m, x, k)] for x in range(-m, m + 1)], 1)
                oq = (R[m].conj() * vq[:, None, :]).sum(2)
                om = (R[m].flip(2).conj() * vm[:, None, :]).sum(2) * (-1) ** m
                om = torch.where(sg[sl][:, None], om.conj(), om)
                dst = [ip[(m, u, k)] for u in range(-m, m + 1)]
                for j, i in enumerate(dst):
                    out[i, a] = oq[:, j]
                    out[i, b] = om[:, j]
    return torch.fft.ifftn(out.reshape(p.shape), dim=(1, 2, 3), norm="forward")


def _evaluate(xi, c):
    """(ff, df, vexc, p) of one field xi (N, no) in 64 bits."""
    n, _ = _grid(c)
    rho0, pref = _solvent(c)
    x = xi.double().reshape(n[0] * n[1] * n[2], -1)
    w, fwd, bwd = _angular(c["mmax"], c["mrso"], x.device)
    np_ = fwd.shape[0] // 2
    f = fwd @ (rho0 * (x * x - 1)).T
    p = torch.complex(f[0::2], f[1::2]).reshape(np_, *n)
    del f
    p = _convolve(p, c, 2.0**-23 if c["form"] == "fp32" else 2.0**-52)
    r = p.reshape(np_, -1)
    vexc = r.real.T @ bwd[0::2] + r.imag.T @ bwd[1::2]
    ff = float((vexc * w * (x * x - 1)).sum() * rho0 * pref)
    return ff, 2 * rho0 * x * vexc, vexc, p


def _exact_vext(c, sol):
    dev = _dev()
    n, L = _grid(c)
    kT = M.kT(TEMP)
    mmax, mrso = c["mmax"], c["mrso"]
    x, _ = np.polynomial.legendre.leggauss(mmax + 1)
    nphi, npsi = 2 * mmax + 1, 2 * (mmax // mrso) + 1
    th, ph, ps = np.meshgrid(np.arccos(x[::-1]), 2 * np.pi * np.arange(nphi) / nphi,
                             2 * np.pi * np.arange(npsi) / (npsi * mrso), indexing="ij")
    ct, st, cp, sp, cs, ss = (f(a).reshape(-1) for a in (th, ph, ps) for f in (np.cos, np.sin))
    rot = np.stack([ct * cp * cs - sp * ss, -ct * cp * ss - sp * cs, st * cp, ct * sp * cs + cp * ss,
                    -ct * sp * ss + cp * cs, st * sp, -st * cs, st * ss, ct], 1).reshape(-1, 3, 3)
    grid = torch.stack(torch.meshgrid(*(torch.arange(v, dtype=torch.float64, device=dev) * (l / v)
                                        for v, l in zip(n, L)), indexing="ij"), -1).reshape(-1, 1, 3)
    e, na, e0 = 1.602176565e-19, 6.02214129e23, 8.854187817e-12
    qfact = e * e * 1e-3 * na / (4 * math.pi * e0 * 1e-10)
    V = torch.zeros((grid.shape[0], rot.shape[0]), dtype=torch.float64, device=dev)
    for sv in WATER:
        off = torch.tensor(rot @ sv[3:], device=dev)[None]
        for so in sol:
            d2 = torch.zeros_like(V)
            for k in range(3):
                dx = grid[:, :, k] + off[:, :, k] - so[3 + k]
                dx = dx - L[k] * torch.round(dx / L[k])
                d2 += dx * dx
            inv = torch.clamp(d2, min=1e-12).rsqrt_()
            if sv[1] > 0 and so[1] > 0:
                s6 = (0.5 * (sv[1] + so[1]) * inv) ** 6
                V += 4 * math.sqrt(sv[2] * so[2]) * (s6 * s6 - s6)
            V += qfact * sv[0] * so[0] * inv
    V = torch.clamp(V, max=VMAX_KT * kT)
    return dict(V=V, xi=torch.exp(-0.5 * torch.clamp(V / kT, min=-600.0)))


def exact(c, seed):
    if c["kind"] in ("solve", "serve"):
        return None  # a minimisation in plain torch takes minutes
    if c["kind"] == "vext":
        return _exact_vext(c, _solute(c, seed))
    xi = prepare(c, seed)["xi"]
    if c["kind"] == "chain":
        ff, df, vexc, p = _evaluate(xi, c)
        return dict(ff=ff, df=df.reshape(xi.shape), vexc=vexc.reshape(xi.shape), p=p)
    got = [_evaluate(x, c)[:2] for x in xi]
    ff = [f for f, _ in got]
    return dict(ff=ff[0] if c["batch"] == 1 else ff, df=torch.stack([d for _, d in got]).reshape(xi.shape))
