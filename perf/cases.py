"""The work a user of qed3_amd has it do, as cases that can be timed: operator applications,
solves, the batched solve, the molecular-dynamics pieces, a trajectory, training steps and the
overlap operator, from lattices of a few thousand points, where a call is a handful of short
launches, to the n=128, Lt=64 lattices the framework is quoted on.

listed() and draw() give cases, prepare() what a program holds before the call (context with
its gauge field, autotuned as the documented adapter does, sources and output buffers on the
device), run() one call, work() the traffic and arithmetic it cannot do without, and exact()
the same outputs in 64 bits by plain torch on the lattice's tables.

Gauge angles are von Mises (kappa = 1.4), sources complex Gaussian: the distributions of the
framework's own benchmark.  at = <ell>/2, r = 1, antiperiodic in time, as there.
"""
import ctypes
import math

import numpy as np
import torch

import qed3_amd as q

TOL = 1e-10  # true residual of every solve
DELTA = 0.001  # reliable-update threshold of the learned method
OPS = {"D": q.OP_D, "Ddag": q.OP_DDAG, "DdagD": q.OP_DDAGD, "DDdag": q.OP_DDDAG}
PRECS = {"f64": (q.F64, torch.complex128), "f32": (q.F32, torch.complex64), "f16": (q.F16, torch.float16)}
SOLVERS = {"f64": q.CG_F64, "mixed": q.CG_MIXED, "half": q.CG_HALF}


def listed():
    return [
        # one D^dag D on a test-sized lattice: launches and the wait are all there is
        {"name": "apply_small", "kind": "apply", "lattice": 0, "n": 8, "Lt": 8, "m": 0.1, "op": "DdagD", "prec": "f64"},
        # D^dag D of the full-size dual lattice, the operator every FP64 residual goes through
        {"name": "apply_large", "kind": "apply", "lattice": 1, "n": 128, "Lt": 64, "m": 0.02, "op": "DdagD",
         "prec": "f64"},
        # the plain FP64 solve at the sizes where a program checks itself
        {"name": "cg_f64_small", "kind": "solve", "lattice": 1, "n": 16, "Lt": 16, "m": 0.1, "solver": "f64"},
        # the half-storage solve, sizes off every power of two
        {"name": "cg_half_odd", "kind": "solve", "lattice": 0, "n": 77, "Lt": 45, "m": 0.05, "solver": "half"},
        # the headline: learned solve, n=128, Lt=64, near-critical
        {"name": "learned_large", "kind": "solve", "lattice": 1, "n": 128, "Lt": 64, "m": 0.02, "solver": "learned"},
        # the solve inside the full HMC run (simplicial n=64, Lt=32, m=0.1)
        {"name": "learned_hmc", "kind": "solve", "lattice": 0, "n": 64, "Lt": 32, "m": 0.1, "solver": "learned"},
        # right-hand sides of uneven lattices in one call (pseudofermions, masses, refinements)
        {"name": "batch_uneven", "kind": "batch", "m": 0.06,
         "systems": "0:32:16 1:32:16 0:48:32 1:24:32 0:64:16 1:40:20 0:21:64 1:17:33"},
        # the molecular-dynamics step's fermion work besides the solve: new links, then the force
        {"name": "update_force", "kind": "force", "lattice": 0, "n": 64, "Lt": 32, "m": 0.1},
        # a short trajectory of the full HMC (compact action, learned solver)
        {"name": "hmc_short", "kind": "hmc", "lattice": 0, "n": 16, "Lt": 16, "m": 0.1, "nsteps": 4, "inner": 25,
         "tau": 0.2},
        # one training step of the learned preconditioner: loss and gradient of a batch
        {"name": "train_learned", "kind": "train", "net": "horner", "lattice": 1, "n": 32, "Lt": 32, "m": 0.02,
         "layers": 4, "batch": 2},
        # one training step of the 16-channel message-passing network (matrix-core layers)
        {"name": "train_channels", "kind": "train", "net": "channels", "lattice": 1, "n": 16, "Lt": 16, "m": 0.02,
         "layers": 4, "batch": 4},
        # the overlap operator (one multi-shift solve) at the overlap benchmark's size
        {"name": "overlap_apply", "kind": "overlap", "lattice": 0, "n": 16, "Lt": 16, "m": -0.5, "degree": 21,
         "op": "D"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["apply"] * 3 + ["solve"] * 4 + ["batch", "force", "hmc", "train", "train", "overlap"])
    c = {"kind": kind, "lattice": rng.randrange(2), "m": round(rng.uniform(0.02, 0.2), 4)}
    if kind == "apply":
        c |= {"n": _log_int(rng, 6, 120), "Lt": _log_int(rng, 6, 64), "op": rng.choice(sorted(OPS)),
              "prec": rng.choice(sorted(PRECS))}
    elif kind == "solve":
        c |= {"n": _log_int(rng, 10, 120), "Lt": _log_int(rng, 8, 64),
              "solver": rng.choice(["f64", "mixed", "half", "learned", "learned"])}
    elif kind == "batch":
        c.pop("lattice")
        c["systems"] = " ".join("%d:%d:%d" % (rng.randrange(2), _log_int(rng, 12, 56), _log_int(rng, 8, 48))
                                for _ in range(rng.randint(3, 10)))
    elif kind == "force":
        c |= {"n": _log_int(rng, 8, 100), "Lt": _log_int(rng, 8, 64)}
    elif kind == "hmc":
        c |= {"n": rng.randint(6, 18), "Lt": rng.randint(8, 20), "nsteps": rng.randint(2, 5),
              "inner": rng.randint(10, 30), "tau": 0.15}
    elif kind == "train":
        c |= {"net": rng.choice(["horner", "channels"]), "layers": rng.randint(2, 5), "batch": rng.randint(1, 4)}
        top = 40 if c["net"] == "horner" else 16
        c |= {"n": _log_int(rng, 6, top), "Lt": _log_int(rng, 8, 32 if c["net"] == "horner" else 16)}
    else:
        c |= {"n": rng.randint(8, 20), "Lt": rng.randint(8, 20), "m": -0.5, "degree": 21,
              "op": rng.choice(["D", "Ddag"])}
    return c


# ---- inputs -------------------------------------------------------------------------------
class _Buf:
    """A torch tensor's device memory under the name the framework's calls take (.ptr)."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


_geo = {}   # refinement -> lattice tables: the same for every gauge field
_tile = {}  # (lattice, n, Lt) -> autotuned launch shapes, tuned once per shape in a program


def _tables(n):
    if n not in _geo:
        _geo[n] = q.Geometry(n)
    return _geo[n]


def _links(g, lattice):
    """sites, links, alpha (both ends), omega and the crossing sites of each link"""
    if lattice == q.SIMPLICIAL:
        return g.sites, g.links, g.alpha, g.omega, g.dual_sites, g.dual_links
    return g.dual_sites, g.dual_links, g.dual_alpha, g.dual_omega, g.sites, g.links


def _lengths(g, lattice):
    s, l = _links(g, lattice)[:2]
    x, y = s[l[:, 0]], s[l[:, 1]]
    return np.arctan2(np.linalg.norm(np.cross(x, y), axis=1), np.einsum("ij,ij->i", x, y))


def _von_mises(shape, gen, kappa=1.4):
    """Best and Fisher's rejection, every entry redrawn until it is accepted."""
    tau = 1 + math.sqrt(1 + 4 * kappa * kappa)
    rho = (tau - math.sqrt(2 * tau)) / (2 * kappa)
    r = (1 + rho * rho) / (2 * rho)
    out = torch.zeros(shape, dtype=torch.float64, device="cuda")
    todo = torch.ones(shape, dtype=torch.bool, device="cuda")
    rand = lambda: torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    for _ in range(24):
        z = torch.cos(math.pi * rand())
        f = (1 + r * z) / (r + z)
        c = kappa * (r - f)
        u = rand()
        ok = todo & ((c * (2 - c) > u) | (torch.log(c / u) + 1 >= c))
        ang = torch.acos(f.clamp(-1, 1))
        out = torch.where(ok, torch.where(rand() < 0.5, ang, -ang), out)
        todo &= ~ok
    return out


def _gauss(shape, gen, dtype=torch.complex128):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)  # unit variance, as the sources'


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return gen


def _at(g, lattice):
    return 0.5 * float(np.mean(_lengths(g, lattice)))


def _set_gauge(D, sp, tp):
    q.check(q.load().qed3_set_gauge(D._h, ctypes.c_void_p(sp.data_ptr()), ctypes.c_void_p(tp.data_ptr()), 1))


def _context(lattice, n, Lt, m, gen, tune=True):
    g = _tables(n)
    V, E, _ = q.lattice_sizes(lattice, n)
    sp, tp = _von_mises((Lt, E), gen), _von_mises((Lt, V), gen)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=m, at=_at(g, lattice), geometry=g)
    torch.cuda.synchronize()
    _set_gauge(D, sp, tp)
    key = (lattice, n, Lt)
    if tune and key not in _tile:
        D.autotune()
        _tile[key] = {(op, prec): D.tile(op, prec) for op in (q.OP_D, q.OP_DDAG) for prec in (q.F64, q.F32)}
    elif tune:
        for (op, prec), t in _tile[key].items():
            D.set_tile(t["block"], t["ts"], t["remap"], t["lds"], ops=(op,), precs=(prec,))
    return D, sp, tp


def _systems(case):
    return [tuple(int(v) for v in s.split(":")) for s in case["systems"].split()]


def _seeded(case, seed):
    """The inputs of a case from its seed alone: everything prepare() and exact() share."""
    gen = _generator(seed)
    k = case["kind"]
    if k == "batch":
        out = []
        for i, (lat, n, Lt) in enumerate(_systems(case)):
            D, sp, tp = _context(lat, n, Lt, round(case["m"] * (1 + 0.1 * i), 4), gen)
            out.append((D, sp, tp, _gauss((D.N,), gen)))
        return out
    if k == "hmc":
        V, E, _ = q.lattice_sizes(case["lattice"], case["n"])
        return [0.1 * torch.randn((case["Lt"], w), dtype=torch.float64, device="cuda", generator=gen) for w in (E, V)]
    D, sp, tp = _context(case["lattice"], case["n"], case["Lt"], case["m"], gen, tune=k != "train")
    if k == "apply":
        dt = PRECS[case["prec"]][1]
        src = _gauss((D.N,), gen, torch.complex64 if dt == torch.float16 else dt)
        return D, sp, tp, torch.view_as_real(src).to(dt).reshape(-1) if dt == torch.float16 else src
    if k == "train":
        e = _gauss((case["batch"], D.N), gen)
        v = torch.empty_like(e)
        torch.cuda.synchronize()
        for b in range(case["batch"]):  # (D e, e): what the solver's own errors give
            D.apply_device(q.OP_D, q.F64, _Buf(v[b]), _Buf(e[b]))
        if case["net"] == "channels":
            return D, sp, tp, v.to(torch.complex64), e.to(torch.complex64)
        return D, sp, tp, v, e
    return D, sp, tp, _gauss((D.N,), gen)


def prepare(case, seed):
    k = case["kind"]
    made = _seeded(case, seed)
    s = {"kind": k, "case": case}
    if k == "batch":
        s["D"] = [m[0] for m in made]
        s["b"] = [_Buf(m[3]) for m in made]
        s["x"] = [_Buf(torch.zeros_like(m[3])) for m in made]
    elif k == "hmc":
        g = _tables(case["n"])
        D = q.WilsonDirac(case["lattice"], case["n"], case["Lt"], r=1.0, M5=case["m"], at=_at(g, case["lattice"]),
                          geometry=g)
        s["u"], s["t"] = (np.ascontiguousarray(a.cpu().numpy()) for a in made)
        D.update(s["u"], s["t"])
        s["D"] = D
        s["hmc"] = q.HMC(D, 1.0 / 1.4, compact=True, npf=1, tau=case["tau"], nsteps=case["nsteps"],
                         nsteps_inner=case["inner"], tol=TOL, solver=q.PCG, seed=int(seed) % 1000003)
    elif k == "train":
        D, _, _, v, e = made
        s |= {"D": D, "v": _Buf(v), "e": _Buf(e)}
        if case["net"] == "horner":
            s["net"] = q.Precond(D, case["layers"])
            p = s["net"].params  # a state in the middle of training
            p = p * (1 + 0.02 * np.random.default_rng(seed).standard_normal(p.size))
            s["net"].params = p
        else:
            s["net"] = q.Net(D, max(case["layers"], 2), seed=1 + int(seed) % 1000003)
    else:
        D, sp, tp, b = made
        s |= {"D": D, "b": _Buf(b), "x": _Buf(torch.zeros_like(b))}
        if k == "solve" and case["solver"] == "learned":
            s["net"] = q.Precond(D, 4)
        if k == "force":
            s |= {"sp": sp, "tp": tp, "fs": _Buf(torch.zeros_like(sp)), "ft": _Buf(torch.zeros_like(tp))}
        if k == "overlap":
            s["ov"] = q.Overlap(D, case["degree"])
    torch.cuda.synchronize()
    return s


def run(s):
    k, c = s["kind"], s["case"]
    if k == "apply":
        s["D"].apply_device(OPS[c["op"]], PRECS[c["prec"]][0], s["x"], s["b"])
        return s["x"].t
    if k == "solve":
        if c["solver"] == "learned":
            s["net"].solve_device(s["x"], s["b"], tol=TOL, delta=DELTA)
        else:
            s["D"].solve_device(s["x"], s["b"], tol=TOL, solver=SOLVERS[c["solver"]])
        return s["x"].t
    if k == "batch":
        q.batch_solve(s["D"], s["x"], s["b"], tol=TOL)
        return [x.t for x in s["x"]]
    if k == "force":
        _set_gauge(s["D"], s["sp"], s["tp"])
        q.check(q.load().qed3_pf_force(s["D"]._h, s["b"].ptr, s["fs"].ptr, s["ft"].ptr))
        return s["fs"].t, s["ft"].t
    if k == "hmc":  # the chain goes on from where the last pass left it
        s["hmc"].trajectory(s["u"], s["t"], no_reject=True)
        return s["u"], s["t"]
    if k == "train":
        if c["net"] == "horner":
            return s["net"].loss_grad_device(s["v"], s["e"], c["batch"])
        loss, g = ctypes.c_double(), np.zeros(s["net"].nparams, np.complex128)
        q.check(q.load().qed3_net_loss_grad(s["net"]._h, s["v"].ptr, s["e"].ptr, c["batch"], ctypes.byref(loss),
                                            g.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        return loss.value, g
    q.check(q.load().qed3_overlap_apply(s["ov"]._h, OPS[c["op"]], s["x"].ptr, s["b"].ptr))
    return s["x"].t


# ---- work ---------------------------------------------------------------------------------
def _vec_links(lattice, n, Lt, real):
    V, E, _ = q.lattice_sizes(lattice, n)
    return 4 * V * Lt * real, (V + E) * Lt * real, V * Lt, 2 * E / V


def work(case):
    """Inputs read once, outputs written once.  A D costs about 48 flop per spatial hop and 36
    per point for the time hops and the diagonal; the iteration counts of solves are not part
    of the case, so one D^dag D (the residual) is all that is counted for them."""
    k = case["kind"]
    if k == "batch":
        parts = [_vec_links(*s, 8) for s in _systems(case)]
        return {"bytes": sum(2 * v + l for v, l, _, _ in parts), "flops": sum(2 * p * (48 * d + 36) for _, _, p, d in parts)}
    real = {"f64": 8, "f32": 4, "f16": 2}[case["prec"]] if k == "apply" else 8
    vec, links, pts, deg = _vec_links(case["lattice"], case["n"], case["Lt"], real)
    flops = pts * (48 * deg + 36)
    if k == "apply":
        return {"bytes": 2 * vec + links, "flops": flops * (2 if len(case["op"]) > 4 else 1)}
    if k == "force":
        return {"bytes": vec + 2 * links, "flops": 2 * flops + pts * deg * 60}
    if k == "hmc":  # links and momenta in and out, one force per gauge step
        steps = case["nsteps"] * case["inner"]
        return {"bytes": 4 * links, "flops": steps * pts * deg * 20 + case["nsteps"] * 2 * flops}
    if k == "train":
        per = flops if case["net"] == "horner" else pts * 2 * 2 * 32 * 160
        return {"bytes": case["batch"] * 2 * vec // (2 if case["net"] == "channels" else 1) + links,
                "flops": 3 * case["layers"] * case["batch"] * per}
    return {"bytes": 2 * vec + links, "flops": 2 * flops}


# ---- the same outputs in 64 bits ------------------------------------------------------------
def _tri_area(a, b, c):
    """spherical triangle (Van Oosterom and Strackee)"""
    num = np.abs(np.einsum("ij,ij->i", a, np.cross(b, c)))
    dot = lambda x, y: np.einsum("ij,ij->i", x, y)  # noqa: E731
    return 2 * np.arctan2(num, 1 + dot(a, b) + dot(b, c) + dot(c, a))


class _Exact:
    """The Wilson-Dirac operator (r = 1, antiperiodic) on psi[..., Lt, V, 2] in complex128,
    a gather over each site's links."""

    def __init__(self, lattice, n, Lt, m, sp, tp):
        g = _tables(n)
        S, L, al, om, T, TL = _links(g, lattice)
        ell = _lengths(g, lattice)
        i, j = L[:, 0], L[:, 1]
        lv = _tri_area(S[i], S[j], T[TL[:, 0]]) + _tri_area(S[i], S[j], T[TL[:, 1]])
        kap = 2 * lv / ell / ell.mean()
        V, E = len(S), len(L)
        # area of the cell dual to a site: half of each adjacent link's two triangles
        area = np.zeros(V)
        if lattice == q.SIMPLICIAL:
            for k in (0, 1):
                t = T[TL]
                a = 0.5 * (_tri_area(S[L[:, k]], t[:, 0], t[:, 1]))
                np.add.at(area, L[:, k], 2 * a)
        else:
            f = g.faces
            area = _tri_area(g.sites[f[:, 0]], g.sites[f[:, 1]], g.sites[f[:, 2]])
        kt = area / ell.mean() / _at(g, lattice)
        diag = kt + m
        M = 6 if lattice == q.SIMPLICIAL else 3
        nbr = np.tile(np.arange(V)[:, None], (1, M))
        lnk, sgn = np.zeros((V, M), int), np.ones((V, M))
        H = np.zeros((V, M, 2, 2), complex)
        order = np.argsort(np.concatenate([i, j]), kind="stable")
        site = np.concatenate([i, j])[order]
        slot = np.arange(2 * E) - np.searchsorted(site, site)
        l = np.concatenate([np.arange(E)] * 2)[order]
        rev = order >= E
        nbr[site, slot] = np.concatenate([j, i])[order]
        lnk[site, slot] = l
        sgn[site, slot] = np.where(rev, -1.0, 1.0)
        w = np.where(rev, -om[l], om[l])
        a = np.where(rev, al[l, 1], al[l, 0])
        # H_xy = kappa/2 (-1 + gamma(alpha)) e^{i omega sigma3 / 2}
        up, dn = 0.5 * kap[l] * np.exp(-0.5j * w), 0.5 * kap[l] * np.exp(0.5j * w)
        H[site, slot, 0, 0], H[site, slot, 1, 1] = -up, -dn
        H[site, slot, 0, 1], H[site, slot, 1, 0] = np.exp(-1j * a) * dn, np.exp(1j * a) * up
        np.add.at(diag, i, 0.5 * kap)
        np.add.at(diag, j, 0.5 * kap)
        # the slot of x at y, for the adjoint: H_yx^dagger
        back = np.zeros((2 * E, 2), int)
        back[l + E * rev] = np.stack([site, slot], 1)
        mate = back[l + E * ~rev]
        Hd = np.zeros_like(H)
        Hd[site, slot] = np.conj(np.swapaxes(H[mate[:, 0], mate[:, 1]], -1, -2))
        cu = lambda v: torch.as_tensor(v, device="cuda")  # noqa: E731
        self.nbr, self.lnk, self.sgn, self.H, self.Hd = cu(nbr), cu(lnk), cu(sgn), cu(H), cu(Hd)
        self.alpha = cu(np.where(sgn > 0, al[lnk, 0], al[lnk, 1]))
        self.alpha_nb = cu(np.where(sgn > 0, al[lnk, 1], al[lnk, 0]))
        live = np.zeros((V, M))
        live[site, slot] = 1
        self.live, self.omega = cu(live), cu(sgn * om[lnk])
        self.kappa = cu(kap[lnk] * live)
        self.diag, self.kt, self.M, self.Lt, self.V = cu(diag), cu(kt), M, Lt, V
        self.sp, self.tp = sp, tp

    def phase(self, k, sp=None):
        """e^{i theta} of slot k as its site sees it, [Lt, V, 1]"""
        sp = self.sp if sp is None else sp
        ang = sp[:, self.lnk[:, k]] * self.sgn[:, k]
        return torch.polar(torch.ones_like(ang), ang)[..., None]

    def spatial(self, v, H, sp=None):
        out = 0
        for k in range(self.M):
            p = v[..., self.nbr[:, k], :] * self.phase(k, sp)
            out = out + (H[:, k] * p[..., None, :]).sum(-1)
        return out

    def time(self, v, tp=None):
        """(e^{-i theta^t_{s-1}} v(s-1), e^{i theta^t_s} v(s+1)) with the sign of the wrap"""
        tp = self.tp if tp is None else tp
        u = torch.polar(torch.ones_like(tp), tp)[..., None].clone()
        sgn = torch.ones(self.Lt, 1, 1, dtype=torch.float64, device="cuda")
        sgn[-1] = -1
        u = u * sgn
        return torch.roll(u.conj() * v, 1, dims=-3), u * torch.roll(v, -1, dims=-3)

    def apply(self, v, dag=False, sp=None, tp=None):
        v = v.reshape(v.shape[:-1] + (self.Lt, self.V, 2)) if v.shape[-1] != 2 or v.dim() < 3 else v
        out = self.diag[:, None] * v + self.spatial(v, self.Hd if dag else self.H, sp)
        back, fwd = self.time(v, tp)
        a = (fwd, back) if dag else (back, fwd)
        return out - self.kt[:, None] * torch.stack([a[0][..., 0], a[1][..., 1]], -1)

    def normal(self, v):
        return self.apply(self.apply(v), dag=True)

    def solve(self, b, tol=1e-13):
        b = b.reshape(self.Lt, self.V, 2)
        x, r = torch.zeros_like(b), b.clone()
        p, rr = r.clone(), float((r.abs() ** 2).sum())
        stop = tol * tol * rr
        for _ in range(20000):
            w = self.apply(p)
            al = rr / float((w.abs() ** 2).sum())
            x += al * p
            r -= al * self.apply(w, dag=True)
            new = float((r.abs() ** 2).sum())
            if new <= stop:
                break
            p = r + (new / rr) * p
            rr = new
        return x.reshape(-1)

    # the learned preconditioner: g <- T^{-1}(c_j v + S g)
    def horner(self, v, p, layers):
        c, A, B = p[:layers], p[layers:layers + 2], p[layers + 2:]
        scale = torch.stack([torch.stack([A[0], B[0]]), torch.stack([B[1], A[1]])])
        u = torch.polar(torch.ones_like(self.tp), self.tp)
        kt, ic = self.kt, 1 / self.diag
        g = None
        for j in range(layers - 1, -1, -1):
            y = c[j] * v
            if g is not None:
                y = y - self.spatial(g, self.H * scale)
                y0 = torch.cat([(y[:1, :, 0] - kt * u[-1].conj() * g[-1:, :, 0]), y[1:, :, 0]])
                y1 = torch.cat([y[:-1, :, 1], y[-1:, :, 1] - kt * u[-1] * g[:1, :, 1]])
            else:
                y0, y1 = y[..., 0], y[..., 1]
            f, b = [ic * y0[0]], [ic * y1[-1]]
            for s in range(1, self.Lt):
                f.append(ic * (y0[s] + kt * u[s - 1].conj() * f[-1]))
                b.append(ic * (y1[-1 - s] + kt * u[-1 - s] * b[-1]))
            g = torch.stack([torch.stack(f), torch.stack(b[::-1])], -1)
        return g

    # the 16-channel network: five feature maps of h[..., channel, Lt, V, 2]
    def maps(self, h):
        F1, F2 = torch.zeros_like(h), torch.zeros_like(h)
        for k in range(self.M):
            y = h[..., self.nbr[:, k], :]
            C, S = (0.5 * self.kappa[:, k] * t(0.5 * self.omega[:, k]) for t in (torch.cos, torch.sin))
            t0, t1 = torch.complex(C, -S)[:, None], torch.complex(C, S)[:, None]
            u = self.phase(k)
            e = torch.polar(torch.ones_like(C), self.alpha[:, k])[:, None]
            F1 = F1 + u * torch.cat([t0, t1], -1) * y
            F2 = F2 + u * torch.cat([e.conj() * t1, e * t0], -1) * y.flip(-1)
        back, fwd = self.time(h)
        kh = 0.5 * self.kt[:, None]
        return [h, F1, F2, kh * fwd, kh * back]

    def channels(self, r, p, layers, skip):
        """r[B, N]; p: v[2][5][16], W[layers-2][2][5][16][16], u[2][5][16]"""
        n = 160
        v, u = p[:n].reshape(2, 5, 16), p[-n:].reshape(2, 5, 16)
        r = r.reshape(-1, 1, self.Lt, self.V, 2)
        F = torch.stack(self.maps(r), 1)[:, :, 0]  # [B, 5, Lt, V, 2]
        h = torch.einsum("akc,bksxa->bcsxa", v, F)
        for l in range(layers - 2):
            W = p[n + l * 2560:n + (l + 1) * 2560].reshape(2, 5, 16, 16)
            h = torch.einsum("akcd,bkdsxa->bcsxa", W, torch.stack(self.maps(h), 1))
        return torch.einsum("akc,bkcsxa->bsxa", u, torch.stack(self.maps(h), 1)) + skip * r[:, 0]


def _sign(op, v, steps=260):
    """op = (apply, normal): X (X^dag X)^{-1/2} v by the Lanczos matrix function"""
    apply, normal = op
    V, al, be = [v / v.norm()], [], []
    for k in range(steps):
        w = normal(V[-1])
        al.append(float((V[-1].conj() * w).sum().real))
        for _ in range(2):  # full orthogonalisation, twice
            Q = torch.stack(V)
            w = w - torch.tensordot(torch.tensordot(Q.conj(), w, dims=w.dim()), Q, dims=1)
        be.append(float(w.norm()))
        V.append(w / be[-1])
    ev, Z = np.linalg.eigh(np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1))
    y = torch.as_tensor((Z * Z[0]) @ ev ** -0.5, device="cuda").to(v.dtype)
    return apply(torch.tensordot(y, torch.stack(V[:-1]), dims=1)) * v.norm()


def exact(case, seed):
    k = case["kind"]
    if k == "hmc":
        return None  # its momenta and noise come from the framework's own streams
    made = _seeded(case, seed)
    if k == "batch":
        return [_Exact(*s, round(case["m"] * (1 + 0.1 * i), 4), m[1], m[2]).solve(m[3])
                for i, (s, m) in enumerate(zip(_systems(case), made))]
    X = _Exact(case["lattice"], case["n"], case["Lt"], case["m"], made[1], made[2])
    shape = (X.Lt, X.V, 2)
    if k == "apply":
        b = made[3]
        b = torch.view_as_complex(b.double().reshape(-1, 2)) if case["prec"] == "f16" else b.to(torch.complex128)
        b = b.reshape(shape)
        for dag in {"D": [0], "Ddag": [1], "DdagD": [0, 1], "DDdag": [1, 0]}[case["op"]]:
            b = X.apply(b, dag=bool(dag))
        return torch.view_as_real(b).reshape(-1) if case["prec"] == "f16" else b.reshape(-1)
    if k == "solve":
        return X.solve(made[3])
    if k == "overlap":
        v = made[3].reshape(shape)
        if case["op"] == "D":
            return (v + _sign((X.apply, X.normal), v)).reshape(-1)
        dag = lambda w: X.apply(w, dag=True)  # noqa: E731
        return (v + _sign((dag, lambda w: X.apply(dag(w))), v)).reshape(-1)
    if k == "force":  # -2 d/dtheta Re <D eta, D(theta) eta> with the left factor fixed
        eta = made[3].reshape(shape)
        sp, tp = made[1].clone().requires_grad_(), made[2].clone().requires_grad_()
        w = X.apply(eta)
        S = (w.conj() * X.apply(eta, sp=sp, tp=tp)).real.sum()
        return tuple(-2 * f for f in torch.autograd.grad(S, (sp, tp)))
    D, v, e = made[0], made[3].to(torch.complex128), made[4].to(torch.complex128)
    if case["net"] == "horner":
        p = np.ones(case["layers"] + 4) * (1 + 0.02 * np.random.default_rng(seed).standard_normal(case["layers"] + 4))
        f = lambda b, p: X.horner(v[b].reshape(shape), p, case["layers"])  # noqa: E731
    else:
        net = q.Net(D, max(case["layers"], 2), seed=1 + int(seed) % 1000003)
        p, skip = net.params, net.skip
        f = lambda b, p: X.channels(v[b], p, net.layers, skip)[0]  # noqa: E731
    p = torch.as_tensor(p, device="cuda").to(torch.complex128).requires_grad_()
    loss = 0.0
    for b in range(case["batch"]):
        t = e[b].reshape(shape)
        part = ((f(b, p) - t).abs() ** 2).sum() / (t.abs() ** 2).sum() / case["batch"]
        part.backward()
        loss += float(part.detach())
    return loss, p.grad.cpu().numpy()
