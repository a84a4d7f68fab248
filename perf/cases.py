"""The work a user of this package has it do, as measurable cases.

A case is a dict of plain values; prepare() makes what a program holds before
the call (meshes and contexts kept in pools, as cfdl.serving keeps them, with
properties from the seed), run() is one pass through the public entry points
and returns whole fields, and exact() restates the pass in 64 bits with torch
(the plain reference algorithm and its colour orders; the multigrid-
preconditioned modes stop on a Krylov path that only the package defines).

Kinds:
  residual  calc_residual on arrays already in device memory;
  run       outer iterations of the SIMPLE loop from rest on one context, then
            the fields and the solver lines, as a batch job reads them;
  dropin    one solve_uvwp the way the Fortran drop-in modules make it: host
            state up, one outer iteration, state and work arrays back;
  batch     one engine step of the serving loop: ten outer iterations of
            several independent requests in the same grouped launches.
"""
import ctypes
import math
import os
import random
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cfd-lite_amd"))
import cfdl  # noqa: E402

FIELDS = ("u", "v", "w", "p")
# what the drop-in modules send and fetch around solve_uvwp
PUT_STATE = ("u", "v", "w", "p", "u0", "v0", "w0", "gu", "gv", "gw", "gp", "mip", "mip0")
GET_STATE = ("u", "v", "w", "p", "gu", "gv", "gw", "gp", "gpc", "mip", "bu", "bv", "bw", "d", "dc",
             "ap", "anb", "b", "phic")


def _run(name, nx, ny, nz, pc, gs, steps, ncoef=1, subd=4, steady=True, jitter=0.0, channel=False,
         energy=False, asm=64):
    return {"name": name, "kind": "run", "nx": nx, "ny": ny, "nz": nz, "pc": pc, "gs": gs,
            "steps": steps, "ncoef": ncoef, "subd": subd, "steady": steady, "jitter": jitter,
            "channel": channel, "energy": energy, "asm": asm}


def listed():
    return [
        # the stand-alone residual check of a caller that owns its arrays: one
        # short call, latency and launches
        {"name": "residual-24", "kind": "residual", "nx": 24, "ny": 24, "nz": 24, "alloc": True},
        # the smallest run: the reference's own loop (one pseudo-time step of
        # three outer iterations), where launches are everything
        _run("cavity16-reference", 16, 16, 16, "reference", "reference", 1, ncoef=3, steady=False),
        # the 32^3, Re 100 cavity of the convergence runs
        _run("cavity32-reference", 32, 32, 32, "reference", "reference", 6),
        # odd edges, distorted cells, two subdomains, the energy equation too
        _run("box61x47x53-energy", 61, 47, 53, "reference", "reference", 1, ncoef=3, subd=2,
             steady=False, jitter=0.15, energy=True),
        # a drop-in host with its state in pageable memory
        {"name": "dropin64-reference", "kind": "dropin", "nx": 64, "ny": 64, "nz": 64, "subd": 4},
        # the benchmark's own configuration, in the reference's order
        _run("cavity128-reference", 128, 128, 128, "reference", "reference", 6),
        # the same loop in colour order, FP64
        _run("cavity96-colored", 96, 96, 96, "colored", "colored", 10),
        # colour order with FP32 sweeps under FP64 defect correction
        _run("cavity128-mixed", 128, 128, 128, "mixed", "colored", 12),
        # multigrid-preconditioned conjugate gradients in FP64, uneven edges
        _run("box80x100x72-mgcg", 80, 100, 72, "mgcg", "colored", 10, subd=1, jitter=0.1),
        # the fastest way through the benchmark's mesh
        _run("cavity128-mgcg-mixed", 128, 128, 128, "mgcg-mixed", "colored", 16),
        # the distorted, renumbered channel
        _run("channel96-mgcg-mixed", 96, 96, 96, "mgcg-mixed", "colored", 12, subd=1, jitter=0.2,
             channel=True),
        # eight serving requests in flight
        {"name": "batch8-serving", "kind": "batch", "sizes": "16,24,32,40,48,64,80,96", "chunk": 10},
    ]


def _edge(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: edges 8 .. 128 spread over their
    logarithm (odd ones among them), every mode and option."""
    kind = rng.choice(["residual", "run", "run", "run", "run", "run", "run", "run", "dropin",
                       "batch"])
    if kind == "batch":
        n = rng.randint(2, 8)
        return {"kind": "batch", "chunk": 10,
                "sizes": ",".join(str(rng.choice(range(16, 81, 8))) for _ in range(n))}
    n = _edge(rng, 8, 112)
    ex = [max(6, min(128, int(round(n * rng.uniform(0.75, 1.3))))) for _ in range(3)]
    if kind == "residual":
        return {"kind": "residual", "nx": ex[0], "ny": ex[1], "nz": ex[2],
                "alloc": rng.random() < 0.5}
    if kind == "dropin":
        return {"kind": "dropin", "nx": ex[0], "ny": ex[1], "nz": ex[2],
                "subd": rng.choice([1, 2, 4])}
    pc = rng.choice(["reference", "reference", "colored", "mixed", "mgcg", "mgcg-mixed"])
    mg = pc.startswith("mgcg")
    ref = pc == "reference"
    steady = rng.random() < 0.6
    cells = ex[0] * ex[1] * ex[2]
    most = 6 if ref else 12
    total = rng.randint(1, max(1, min(most, int(most * 1.2e6 / cells) or 1)))
    ncoef = 1 if steady else min(3, total)
    c = _run("", *ex, pc, "reference" if ref else "colored", max(1, total // ncoef), ncoef,
             subd=1 if mg else rng.choice([2, 4]), steady=steady,
             jitter=rng.choice([0.0, 0.1, 0.2]), channel=mg and rng.random() < 0.4,
             energy=rng.random() < 0.2, asm=32 if mg and rng.random() < 0.5 else 64)
    del c["name"]
    return c


# ---- what a program keeps: one mesh per shape, contexts reused between cases
_meshes = {}
_idle = {}
IDLE_CELLS = 1 << 23


def _mesh(nx, ny, nz, jitter, renumber, subd):
    key = (nx, ny, nz, jitter, renumber, subd)
    if key not in _meshes:
        if len(_meshes) > 12:
            _meshes.clear()
        m = cfdl.Mesh.box(nx, ny, nz, jitter=jitter)
        if renumber:
            m.renumber(20261202)
        _meshes[key] = m.partition(subd)
    return _meshes[key]


class _Context:
    """One context out of the pool, given back when the state goes."""

    def __init__(self, nx, ny, nz, jitter, subd, channel, steady, pc, gs, asm):
        key = (nx, ny, nz, jitter, subd, channel, steady, pc, gs, asm)
        self.mesh = _mesh(nx, ny, nz, jitter, channel, subd)
        if _idle.get(key):
            self.eq = _idle[key].pop()
        else:
            make = cfdl.UVWP.channel if channel else cfdl.UVWP.cavity
            self.eq = make(self.mesh, rho=1.0, mu=0.01, dt=math.inf if steady else 0.01)
            if steady:
                self.eq.set_relaxation(0.7, 0.3)
            self.eq.set_gs_order(gs)
            self.eq.set_pc_order(pc)
            if asm == 32:
                self.eq.set_assembly_precision(32)
        weakref.finalize(self, _give_back, key, self.eq)


def _give_back(key, eq):
    """Back to the idle set; other shapes' contexts, oldest first, make room."""
    _idle.setdefault(key, []).append(eq)
    held = sum(e.sizes["ap"] for l in _idle.values() for e in l)
    for k in list(_idle):
        while held > IDLE_CELLS and k != key and _idle[k]:
            e = _idle[k].pop()
            held -= e.sizes["ap"]
            e.close()


def _reynolds(seed):
    return math.exp(random.Random(seed).uniform(math.log(100.0), math.log(400.0)))


def _properties(eq, seed):
    """Uniform density and viscosity of the seed's Reynolds number."""
    ne = eq.sizes["ap"]
    eq.set_properties(np.ones(ne), np.full(ne, 1.0 / _reynolds(seed)))


def _lines(eq):
    """The solver lines: iterations, and initial / final / largest residual."""
    log = eq.log()
    return {"iterations": np.array([line[1] for line in log], np.int64),
            "residuals": np.array([line[2:] for line in log], np.float64)}


def _context(case):
    return _Context(case["nx"], case["ny"], case["nz"], case["jitter"], case["subd"],
                    case["channel"], case["steady"], case["pc"], case["gs"], case["asm"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "residual":
        return _residual_state(case, seed)
    if kind == "dropin":
        ctx = _Context(case["nx"], case["ny"], case["nz"], 0.0, case["subd"], False, True,
                       "reference", "reference", 64)
        eq = ctx.eq
        eq.reset()
        _properties(eq, seed)
        eq.run(1, 2)  # the host's state part-way through a run
        eq.clear_log()
        ne = eq.sizes["ap"]
        return {"kind": kind, "ctx": ctx, "host": {k: eq.get(k) for k in PUT_STATE},
                "rho": np.ones(ne), "mu": np.full(ne, 1.0 / _reynolds(seed))}
    if kind == "batch":
        ctxs = []
        for k, n in enumerate(int(s) for s in case["sizes"].split(",")):
            ctxs.append(_Context(n, n, n, 0.0, 1, False, True, "mgcg-mixed", "colored", 32))
            ctxs[-1].eq.reset()
            _properties(ctxs[-1].eq, seed + 7919 * k)
        batch = cfdl.Batch()
        for c in ctxs:
            batch.attach(c.eq)
        return {"kind": kind, "batch": batch, "ctxs": ctxs, "chunk": case["chunk"]}
    ctx = _context(case)
    _properties(ctx.eq, seed)
    return {"kind": kind, "ctx": ctx, "steps": case["steps"], "ncoef": case["ncoef"],
            "energy": case["energy"]}


def run(state):
    kind = state["kind"]
    if kind == "residual":
        return _residual_run(state)
    if kind == "batch":
        eqs = [c.eq for c in state["ctxs"]]
        for eq in eqs:
            eq.reset()
        state["batch"].run(1, state["chunk"])
        return [dict({k: eq.get(k) for k in FIELDS}, **_lines(eq)) for eq in eqs]
    eq = state["ctx"].eq
    if kind == "dropin":
        for k in PUT_STATE:
            eq.set(k, state["host"][k])
        eq.set_properties(state["rho"], state["mu"])
        eq.update_boundaries()
        eq.solve_uvwp()
        out = _lines(eq)
        eq.clear_log()
        out.update({k: eq.get(k) for k in GET_STATE})
        return out
    eq.reset()
    eq.run(state["steps"], state["ncoef"], energy=state["energy"])
    out = _lines(eq)
    out.update({k: eq.get(k) for k in FIELDS + (("t",) if state["energy"] else ())})
    return out


# ---- calc_residual on device arrays
def _residual_state(case, seed):
    m = _mesh(case["nx"], case["ny"], case["nz"], 0.0, False, 1)
    i = m.info()
    ne, nbf = i["ne"], i["nbf"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(n, lo, hi):
        return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo

    row = torch.from_numpy(m.get("ef2nb_idx") - 1).cuda()
    packed = m.get("ef2nb")[:row[-1].item()].view(np.uint32)
    nbr = torch.from_numpy((packed >> 5).astype(np.int32) - 1).cuda()
    s = {"kind": "residual", "ne": ne, "row": row, "nbr": nbr, "ap": uniform(ne, 3.0, 7.0),
         "anb": uniform(nbr.numel(), 0.0, 1.0), "b": uniform(ne, -1.0, 1.0),
         "phi": uniform(ne + nbf, -1.0, 1.0)}
    lib = cfdl.load_library()
    s["call"] = lib.cfdl_calc_residual if case["alloc"] else lib.cfdl_calc_residual_noalloc
    s["ptr"] = [s[k].data_ptr() for k in ("row", "nbr", "ap", "anb", "b", "phi")]
    return s


def _residual_run(s):
    res, res_max = ctypes.c_double(), ctypes.c_double()
    if s["call"](s["ne"], *s["ptr"], ctypes.byref(res), ctypes.byref(res_max),
                 torch.cuda.current_stream().cuda_stream):
        raise cfdl.CfdlError("calc_residual failed")
    return {"rms": res.value, "max": res_max.value}


# ---- the work a pass cannot do without: each field, coefficient and index a
# step reads or writes counted once per step (FP64 8 B, FP32 and int32 4 B),
# with the solvers' usual iteration counts
def work(case):
    kind = case["kind"]
    if kind == "residual":
        ne = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 100.0 * ne, "flops": 16.0 * ne}
    if kind == "batch":
        ne = sum(int(s) ** 3 for s in case["sizes"].split(","))
        return {"bytes": ne * (case["chunk"] * (2108.0 + 416.0 + 274.0 + 442.0 * 6) + 32.0),
                "flops": ne * case["chunk"] * 4000.0}
    ne = case["nx"] * case["ny"] * case["nz"]
    if kind == "dropin":
        return {"bytes": ne * (2108.0 + 416.0 + 22700.0 + 260.0 + 360.0), "flops": ne * 6500.0}
    pc = {"reference": 22700.0, "colored": 22700.0, "mixed": 14800.0, "mgcg": 190.0 + 580.0 * 7,
          "mgcg-mixed": 274.0 + 442.0 * 7}[case["pc"]]
    outer = case["steps"] * case["ncoef"]
    per = 2108.0 + 416.0 + pc + (900.0 if case["energy"] else 0.0)
    return {"bytes": ne * (outer * per + 32.0),
            "flops": ne * outer * (4000.0 if case["pc"].startswith("mgcg") else 6500.0)}


# ---- the pass in 64 bits, by torch alone
def exact(case, seed):
    if case["kind"] == "residual":
        s = _residual_state(case, seed)
        ne, row, nbr = s["ne"], s["row"].long(), s["nbr"].long()
        owner = torch.repeat_interleave(torch.arange(ne, device="cuda"), row[1:] - row[:-1])
        r = s["b"].clone()
        r.index_add_(0, owner, s["anb"] * s["phi"][nbr])
        r -= s["ap"] * s["phi"][:ne]
        return {"rms": math.sqrt((r * r).sum().item() / ne), "max": max(r.max().item(), 0.0)}
    if case["kind"] != "run" or case["pc"].startswith("mgcg") or case["channel"]:
        return None
    ne = case["nx"] * case["ny"] * case["nz"]
    outer = case["steps"] * case["ncoef"]
    # sweeps in the reference's order take one step per dependency level
    if ne > 900000 or (case["pc"] == "reference" and 0.05 * ne ** (1 / 3) * outer > 12.0):
        return None
    m = _mesh(case["nx"], case["ny"], case["nz"], case["jitter"], False, case["subd"])
    x = _Exact(m, 1.0 / _reynolds(seed), math.inf if case["steady"] else 0.01,
               (0.7, 0.3) if case["steady"] else (1.0, 1.0), case["pc"] != "reference")
    for _ in range(case["steps"]):
        for _ in range(case["ncoef"]):
            x.iteration()
        x.u0, x.mip0 = x.u.clone(), x.mip.clone()
    out = {"iterations": None, "residuals": np.array(x.log, np.float64)}
    out.update(u=x.u[0], v=x.u[1], w=x.u[2], p=x.p)
    if case["energy"]:
        out["t"] = None
    return out


class _Exact:
    """SIMPLE outer iterations of the lid-driven cavity on a hexahedral mesh,
    Gauss-Seidel in the given visiting order, as tensor operations."""

    def __init__(self, mesh, mu, dt, alpha, colored, nit=100):
        def dev(a):
            return torch.from_numpy(np.ascontiguousarray(a)).cuda()

        i = mesh.info()
        ne, nf, nbf = self.ne, self.nf, self.nbf = i["ne"], i["nf"], i["nbf"]
        ef = mesh.get("ef2nb")
        nb = ((ef[:6 * ne].view(np.uint32) >> 5).astype(np.int64) - 1).reshape(ne, 6)
        fs = ef[6 * ne:].astype(np.int64).reshape(ne, 6)
        self.mu, self.dt, self.alpha, self.nit = mu, dt, alpha, nit
        self.nb, self.fg = dev(nb), dev(np.abs(fs) - 1)
        self.sg = dev(np.sign(fs).astype(np.float64))
        self.inner = self.nb < ne
        self.x = dev(np.stack([mesh.get(k) for k in ("xc", "yc", "zc")], 1))
        self.vol = dev(mesh.get("vol"))
        aip = dev(mesh.get("aip").reshape(nf, 3))
        self.area = aip.norm(dim=1)
        self.nrm, self.rip = aip / self.area[:, None], dev(mesh.get("rip").reshape(nf, 3))
        own = self.sg > 0
        cell = torch.arange(ne, device="cuda")[:, None].expand(ne, 6)
        self.P = torch.zeros(nf, dtype=torch.int64, device="cuda")
        self.N = torch.zeros_like(self.P)
        self.P[self.fg[own]], self.N[self.fg[own]] = cell[own], self.nb[own]
        self.fin = (self.N < ne).nonzero().flatten()
        self.hown = torch.zeros(nbf, dtype=torch.int64, device="cuda")
        self.hown[self.nb[~self.inner] - ne] = cell[~self.inner]
        self.lid = torch.zeros(nbf, dtype=torch.bool, device="cuda")
        lo, hi = mesh.get("esec").reshape(-1, 2)[mesh.names.index("top")]
        self.lid[lo - ne - 1:hi - ne] = True
        n = ne + nbf
        z = dict(dtype=torch.float64, device="cuda")
        self.u, self.u0, self.p = torch.zeros(3, n, **z), torch.zeros(3, n, **z), torch.zeros(n, **z)
        self.gu, self.gp = torch.zeros(3, n, 3, **z), torch.zeros(n, 3, **z)
        self.mip, self.mip0 = torch.zeros(nf, **z), torch.zeros(nf, **z)
        # visiting orders: the whole mesh, and inside each subdomain
        sub, order = np.zeros(ne, np.int64), np.arange(ne)
        self.nsubd = i["nsubd"]
        if self.nsubd > 1:
            order, sub = mesh.get("g2gf").astype(np.int64) - 1, mesh.get("gf2g").astype(np.int64) - 1
        place = np.empty(ne, np.int64)
        place[order] = np.arange(ne)
        whole = np.arange(ne)
        self.all = self._groups(nb, whole, np.zeros(ne, np.int64), colored)
        # a subdomain's colours follow the global order
        self.parts = self._groups(nb, whole if colored else place, sub, colored)
        self.sub = dev(sub)
        nbc = self.nb.clamp(max=ne - 1)
        self.same = self.inner & (self.sub[nbc] == self.sub[:, None])
        self.slot = torch.where(self.same, self.nb,
                                ne + torch.arange(6 * ne, device="cuda").reshape(ne, 6))
        self.cross = (self.inner & ~self.same).flatten().nonzero().flatten()
        self.size = torch.bincount(self.sub, minlength=self.nsubd).double()
        self.log = []

    def _groups(self, nb, place, sub, colored):
        """Cells that may be updated together, in visiting order: greedy
        colours, or dependency levels of the sequential order."""
        ne = self.ne
        key = np.zeros(ne, np.int64)
        order = np.argsort(place, kind="stable")
        nbl, pl, sl = nb.tolist(), place.tolist(), sub.tolist()
        kl = [0] * ne
        for e in order.tolist():
            seen = [kl[d] for d in nbl[e] if d < ne and sl[d] == sl[e] and pl[d] < pl[e]]
            if colored:
                c = 0
                while c in seen:
                    c += 1
                kl[e] = c
            else:
                kl[e] = max(seen) + 1 if seen else 0
        key[:] = kl
        by = np.argsort(key, kind="stable")
        cut = np.flatnonzero(np.diff(key[by])) + 1
        return [torch.from_numpy(g).cuda() for g in np.split(by, cut)]

    @staticmethod
    def _sweeps(groups, nb, ap, anb, b, phi, sor):
        packed = [(g, nb[g], ap[g], anb[g], b[g]) for g in groups]
        return [(g, n, a, an / a[:, None] / sor, bb / a / sor) for g, n, a, an, bb in packed]

    @staticmethod
    def _symmetric(packed, phi, sor):
        for some in (packed, packed[::-1]):
            for g, n, _, an, bb in some:
                v = (an * phi[n]).sum(1) + bb
                phi[g] = v + (1.0 - 1.0 / sor) * phi[g] if sor != 1.0 else v

    def _solve_gs(self, ap, anb, b, phi, sor):
        packed = self._sweeps(self.all, self.nb, ap, anb, b, phi, sor)

        def resid():
            return b + (anb * phi[self.nb]).sum(1) - ap * phi[:self.ne]

        ri = rf = resid().square().mean().sqrt().item()
        it, rm = 0, 0.0
        while it < self.nit and rf > ri / 10.0:
            it += 1
            self._symmetric(packed, phi, sor)
            r = resid().abs()
            rf, rm = r.square().mean().sqrt().item(), r.max().item()
        self.log.append((ri, rf, rm))

    def _solve_parts(self, ap, anb, b):
        ne, ns = self.ne, self.nsubd
        phi = torch.zeros(7 * ne, dtype=torch.float64, device="cuda")
        packed = self._sweeps(self.parts, self.slot, ap, anb, b, phi, 1.02)
        src = self.nb.flatten()[self.cross]

        def resid():
            r = b + (anb * phi[self.slot]).sum(1) - ap * phi[:ne]
            s = torch.zeros(ns, dtype=torch.float64, device="cuda").index_add_(0, self.sub, r * r)
            return (s / self.size).sum().item(), max(r.max().item(), 0.0)

        s, rm = resid()
        ri = rf = math.sqrt(s / ns)
        it = 0
        while it < self.nit and rf > ri / 10.0:
            for _ in range(2):
                self._symmetric(packed, phi, 1.02)
            it += 2
            phi[ne + self.cross] = phi[src]
            if it % 10 == 0:
                s, m = resid()
                rf, rm = math.sqrt((rf + s) / ns), max(rm, m)
        self.log.append((ri, rf, rm))
        return phi[:ne]

    def _grad(self, phi):
        ne = self.ne
        dr = self.x[self.nb] - self.x[:ne, None]
        w = 1.0 / dr.square().sum(2)
        g = (w * (phi[self.nb] - phi[:ne, None]))[:, :, None] * dr
        a = [[(w * dr[:, :, i] * dr[:, :, j]).sum(1) for j in range(3)] for i in range(3)]
        g = g.sum(1)

        def minor(i, j):
            (p, q), (r, s) = [[k for k in range(3) if k != m] for m in (i, j)]
            return (a[p][r] * a[q][s] - a[p][s] * a[q][r]) * (-1.0) ** (i + j)

        det = sum(a[0][j] * minor(0, j) for j in range(3))
        out = torch.zeros(ne + self.nbf, 3, dtype=torch.float64, device="cuda")
        for i in range(3):
            out[:ne, i] = sum(minor(j, i) * g[:, j] for j in range(3)) / det
        return out

    def _weight(self, e, nb, f):
        la = (self.x[e] - self.rip[f]).norm(dim=-1)
        lb = (self.x[nb] - self.rip[f]).norm(dim=-1)
        return la / (la + lb)

    def iteration(self):
        ne, mu, inner = self.ne, self.mu, self.inner
        n = ne + self.nbf
        u, H = self.u, slice(self.ne, n)
        # boundary values: the lid moves, walls stand, no flux through either
        u[:, H] = 0.0
        u[0, H] = self.lid.double()
        self.p[H] = self.p[self.hown]
        bface = self.fg[~inner]
        self.mip[bface] = 0.0
        # momentum coefficients
        e = torch.arange(ne, device="cuda")[:, None].expand(ne, 6)
        area, sg = self.area[self.fg], self.sg
        nrm = sg[:, :, None] * self.nrm[self.fg]
        dr = self.x[self.nb] - self.x[:ne, None]
        ds = dr.norm(dim=2)
        nbc = torch.where(inner, self.nb, e)
        wt = torch.where(inner, self._weight(e, nbc, self.fg), torch.zeros_like(ds))
        flux = -(sg * self.mip[self.fg]) * inner
        d = mu * area / ds
        anb = (d + flux.clamp(min=0.0)) * inner
        rip = self.rip[self.fg]
        foot_p = rip - ((rip - self.x[:ne, None]) * nrm).sum(2, keepdim=True) * nrm
        foot_n = rip - ((rip - self.x[self.nb]) * nrm).sum(2, keepdim=True) * nrm
        drp = torch.where(inner[:, :, None], foot_n - foot_p, torch.ones_like(foot_n))
        dsp = drp.norm(dim=2)
        wt3 = wt[None, :, :, None]
        gip = (1.0 - wt3) * self.gu[:, :ne, None] + wt3 * self.gu[:, nbc]  # component, cell, face, axis
        ap0 = self.vol / self.dt
        src = ap0 * self.u0[:, :ne] + flux.sum(1) * u[:, :ne] - self.vol * self.gp[:ne].T
        along = (gip * dr).sum(3) / ds
        across = (gip * dr.permute(2, 0, 1)[:, :, :, None]).sum(0).permute(2, 0, 1) / ds
        src = src + (mu * area * inner * across).sum(2)
        src = src + (mu * area * inner * ((gip * drp).sum(3) / dsp - along)).sum(2)
        ap = anb.sum(1) + ap0
        # walls: the tangential part enters explicitly, the rest implicitly
        ob = (~inner).double() * d
        un = (u[:, :ne].T[:, None] * nrm).sum(2)
        tang = u[:, :ne, None] - un[None] * nrm.permute(2, 0, 1)
        uh = torch.where(inner[None], torch.zeros_like(tang), u[:, self.nb])
        src = src + (ob * (uh - tang) - ob * u[:, :ne, None]).sum(2)
        anb = anb + ob
        ap = ap + ob.sum(1)
        if self.alpha[0] != 1.0:
            relaxed = ap / self.alpha[0]
            src = src + (relaxed - ap) * u[:, :ne]
            ap = relaxed
        dd, dc = self.vol / ap, self.vol / (ap - anb.sum(1))
        for k in range(3):
            self._solve_gs(ap, anb, src[k], u[k], 1.0)
        for k in range(3):
            self.gu[k] = self._grad(u[k])
        # face fluxes
        f = self.fin
        P, N = self.P[f], self.N[f]
        A, nf = self.area[f], self.nrm[f]
        w = self._weight(P, N, f)
        drf = self.x[N] - self.x[P]

        def face(q):
            return (1.0 - w) * q[..., P] + w * q[..., N]

        gpf = face(self.gp.T).T
        dot = (drf * nf).sum(1)
        m = (face(u).T * nf).sum(1) * A
        df = face(dd)
        m = m - A * df / dot * (self.p[N] - self.p[P] - (gpf * drf).sum(1))
        m = m - df / self.dt * (self.mip0[f] - (face(self.u0).T * nf).sum(1) * A)
        self.mip[f] = m
        # pressure correction
        coef = face(dc) / dot * A
        per_face = torch.zeros(self.nf, dtype=torch.float64, device="cuda")
        per_face[f] = coef
        anb = per_face[self.fg]
        b = -(sg * self.mip[self.fg]).sum(1)
        ap = anb.sum(1)
        if self.nsubd > 1:
            pc = self._solve_parts(ap, anb, b)
        else:
            full = torch.zeros(n, dtype=torch.float64, device="cuda")
            self._solve_gs(ap, anb, b, full, 1.02)
            pc = full[:ne]
        pc = pc - pc[0]
        pc = torch.cat([pc, pc[self.hown]])
        gpc = self._grad(pc)
        self.p[:ne] += self.alpha[1] * pc[:ne]
        self.gp[:ne] += self.alpha[1] * gpc[:ne]
        self.mip[f] -= A * face(dc) * (pc[N] - pc[P]) / dot
