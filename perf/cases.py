"""Performance cases of the MHD pipeline: what is timed, and on which inputs.

A case is one piece of work as a user's program asks for it: a single mesh that is filled from
host memory, advanced some RK steps and read back (`Mesh`), or a batch of many meshes that is
advanced some steps and read back (`Batch`). The states live in pinned host buffers that are
kept between passes, as a program that feeds and reads runs all the time keeps them.

FP64 runs return the conserved state and the face field in FP64. Mixed-precision runs return
them in FP32, the precision of their fluxes.
"""
import ctypes as C
import math
import random

import torch

import chasqui_amd


def _case(name, **kw):
    c = dict(kind="solo", problem="blast", nx1=64, nx2=1, nx3=1, recon="ppm", rsolver="hlld", integrator="rk3",
             precision="fp64", fofc=True, flatten=True, preset=False, steps=20, runs=1)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest run: the 1D circularly polarised Alfven wave of the convergence tests
        _case("cpaw_1d_128", problem="cpaw", nx1=128, steps=100),
        # a long shock tube with outflow boundaries, at the upper end of the served tubes; odd size
        _case("tube_1d_3999_mixed", problem="tube", nx1=3999, precision="mixed", steps=60),
        # a small 2D vortex of odd, unequal sizes: launches and latency
        _case("vortex_2d_150x129", problem="orszag_tang", nx1=150, nx2=129, recon="ppmx", steps=50),
        # the upper end of the ensembles' sizes, alone, in mixed precision
        _case("vortex_2d_512_mixed", problem="orszag_tang", nx1=512, nx2=512, recon="ppmx", precision="mixed", steps=50),
        # a large 2D run with the most expensive reconstruction
        _case("vortex_2d_1000x1024_wenoz", problem="orszag_tang", nx1=1000, nx2=1024, recon="wenoz", steps=20),
        # the smallest served 3D blast, ragged; the positivity fallback fires
        _case("blast_3d_64x56x45", problem="blast", nx1=64, nx2=56, nx3=45, steps=40),
        # the headline run: 256^3 blast, PPM + HLLD + RK3 + CT + positivity fallback + flattening
        _case("blast_3d_256", problem="blast", nx1=256, nx2=256, nx3=256, steps=20),
        # the largest served blast, in the served precision
        _case("blast_3d_192_mixed", problem="blast", nx1=192, nx2=192, nx3=192, precision="mixed", steps=30),
        # the oblique wave of the mixed-precision accuracy table
        _case("cpaw_3d_128_wenoz_mixed", problem="cpaw", nx1=128, nx2=128, nx3=128, recon="wenoz", precision="mixed",
              steps=20),
        # the recommended robust options: PPMX in characteristic variables, LHLLD, dual energy
        _case("robust_3d_80x72x64", problem="blast", nx1=80, nx2=72, nx3=64, recon="ppmx", rsolver="lhlld", preset=True,
              steps=15),
        # an ensemble of 2D vortices of the ensemble's sizes (64^2 to 512^2), one shared step
        _case("ensemble_48_vortices", kind="batch", problem="orszag_tang", nx1=64, nx2=512, recon="ppmx", runs=48,
              steps=40),
        # an ensemble of small 1D and 2D runs in mixed precision, as a server holds them
        _case("ensemble_64_small_mixed", kind="batch", problem="tube", nx1=32, nx2=128, precision="mixed", runs=64,
              steps=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges; sizes over their logarithm, odd ones among them."""
    family = rng.choice(("1d", "1d", "2d", "2d", "3d", "3d", "robust", "ensemble"))
    recon = rng.choice(("plm", "ppm", "ppmx", "wenoz"))
    precision = rng.choice(("fp64", "mixed"))
    integrator = rng.choice(("rk2", "rk3"))
    common = dict(recon=recon, precision=precision, integrator=integrator)
    if family == "1d":
        return _case(None, problem=rng.choice(("cpaw", "tube")), nx1=_log(rng, 100, 4000), steps=rng.randint(60, 100),
                     **common)
    if family == "2d":
        return _case(None, problem="orszag_tang", nx1=_log(rng, 64, 1024), nx2=_log(rng, 64, 1024),
                     steps=rng.randint(20, 50), **common)
    if family == "3d":
        return _case(None, problem=rng.choice(("cpaw", "blast")), nx1=_log(rng, 32, 192), nx2=_log(rng, 32, 192),
                     nx3=_log(rng, 32, 192), steps=rng.randint(10, 25), **common)
    if family == "robust":
        return _case(None, problem="blast", nx1=_log(rng, 32, 96), nx2=_log(rng, 32, 96), nx3=_log(rng, 32, 96),
                     recon="ppmx", rsolver="lhlld", preset=True, steps=rng.randint(8, 15))
    return _case(None, kind="batch", problem=rng.choice(("orszag_tang", "tube")), nx1=32, nx2=rng.choice((128, 256, 400)),
                 runs=_log(rng, 12, 64), steps=rng.randint(20, 40), **common)


# ---------------------------------------------------------------- the runs of a case
def _runs(case, seed):
    """The meshes of a case: problem, cells, extents, adiabatic index, CFL number, boundaries."""
    if case["kind"] == "solo":
        return [_run(case["problem"], case["nx1"], case["nx2"], case["nx3"], seed * 1000)]
    r = random.Random(97)   # the sizes are the case's own, the states are the seed's
    lo, hi = case["nx1"], case["nx2"]
    if case["problem"] == "orszag_tang":
        sizes = [n for n in (32, 48, 64, 96, 128, 192, 256, 384, 512) if lo <= n <= hi]
        return [_run("orszag_tang", n, n, 1, seed * 1000 + q)
                for q, n in enumerate(r.choice(sizes) for _ in range(case["runs"]))]
    out = []   # tubes of 400 to 4000 cells and vortices of lo^2 to hi^2, alternating
    for q in range(case["runs"]):
        if q % 2 == 0:
            out.append(_run("tube", _log(r, 400, 4000), 1, 1, seed * 1000 + q))
        else:
            n = _log(r, lo, hi)
            out.append(_run("orszag_tang", n, n, 1, seed * 1000 + q))
    return out


def _run(problem, nx1, nx2, nx3, seed):
    n = (nx1, nx2, nx3)
    if problem == "blast":   # equal cells: the longest axis spans 1
        h = 1.0 / max(n)
        ext = [(-0.5 * h * q, 0.5 * h * q) if q > 1 else (0.0, 1.0) for q in n]
        gamma, cfl, bc = 5.0 / 3.0, 0.3, "periodic"
    elif problem == "tube":
        ext, gamma, cfl, bc = [(-0.5, 0.5), (0.0, 1.0), (0.0, 1.0)], 2.0, 0.4, "outflow"
    else:
        ext, gamma, cfl, bc = [(0.0, 1.0)] * 3, 5.0 / 3.0, 0.4 if nx2 == 1 else 0.3, "periodic"
    return dict(problem=problem, n=n, ext=ext, gamma=gamma, cfl=cfl, bc=bc, seed=seed, ng=3)


def _cells(run):
    return [q + 2 * run["ng"] if q > 1 or d == 0 else 1 for d, q in enumerate(run["n"])]


def _initial(run, device):
    """Conserved state (6, nk, nj, ni) and face fields (nk+1, nj+1, ni+1), ghost cells zero.

    The face field is the discrete curl of a vector potential on the edges plus a constant, so
    its divergence vanishes to round-off."""
    n, ext, ng, seed = run["n"], run["ext"], run["ng"], run["seed"]
    rnd = random.Random(seed)
    f8 = dict(dtype=torch.float64, device=device)
    dx = [(ext[d][1] - ext[d][0]) / n[d] for d in range(3)]
    has = [n[0] > 1, n[1] > 1, n[2] > 1]
    cen = [ext[d][0] + (torch.arange(n[d], **f8) + 0.5) * dx[d] for d in range(3)]
    edg = [ext[d][0] + torch.arange(n[d] + 1, **f8) * dx[d] for d in range(3)]
    view = [lambda v: v.view(1, 1, -1), lambda v: v.view(1, -1, 1), lambda v: v.view(-1, 1, 1)]
    X, Y, Z = (view[d](cen[d]) for d in range(3))

    def noise(amp):
        g = torch.Generator(device=device)
        g.manual_seed(seed + 1)
        return 1.0 + amp * (2.0 * torch.rand((n[2], n[1], n[0]), generator=g, **f8) - 1.0)

    const = [0.0, 0.0, 0.0]
    zero = torch.zeros((), **f8)
    pot = [lambda x, y, z: zero, lambda x, y, z: zero, lambda x, y, z: zero]
    one = torch.ones((n[2], n[1], n[0]), **f8)
    if run["problem"] == "cpaw":
        kv = [2.0 * math.pi * has[d] / (ext[d][1] - ext[d][0]) for d in range(3)]
        kn = math.sqrt(sum(q * q for q in kv))
        e1 = [q / kn for q in kv]
        e2 = [-e1[1], e1[0], 0.0]
        s = math.hypot(e2[0], e2[1])
        e2 = [q / s for q in e2]
        e3 = [e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]]
        amp, ph = 0.1 * rnd.uniform(0.95, 1.05), rnd.uniform(0.0, 2.0 * math.pi)

        def wave(d, x, y, z):   # a helical field: its curl is kn times itself
            a = kv[0] * x + kv[1] * y + kv[2] * z + ph
            return amp * (e2[d] * torch.sin(a) + e3[d] * torch.cos(a))

        pot = [lambda x, y, z, d=d: wave(d, x, y, z) / kn for d in range(3)]
        const = e1
        rho, prs = one, 0.1 * one
        vel = [wave(d, X, Y, Z) * one for d in range(3)]
    elif run["problem"] == "orszag_tang":
        p0 = 5.0 / (12.0 * math.pi) * rnd.uniform(0.95, 1.05)
        b0 = rnd.uniform(0.95, 1.05) / math.sqrt(4.0 * math.pi)
        tp = 2.0 * math.pi
        pot[2] = lambda x, y, z: b0 * (torch.cos(2 * tp * x) / (2 * tp) + torch.cos(tp * y) / tp)
        rho, prs = 25.0 / (36.0 * math.pi) * one, p0 * one
        vel = [-torch.sin(tp * Y) * one, torch.sin(tp * X) * one, 0.0 * one]
    elif run["problem"] == "blast":
        s = math.sqrt(0.5)
        const = [s, s, 0.0]
        r2 = X * X + (Y * Y if has[1] else 0.0) + (Z * Z if has[2] else 0.0)
        rho = noise(1e-3)
        prs = torch.where(r2 < 0.01, 10.0, 0.1) * one
        vel = [0.0 * one] * 3
    else:   # Brio-Wu tube
        const = [0.75, 0.0, 0.0]
        pot[2] = lambda x, y, z: torch.abs(x)
        left = X < 0.0
        rho = torch.where(left, 1.0, 0.125) * noise(1e-3)
        prs = torch.where(left, 1.0, 0.1) * one
        vel = [0.0 * one] * 3

    def edge(d):   # the potential on the edges along d
        at = [cen[q] if q == d else edg[q] for q in range(3)]
        v = pot[d](*(view[q](at[q]) for q in range(3)))
        return v.expand(len(at[2]), len(at[1]), len(at[0]))

    def diff(a, d):   # along d, zero where the mesh has no such direction
        ax = 2 - d
        lo, hi = a.narrow(ax, 0, n[d]), a.narrow(ax, 1, n[d])
        return (hi - lo) / dx[d] if has[d] else torch.zeros_like(lo)

    A = [edge(d) for d in range(3)]
    B = [const[0] + (diff(A[2], 1) - diff(A[1], 2)), const[1] + (diff(A[0], 2) - diff(A[2], 0)),
         const[2] + (diff(A[1], 0) - diff(A[0], 1))]
    bc = [0.5 * (B[d].narrow(2 - d, 0, n[d]) + B[d].narrow(2 - d, 1, n[d])) for d in range(3)]
    eng = prs / (run["gamma"] - 1.0) + 0.5 * rho * sum(v * v for v in vel) + 0.5 * sum(b * b for b in bc)
    ni, nj, nk = _cells(run)
    off = [ng, ng if has[1] else 0, ng if has[2] else 0]
    u = torch.zeros((6, nk, nj, ni), **f8)
    act = (slice(off[2], off[2] + n[2]), slice(off[1], off[1] + n[1]), slice(off[0], off[0] + n[0]))
    for q, v in enumerate([rho, rho * vel[0], rho * vel[1], rho * vel[2], eng]):
        u[q][act] = v
    faces = []
    for d in range(3):
        f = torch.zeros((nk + 1, nj + 1, ni + 1), **f8)
        s = [slice(off[2 - ax], off[2 - ax] + n[2 - ax] + (1 if 2 - ax == d else 0)) for ax in range(3)]
        f[tuple(s)] = B[d]
        faces.append(f)
    return u, faces


# ---------------------------------------------------------------- the framework's side
ARRAYS = ("u0", "b1f0", "b2f0", "b3f0")


def _config(case, run):
    kw = dict(recon=case["recon"], rsolver=case["rsolver"], integrator=case["integrator"], gamma=run["gamma"],
              cfl=run["cfl"], flatten=case["flatten"], fofc=case["fofc"], precision=case["precision"],
              bc=(run["bc"],) * 3)
    if case["preset"]:
        kw.update(characteristic=True, dual_energy=True)
    return chasqui_amd.make_config(**kw)


def _pinned(n, dtype=torch.float64):
    return torch.empty(n, dtype=dtype, pin_memory=torch.cuda.is_available())


def prepare(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    meshes, slots, parts = [], [], []
    nu = nb = 0
    for run in _runs(case, seed):
        desc = chasqui_amd.make_mesh_desc(*run["n"], ng=run["ng"], x1=run["ext"][0], x2=run["ext"][1], x3=run["ext"][2])
        meshes.append(chasqui_amd.Mesh(desc, _config(case, run)))
        u, faces = _initial(run, device)
        slots.append((nu, u.numel(), nb, faces[0].numel()))
        nu += u.numel()
        nb += 3 * faces[0].numel()
        parts.append([u] + faces)
    u_in, b_in, u_out, b_out = _pinned(nu), _pinned(nb), _pinned(nu), _pinned(nb)
    for (ou, cu, ob, cb), part in zip(slots, parts):
        u_in[ou:ou + cu].copy_(part[0].view(-1))
        for d in range(3):
            b_in[ob + d * cb:ob + (d + 1) * cb].copy_(part[1 + d].reshape(-1))
    del parts
    state = dict(case=case, meshes=meshes, slots=slots, u_in=u_in, b_in=b_in, u_out=u_out, b_out=b_out)
    if case["precision"] == "mixed":
        state.update(u32=torch.empty(nu, dtype=torch.float32), b32=torch.empty(nb, dtype=torch.float32))
    if case["kind"] == "batch":
        for q in range(len(meshes)):
            _fill(state, q)
        batch = chasqui_amd.Batch(len(meshes))
        for m in meshes:
            batch.add(m)
        batch.tune()
        state["batch"] = batch
    return state


def _transfer(fn, mesh, name, buf, at, count):
    aid = ARRAYS.index(name)
    aid = 0 if aid == 0 else 4 + aid   # CHQ_U0, CHQ_B1F0 .. CHQ_B3F0
    if fn(mesh.h, aid, C.c_void_p(buf.data_ptr() + 8 * at), C.c_size_t(count)) != 0:
        raise RuntimeError(mesh.L.chq_last_error().decode())


def _fill(state, q):
    """Initial state of run q from host memory into its mesh, ready to step."""
    m = state["meshes"][q]
    ou, cu, ob, cb = state["slots"][q]
    _transfer(m.L.chq_upload, m, "u0", state["u_in"], ou, cu)
    for d in range(3):
        _transfer(m.L.chq_upload, m, ARRAYS[1 + d], state["b_in"], ob + d * cb, cb)
    m.init(t=0.0, tlim=1e30)


def _read(state):
    for m, (ou, cu, ob, cb) in zip(state["meshes"], state["slots"]):
        _transfer(m.L.chq_download, m, "u0", state["u_out"], ou, cu)
        for d in range(3):
            _transfer(m.L.chq_download, m, ARRAYS[1 + d], state["b_out"], ob + d * cb, cb)
    if "u32" in state:
        return {"u": state["u32"].copy_(state["u_out"]), "b": state["b32"].copy_(state["b_out"])}
    return {"u": state["u_out"], "b": state["b_out"]}


def run(state):
    steps = state["case"]["steps"]
    if "batch" in state:   # a batch keeps running: some more steps, then every run's state
        state["batch"].step(steps)
        return _read(state)
    _fill(state, 0)        # one run from its initial state
    mesh = state["meshes"][0]
    mesh.step(steps)
    out = _read(state)
    out["t"] = mesh.status()["t"]
    return out


# ---------------------------------------------------------------- bytes and operations
# FP64 or FP32 operations of one face: the two half-states a cell's reconstruction gives (seven
# variables) and one Riemann solve
FACE_FLOPS = {"dc": 250, "plm": 330, "ppm": 600, "ppmx": 800, "wenoz": 1100}


def work(case):
    nst = {"rk1": 1, "rk2": 2, "rk3": 3}[case["integrator"]]
    byts = flops = 0.0
    for r in _runs(case, 1):
        cells = float(r["n"][0] * r["n"][1] * r["n"][2])
        ndim = sum(q > 1 for q in r["n"])
        # a stage reads its input state (5 conserved values and 3 face fields), writes its output
        # and, after the first, reads the step's start as well; plus the state in and out
        byts += cells * 64.0 * (case["steps"] * (2 * nst + nst - 1) + 2)
        face = FACE_FLOPS[case["recon"]] + (900 if case["preset"] else 0)
        flops += cells * case["steps"] * nst * (ndim * face + 150)
    return {"bytes": byts, "flops": flops}


# ---------------------------------------------------------------- the same runs in plain torch
def exact(case, seed):
    """The pass in FP64 with plain torch: PLM/PPM/PPMX/WENO-Z + flattening + HLLD + upwind CT +
    RK2/RK3 with the positivity fallback. Single meshes without the robust options, up to the
    size that takes some seconds."""
    updates = case["steps"] * case["nx1"] * case["nx2"] * case["nx3"]
    if case["kind"] != "solo" or case["preset"] or updates > 2.6e8:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    r = _runs(case, seed)[0]
    sim = _Method(r, case["recon"], case["flatten"], case["fofc"])
    u, b = _initial(r, device)
    t = sim.advance(u, b, case["steps"], 3 if case["integrator"] == "rk3" else 2)
    return {"u": sim.u.reshape(-1), "b": torch.stack(sim.b).reshape(-1), "t": t}


def _sh(q, s, ax):
    """q at index + s along axis ax (periodic over the array; only interior values are used)."""
    return torch.roll(q, -s, ax)


class _Method:
    FLOORS = (1e-10, 1e-12)   # density and pressure floors

    def __init__(self, run, recon, flatten, fofc):
        self.r, self.recon, self.flatten, self.fofc = run, recon, flatten, fofc
        self.n, self.ng, self.gamma = run["n"], run["ng"], run["gamma"]
        self.ndim = sum(q > 1 for q in self.n)
        self.dx = [(run["ext"][d][1] - run["ext"][d][0]) / self.n[d] for d in range(3)]
        self.lo = [self.ng if d == 0 or self.n[d] > 1 else 0 for d in range(3)]
        self.dims = [d for d in range(3) if self.n[d] > 1]
        self.dfl, self.pfl = self.FLOORS

    def box(self, up=()):
        """Active cells; one more along each direction of `up`."""
        return tuple(slice(self.lo[d], self.lo[d] + self.n[d] + (d in up)) for d in (2, 1, 0))

    # ---- boundaries, x1 then x2 then x3, whole slabs
    def fill(self, u, b):
        per = self.r["bc"] == "periodic"
        for d in self.dims:
            ax, lo, n, ng = 2 - d, self.lo[d], self.n[d], self.ng
            hi = lo + n - 1
            cellwise = [u] + [b[q].unsqueeze(0) for q in range(3) if q != d]
            nk, nj, ni = u.shape[1:]
            for a in cellwise:
                v = a
                if a is not u and d == 0:
                    v = a[:, :nk, :nj, :ni]
                elif a is not u and d == 1:
                    v = a[:, :nk]
                for g in range(ng):
                    v.select(ax + 1, g).copy_(v.select(ax + 1, g + n if per else lo))
                    v.select(ax + 1, hi + 1 + g).copy_(v.select(ax + 1, hi + 1 + g - n if per else hi))
            f = b[d]
            if per:
                f.select(ax, hi + 1).copy_(f.select(ax, lo))
            for g in range(ng):
                f.select(ax, g).copy_(f.select(ax, g + n if per else lo))
                f.select(ax, hi + 2 + g).copy_(f.select(ax, hi + 2 + g - n if per else hi + 1))

    # ---- conserved to primitive
    def centre(self, b):
        nk, nj, ni = self.u.shape[1:]
        out = []
        for d in range(3):
            f = b[d][:nk, :nj, :ni]
            out.append(0.5 * (f + b[d].narrow(2 - d, 1, (ni, nj, nk)[d])[:nk, :nj, :ni]) if d in self.dims else f)
        return out

    def prim(self, u, b):
        bc = self.centre(b)
        d = torch.clamp(u[0], min=self.dfl)
        v = [u[1 + q] / d for q in range(3)]
        bsq = bc[0] ** 2 + bc[1] ** 2 + bc[2] ** 2
        p = (self.gamma - 1.0) * (u[4] - 0.5 * d * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) - 0.5 * bsq)
        p = torch.clamp(p, min=self.pfl)
        self.w = [d] + v + [p]
        self.bc = bc
        self.ec = [v[2] * bc[1] - v[1] * bc[2], v[0] * bc[2] - v[2] * bc[0], v[1] * bc[0] - v[0] * bc[1]]

    def cfl_dt(self):
        a, dt = self.box(), None
        d, p, bc = self.w[0][a], self.w[4][a], [q[a] for q in self.bc]
        for q in self.dims:
            s = torch.abs(self.w[1 + q][a]) + self.fast(d, p, bc[q], bc[(q + 1) % 3], bc[(q + 2) % 3])
            m = float((self.dx[q] / s).min())
            dt = m if dt is None else min(dt, m)
        return dt

    def fast(self, d, p, bn, b1, b2):
        gp = self.gamma * p
        a = (gp + bn * bn + b1 * b1 + b2 * b2) / d
        return torch.sqrt(0.5 * (a + torch.sqrt(torch.clamp(a * a - 4.0 * gp * bn * bn / (d * d), min=0.0))))

    # ---- reconstruction of one variable along ax: (value at the cell's left face, at its right)
    def halves(self, q, ax):
        m2, m1, p1, p2 = (_sh(q, s, ax) for s in (-2, -1, 1, 2))
        if self.recon == "plm":
            l, r = q - m1, p1 - q
            s = torch.where(l * r > 0, 2.0 * (l * r) / (l + r), 0.0)
            return q - 0.5 * s, q + 0.5 * s
        if self.recon == "ppm":
            l, r = q - m1, p1 - q
            m = 0.5 * (p1 - m1)
            s = torch.sign(m) * torch.minimum(torch.abs(m), 2.0 * torch.minimum(torch.abs(l), torch.abs(r)))
            s = torch.where(l * r <= 0, 0.0, s)
            hi = 0.5 * (q + p1) + (s - _sh(s, 1, ax)) / 6.0
            lo = _sh(hi, -1, ax)
            flat = (hi - q) * (q - lo) <= 0
            d, c = hi - lo, q - 0.5 * (lo + hi)
            t = d * d / 6.0
            nlo = torch.where(d * c > t, 3.0 * q - 2.0 * hi, lo)
            nhi = torch.where(~(d * c > t) & (d * c < -t), 3.0 * q - 2.0 * lo, hi)
            return torch.where(flat, q, nlo), torch.where(flat, q, nhi)
        if self.recon == "ppmx":
            f = (7.0 / 12.0) * (q + p1) - (1.0 / 12.0) * (m1 + p2)
            d2, dl, dr = 3.0 * (q + p1 - 2.0 * f), m1 + p1 - 2.0 * q, q + p2 - 2.0 * p1
            lim = torch.sign(d2) * torch.minimum(torch.minimum(1.25 * dl.abs(), 1.25 * dr.abs()), d2.abs())
            lim = torch.where((d2 * dl > 0) & (d2 * dr > 0), lim, 0.0)
            hi = torch.where((f - q) * (p1 - f) < 0, 0.5 * (q + p1) - lim / 6.0, f)
            lo = _sh(hi, -1, ax)
            dm, dp = q - lo, hi - q
            ext = (dm * dp <= 0) | ((p1 - q) * (q - m1) <= 0)
            d2, dc = 6.0 * (lo + hi - 2.0 * q), m1 + p1 - 2.0 * q
            dl, dr = m2 + q - 2.0 * m1, q + p2 - 2.0 * p1
            lim = torch.sign(d2) * torch.minimum(torch.minimum(1.25 * dl.abs(), 1.25 * dr.abs()),
                                                 torch.minimum(1.25 * dc.abs(), d2.abs()))
            lim = torch.where((d2 * dc > 0) & (d2 * dl > 0) & (d2 * dr > 0), lim, 0.0)
            big = d2.abs() > 1e-12 * (q.abs() + m1.abs() + p1.abs()) + 1e-300
            rho = torch.where(big, lim / torch.where(big, d2, 1.0), 0.0)
            cut = rho < 1.0 - 1e-12
            xlo, xhi = torch.where(cut, q - rho * dm, lo), torch.where(cut, q + rho * dp, hi)
            mlo = torch.where(dm.abs() >= 2.0 * dp.abs(), q - 2.0 * dp, lo)
            mhi = torch.where(dp.abs() >= 2.0 * dm.abs(), q + 2.0 * dm, hi)
            return torch.where(ext, xlo, mlo), torch.where(ext, xhi, mhi)
        return self.wz(p2, p1, q, m1, m2), self.wz(m2, m1, q, p1, p2)

    @staticmethod
    def wz(a, b, c, d, e):
        s = [13.0 / 12.0 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2,
             13.0 / 12.0 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2,
             13.0 / 12.0 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2]
        tau = torch.abs(s[0] - s[2])
        w = [g * (1.0 + tau / (v + 1e-36)) for g, v in zip((0.1, 0.6, 0.3), s)]
        p = [(2 * a - 7 * b + 11 * c) / 6.0, (-b + 5 * c + 2 * d) / 6.0, (2 * c + 5 * d - e) / 6.0]
        return (w[0] * p[0] + w[1] * p[1] + w[2] * p[2]) / (w[0] + w[1] + w[2])

    # ---- fluxes of direction d at the lower face of every cell, in x, y, z order
    def states(self, d, donor):
        ax = 2 - d
        t1, t2 = (d + 1) % 3, (d + 2) % 3
        q = [self.w[0], self.w[1 + d], self.w[1 + t1], self.w[1 + t2], self.w[4], self.bc[t1], self.bc[t2]]
        if donor:
            return [_sh(v, -1, ax) for v in q], q
        pairs = [self.halves(v, ax) for v in q]
        lo, hi = [a for a, _ in pairs], [b for _, b in pairs]
        if self.flatten and self.recon != "plm":
            p, u = q[4], q[1]
            pm, pp = _sh(p, -1, ax), _sh(p, 1, ax)
            dp, dp2 = pp - pm, _sh(p, 2, ax) - _sh(p, -2, ax)
            on = (dp.abs() > 0.33 * torch.minimum(pm, pp)) & (_sh(u, -1, ax) > _sh(u, 1, ax))
            ratio = torch.where(dp2.abs() > 1e-300, dp / torch.where(dp2 == 0, 1.0, dp2), 0.0)
            f = torch.where(on, torch.clamp(10.0 * (ratio - 0.75), 0.0, 1.0), 0.0)
            lo = [torch.where(f > 0, a + f * (v - a), a) for a, v in zip(lo, q)]
            hi = [torch.where(f > 0, a + f * (v - a), a) for a, v in zip(hi, q)]
        bl, bh = (lo[0] <= self.dfl) | (lo[4] <= self.pfl), (hi[0] <= self.dfl) | (hi[4] <= self.pfl)
        lo = [torch.where(bl, v, a) for a, v in zip(lo, q)]
        hi = [torch.where(bh, v, a) for a, v in zip(hi, q)]
        return [_sh(v, -1, ax) for v in hi], lo

    def cons_flux(self, s, bn):
        d, u, v, w, p, b1, b2 = s
        e = p / (self.gamma - 1.0) + 0.5 * (d * (u * u + v * v + w * w) + (bn * bn + b1 * b1 + b2 * b2))
        pt = p + 0.5 * (bn * bn + b1 * b1 + b2 * b2)
        vb = u * bn + v * b1 + w * b2
        U = [d, d * u, d * v, d * w, e, b1, b2]
        F = [d * u, d * u * u + pt - bn * bn, d * u * v - bn * b1, d * u * w - bn * b2, (e + pt) * u - bn * vb,
             b1 * u - bn * v, b2 * u - bn * w]
        return U, F, e, pt

    def flux(self, d, b, donor=False):
        nk, nj, ni = self.u.shape[1:]
        bn = b[d][:nk, :nj, :ni]
        L, R = self.states(d, donor)
        f = (self.hlle if donor else self.hlld)(L, R, bn)
        t1, t2 = (d + 1) % 3, (d + 2) % 3
        out = [f[0], None, None, None, f[4]]
        out[1 + d], out[1 + t1], out[1 + t2] = f[1], f[2], f[3]
        return out, {t2: -f[5], t1: f[6]}   # face EMFs by component

    def hlle(self, L, R, bn):
        UL, FL, _, _ = self.cons_flux(L, bn)
        UR, FR, _, _ = self.cons_flux(R, bn)
        cl, cr = self.fast(L[0], L[4], bn, L[5], L[6]), self.fast(R[0], R[4], bn, R[5], R[6])
        sl, sr = torch.minimum(L[1] - cl, R[1] - cr), torch.maximum(L[1] + cl, R[1] + cr)
        out = []
        for q in range(7):
            m = (sr * FL[q] - sl * FR[q] + sl * sr * (UR[q] - UL[q])) / (sr - sl)
            out.append(torch.where(sl >= 0, FL[q], torch.where(sr <= 0, FR[q], m)))
        return out

    def hlld(self, L, R, bn):
        UL, FL, el, ptl = self.cons_flux(L, bn)
        UR, FR, er, ptr = self.cons_flux(R, bn)
        cl, cr = self.fast(L[0], L[4], bn, L[5], L[6]), self.fast(R[0], R[4], bn, R[5], R[6])
        sl, sr = torch.minimum(L[1] - cl, R[1] - cr), torch.maximum(L[1] + cl, R[1] + cr)
        bn2, al, ar = bn * bn, sl - L[1], sr - R[1]
        ml, mr = L[0] * al, R[0] * ar
        sm = (mr * R[1] - ml * L[1] + (ptl - ptr)) / (mr - ml)
        pts = (mr * ptl - ml * ptr + L[0] * R[0] * ar * al * (R[1] - L[1])) / (mr - ml)

        def star(S, a, s, e, pt):
            bs = s - sm
            ds = S[0] * a / bs
            den = S[0] * a * bs - bn2
            deg = den.abs() <= 1e-12 * ((S[0] * a * bs).abs() + bn2) + 1e-300
            sden = torch.where(deg, 1.0, den)
            nv, nb = bn * (sm - S[1]) / sden, (S[0] * a * a - bn2) / sden
            vs, ws = torch.where(deg, S[2], S[2] - S[5] * nv), torch.where(deg, S[3], S[3] - S[6] * nv)
            b1, b2 = torch.where(deg, S[5], S[5] * nb), torch.where(deg, S[6], S[6] * nb)
            vb, vbs = S[1] * bn + S[2] * S[5] + S[3] * S[6], sm * bn + vs * b1 + ws * b2
            es = (a * e - pt * S[1] + pts * sm + bn * (vb - vbs)) / bs
            return ds, vs, ws, es, b1, b2, vbs

        dl, vl, wl, esl, b1l, b2l, vbl = star(L, al, sl, el, ptl)
        dr, vr, wr, esr, b1r, b2r, vbr = star(R, ar, sr, er, ptr)
        ql, qr = torch.sqrt(torch.clamp(dl, min=0.0)), torch.sqrt(torch.clamp(dr, min=0.0))
        sls, srs = sm - bn.abs() / ql, sm + bn.abs() / qr
        sg, qs = torch.sign(bn), ql + qr
        vss = (ql * vl + qr * vr + (b1r - b1l) * sg) / qs
        wss = (ql * wl + qr * wr + (b2r - b2l) * sg) / qs
        b1ss = (ql * b1r + qr * b1l + ql * qr * (vr - vl) * sg) / qs
        b2ss = (ql * b2r + qr * b2l + ql * qr * (wr - wl) * sg) / qs
        vbss = sm * bn + vss * b1ss + wss * b2ss
        ell, err = esl - ql * (vbl - vbss) * sg, esr + qr * (vbr - vbss) * sg
        usl = [dl, dl * sm, dl * vl, dl * wl, esl, b1l, b2l]
        usr = [dr, dr * sm, dr * vr, dr * wr, esr, b1r, b2r]
        ull = [dl, dl * sm, dl * vss, dl * wss, ell, b1ss, b2ss]
        urr = [dr, dr * sm, dr * vss, dr * wss, err, b1ss, b2ss]
        double = bn2 > 1e-12 * (ptl + ptr)
        out = []
        for q in range(7):
            fl, fr = FL[q] + sl * (usl[q] - UL[q]), FR[q] + sr * (usr[q] - UR[q])
            fll = torch.where(double, fl + sls * (ull[q] - usl[q]), fl)
            frr = torch.where(double, fr + srs * (urr[q] - usr[q]), fr)
            m = torch.where(sm > 0, fll, torch.where(sm < 0, frr, 0.5 * (fll + frr)))
            m = torch.where(sls > 0, fl, torch.where(srs < 0, fr, m))
            out.append(torch.where(sl >= 0, FL[q], torch.where(sr <= 0, FR[q], m)))
        return out

    # ---- edge EMFs from the face EMFs, upwinded with the mass fluxes
    def edges(self, f, em):
        e = [None, None, None]
        for c in range(3):
            a, b = (c + 1) % 3, (c + 2) % 3   # the edge's two transverse directions
            if a not in self.dims or b not in self.dims:   # a copy, or no such EMF in 1D
                e[c] = em[a][c] if a in self.dims else em[b][c] if b in self.dims else None
                continue
            axa, axb = 2 - a, 2 - b
            fa, fb, ec = em[a][c], em[b][c], self.ec[c]   # EMF c on a-faces and on b-faces

            def up(flux, left, right):
                return torch.where(flux > 1e-14, left, torch.where(flux < -1e-14, right, 0.5 * (left + right)))

            ga, gb = f[a][0], f[b][0]
            fam, fbm, ecam, ecbm = _sh(fa, -1, axb), _sh(fb, -1, axa), _sh(ec, -1, axa), _sh(ec, -1, axb)
            ecabm = _sh(ecam, -1, axb)
            # derivatives along a, on the cells below and above the edge in b
            l1 = up(_sh(ga, -1, axb), fbm - ecabm, fb - ecbm)
            r1 = up(ga, fbm - ecam, fb - ec)
            l2 = up(_sh(gb, -1, axa), fam - ecabm, fa - ecam)
            r2 = up(gb, fam - ecbm, fa - ec)
            e[c] = 0.25 * (l1 + r1 + l2 + r2 + fbm + fb + fam + fa)
        return e

    # ---- out = g0 a + g1 b - bdt (div F, curl E)
    def update(self, out, g0, A, g1, B, bdt, f, e):
        (uo, bo), (ua, ba), (ub, bb) = out, A, B
        c = self.box()
        div = [0.0] * 5
        for d in self.dims:
            for q in range(5):
                div[q] = div[q] + ((_sh(f[d][q], 1, 2 - d) - f[d][q]) / self.dx[d])[c]
        new = [g0 * ua[q][c] + g1 * ub[q][c] - bdt * div[q] for q in range(5)]
        for d in range(3):
            t1, t2 = (d + 1) % 3, (d + 2) % 3
            curl = 0.0
            if t1 in self.dims:
                curl = curl + (_sh(e[t2], 1, 2 - t1) - e[t2]) / self.dx[t1]
            if t2 in self.dims:
                curl = curl - (_sh(e[t1], 1, 2 - t2) - e[t1]) / self.dx[t2]
            s = self.box((d,) if d in self.dims else ())
            val = g0 * ba[d][s] + g1 * bb[d][s]
            if torch.is_tensor(curl):
                val = val - bdt * curl[s]
            bo[d][s] = val
            if d not in self.dims:   # both faces of the single layer
                bo[d][self.shift(s, d)] = val
        for q in range(5):
            uo[q][c] = new[q]

    def shift(self, s, d):
        return tuple(slice(v.start + 1, v.stop + 1) if q == 2 - d else v for q, v in enumerate(s))

    def bad(self, u, b):
        c = self.box()
        d = u[0][c]
        bc = [q[c] for q in self.centre(b)]
        p = (self.gamma - 1.0) * (u[4][c] - 0.5 * (u[1][c] ** 2 + u[2][c] ** 2 + u[3][c] ** 2) / d
                                  - 0.5 * (bc[0] ** 2 + bc[1] ** 2 + bc[2] ** 2))
        flag = torch.zeros_like(u[0], dtype=torch.bool)
        flag[c] = (d <= self.dfl) | (p <= self.pfl)
        return flag

    def stage(self, S, cur, out, g0, g1, bdt):
        b = S[cur][1]
        f, em = {}, {}
        for d in self.dims:
            f[d], em[d] = self.flux(d, b)
        e = self.edges(f, em)
        self.update(S[out], g0, S[0], g1, S[1], bdt, f, e)
        if self.fofc:
            flag = self.bad(*S[out])
            if bool(flag.any()):   # donor-cell HLLE on the faces of flagged cells, then again
                for d in self.dims:
                    m = flag | _sh(flag, -1, 2 - d)
                    g, gm = self.flux(d, b, donor=True)
                    f[d] = [torch.where(m, x, y) for x, y in zip(g, f[d])]
                    em[d] = {c: torch.where(m, gm[c], em[d][c]) for c in gm}
                self.update(S[out], g0, S[0], g1, S[1], bdt, f, self.edges(f, em))
        self.fill(*S[out])
        self.prim(*S[out])

    def advance(self, u, b, steps, nst):
        self.u, self.b = u, b
        S = [(u, b), (u.clone(), [q.clone() for q in b])]
        self.fill(u, b)
        self.prim(u, b)
        t, mdt = 0.0, self.cfl_dt()
        table = {2: [(1.0, 0.0, 1.0, 0, 1), (0.5, 0.5, 0.5, 1, 0)],
                 3: [(1.0, 0.0, 1.0, 0, 1), (0.75, 0.25, 0.25, 1, 1), (1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0, 1, 0)]}[nst]
        for _ in range(steps):
            dt = self.r["cfl"] * mdt
            for g0, g1, beta, cur, out in table:
                self.stage(S, cur, out, g0, g1, beta * dt)
            t += dt
            mdt = self.cfl_dt()
        u[5] = self.w[0] * (self.w[4] / self.w[0] ** self.gamma)
        return t
