"""Performance cases of the DFSPH solver: the calls that a simulation makes, over the sizes it makes them at.

A case is a scene (fluid lattice, walls, options) and the call that is made on it:

  step        SPH::DFSPHCUDA::step() through HostSolver.step(): one whole time step, tolerances 0.1 %, CFL time step
  search      dfsph_neighbor_search: sort, reorder, neighbor lists
  divergence  dfsph_divergence_solve: density, factor, warm start and the divergence iterations
  pressure    density and factor, XSPH + gravity, velocity update and dfsph_pressure_solve
  forces      dfsph_external_forces and dfsph_cfl
  train       dfsph_mlp_train and the parameters read back: fitting the learned warm start

The solver keeps its particles on the device.  What a call leaves there is returned as a mapping that reads a field when
the field is asked for, as a program does: a simulation loop downloads nothing between its steps.
"""
import math

import numpy as np
import torch

import splishsplash_for_cuda_amd as S
from splishsplash_for_cuda_amd import learned, wave_tank

RHO0 = 1000.0
EPS = 1.0e-5


def listed():
    return [
        # the smallest scene of the tests and of the smoke test: launches and the host's two waits per step
        dict(name="step_1600", kind="step", nx=10, ny=16, nz=10, r=0.025, lx=1.0, ly=1.2, lz=0.6, wall=2, packing=1.0),
        # the 16,000-particle dam break of the reference's demo scene
        dict(name="step_16k", kind="step", nx=20, ny=40, nz=20, r=0.025, lx=4.0, ly=3.0, lz=1.5, wall=2, packing=1.0),
        # the 1M dam break, walls sampled at spacing r (about 47 wall neighbors on the floor)
        dict(name="step_1m", kind="step", nx=128, ny=128, nz=64, r=0.01, lx=6.0, ly=3.0, lz=2.0, wall=1, packing=1.0),
        # the wave tank at half its resolution: piston, floating box, open boundary
        dict(name="step_tank_260k", kind="step", tank=True, r=0.016, length=10.0, depth=0.9),
        # a training-scene dam break with the learned warm start on every step (features and network)
        dict(name="step_learned_150k", kind="step", nx=57, ny=51, nz=53, r=0.0125, lx=3.0, ly=1.9, lz=1.7, wall=2,
             packing=1.0, learned=True),
        # the 4M dam break: the largest search
        dict(name="search_4m", kind="search", nx=256, ny=128, nz=128, r=0.0075, lx=6.0, ly=3.0, lz=2.0, wall=2, packing=1.0),
        # a pool under spray: sparse blocks, ragged counts, both list forms
        dict(name="search_spray_200k", kind="search", nx=75, ny=13, nz=107, r=0.0125, lx=1.95, ly=1.6, lz=2.8, wall=2,
             packing=0.95, spray=97001),
        # the 4M dam break's divergence solve
        dict(name="divergence_4m", kind="divergence", nx=256, ny=128, nz=128, r=0.0075, lx=6.0, ly=3.0, lz=2.0, wall=2, packing=1.0),
        # two liquids: particles of unlike mass
        dict(name="divergence_masses_130k", kind="divergence", nx=51, ny=50, nz=51, r=0.0125, lx=3.1, ly=1.9, lz=1.4, wall=2,
             packing=1.0, masses=True),
        # fluid near its rest density, odd extents: the density solver has work to do
        dict(name="pressure_700k", kind="pressure", nx=97, ny=71, nz=101, r=0.01, lx=4.0, ly=2.2, lz=2.06, wall=2, packing=0.93),
        # viscosity and time step of a 0.5M block
        dict(name="forces_500k", kind="forces", nx=80, ny=79, nz=79, r=0.01, lx=4.0, ly=2.4, lz=1.7, wall=2, packing=0.97),
        # a few mini-batches of the warm-start training
        dict(name="train_4096", kind="train", samples=200000, batch=4096, steps=20),
    ]


def draw(rng):
    kind = rng.choice(["step", "step", "search", "divergence", "pressure", "forces", "train"])
    if kind == "train":
        return dict(kind="train", samples=int(math.exp(rng.uniform(math.log(20000), math.log(500000)))),
                    batch=64 * int(math.exp(rng.uniform(math.log(4), math.log(256)))), steps=rng.randint(5, 40))
    if kind == "step" and rng.random() < 0.2:
        return dict(kind="step", tank=True, r=rng.uniform(0.016, 0.03), length=rng.uniform(4.0, 10.0), depth=rng.uniform(0.4, 0.9))
    top = {"step": 1.0e6, "search": 3.0e6}.get(kind, 2.0e6)
    n = math.exp(rng.uniform(math.log(1500), math.log(top)))
    ax, az = rng.uniform(0.5, 2.0), rng.uniform(0.5, 2.0)
    ny = max(6, round((n / (ax * az)) ** (1.0 / 3.0)))
    nx, nz = max(5, round(ax * ny)), max(5, round(az * ny))
    r = rng.uniform(0.0075, 0.025)
    d = 2.0 * r
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, r=r, lx=(rng.uniform(1.3, 2.5) * nx + 2) * d,
             ly=(1.5 * ny + 4) * d, lz=(rng.uniform(1.0, 1.3) * nz + 2) * d, wall=rng.choice([1, 2, 2]),
             packing=rng.uniform(0.92, 0.98) if kind in ("pressure", "forces") else 1.0)
    if kind == "search" and rng.random() < 0.4:
        c["spray"] = int(n * rng.uniform(0.1, 0.8))
    if kind == "divergence" and rng.random() < 0.4:
        c["masses"] = True
    if kind == "step" and rng.random() < 0.25:
        c["learned"] = True
    return c


# ---- inputs ------------------------------------------------------------------

def _walls(lx, ly, lz, spacing):
    """Lattice points on the faces of the box [0, l]."""
    l = (lx, ly, lz)
    m = [max(int(round(v / spacing)), 1) for v in l]
    ax = [l[a] * np.arange(m[a] + 1) / m[a] for a in range(3)]
    out = []
    for a in range(3):
        b, c = [k for k in range(3) if k != a]
        # the edges shared with the faces before are left out
        sb = slice(None) if b > a else slice(1, -1)
        sc = slice(None) if c > a else slice(1, -1)
        B, C = np.meshgrid(ax[b][sb], ax[c][sc], indexing="ij")
        for v in (0.0, l[a]):
            p = np.empty((B.size, 3))
            p[:, a], p[:, b], p[:, c] = v, B.ravel(), C.ravel()
            out.append(p)
    return np.concatenate(out).astype(np.float32)


def _motion(x, seed, speed):
    """A smooth flow with eddies and compression over the scene, and a little noise."""
    rng = np.random.default_rng(seed + 77)
    span = np.maximum(x.max(0) - x.min(0), 1e-3)
    v = np.empty_like(x)
    for a in range(3):
        k = rng.uniform(2.0, 5.0, 3) / span
        v[:, a] = speed * np.sin(x @ k.astype(np.float32) + np.float32(rng.uniform(0.0, 6.28)))
    return v + rng.standard_normal(x.shape, dtype=np.float32) * np.float32(0.02 * speed)


def _scene(case, seed):
    """fluid, walls, velocities, masses (or None) of a dam break, as float32 arrays."""
    rng = np.random.default_rng(seed)
    r, d = case["r"], 2.0 * case["r"]
    s = d * case["packing"]
    g = np.meshgrid(*[np.arange(case[k], dtype=np.float32) for k in ("nx", "ny", "nz")], indexing="ij")
    x = np.stack([a.ravel() for a in g], 1) * np.float32(s) + np.float32(d)
    x += (rng.random(x.shape, dtype=np.float32) - np.float32(0.5)) * np.float32(0.1 * r)
    if case.get("spray"):
        # droplets (small jittered lattice balls) over the block, thinning upward
        o = np.stack(np.meshgrid(*[np.arange(-3, 4)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
        lo = x[:, 1].max() + d
        drops, left = [], case["spray"]
        while left > 0:
            c = np.array([rng.uniform(4 * d, case["lx"] - 4 * d), lo + (case["ly"] - 4 * d - lo) * rng.random() ** 2,
                          rng.uniform(4 * d, case["lz"] - 4 * d)])
            b = o[(o * o).sum(1) <= rng.uniform(0.0, 9.0)] * s + c
            b = b[:left] + rng.uniform(-0.3 * r, 0.3 * r, (min(len(b), left), 3))
            drops.append(b.astype(np.float32))
            left -= len(b)
        x = np.concatenate([x] + drops)
        x = x[rng.permutation(len(x))]
    x = np.ascontiguousarray(x)
    m = None
    if case.get("masses"):
        m = (0.8 * d ** 3 * RHO0 * np.where(rng.random(len(x)) < 0.5, 1.0, 0.9)).astype(np.float32)
    return x, _walls(case["lx"], case["ly"], case["lz"], case["wall"] * r), _motion(x, seed, 0.5), m


def _tank(case, seed):
    t = wave_tank.build(r=case["r"], length=case["length"], depth=case["depth"], seed=seed)
    return t, _motion(t.fluid, seed, 0.2)


def _dataset(case, seed):
    """Features and targets of the warm start's sizes, and initial weights."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    mean = np.array([-0.05, 0.0, 0.8, 0.1, -0.002, -0.005, 0.1, 0.0, 0.0, 0.0, 0.7, 0.95])
    std = np.array([0.1, 0.01, 0.15, 0.08, 0.003, 0.01, 0.15, 0.1, 0.1, 0.1, 0.03, 0.1])
    z = rng.standard_normal((n, 12))
    w = rng.standard_normal((12, 2)) / 3.0
    t = np.tanh(z @ w) * [0.004, 0.001] + rng.standard_normal((n, 2)) * [4e-4, 1e-4]
    p = []
    for s in ((64, 12), (64,), (64, 64), (64,), (64, 64), (64,), (2, 64), (2,)):
        lim = math.sqrt(6.0 / sum(s)) if len(s) == 2 else 0.0
        p.append(rng.uniform(-lim, lim, s).ravel())
    return (z * std + mean).astype(np.float32), t.astype(np.float32), np.concatenate(p).astype(np.float32)


def _params(case):
    return S.default_params(
        particle_radius=case["r"], dt=0.001, use_cfl=1, cfl_factor=1.0, dt_min=1e-4, dt_max=5e-3, max_error=0.1,
        max_error_v=0.1, max_neighbors=128,
        warm_start_mode=S.WARMSTART_LEARNED if case.get("learned") else S.WARMSTART_REFERENCE,
        learned_gate=S.LEARNED_ALWAYS)


# ---- the calls -----------------------------------------------------------------

class Fields(dict):
    """What a call left on the device, by name: reading an entry downloads it.

    Fields of the fluid come in the order of the particles' ids, the others (search) in device order.  The mapping keeps
    the state alive that owns the solver."""

    def __init__(self, state, by_id, raw, values):
        super().__init__({k: None for k in list(by_id) + list(raw)})
        self.update(values)
        self._state, self._solver = state, state["solver"]
        self._by_id, self._raw, self._order = by_id, raw, None

    def __getitem__(self, name):
        if name in self._by_id:
            if self._order is None:
                self._order = np.argsort(self._solver.download(S.FIELD_ID), kind="stable")
            return self._solver.download(self._by_id[name])[self._order]
        if name in self._raw:
            return self._raw[name]()
        return super().__getitem__(name)


def prepare(case, seed):
    if case["kind"] == "train":
        x, t, w = _dataset(case, seed)
        s = S.Solver()
        s.mlp_set_params(w)
        s.mlp_dataset_upload(x, t)
        s.mlp_fit_normalization()
        return dict(case=case, solver=s, seed=seed & 0xffff)
    p = _params(case)
    if case.get("tank"):
        t, v = _tank(case, seed)
        hs = wave_tank.make_solver(t, p)
        hs.view.upload_field(S.FIELD_VEL, v)
        return dict(case=case, host=hs, solver=hs.view)
    x, walls, v, m = _scene(case, seed)
    if case["kind"] == "step":
        hs = S.HostSolver(p, walls, x, v)
        if case.get("learned"):
            learned.attach(hs.view)
        return dict(case=case, host=hs, solver=hs.view)
    s = S.Solver(p)
    s.upload_boundary(walls)
    s.upload_fluid(x, v, m)
    if case["kind"] != "search":
        s.neighbor_search()
    if case["kind"] == "forces":
        s.compute_density_factor()
    return dict(case=case, solver=s)


def run(state):
    case, s = state["case"], state["solver"]
    kind = case["kind"]
    if kind == "step":
        st = state["host"].step()
        raw = {}
        if case.get("tank"):
            def box():
                b, f, t = s.rigid_body(1)
                return {"force": f.astype(np.float32), "torque": t.astype(np.float32),
                        "velocity": np.array(b.velocity[:], np.float32), "position": np.array(b.position[:], np.float32)}
            raw = {"box": box}
        return Fields(state, {"position": S.FIELD_POS, "velocity": S.FIELD_VEL, "density": S.FIELD_DENSITY}, raw,
                      {"iterations": [st.iters_v, st.iters], "n": st.n_fluid, "dt": st.h})
    if kind == "search":
        s.neighbor_search()
        raw = {"id": lambda: s.download(S.FIELD_ID), "fluid": lambda: s.download(S.FIELD_NBR_FLUID),
               "walls": lambda: s.download(S.FIELD_NBR_BOUNDARY), "position": lambda: s.download(S.FIELD_POS)}
        if case["nx"] * case["ny"] * case["nz"] + case.get("spray", 0) <= 400000:
            raw["lists"] = lambda: s.neighbors()[2]
        return Fields(state, {}, raw, {})
    if kind == "divergence":
        it, err = s.divergence_solve()
        return Fields(state, {"velocity": S.FIELD_VEL, "density": S.FIELD_DENSITY, "factor": S.FIELD_FACTOR,
                          "kappaV": S.FIELD_KAPPAV}, {}, {"iterations": it, "error": err})
    if kind == "pressure":
        s.compute_density_factor()
        s.external_forces()
        s.update_vel()
        it, err = s.pressure_solve()
        return Fields(state, {"velocity": S.FIELD_VEL, "density": S.FIELD_DENSITY, "factor": S.FIELD_FACTOR}, {},
                      {"iterations": it})
    if kind == "forces":
        s.external_forces()
        s.cfl(wait=False)
        return Fields(state, {"acceleration": S.FIELD_ACC}, {"dt": lambda: float(s.get_time()[1])}, {})
    first, last = s.mlp_train(case["steps"], case["batch"], 2e-3, state["seed"])
    w, _ = s.mlp_get_params()
    return {"loss_first": first, "loss_last": last, "params": w}


def work(case):
    """Each particle's state once in and once out, and the pair sums that cannot be avoided (about 30 neighbors)."""
    if case["kind"] == "train":
        # forward and backward of 9,152 weights, 56 bytes of features and targets a sample
        k = case["steps"] * case["batch"]
        return {"bytes": k * 56 + 2 * 4 * 9282, "flops": 6.0 * 9152 * k}
    if case.get("tank"):
        d = 2.0 * case["r"]
        n = (case["length"] - 0.15) * case["depth"] * 1.0 / d ** 3
    else:
        n = case["nx"] * case["ny"] * case["nz"] + case.get("spray", 0)
    pairs = 30.0 * n
    # bytes a particle, flops a pair (distance 8, gradient 10, update or source 8), sweeps
    b, f = {
        "step": (2 * (16 + 12 + 4 * 6), 8 + 13 * 26),      # state in and out; search and 13 sweeps
        "search": (2 * (16 + 12 + 4 * 6) + 4 * 30, 8),     # reordered state and one index a neighbor
        "divergence": (16 + 12 + 4 + 12 + 4 * 4 + 4 * 30, 8 * 26),
        "pressure": (16 + 12 + 4 + 12 + 4 * 4 + 4 * 30, 8 * 26),
        "forces": (16 + 12 + 4 + 12 + 4 * 30, 26),
    }[case["kind"]]
    return {"bytes": float(b * n), "flops": f * pairs}


# ---- the same in 64 bits ---------------------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs(a, b, h):
    """Index pairs (i, j) with |a_i - b_j| < h: a grid of edge h over b, rows of three cells."""
    lo = torch.minimum(a.min(0).values, b.min(0).values) - 1.5 * h
    ca, cb = ((a - lo) / h).long(), ((b - lo) / h).long()
    dim = torch.maximum(ca.max(0).values, cb.max(0).values) + 2
    nx, ny, nz = (int(v) for v in dim)
    kb = cb[:, 0] + nx * (cb[:, 1] + ny * cb[:, 2])
    order = torch.argsort(kb)
    start = torch.zeros(nx * ny * nz + 1, dtype=torch.int64, device=a.device)
    start[1:] = torch.cumsum(torch.bincount(kb, minlength=nx * ny * nz), 0)
    I, J = [], []
    for c0 in range(0, len(a), 1 << 18):
        c = ca[c0:c0 + (1 << 18)]
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                k = c[:, 0] + nx * ((c[:, 1] + dy) + ny * (c[:, 2] + dz))
                s, e = start[k - 1], start[k + 2]
                cnt = e - s
                i = torch.repeat_interleave(torch.arange(len(c), device=a.device), cnt)
                off = torch.arange(len(i), device=a.device) - torch.repeat_interleave(torch.cumsum(cnt, 0) - cnt, cnt)
                j = order[s[i] + off]
                i = i + c0
                near = ((a[i] - b[j]) ** 2).sum(1) < h * h
                I.append(i[near])
                J.append(j[near])
    return torch.cat(I), torch.cat(J)


class _Exact:
    """One DFSPH step in 64 bits on pair lists, warm starts zero (a freshly uploaded fluid)."""

    def __init__(self, r, x, v, m, walls, bodies=(), gravity=-9.81, dt=1e-3):
        t = lambda a: torch.as_tensor(np.asarray(a), device=_dev()).double()  # noqa: E731
        self.r, self.hk, self.h, self.nu = r, 4.0 * r, dt, 0.01
        self.x, self.v = t(x), t(v)
        self.n = len(self.x)
        m0 = 0.8 * (2.0 * r) ** 3 * RHO0
        self.m = torch.full((self.n,), m0, dtype=torch.float64, device=_dev()) if m is None else t(m)
        self.g = torch.tensor([0.0, gravity, 0.0], dtype=torch.float64, device=_dev())
        self.kc = 8.0 / (math.pi * self.hk ** 3)
        # walls, then the bodies' particles; psi of each set over those before it and itself
        bx, psi = t(walls), None
        psi = self._psi(bx)
        bv = torch.zeros_like(bx)
        self.body = torch.zeros(len(bx), dtype=torch.int64, device=_dev())
        for k, (pts, center, vel) in enumerate(bodies):
            p = torch.as_tensor(np.asarray(pts), device=_dev()).double() + torch.tensor(center, dtype=torch.float64, device=_dev())
            p = p.float().double()
            bx = torch.cat([bx, p])
            psi = torch.cat([psi, self._psi(bx)[-len(p):]])
            bv = torch.cat([bv, torch.tensor(vel, dtype=torch.float64, device=_dev()).expand(len(p), 3)])
            self.body = torch.cat([self.body, torch.full((len(p),), k + 1, dtype=torch.int64, device=_dev())])
        self.bx, self.bv, self.psi = bx, bv, psi
        self.i, self.j = _pairs(self.x, self.x, self.hk)
        keep = self.i != self.j
        self.i, self.j = self.i[keep], self.j[keep]
        self.ib, self.jb = _pairs(self.x, bx, self.hk)
        self.dx = self.x[self.i] - self.x[self.j]
        self.db = self.x[self.ib] - bx[self.jb]
        q, qb = self.dx.norm(dim=1) / self.hk, self.db.norm(dim=1) / self.hk
        self.w, self.wb = self._W(q), self._W(qb)
        self.gf, self.gb = self._G(q, self.dx), self._G(qb, self.db)
        self.count = torch.bincount(self.i, minlength=self.n) + torch.bincount(self.ib, minlength=self.n)
        self.reaction = torch.zeros_like(bx)

    def _W(self, q):
        return self.kc * torch.where(q <= 0.5, 6 * q ** 3 - 6 * q ** 2 + 1, 2 * (1 - q) ** 3)

    def _G(self, q, d):
        l = 6.0 * self.kc / self.hk
        r = torch.clamp(q * self.hk, min=1e-30)
        c = torch.where(q <= 0.5, l * (3 * q * q - 2 * q), -l * (1 - q) ** 2) / r
        return torch.where(r > 1e-6, c, torch.zeros_like(c))[:, None] * d

    def _psi(self, b):
        i, j = _pairs(b, b, self.hk)
        far = i != j
        i, j = i[far], j[far]
        s = torch.full((len(b),), self.kc, dtype=torch.float64, device=b.device)
        s.index_add_(0, i, self._W((b[i] - b[j]).norm(dim=1) / self.hk))
        return RHO0 / s

    def _sum(self, i, values):
        return torch.zeros((self.n,) + values.shape[1:], dtype=torch.float64, device=values.device).index_add_(0, i, values)

    def density(self):
        m, psi = self.m[self.j], self.psi[self.jb]
        self.rho = self.m * self.kc + self._sum(self.i, m * self.w) + self._sum(self.ib, psi * self.wb)
        gf, gb = m[:, None] * self.gf, psi[:, None] * self.gb
        s2 = self._sum(self.i, (gf * gf).sum(1)) + self._sum(self.ib, (gb * gb).sum(1))
        s = self._sum(self.i, gf) + self._sum(self.ib, gb)
        self.alpha = -(1.0 / self.h) / torch.clamp(s2 + (s * s).sum(1), min=EPS)

    def _rate(self):
        return (self._sum(self.i, self.m[self.j] * ((self.v[self.i] - self.v[self.j]) * self.gf).sum(1)) +
                self._sum(self.ib, self.psi[self.jb] * ((self.v[self.ib] - self.bv[self.jb]) * self.gb).sum(1)))

    def _apply(self, k, step):
        s = k[self.i] + k[self.j]
        s = torch.where(s.abs() > EPS, s, torch.zeros_like(s)) * self.m[self.j]
        kb = torch.where(k.abs() > EPS, k, torch.zeros_like(k))[self.ib] * self.psi[self.jb]
        f = kb[:, None] * self.gb
        self.v = self.v + step * (self._sum(self.i, s[:, None] * self.gf) + self._sum(self.ib, f))
        self.reaction.index_add_(0, self.jb, -self.m[self.ib][:, None] * f)

    def _loop(self, source, alpha, step, eta, floor):
        """Jacobi iterations while ((error > eta) or (it < floor)) and it < 100; the increments' sum and the count."""
        k = source() * alpha
        total, it, err = (torch.zeros_like(k) if floor == 3 else k.clone()), 0, 0.0
        while (err > eta or it < floor) and it < 100:
            self._apply(k, step)
            if floor == 3:
                total = total + k
            s = source()
            k = s * alpha
            if floor == 2:
                total = total + k
            err = float(s.sum()) / self.n
            it += 1
        return total, it, err

    def divergence(self):
        self.density()
        source = lambda: torch.where(self.count < 20, torch.zeros_like(self.rho), torch.clamp(self._rate(), min=0.0))  # noqa: E731
        self.kappaV, self.iters_v, self.err_v = self._loop(source, self.alpha, self.h, 0.001 * RHO0 / self.h, 3)

    def forces(self):
        c = (1.0 / self.h) * self.nu * self.m[self.j] / self.rho[self.j] * self.w
        self.acc = self.g - self._sum(self.i, c[:, None] * (self.v[self.i] - self.v[self.j]))

    def cfl(self):
        top = float(((self.v + self.h * self.acc) ** 2).sum(1).max())
        self.hf = min(max(0.4 * 2.0 * self.r / math.sqrt(top), 1e-4), 5e-3)

    def pressure(self):
        self.v = self.v + self.h * self.acc
        self.alpha = self.alpha / self.hf
        source = lambda: torch.clamp(self.rho + self.hf * self._rate() - RHO0, min=0.0)  # noqa: E731
        _, self.iters, self.err = self._loop(source, self.alpha, self.hf, 0.001 * RHO0, 2)


def _exact_train(case, seed):
    """Adam on the normalised loss in 64 bits, the batches drawn as dfsph_mlp_train draws them."""
    x, t, w = _dataset(case, seed)
    dev, n = _dev(), len(x)

    def norm(a):
        a = torch.as_tensor(a, device=dev).double()
        return (a - a.mean(0)) / a.std(0, unbiased=False)

    x, t = norm(x), norm(t)
    p = torch.as_tensor(w, device=dev).double().requires_grad_()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    shapes = ((64, 12), (64,), (64, 64), (64,), (64, 64), (64,), (2, 64), (2,))
    steps, batch = case["steps"], case["batch"]
    losses = []
    mask = (1 << 64) - 1
    for it in range(steps):
        s = ((seed & 0xffff) << 32) ^ ((it * 0x632be59bd9b4e019) & mask)
        with np.errstate(over="ignore"):
            z = np.uint64(s) + np.uint64(0x9e3779b97f4a7c15) * np.arange(1, batch + 1, dtype=np.uint64)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
            z = (z ^ (z >> np.uint64(31))) % np.uint64(n)
        i = torch.as_tensor(z.astype(np.int64), device=dev)
        a, at = x[i], 0
        for k, shape in enumerate(shapes):
            q = p[at:at + math.prod(shape)].reshape(shape)
            at += math.prod(shape)
            if len(shape) == 2:
                y = a @ q.T
            else:
                y = y + q
                a = torch.nn.functional.silu(y)
        loss = 0.5 * ((y - t[i]) ** 2).sum() / batch
        g, = torch.autograd.grad(loss, p)
        losses.append(float(loss.detach()))
        with torch.no_grad():
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            lr = 2e-3 * (1.0 - 0.9 * it / max(steps - 1, 1))
            p -= lr * (m / (1.0 - 0.9 ** (it + 1))) / (torch.sqrt(v / (1.0 - 0.999 ** (it + 1))) + 1e-8)
    return {"loss_first": losses[0], "loss_last": losses[-1], "params": p.detach()}


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "search":
        return None
    if case.get("tank"):
        t, v = _tank(case, seed)
        w = 2.0 * math.pi / t.piston["period"]
        e = _Exact(case["r"], t.fluid, v, None, t.walls,
                   [(t.bodies[0][1], t.piston["position"], (t.piston["amplitude"] * w, 0.0, 0.0)),
                    (t.bodies[1][1], t.box["position"], (0.0, 0.0, 0.0))])
    else:
        x, walls, v, m = _scene(case, seed)
        e = _Exact(case["r"], x, v, m, walls)
    kind = case["kind"]
    if kind == "divergence":
        e.divergence()
        return {"velocity": e.v, "density": e.rho, "factor": e.alpha, "kappaV": e.kappaV, "iterations": None, "error": e.err_v}
    if kind == "forces":
        e.density()
        e.forces()
        e.cfl()
        return {"acceleration": e.acc, "dt": e.hf}
    if kind == "pressure":
        e.density()
        e.forces()
        e.hf = e.h
        e.pressure()
        return {"velocity": e.v, "density": e.rho, "factor": e.alpha, "iterations": None}
    e.divergence()
    e.forces()
    e.cfl()
    e.pressure()
    out = {"position": e.x + e.h * e.v, "velocity": e.v, "density": e.rho, "iterations": [None, None], "n": None, "dt": e.h}
    if case.get("tank"):
        f = e.reaction[e.body == 2]
        arm = e.bx[e.body == 2] - torch.tensor(t.box["position"], dtype=torch.float64, device=_dev())
        force = f.sum(0)
        vel = e.h * (force / t.box["mass"] + e.g)
        out["box"] = {"force": force, "torque": torch.linalg.cross(arm, f).sum(0), "velocity": vel,
                      "position": torch.tensor(t.box["position"], dtype=torch.float64, device=_dev()) + e.h * vel}
    return out
