"""What a user of this library has it do, as timed cases.

Each case is a pass of a user's program through the Python API: lattices are
created, given their geometry and their initial state in `prepare` (except
where a whole short job is the case), `run` advances them and takes the
results that such a program takes, and `exact` computes the same results with
plain torch in 64 bits, without the library.

Moments and velocities come back at the precision at which the lattice holds
them: the 64-bit arrays of the API for 32-bit storage, and the 16-bit values
of the storage format for FP16 and BF16 lattices.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mr-lbm_amd"))

import mrlbm  # noqa: E402
from mrlbm import geometry, serve  # noqa: E402

STORE = {"fp32": mrlbm.STORE_FP32, "fp16": mrlbm.STORE_FP16, "bf16": mrlbm.STORE_BF16}
WORD = {"fp32": 4, "fp16": 2, "bf16": 2}
CAVITY_EDGES = (32, 48, 64, 96, 128)
EXACT_LU_MAX = 17e9  # lattice updates that `exact` takes on (about 20 s at 256^3)


def listed():
    return [
        # one time step and the probe points of a small cavity: the time
        # series a user records; launches and latency are all of it
        dict(name="probe_series_32", kind="probe", nx=32, ny=32, nz=32, storage="fp32", points=16),
        # the 64^3 Re = 100 cavity advanced by 1000 steps, its convergence
        # residual and its fields: the commonest small run
        dict(name="cavity_64", kind="cavity", nx=64, ny=64, nz=64, storage="fp32", steps=1000),
        # a short parameter-study job from start to end: create, initial
        # fields from host arrays, 400 steps, density and velocity, release
        dict(name="job_96x72x80", kind="job", nx=96, ny=72, nz=80, storage="fp32", steps=400),
        # the headline lattice: Taylor-Green vortex at 256^3, FP32 moments,
        # fields and kinetic energy every 500 steps
        dict(name="tgv_256_fp32", kind="tgv", nx=256, ny=256, nz=256, storage="fp32", steps=500),
        # Taylor-Green vortex with FP16 moments on a larger non-cubic lattice
        dict(name="tgv_256x192x160_fp16", kind="tgv", nx=256, ny=192, nz=160, storage="fp16", steps=1000),
        # duct with voxelised spheres, BF16 moments, extents that are odd
        # multiples of the tile
        dict(name="duct_200x72x104_bf16", kind="duct", nx=200, ny=72, nz=104, q=19, storage="bf16", steps=1000,
             spheres=6),
        # D3Q27 forced duct, FP32 moments
        dict(name="duct_q27_256x128x128_fp32", kind="duct", nx=256, ny=128, nz=128, q=27, storage="fp32", steps=500,
             spheres=0),
        # the largest: D3Q27 duct 512x256x256 with FP16 moments, a window of
        # flow statistics (mean flow sampled every 10 steps) and the mean flow
        dict(name="stats_q27_512x256x256_fp16", kind="stats", nx=512, ny=256, nz=256, q=27, storage="fp16",
             samples=10, every=10),
        # in-situ monitoring of a channel every 20 steps: mass, energy,
        # non-finite check, moment means and convergence residual
        dict(name="monitor_192x160x128", kind="monitor", nx=192, ny=160, nz=128, storage="fp32", steps=20),
        # twelve lid-driven cavities of different sizes in one batch
        dict(name="batch_12_cavities", kind="batch", edges="32,32,32,32,32,48,48,48,64,64,96,128", storage="fp32",
             steps=400),
        # a served stream of duct requests with FP16 moments, fields returned
        dict(name="serve_6_ducts_fp16", kind="serve", requests=6, ny_max=64, nx_max=128, steps=400, pick=7,
             storage="fp16"),
    ]


def _extent(rng, lo, hi):
    """A multiple of 8, spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, 8 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 8)))


def draw(rng):
    kind = rng.choice(["probe", "cavity", "job", "tgv", "tgv", "duct", "duct", "stats", "monitor", "batch", "serve"])
    storage = rng.choice(["fp32", "fp16", "bf16"])

    def shape(lo, hi, most):
        while True:
            s = [_extent(rng, lo, hi) for _ in range(3)]
            if s[0] * s[1] * s[2] <= most:
                return dict(nx=s[0], ny=s[1], nz=s[2])

    if kind == "probe":
        return dict(kind=kind, storage="fp32", points=rng.choice([1, 5, 16, 64, 200]), **shape(16, 64, 1 << 18))
    if kind == "cavity":
        return dict(kind=kind, storage=storage, steps=50 * rng.randint(4, 30), **shape(24, 128, 1 << 20))
    if kind == "job":
        return dict(kind=kind, storage=storage, steps=rng.randint(100, 900), **shape(32, 144, 1 << 20))
    if kind == "tgv":
        return dict(kind=kind, storage=storage, steps=rng.randint(200, 600), **shape(48, 256, 1 << 23))
    if kind == "duct":
        return dict(kind=kind, storage=storage, q=rng.choice([19, 27]), steps=rng.randint(100, 800),
                    spheres=rng.randint(0, 8), **shape(40, 256, 3 << 20))
    if kind == "stats":
        return dict(kind=kind, storage=storage, q=rng.choice([19, 27]), samples=rng.randint(4, 12),
                    every=rng.randint(5, 20), **shape(64, 320, 12 << 20))
    if kind == "monitor":
        return dict(kind=kind, storage=storage, steps=rng.randint(5, 40), **shape(48, 256, 1 << 23))
    if kind == "batch":
        n = rng.randint(3, 12)
        edges = sorted(rng.choice(CAVITY_EDGES) for _ in range(n))
        return dict(kind=kind, storage=storage, edges=",".join(str(e) for e in edges), steps=50 * rng.randint(3, 8))
    return dict(kind="serve", requests=rng.randint(2, 8), ny_max=16 * rng.randint(3, 5), nx_max=16 * rng.randint(6, 10),
                steps=rng.randint(150, 400), pick=rng.randint(1, 10**6), storage=storage)


# ---------------------------------------------------------------------------
# inputs: physical parameters drawn from the seed


def _shape(c):
    return c["nx"], c["ny"], c["nz"]


def _spheres(rng, shape, n):
    """n spheres inside the duct, of radii as the served ducts have them."""
    out = []
    for _ in range(n):
        r = rng.uniform(3.0, max(3.5, min(shape[1], shape[2]) / 6.0))
        out.append(((rng.uniform(0, shape[0]), rng.uniform(0, shape[1]), rng.uniform(0, shape[2])), r))
    return out


def _edges(c):
    return [int(e) for e in c["edges"].split(",")]


def _inputs(c, seed):
    """Physical parameters of the case: what both `prepare` and `exact` start from."""
    rng = random.Random(f"{c['kind']} {seed}")
    k = c["kind"]
    if k in ("probe", "cavity"):
        lid = rng.uniform(0.04, 0.06)
        d = dict(lid=lid, tau=0.5 + 3.0 * lid * c["nz"] / rng.uniform(80.0, 120.0))
        if k == "probe":
            d["points"] = np.array([[rng.randrange(e) for e in _shape(c)] for _ in range(c["points"])], np.int32)
        return d
    if k == "tgv":
        return dict(u0=rng.uniform(0.04, 0.06), tau=rng.uniform(0.53, 0.56))
    if k == "job":
        modes = [([rng.randint(1, 3) for _ in range(3)], [rng.uniform(0, 2 * math.pi) for _ in range(3)],
                  rng.uniform(0.005, 0.02)) for _ in range(3)]
        return dict(modes=modes, tau=rng.uniform(0.53, 0.6))
    if k == "duct":
        return dict(g=10 ** rng.uniform(-5.5, -4.5), tau=0.5 + 3.0 * rng.uniform(0.03, 0.1),
                    spheres=_spheres(rng, _shape(c), c["spheres"]))
    if k == "stats":
        return dict(g=10 ** rng.uniform(-5.3, -4.7), tau=0.5 + 3.0 * rng.uniform(0.03, 0.1), spheres=[])
    if k == "monitor":
        return dict(g=10 ** rng.uniform(-6, -5), tau=0.5 + 3.0 * rng.uniform(0.02, 0.06), u=rng.uniform(0.03, 0.06),
                    spheres=[])
    if k == "batch":
        lid = 0.05
        return dict(lid=lid, tau=[0.5 + 3.0 * lid * n / rng.uniform(50.0, 400.0) for n in _edges(c)])
    return dict(gx=[10 ** rng.uniform(-5.5, -4.5) for _ in range(c["requests"])],
                nu=[rng.uniform(0.03, 0.1) for _ in range(c["requests"])])


def _job_fields(c, p, xp):
    """Initial density and velocity of the short job: a few Fourier modes."""
    nx, ny, nz = _shape(c)
    if xp is np:
        grid = np.meshgrid(*[2 * np.pi * np.arange(e, dtype=np.float64) / e for e in (nx, ny, nz)], indexing="ij")
    else:
        grid = torch.meshgrid(*[2 * math.pi * torch.arange(e, dtype=torch.float64, device="cuda") / e
                                for e in (nx, ny, nz)], indexing="ij")
    x, y, z = grid
    rho, u, v, w = 1.0 + 0 * x, 0 * x, 0 * x, 0 * x
    for (a, b, d), (pa, pb, pd), amp in p["modes"]:
        u = u + amp * xp.sin(b * y + pa) * xp.cos(d * z + pb)
        v = v + amp * xp.sin(d * z + pb) * xp.cos(a * x + pd)
        w = w + amp * xp.sin(a * x + pd) * xp.cos(b * y + pa)
        rho = rho + amp * amp * xp.cos(a * x + pa) * xp.cos(b * y + pb) * xp.cos(d * z + pd)
    return rho, u, v, w


def _requests(c, seed):
    """Duct requests of the library's stream that are small enough, with the
    case's step budget; the force and viscosity come from the seed (the sizes
    and spheres are the case's)."""
    p = _inputs(c, seed)
    out = []
    for r in serve.duct_requests(200, seed=c["pick"]):
        if r.nx <= c["nx_max"] and r.ny <= c["ny_max"]:
            out.append(r)
        if len(out) == c["requests"]:
            break
    arr = (type(out[0]) * len(out))(*out)
    for i, r in enumerate(arr):
        r.steps, r.gx, r.nu, r.seed = c["steps"], p["gx"][i], p["nu"][i], seed & 0xFFFF
    return arr


# ---------------------------------------------------------------------------
# the library's side


class _State(dict):
    """What the program holds between passes; releases its lattices."""

    def __del__(self):
        if self.get("batch"):
            self["batch"].close()
        for lat in self.get("lats", []):
            lat.close()


def _cavity(shape, tau, lid, storage, seed, tile=None, types=None):
    lat = mrlbm.Lattice(shape, q=19, tau=tau, walls=(1, 1, 1), storage=STORE[storage], seed=seed, tile=tile)
    lat.set_bc_velocity(0, (lid, 0.0, 0.0))
    lat.set_node_types(geometry.classify(shape, (1, 1, 1), None, [(2, +1, 0)]) if types is None else types)
    lat.init_uniform()
    return lat


def prepare(case, seed):
    c, p, k = case, _inputs(case, seed), case["kind"]
    key = seed & 0xFFFF
    s = _State(case=c)
    if k in ("probe", "cavity"):
        lat = _cavity(_shape(c), p["tau"], p["lid"], c["storage"], key)
        lat.step(100)
        if k == "probe":
            s["points"] = p["points"]
        else:
            lat.velocity_residual()
    elif k == "tgv":
        lat = mrlbm.Lattice(_shape(c), q=19, tau=p["tau"], storage=STORE[c["storage"]], seed=key)
        lat.init_taylor_green(p["u0"])
    elif k in ("duct", "stats", "monitor"):
        lat = mrlbm.Lattice(_shape(c), q=c.get("q", 19), tau=p["tau"], walls=(0, 1, 1), force=(p["g"], 0.0, 0.0),
                            storage=STORE[c["storage"]], seed=key)
        lat.set_geometry(centres=[ctr for ctr, _ in p["spheres"]], radii=[r for _, r in p["spheres"]])
        lat.init_uniform(u=(p.get("u", 0.0), 0.0, 0.0))
        if k == "monitor":
            lat.velocity_residual()
    elif k == "batch":
        tile = (8, 8, 8)
        types = {n: geometry.cavity(n) for n in set(_edges(c))}
        s["lats"] = [_cavity((n, n, n), t, p["lid"], c["storage"], key, tile, types[n])
                     for n, t in zip(_edges(c), p["tau"])]
        s["batch"] = mrlbm.Batch(q=19, tile=tile, storage=STORE[c["storage"]])
        for lat in s["lats"]:
            s["batch"].add(lat)
        return s
    elif k == "job":
        s["fields"] = [np.asfortranarray(f) for f in _job_fields(c, p, np)]  # x fastest, as the library takes them
        s["tau"], s["key"] = p["tau"], key
        return s
    else:
        s["requests"] = _requests(c, seed)
        s["moments"] = [serve.attach_output(r) for r in s["requests"]]
        return s
    s["lats"] = [lat]
    lat.synchronize()
    return s


def _held(a, storage):
    """Moments or velocities at the precision at which the lattice holds them."""
    if storage == "fp32":
        return a
    return torch.from_numpy(a).to(torch.float16 if storage == "fp16" else torch.bfloat16)


def run(state):
    c = state["case"]
    k, st = c["kind"], c["storage"]
    if k == "job":
        with mrlbm.Lattice(_shape(c), q=19, tau=state["tau"], storage=STORE[st], seed=state["key"]) as lat:
            lat.init_fields(*state["fields"])
            lat.step(c["steps"])
            rho, *u = lat.macroscopic()
            return [rho] + [_held(f, st) for f in u]
    if k == "batch":
        state["batch"].step(c["steps"], graph_steps=50)
        return [_held(lat.moments(), st) for lat in state["lats"]]
    if k == "serve":
        serve.run(state["requests"], storage=STORE[st], realtime=False, quantum=100, graph_steps=50, max_batch=6)
        return {"moments": [_held(m, st) for m in state["moments"]], "ke": [r.ke1 for r in state["requests"]]}
    lat = state["lats"][0]
    if k == "probe":
        lat.step(1)
        return lat.sample(state["points"])
    if k == "cavity":
        lat.step(c["steps"])
        return {"residual": lat.velocity_residual(), "moments": _held(lat.moments(), st)}
    if k == "tgv":
        lat.step(c["steps"])
        return {"reduce": np.array(lat.reduce()), "moments": _held(lat.moments(), st)}
    if k == "duct":
        lat.step(c["steps"])
        return _held(lat.moments(), st)
    if k == "monitor":
        lat.step(c["steps"])
        return {"reduce": np.array(lat.reduce_checked(), np.float64), "means": lat.moment_means(),
                "residual": lat.velocity_residual()}
    lat.mean_flow_reset()
    for _ in range(c["samples"]):
        lat.step(c["every"])
        lat.mean_flow_accumulate()
    tke = lat.turbulent_ke()
    (rho, *u), _ = lat.mean_flow()
    return {"tke": tke, "rho": rho, "u": torch.stack([torch.as_tensor(_held(f, st)) for f in u])}


def _lattices(c):
    """(nodes, Q, steps) of every lattice that a pass advances."""
    k = c["kind"]
    if k == "batch":
        return [(n ** 3, 19, c["steps"]) for n in _edges(c)]
    if k == "serve":
        return [(r.nx * r.ny * r.nz, 19, c["steps"]) for r in _requests(c, 0)]
    steps = c["samples"] * c["every"] if k == "stats" else c.get("steps", 1)
    return [(c["nx"] * c["ny"] * c["nz"], c.get("q", 19), steps)]


def work(case):
    """Every step reads and writes the ten moments of every node once; about
    350 (D3Q19) or 500 (D3Q27) operations per node. Read-back, monitors and
    initial fields read or write each of their values once."""
    c, k = case, case["kind"]
    w = WORD[c["storage"]]
    b = f = 0.0
    for n, q, steps in _lattices(c):
        b += steps * n * 20.0 * w
        f += steps * n * (350.0 if q == 19 else 500.0)
        if k in ("cavity", "tgv", "duct", "batch", "serve"):
            b += n * (10.0 * w + 80.0)
        if k == "tgv":
            b += n * 4.0 * w
        if k == "cavity":
            b += n * (3.0 * w + 24.0)
        if k == "job":
            b += n * (10.0 * w + 32.0 + 10.0 * w + 32.0)
        if k == "monitor":
            b += n * (10.0 * w + 24.0)
        if k == "stats":
            b += n * (c["samples"] * (4.0 * w + 64.0) + 4.0 * w + 24.0 + 64.0)
        if k == "probe":
            b += c["points"] * (10.0 * w + 80.0)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch

_CX = [0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0, 1, -1, 1, -1, 1, -1, -1, 1]
_CY = [0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 1, -1, 1, -1, 1, -1, -1, 1, 1, -1]
_CZ = [0, 0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0, -1, 1, -1, 1, 1, -1, -1, 1, 1, -1, 1, -1]
_PAIRS = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]


def _octants(d):
    m = 0
    for o in range(8):
        corner = [1 if (o >> a) & 1 else -1 for a in range(3)]
        if all(d[a] in (0, corner[a]) for a in range(3)):
            m |= 1 << o
    return m


class _Exact:
    """The moment-representation scheme on one lattice, in 64 bits: fields of
    index [z, y, x] (x fastest), moments unscaled."""

    def __init__(self, shape, q, tau, walls=(0, 0, 0), force=0.0, spheres=(), lid=None):
        self.shape, self.q, self.om, self.force = shape, q, 1.0 / tau, force
        nx, ny, nz = shape
        self.n = nx * ny * nz
        dev = dict(dtype=torch.float64, device="cuda")
        w = [1 / 3, 1 / 18, 1 / 36, 0] if q == 19 else [8 / 27, 2 / 27, 1 / 54, 1 / 216]
        cls = [0 if i == 0 else 1 if i < 7 else 2 if i < 19 else 3 for i in range(27)]
        self.cv = np.array([_CX, _CY, _CZ])[:, :q]
        self.w = np.array([w[cls[i]] for i in range(q)])
        c = self.cv.astype(float)
        self.h = np.stack([c[a] * c[b] - (1 / 3 if a == b else 0.0) for a, b in _PAIRS])
        # f = rho [w (1 + 3 c.u + 4.5 sum_ab (2 - d_ab) H_ab m_ab)]
        coef = np.array([1.0 if a == b else 2.0 for a, b in _PAIRS])
        self.recon = torch.tensor(np.concatenate([self.w[:, None], (3 * self.w * c).T,
                                                  (4.5 * self.w * self.h * coef[:, None]).T], 1), **dev)
        self.project = torch.tensor(np.concatenate([np.ones((1, q)), c, self.h]), **dev)
        self.solid = self.bc = None
        if any(walls) or spheres:
            self._boundaries(walls, spheres, lid, coef)
        self.pull = None
        if self.n <= 1 << 21:  # one gather instead of a roll per population
            j = torch.arange(self.n, device="cuda").view(nz, ny, nx)
            self.pull = torch.stack([torch.roll(j, (int(self.cv[2, i]), int(self.cv[1, i]), int(self.cv[0, i])),
                                                (0, 1, 2)).reshape(-1) for i in range(q)])
        self.m = torch.zeros((10, self.n), **dev)  # rho, u, m_ab
        self.m[0] = 1.0

    def _boundaries(self, walls, spheres, lid, coef):
        nx, ny, nz = self.shape
        z, y, x = torch.meshgrid(*[torch.arange(e, device="cuda") for e in (nz, ny, nx)], indexing="ij")
        solid = torch.zeros((nz, ny, nx), dtype=torch.bool, device="cuda")
        for (sx, sy, sz), r in spheres:
            solid |= ((x - sx) ** 2 + (y - sy) ** 2 + (z - sz) ** 2).double() <= r * r
        bits = torch.zeros((nz, ny, nx), dtype=torch.int64, device="cuda")
        pos, ext = (x, y, z), (nx, ny, nz)
        for a in range(3):
            if walls[a]:
                for side, at in ((-1, 0), (1, ext[a] - 1)):
                    d = [0, 0, 0]
                    d[a] = side
                    bits |= torch.where(pos[a] == at, _octants(d), 0)
        if spheres:
            for d in [(i, j, k) for i in (-1, 0, 1) for j in (-1, 0, 1) for k in (-1, 0, 1) if i or j or k]:
                near = torch.roll(solid, (-d[2], -d[1], -d[0]), (0, 1, 2))
                for a in range(3):
                    if walls[a] and d[a]:
                        near = near & (pos[a] != (ext[a] - 1 if d[a] > 0 else 0))
                bits |= torch.where(near, _octants(d), 0)
        solid |= bits == 255  # no fluid neighbour: solid too
        moving = (z == nz - 1) & ~solid if lid is not None else torch.zeros_like(solid)
        bits = torch.where(solid, 0, bits + 256 * moving).reshape(-1)
        self.solid = solid.reshape(-1) if spheres else None
        self.bc = torch.nonzero(bits).reshape(-1)
        keys, at = torch.unique(bits[self.bc], return_inverse=True)
        known, inv, vel = [], [], []
        for key in keys.tolist():
            oct_, u = key & 255, np.array([lid if key & 256 else 0.0, 0.0, 0.0])
            kn = np.array([any(not (oct_ >> o) & 1 for o in range(8)
                               if all(-self.cv[a, i] in (0, 1 if (o >> a) & 1 else -1) for a in range(3)))
                           for i in range(self.q)])
            # single plane walls of D3Q27 keep the D3Q19 closure
            qc = 19 if self.q == 27 and oct_ in (0xCC, 0x33, 0x55, 0xAA, 0xF0, 0x0F) else self.q
            wc = self.w if qc == self.q else np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12)
            k = kn[:qc]
            h, cu, wk = self.h[:, :qc][:, k], 3 * (u @ self.cv[:, :qc])[k], wc[k]
            uu = np.array([u[a] * u[b] for a, b in _PAIRS])
            A = np.zeros((7, 7))
            A[0, 0] = (wk * (1 + cu + 4.5 * self.om * ((coef * uu) @ h))).sum()
            A[0, 1:] = 4.5 * (1 - self.om) * coef * (h @ wk)
            A[1:, 0] = h @ (wk * (1 + cu))
            A[1:, 1:] = 4.5 * (h * wk) @ h.T * coef
            known.append(kn)
            inv.append(np.linalg.inv(A))
            vel.append(u)
        dev = dict(dtype=torch.float64, device="cuda")
        self.known = torch.tensor(np.array(known).T.astype(float), **dev)[:, at]
        self.inv = torch.tensor(np.array(inv), **dev)[at]
        self.vel = torch.tensor(np.array(vel).T, **dev)[:, at]

    def set_fields(self, rho, ux, uy, uz):
        """Density and velocity with equilibrium second moments."""
        self.m[0], self.m[1], self.m[2], self.m[3] = rho, ux, uy, uz
        for k, (a, b) in enumerate(_PAIRS):
            self.m[4 + k] = self.m[1 + a] * self.m[1 + b]

    def step(self, steps):
        nx, ny, nz = self.shape
        om, g = self.om, self.force
        for _ in range(steps):
            terms = self.m.clone()
            terms[1:] *= terms[0]
            f = self.recon @ terms
            if self.pull is not None:
                f = torch.gather(f, 1, self.pull)
            else:
                for i in range(1, self.q):
                    f[i] = torch.roll(f[i].view(nz, ny, nx), (int(self.cv[2, i]), int(self.cv[1, i]),
                                                              int(self.cv[0, i])), (0, 1, 2)).reshape(-1)
            s = self.project @ f
            s[1:] /= s[0]
            if self.bc is not None:
                b = self.project @ (f[:, self.bc] * self.known)
                x = torch.matmul(self.inv, torch.cat([b[:1], b[4:]]).T.unsqueeze(2)).squeeze(2).T
                s[:, self.bc] = torch.cat([x[:1], self.vel, x[1:] / x[:1]])
            del f
            if g:
                s[1] += g / s[0]
            new = s.clone()
            for k, (a, c) in enumerate(_PAIRS):
                t = (1 - om) * s[4 + k] + om * s[1 + a] * s[1 + c]
                if g and a == 0:
                    t += (1 - om / 2) * g / s[0] * (2 * s[1] if c == 0 else s[1 + c])
                new[4 + k] = t
            if self.solid is not None:
                new = torch.where(self.solid, self.m, new)
            self.m = new

    def stored(self):
        """The ten moments as the library stores them: rho - 1, 3u, 4.5 m_aa, 9 m_ab."""
        scale = [1, 3, 3, 3] + [4.5 if a == b else 9.0 for a, b in _PAIRS]
        out = self.m * torch.tensor(scale, dtype=torch.float64, device="cuda")[:, None]
        out[0] -= 1.0
        return out

    def ke(self):
        return float((self.m[0] * (self.m[1:4] ** 2).sum(0)).mean() / 2)


def _exact_taylor_green(shape, u0):
    ax = [2 * math.pi * torch.arange(e, dtype=torch.float64, device="cuda") / e for e in shape]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    rho = 1 + 3 / 16 * u0 * u0 * (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2)
    u = u0 * torch.sin(x) * torch.cos(y) * torch.cos(z)
    v = -u0 * torch.cos(x) * torch.sin(y) * torch.cos(z)
    return [f.reshape(-1) for f in (rho, u, v, torch.zeros_like(u))]


def exact(case, seed):
    c, k = case, case["kind"]
    # time goes with the lattice updates, and for small lattices with the steps
    if sum(s * max(n, 1 << 18) * q / 19 for n, q, s in _lattices(c)) > EXACT_LU_MAX:
        return None
    p = _inputs(c, seed)
    if k == "batch":
        out = []
        for n, tau in zip(_edges(c), p["tau"]):
            e = _Exact((n, n, n), 19, tau, walls=(1, 1, 1), lid=p["lid"])
            e.step(c["steps"])
            out.append(e.stored().cpu())
        return out
    if k == "serve":
        out, ke = [], []
        for r in _requests(c, seed):
            sp = [((r.sphere[i][0], r.sphere[i][1], r.sphere[i][2]), r.sphere[i][3]) for i in range(r.nspheres)]
            e = _Exact((r.nx, r.ny, r.nz), 19, 0.5 + 3.0 * r.nu, walls=(0, 1, 1), force=r.gx, spheres=sp)
            e.step(c["steps"])
            out.append(e.stored().reshape(-1).cpu())
            ke.append(e.ke())
        return {"moments": out, "ke": ke}
    q = c.get("q", 19)
    if k in ("probe", "cavity"):
        e = _Exact(_shape(c), q, p["tau"], walls=(1, 1, 1), lid=p["lid"])
        e.step(100)
    elif k in ("tgv", "job"):
        e = _Exact(_shape(c), q, p["tau"])
        if k == "tgv":
            e.set_fields(*_exact_taylor_green(_shape(c), p["u0"]))
        else:
            e.set_fields(*[f.permute(2, 1, 0).reshape(-1) for f in _job_fields(c, p, torch)])
    else:
        e = _Exact(_shape(c), q, p["tau"], walls=(0, 1, 1), force=p["g"], spheres=p["spheres"])
        zero = torch.zeros_like(e.m[0])
        e.set_fields(zero + 1, zero + p.get("u", 0.0), zero, zero)
        del zero
    if k == "stats":
        acc = torch.zeros_like(e.m[:4])
        for _ in range(c["samples"]):
            e.step(c["every"])
            acc += e.m[:4]
        acc /= c["samples"]
        tke = float((e.m[0] * ((e.m[1:4] - acc[1:]) ** 2).sum(0)).mean() / 2)
        rho, *u = [f.view(_shape(c)[::-1]).permute(2, 1, 0).cpu() for f in acc]
        return {"tke": tke, "rho": rho, "u": torch.stack(u)}
    before = e.m[1:4].clone()
    e.step(c.get("steps", 1))
    res = float((e.m[1:4] - before).norm() / e.m[1:4].norm())
    if k == "probe":
        pt = torch.from_numpy(p["points"]).long().cuda()
        at = pt[:, 0] + c["nx"] * (pt[:, 1] + c["ny"] * pt[:, 2])
        return e.stored()[:, at].T.contiguous().cpu()
    if k == "job":
        return [f.view(_shape(c)[::-1]).permute(2, 1, 0).cpu() for f in e.m[:4]]
    if k == "monitor":
        return {"reduce": np.array([float((e.m[0] - 1).mean()), e.ke(), 0.0]),
                "means": e.stored().mean(1).cpu(), "residual": res}
    if k == "cavity":
        return {"residual": res, "moments": e.stored().cpu()}
    if k == "tgv":
        return {"reduce": np.array([float((e.m[0] - 1).mean()), e.ke()]), "moments": e.stored().cpu()}
    return e.stored().cpu()
