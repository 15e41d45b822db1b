"""What a user of the step library has it do, as cases that can be timed.

A case is one call cycle of a program that steps site-response models: dmp_run
of some steps through the Python binding, the seismograms it returns, and in
some cases the state download with which the drop-in run_explicit saves a
snapshot after each such call.  The sites are those of damian_hip.cases (the
homogeneous layer, the two-material valley, the canyon quadtree and its
uniform mesh, the random sediment basins and sweeps of them), at their own and
at other sizes.  The source (incidence, arrival time, frequency, amplitude)
comes from the seed; the mesh belongs to the case and is built once.
"""
import copy
import functools
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "damian.par_amd" / "python"))

from damian_hip import cases as sites  # noqa: E402
from damian_hip import lib  # noqa: E402

PRECISIONS = {"fp64": lib.DMP_FP64, "fp32c": lib.DMP_FP32C}


def listed():
    """`site` and its sizes say what is stepped; `steps` a call's length;
    `interval` the sampling interval in steps (0: no receivers); `snapshot`
    whether the state is downloaded after the call; `tuned` whether the
    program has had the library pick the launch shape for such calls."""
    def case(name, site, precision, steps, interval=1, snapshot=False, tuned=False, **sizes):
        return dict(name=name, site=site, precision=precision, steps=steps, interval=interval,
                    snapshot=snapshot, tuned=tuned, **sizes)

    return [
        # a program that looks at every step of a small model: only latency
        case("layer_800_fp64_1_step", "layer", "fp64", 1, nx=40, nz=20),
        # a quick look at a small valley with hanging nodes
        case("valley_332_fp32c_20_steps", "valley", "fp32c", 20),
        # the drop-in run_explicit: steps up to the next saved snapshot, no receivers
        case("layer_40k_fp64_save_cycle", "layer", "fp64", 50, interval=0, snapshot=True, nx=400, nz=100),
        # the canyon benchmark in a short call, as an interactive program makes
        case("canyon_fp32c_20_steps", "canyon", "fp32c", 20, tuned=True, band=50.0),
        # the canyon benchmark proper, in both precisions
        case("canyon_fp32c_1000_steps", "canyon", "fp32c", 1000, tuned=True, band=50.0),
        case("canyon_fp64_1000_steps", "canyon", "fp64", 1000, snapshot=True, tuned=True, band=50.0),
        # the canyon on its uniform 2.5 m grid: bound by memory
        case("canyon_944k_fp32c_100_steps", "uniform_canyon", "fp32c", 100, tuned=True),
        case("canyon_944k_fp64_save_cycle", "uniform_canyon", "fp64", 80, interval=20, snapshot=True),
        # a random basin (moduli per element) with a coarser seismogram
        case("basin_141k_fp32c_200_steps", "basin", "fp32c", 200, interval=10, snapshot=True, depth=200.0),
        case("basin_141k_fp64_200_steps", "basin", "fp64", 200, tuned=True, depth=200.0),
        # sweeps: uneven basins advanced together
        case("sweep_16_fp32c_50_steps", "sweep", "fp32c", 50, tuned=True, depth=100.0, deepest=300.0, count=16),
        case("sweep_6_fp64_100_steps", "sweep", "fp64", 100, depth=80.0, deepest=160.0, count=6),
    ]


def draw(rng):
    def log_uniform(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    site = rng.choice(["layer", "layer", "canyon", "basin", "sweep"])
    if site == "layer":
        n = log_uniform(200, 900e3)
        nz = max(5, int(math.sqrt(n / rng.uniform(2.0, 5.0))))
        sizes = {"nx": max(20, int(n / nz)), "nz": nz}
        most = min(1000, max(20, int(100e6 / n)))
    elif site == "canyon":
        sizes, most = {"band": round(rng.uniform(15.0, 90.0), 1)}, 1000
    elif site == "basin":
        d = round(log_uniform(45.0, 300.0), 1)
        sizes, most = {"depth": d}, min(1000, int(100e6 / (3.5 * d * d)))
    else:
        d = rng.uniform(40.0, 90.0)
        sizes = {"depth": round(d, 1), "deepest": round(d * rng.uniform(1.2, 2.5), 1), "count": rng.randint(2, 12)}
        most = 50
    steps = int(log_uniform(1, most))
    return dict(site=site, precision=rng.choice(["fp64", "fp32c"]), steps=steps,
                interval=min(steps, rng.choice([1, 1, 5, 10])), snapshot=rng.random() < 0.4,
                tuned=rng.random() < 0.4, **sizes)


# ---------------------------------------------------------------------------
# the models
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def layer(nx, nz):
    """Homogeneous layer of 5 m cells (Vs 500, Vp 1000, rho 2000)."""
    w, h = 5.0 * nx, 5.0 * nz
    pulse = 0.25 + 0.6 * h / 500.0
    text = sites.problem_text(w, h, 10.0, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                              [0.5 * w, 0.6 * h, 0.5 * w, 0, 1, pulse, 0.0, 1.0, 4.0])
    n = min(101, max(10, nx))
    return sites.S.case_from_problem_text(text, sheet=(-0.9 * w / n, w - 1.8 * w / n, w / n), name="layer")


@functools.lru_cache(maxsize=None)
def canyon(band, uniform=False):
    return sites.c2(uniform=True) if uniform else sites.c2(band=band)


@functools.lru_cache(maxsize=None)
def basin(depth, field):
    return sites.c4_valley(depth, "P", 0.0, nsteps=10000, field_seed=field)


def models(case):
    """The case's models, with the source that the case's site comes with."""
    site = case["site"]
    if site == "layer":
        return [layer(case["nx"], case["nz"])]
    if site == "valley":
        return [sites.f2()]
    if site == "canyon":
        return [canyon(case["band"])]
    if site == "uniform_canyon":
        return [canyon(0.0, uniform=True)]
    if site == "basin":
        return [basin(case["depth"], 3003)]
    step = (case["deepest"] - case["depth"]) / max(1, case["count"] - 1)
    return [basin(case["depth"] + k * step, 3003 + k) for k in range(case["count"])]


def sourced(case, seed):
    """The models with sources of their own from the seed."""
    rng = random.Random(seed)
    out = []
    for m in models(case):
        m, mdl = copy.copy(m), copy.copy(m.model)
        m.model = mdl
        mdl.prob = rng.choice(["WAVEP ", "WAVESV"])
        mdl.wangle = math.radians(rng.uniform(0.0, 60.0 if mdl.prob == "WAVEP " else 28.0))
        mdl.wamp = rng.uniform(0.5, 2.0)
        mdl.wfreq *= rng.uniform(0.8, 1.1)
        mdl.wt0 *= rng.uniform(1.0, 1.05)
        out.append(m)
    return out


def arrival(built):
    """Steps until the pulses are at the surface: the calls start there."""
    return max(int(m.model.wt0 / m.dt) for m in built)


# ---------------------------------------------------------------------------
# one call cycle
# ---------------------------------------------------------------------------
SHAPES = {}   # launch shapes picked for a case by the library, kept like a program's configuration


def prepare(case, seed):
    built = sourced(case, seed)
    many, interval = case["site"] == "sweep", case["interval"]
    solvers = [lib.Solver(m, precision=PRECISIONS[case["precision"]], io_interval=max(1, interval),
                          receivers=interval > 0, init=not many) for m in built]
    handle = lib.Batch(solvers) if many else solvers[0]
    if case["tuned"]:
        key = repr(sorted(case.items()))
        if key not in SHAPES:
            SHAPES[key] = handle.autotune(min(case["steps"], 60))
        handle.set_tuning(*SHAPES[key])
    handle.run(arrival(built), record=False)
    return {"case": case, "handle": handle, "solvers": solvers}


def run(state):
    case, handle = state["case"], state["handle"]
    out = {}
    samples = handle.run(case["steps"], record=case["interval"] > 0)
    if samples is not None and len(samples):
        out["samples"] = samples
    if case["snapshot"] or not out:
        if case["site"] == "sweep":
            out["state"] = [handle.state(q) for q in range(len(state["solvers"]))]
        else:
            out["state"] = handle.state()
    return out


def work(case):
    """A pass reads two state levels and the elements' moduli and densities
    and writes two levels; per step a node takes its mass term and, from each
    element, two rows of eight."""
    built = models(case)
    nodes, elems = sum(m.mesh.nnodes for m in built), sum(m.nelems for m in built)
    material = 16 if case["precision"] == "fp64" else 8
    heterogeneous = any(m.elem_props is not None for m in built)
    out = 0
    if case["interval"]:
        out += 16 * sum(len(m.recv_elem) for m in built) * (case["steps"] // case["interval"])
    if case["snapshot"]:
        out += 48 * nodes
    return {"bytes": 64 * nodes + (material * elems if heterogeneous else 0) + out,
            "flops": case["steps"] * (128 * elems + 12 * nodes)}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def element_matrices():
    """K_lambda, K_mu (plane strain) and the mass pattern of the unit square,
    corners (0,0), (1,0), (1,1), (0,1), by 2 x 2 Gauss points."""
    cx, cz = np.array([0, 1, 1, 0]), np.array([0, 0, 1, 1])
    kl, km, mm = np.zeros((8, 8)), np.zeros((8, 8)), np.zeros((4, 4))
    dl = np.array([[1.0, 1, 0], [1, 1, 0], [0, 0, 0]])
    dm = np.diag([2.0, 2, 1])
    for x in (0.5 - math.sqrt(1 / 12), 0.5 + math.sqrt(1 / 12)):
        for z in (0.5 - math.sqrt(1 / 12), 0.5 + math.sqrt(1 / 12)):
            nx, nz = np.where(cx, x, 1 - x), np.where(cz, z, 1 - z)
            b = np.zeros((3, 8))
            b[0, 0::2] = b[2, 1::2] = np.where(cx, 1, -1) * nz
            b[1, 1::2] = b[2, 0::2] = np.where(cz, 1, -1) * nx
            kl += b.T @ dl @ b / 4
            km += b.T @ dm @ b / 4
            mm += np.outer(nx * nz, nx * nz)
    return kl, km, np.kron(mm, np.eye(2))


def trains(mdl):
    """Incident wave and its two reflections at the free surface:
    (propagation direction, speed, amplitude, motion) of each."""
    vp, vs = mdl.wvelo
    r = vp / vs
    if mdl.prob == "WAVEP ":
        e = mdl.wangle
        f = math.asin(math.sin(e) / r)
    else:
        f = mdl.wangle
        e = math.asin(math.sin(f) * r)
    se, ce, sf, cf = math.sin(e), math.cos(e), math.sin(f), math.cos(f)
    s2e, s2f, c2f = math.sin(2 * e), math.sin(2 * f), math.cos(2 * f)
    den = s2e * s2f + r * r * c2f * c2f
    back = (s2e * s2f - r * r * c2f * c2f) / den
    p_down, s_down = ((se, ce), vp, (se, ce)), ((sf, cf), vs, (-cf, sf))
    if mdl.prob == "WAVEP ":
        parts = [((se, -ce), vp, (se, -ce)) + (1.0,), p_down + (back,), s_down + (-2 * r * s2e * c2f / den,)]
    else:
        parts = [((sf, -cf), vs, (cf, sf)) + (1.0,), p_down + (r * math.sin(4 * f) / den,), s_down + (back,)]
    return [(d, v, m, a * mdl.wamp) for d, v, m, a in parts]


def free_field(mdl, xz, t):
    """Displacement and acceleration at points (n, 2) and times (k,): (k, n, 2) each."""
    u = torch.zeros(len(t), len(xz), 2, dtype=torch.float64, device=t.device)
    acc = torch.zeros_like(u)
    w = math.pi * mdl.wfreq
    rel = xz - torch.tensor(mdl.worigin, dtype=torch.float64, device=t.device)
    for d, v, motion, amp in trains(mdl):
        s = (w * (t[:, None] - mdl.wt0 - ((rel[:, 0] * d[0] + rel[:, 1] * d[1]) / v)[None])) ** 2
        e = amp * torch.exp(-s)
        m = torch.tensor(motion, dtype=torch.float64, device=t.device)
        u += ((1 - 2 * s) * e)[..., None] * m
        acc += (-2 * (4 * s * s - 12 * s + 3) * w * w * e)[..., None] * m
    return u, acc


class Model64:
    """One model's share of the joined arrays (nodes from `base` on)."""

    EXTERIOR = {2: (0, 3), 4: (1, 2), 1: (2, 3), 6: (0, 2, 3), 5: (1, 2, 3)}   # corners by layer kind

    def __init__(self, m, base, dev):
        def on(a, dtype=torch.float64):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=dev)

        self.m, self.base, self.dev = m, base, dev
        mesh = m.mesh
        c = mesh.corners().astype(np.int64) - 1
        p = m.elem_props if m.elem_props is not None else m.model.matconst[mesh.ematprop - 1]
        mu, lam, rho, vp, vs = p.T
        h = mesh.elength()
        mass = (h / 2) ** 2 * rho
        a1, a2 = 1 / m.dt ** 2, 1 / (2 * m.dt)
        kl, km, mm = element_matrices()
        n = mesh.nnodes
        ab = m.absorbing[c]
        along, across = (vs * rho * h)[:, None] * (ab > 0), (vp * rho * h)[:, None] * (ab > 0)
        damp = np.stack([np.where(ab == 1, along, across), np.where(ab == 1, across, along)], axis=-1)
        self.nodes, self.dof = on(mesh.nodes), 2 * n
        md, cd = np.zeros((n, 2)), np.zeros((n, 2))
        np.add.at(md, c, np.repeat(mass, 8).reshape(-1, 4, 2))
        np.add.at(cd, c, damp)
        full = a1 * md + a2 * cd
        hang = m.hanging.astype(np.int64).reshape(-1, 3) - 1
        for k in (1, 2):
            np.add.at(full, hang[:, k], full[hang[:, 0]] / 2)
        self.md, self.cd, self.full = on(a1 * md).ravel(), on(a2 * cd).ravel(), on(full).ravel()
        self.hang = on(hang, torch.int64) + base
        d = (2 * c[:, :, None] + np.arange(2)).reshape(-1, 8) + 2 * base
        self.rows, self.cols = on(np.repeat(d, 8, axis=1).ravel(), torch.int64), on(np.tile(d, (1, 8)).ravel(), torch.int64)
        self.vals = (on(lam)[:, None] * on(kl.ravel()) + on(mu)[:, None] * on(km.ravel())).ravel()
        # plane-wave layer: per kind, its elements and the rows between exterior and interior corners
        self.layer = []
        for kind, ext in self.EXTERIOR.items():
            e = m.seismic[m.seismic[:, 1] == kind, 0].astype(np.int64) - 1 if len(m.seismic) else np.zeros(0, np.int64)
            x = np.repeat(np.isin(np.arange(4), ext), 2)
            mask = np.where(x[:, None] != x[None], np.where(x[:, None], 1.0, -1.0), 0.0)
            if len(e):
                self.layer.append((on(c[e], torch.int64), on(d[e].ravel(), torch.int64), on(lam[e])[:, None],
                                   on(mu[e])[:, None], on(mass[e])[:, None], on(mask * kl).T, on(mask * km).T, on(mask * mm).T))
        # receivers: corners and bilinear weights
        r = m.recv_elem.astype(np.int64) - 1
        lo, hi = mesh.nodes[c[r, 0]], mesh.nodes[c[r, 2]]
        s = np.clip((m.recv_xy - lo) / (hi - lo), 0, 1)
        x, z = s.T
        w = np.stack([(1 - x) * (1 - z), x * (1 - z), x * z, (1 - x) * z], axis=1) * (r >= 0)[:, None]
        self.rc, self.rw, self.rxy = on(c[r], torch.int64) + base, on(w)[..., None], on(m.recv_xy)
        self.rff = on(m.recv_ff.astype(bool) & (r >= 0))[:, None]

    def forces(self, steps):
        """(dof indices, values (steps, n)) of the layer's forces."""
        t = torch.tensor(steps, dtype=torch.float64, device=self.dev) * self.m.dt
        index, value = [], []
        for c, d, lam, mu, mass, kl, km, mm in self.layer:
            u, a = free_field(self.m.model, self.nodes[c.ravel()], t)
            u, a = u.reshape(len(t), -1, 8), a.reshape(len(t), -1, 8)
            f = lam * (u @ kl) + mu * (u @ km) + mass * (a @ mm)
            index.append(d)
            value.append(f.reshape(len(t), -1))
        return torch.cat(index), torch.cat(value, dim=1)

    def sample(self, u, j):
        t = torch.tensor([j * self.m.dt], dtype=torch.float64, device=self.dev)
        return (self.rw * u.view(-1, 2)[self.rc]).sum(1) + self.rff * free_field(self.m.model, self.rxy, t)[0][0]


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    built, parts, base = sourced(case, seed), [], 0
    for m in built:
        parts.append(Model64(m, base, dev))
        base += m.mesh.nnodes
    n = 2 * base
    k = torch.sparse_coo_tensor(torch.stack([torch.cat([p.rows for p in parts]), torch.cat([p.cols for p in parts])]),
                                torch.cat([p.vals for p in parts]), (n, n)).coalesce().to_sparse_csr()
    md, cd, full = (torch.cat([getattr(p, a) for p in parts]) for a in ("md", "cd", "full"))
    hang = torch.cat([p.hang for p in parts])
    u, up = torch.zeros(n, dtype=torch.float64, device=dev), torch.zeros(n, dtype=torch.float64, device=dev)
    s0 = arrival(built)
    interval, samples = case["interval"], []
    for j in range(1, s0 + case["steps"] + 1):
        if j % 64 == 1:
            f = [p.forces(range(j, j + 64)) for p in parts]
            findex, fvalue = torch.cat([x[0] for x in f]), torch.cat([x[1] for x in f], dim=1)
        r = md * (2 * u - up) + cd * up - torch.mv(k, u)
        r.index_add_(0, findex, fvalue[(j - 1) % 64])
        new = r.view(-1, 2)
        half = new[hang[:, 0]] / 2
        new = new.index_add(0, hang[:, 1], half).index_add_(0, hang[:, 2], half) / full.view(-1, 2)
        new[hang[:, 0]] = (new[hang[:, 1]] + new[hang[:, 2]]) / 2
        u, up = new.view(-1), u
        if interval and j > s0 and j % interval == 0:
            samples.append(torch.cat([p.sample(u, j) for p in parts]).cpu().numpy())
    out = {}
    if samples:
        out["samples"] = np.stack(samples)
    if case["snapshot"] or not out:
        at = [2 * p.base for p in parts]
        state = [[x[a:a + p.dof].cpu().numpy() for x in (u, up)] for a, p in zip(at, parts)]
        out["state"] = state if case["site"] == "sweep" else state[0] + [parts[0].full.cpu().numpy()]
    return out
