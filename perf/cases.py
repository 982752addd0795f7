"""Workloads for timing the framework through its public entry points.

Four kinds of work, each over the range of sizes that users run:

  solve   one case advanced a number of time steps (GpuSolver.run or
          run_noalloc) and its fields read back, from a cavity of a few hundred
          cells to the 4.1M-tet channel with an immersed sphere; FP64 and FP32
          storage, hexes and tets, walls, in- and outlets and periodic sides
  batch   independent cases on one mesh advanced together (GpuBatch.run) and
          every case's fields read back: the training-data generator
  infer   the warm-start network's prediction of a start state (Mpnn.forward)
  train   loss and gradients of the network (Mpnn.loss_grad), the pass that a
          training step repeats

A case is a dict of plain values; prepare() builds the mesh, the solver or the
network and the seeded inputs, run() is one pass, exact() the same result in
64 bits with plain torch.  Fields of FP32-storage solvers are handed on as
float32, the precision their users keep (training targets, saved velocities).
"""
import math
import os
import sys
from functools import lru_cache

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "3d-plfbs-gpu_amd"))

from plbfs import case as pc  # noqa: E402
from plbfs import meshgen, mpnn, objects  # noqa: E402
from plbfs import warmstart as ws  # noqa: E402
from plbfs.solver import GpuBatch, GpuSolver, HostMesh  # noqa: E402

PERIODIC_PATCHES = {"x0": "inlet", "x1": "outlet", "y0": "farfield", "y1": "farfield", "z0": "zlow", "z1": "zhigh"}


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def solve_case(flow, n, tets=False, precision="fp64", nodes=0, steps=100, call="run", gradient="LS",
               stepping="local", **more):
    return dict(more, kind="solve", flow=flow, nx=n[0], ny=n[1], nz=n[2], tets=tets, precision=precision,
                nodes=nodes, steps=steps, call=call, gradient=gradient, stepping=stepping)


def batch_case(n, cases, precision="fp32", spheres=True, steps=100, block_cells=64, cases_per_block=8, **more):
    return dict(more, kind="batch", flow="channel", nx=n[0], ny=n[1], nz=n[2], tets=False, precision=precision,
                cases=cases, spheres=spheres, steps=steps, block_cells=block_cells, cases_per_block=cases_per_block)


def net_case(kind, n, tets=False, **more):
    return dict(more, kind=kind, flow="channel", nx=n[0], ny=n[1], nz=n[2], tets=tets)


def listed():
    return [
        # the smallest call: a cavity of 216 cells, as a first run or a sweep of tiny cases makes it
        solve_case("cavity", (6, 6, 6), steps=20, name="cavity 216 hex fp64"),
        # the lid-driven cavity of the benchmark set
        solve_case("cavity", (32, 32, 32), steps=200, name="cavity 32k hex fp64"),
        # the 96x48x48 sphere channel on which the time to residual 1e-6 is measured, in both precisions
        solve_case("channel", (96, 48, 48), nodes=450, steps=200, name="channel 221k hex fp64"),
        solve_case("channel", (96, 48, 48), precision="fp32", nodes=450, steps=200, name="channel 221k hex fp32"),
        # the headline workload: 4,088,832 tets with a 2,000-node sphere
        solve_case("channel", (88, 88, 88), tets=True, nodes=2000, steps=100, name="channel 4.1M tet fp64"),
        # FP32 storage on a tet mesh of an odd size that no block divides
        solve_case("channel", (57, 57, 57), tets=True, precision="fp32", nodes=900, steps=50,
                   name="channel 1.1M tet fp32"),
        # allocation-free steps on a ragged periodic mesh, hybrid gradients, one global time step
        solve_case("periodic", (37, 19, 23), steps=100, call="run_noalloc", gradient="hybrid", stepping="min",
                   name="periodic 16k hex fp64 noalloc"),
        # the batch of the benchmark set: 128 Reynolds numbers and spheres on one 64x32x32 mesh
        batch_case((64, 32, 32), 128, name="batch 128 x 65k hex fp32"),
        # a small FP64 batch: a parameter study without an immersed body, case count not a power of two
        batch_case((25, 12, 13), 11, precision="fp64", spheres=False, cases_per_block=4,
                   name="batch 11 x 3.9k hex fp64"),
        # the warm start's inference on the 96x48x48 channel
        net_case("infer", (96, 48, 48), name="network forward 221k"),
        # a training pass on the 64x32x32 mesh that the shipped parameters were trained on
        net_case("train", (64, 32, 32), name="network gradient 65k"),
        # a training pass on a small tet mesh
        net_case("train", (11, 9, 10), tets=True, name="network gradient 5.9k tet"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "solve", "batch", "infer", "train"])
    if kind == "solve":
        flow = rng.choice(["cavity", "channel", "channel", "periodic"])
        tets = rng.random() < 0.5 and flow != "periodic"  # a split face has no single partner across the box
        cells = size(216, 700000)
        edge = (cells / (6.0 if tets else 1.0)) ** (1.0 / 3.0)
        n = [max(3, int(round(edge * rng.uniform(0.8, 1.25)))) for _ in range(3)]
        if flow == "channel" and not tets:
            n = [max(3, int(round(2 * edge / 2 ** (1 / 3)))), *(max(3, int(round(q / 2 ** (1 / 3)))) for q in n[1:])]
        nodes = int(round(math.pi * (0.25 * n[1]) ** 2)) * (4 if tets else 1) if flow == "channel" and n[1] >= 24 else 0
        return solve_case(flow, n, tets=tets, precision=rng.choice(["fp64", "fp32"]), nodes=nodes,
                          steps=rng.randint(20, 60), call=rng.choice(["run", "run", "run_noalloc"]),
                          gradient=rng.choice(["LS", "LS", "hybrid"]),
                          stepping=rng.choice(["local", "local", "min"]))
    if kind == "batch":
        ny = size(6, 28)
        n = (2 * ny + rng.randint(-1, 1), ny, ny + rng.randint(-1, 1))
        precision = rng.choice(["fp32", "fp32", "fp64"])
        bc, cp = rng.choice([(64, 4), (64, 8), (128, 4)])
        return batch_case(n, rng.randint(2, 40), precision=precision, spheres=ny >= 24, steps=rng.randint(20, 60),
                          block_cells=bc, cases_per_block=cp)
    tets = rng.random() < 0.4
    cells = size(500, 150000 if kind == "infer" else 60000)
    edge = (cells / (12.0 if tets else 2.0)) ** (1.0 / 3.0)
    return net_case(kind, (max(3, int(2 * edge)), max(3, int(edge)), max(3, int(edge * rng.uniform(0.9, 1.2)))),
                    tets=tets)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def physics(c):
    """(Case, patch types, box lengths, sphere diameter) of a workload."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    sphere = bool(c.get("nodes") or c.get("spheres"))
    lengths = (2.0 * nx, float(ny), float(nz)) if c["tets"] else (float(nx), float(ny), float(nz))
    dia = (0.15 if c["tets"] else 0.25) * ny
    if c["flow"] == "cavity":
        lengths = (1.0, ny / nx, nz / nx)
        case, patches = pc.cavity_case(re=100.0), pc.CAVITY_PATCHES
    else:
        # fneq_min 0.55: the floor of the non-equilibrium weight without which wakes at these cell sizes diverge
        case = pc.channel_case(re=100.0 if c["tets"] else 40.0, length_scale=dia if sphere else 4.0, fneq_min=0.55)
        patches = pc.CHANNEL_PATCHES
        if c["flow"] == "periodic":
            per = dict(rho=1.0, u=0.0, v=0.0, w=0.0, vel_type="periodic", rho_type="periodic")
            case.bcs["zlow"] = dict(per, per_translate=(0.0, 0.0, lengths[2]))
            case.bcs["zhigh"] = dict(per, per_translate=(0.0, 0.0, -lengths[2]))
            patches = PERIODIC_PATCHES
    case.lsq_exact_det = 1 if c["tets"] else 0  # the reference's LSQ determinant diverges on jittered tets
    case.gradient_calc = c.get("gradient", "LS")
    case.time_stepping = c.get("stepping", "local")
    case.precision = 1 if c.get("precision") == "fp32" else 0
    case.tolerance = 0.0
    case.check_interval = 100
    return case, patches, lengths, dia


@lru_cache(maxsize=1)
def host_mesh(flow, nx, ny, nz, tets, sphere, batch):
    """The mesh as a program has it in hand: read (here generated) once, with its geometry."""
    c = dict(flow=flow, nx=nx, ny=ny, nz=nz, tets=tets, nodes=int(sphere))
    case, patches, lengths, _ = physics(c)
    # hex cavities are regular, as the benchmark's is (the reference's scheme does not hold on jittered ones)
    jitter = 0.10 if tets else 0.15 if flow != "cavity" else 0.0
    pm = meshgen.box_mesh(nx, ny, nz, lengths=lengths, tets=tets, jitter=jitter, jitter_seed=2, permute_seed=3,
                          patch_types=patches)
    hm = HostMesh.from_polymesh(pm, 0.01 if batch else case.visc, case.gamma, 0.0 if batch else case.fneq_min)
    return pm, hm, hm.geometry()


def mesh_of(c):
    return host_mesh(c["flow"], c["nx"], c["ny"], c["nz"], bool(c["tets"]), bool(c.get("nodes")),
                     c["kind"] == "batch")


def start_state(case, geo, n, rng):
    """The case's initial state with a smooth seeded disturbance, as a flow on its way has it."""
    x = np.stack([geo["cx"][:n], geo["cy"][:n], geo["cz"][:n]], 1)
    lo, hi = x.min(0), x.max(0)
    x = (x - lo) / np.maximum(hi - lo, 1e-30)
    k, ph = rng.uniform(1.0, 6.0, size=(4, 3)), rng.uniform(0, 2 * np.pi, size=4)
    wave = [np.sin(x @ k[q] + ph[q]) for q in range(4)]
    rho, u, v, w = case.initial_state(geo["cx"][:n], geo["cy"][:n], geo["cz"][:n])
    U = case.mach_no
    return rho + 1e-3 * wave[0], u + 0.02 * U * wave[1], v + 0.02 * U * wave[2], w + 0.02 * U * wave[3]


def sphere_nodes(c, case, lengths, dia, rng, n_nodes):
    """set_ibm arguments of a sphere in the upstream third, near the axis."""
    H = lengths[1]
    centre = (float(rng.uniform(0.5 * dia + 0.1 * H, max(lengths[0] / 3.0, 0.5 * dia + 0.2 * H))),
              0.5 * lengths[1] + float(rng.uniform(-1, 1)) * H / 16, 0.5 * lengths[2] + float(rng.uniform(-1, 1)) * H / 16)
    X, dA = objects.fibonacci_sphere(n_nodes, centre, 0.5 * dia)
    return dict(x_ref=X, x=X, stiffness=5.0, node_area=dA, dt=case.time_marching_step, h=1.0, kernel=1)


def inputs(c, seed):
    """Everything that the seed decides, as host arrays (shared by prepare and exact)."""
    rng = np.random.default_rng(seed)
    case, _, lengths, dia = physics(c)
    pm, hm, geo = mesh_of(c)
    n = pm.n_cells
    if c["kind"] == "solve":
        state = start_state(case, geo, n, rng)
        ibm = sphere_nodes(c, case, lengths, dia, rng, c["nodes"]) if c["nodes"] else None
        return dict(case=case, state=state, ibm=ibm)
    if c["kind"] == "batch":
        each = []
        for _ in range(c["cases"]):
            d = float(rng.uniform(6.0, 0.44 * c["ny"])) if c["spheres"] else 4.0
            k = pc.channel_case(re=float(rng.uniform(20.0, 200.0)) if c["spheres"] else float(rng.uniform(10.0, 40.0)),
                                length_scale=d, fneq_min=case.fneq_min)
            ibm = sphere_nodes(c, case, lengths, d, rng, objects.sphere_nodes_for_diameter(d)) if c["spheres"] else None
            each.append(dict(visc=k.visc, state=start_state(case, geo, n, rng), ibm=ibm))
        return dict(case=case, each=each)
    dia = float(rng.uniform(0.14, 0.44)) * lengths[1]
    centre = (lengths[0] * float(rng.uniform(0.2, 0.33)), 0.5 * lengths[1], 0.5 * lengths[2])
    x = mpnn.node_inputs(geo, n, centre, dia, float(rng.uniform(20.0, 200.0)))
    t = mpnn.targets(*start_state(case, geo, n, rng), case.mach_no)
    return dict(x=x, target=t, mask=mpnn.output_mask(n))


def prepare(case, seed):
    pm, hm, geo = mesh_of(case)
    d = inputs(case, seed)
    if case["kind"] == "solve":
        s = GpuSolver(hm, d["case"].params, d["case"].patches_for(pm.patch_names))
        s.set_state(*d["state"])
        if d["ibm"]:
            s.set_ibm(**d["ibm"])
        return dict(c=case, s=s)
    if case["kind"] == "batch":
        b = GpuBatch(hm, d["case"].params, d["case"].patches_for(pm.patch_names), [e["visc"] for e in d["each"]])
        b.set_tiling(case["block_cells"], case["cases_per_block"], 0)
        for k, e in enumerate(d["each"]):
            b.set_state(k, *e["state"])
            if e["ibm"]:
                b.set_ibm(k, **e["ibm"])
        return dict(c=case, s=b)
    src, dst, ef, _ = mpnn.graph_from_geometry(geo, pm.n_cells)
    net = mpnn.Mpnn(pm.n_cells, src, dst, ef, train=case["kind"] == "train")
    net.set_params(ws.load_params())
    return dict(d, c=case, s=net)


def kept(c, arrays):
    """Fields in the precision that the solver stores."""
    return [np.asarray(a, dtype=np.float32 if c["precision"] == "fp32" else np.float64) for a in arrays]


def run(state):
    c, s = state["c"], state["s"]
    if c["kind"] == "solve":
        r = s.run(c["steps"]) if c["call"] == "run" else s.run_noalloc(c["steps"])
        out = dict(fields=kept(c, s.state()), hist=kept(c, [r["hist"]])[0], steps=r["steps"], rc=r["rc"])
        if c["nodes"]:
            out["nodes"] = kept(c, s.ibm_state())
        return out
    if c["kind"] == "batch":
        rc, res = s.run(c["steps"])
        fields = np.empty((s.B, 4, s.N), dtype=np.float32 if c["precision"] == "fp32" else np.float64)
        for b in range(s.B):
            fields[b] = s.state(b)
        return dict(fields=fields, residual=kept(c, [[r["residual"] for r in res]])[0], rc=rc,
                    status=np.array([r["status"] for r in res]))
    if c["kind"] == "infer":
        return s.forward(state["x"])
    loss, grads = s.loss_grad(state["x"], state["target"], state["mask"])
    return dict(loss=loss, grads=grads)


def sizes(c):
    """(cells, faces, directed interior edges)"""
    n = (c["nx"], c["ny"], c["nz"])
    box = n[0] * n[1] * n[2]
    side = 2 * (n[0] * n[1] + n[1] * n[2] + n[0] * n[2])
    if c["tets"]:
        cells, inner = 6 * box, (24 * box - 2 * side) // 2
        return cells, inner + 2 * side, 2 * inner
    inner = (6 * box - side) // 2
    return box, inner + side, 2 * inner


def work(case):
    """Least traffic and arithmetic of one pass.  Solver, per RK stage: the state read and the next one written,
    the step's start state and the RK accumulator (8P + 12P per cell, P bytes a value; volume and time step 2P)
    and each face's indices and geometry once (8 + 10P); about 450 operations a face and 150 a cell.  A batch
    reads the geometry once for all its cases.  Network, per layer: node states read and written, edge inputs
    and indices read; two products per MLP, three times that with the backward pass."""
    n, f, e = sizes(case)
    if case["kind"] in ("solve", "batch"):
        P = 4 if case["precision"] == "fp32" else 8
        b = case.get("cases", 1)
        stages = 4 * case["steps"]
        return dict(bytes=stages * (b * n * 20 * P + n * 2 * P + f * (8 + 10 * P)) + b * n * 4 * P,
                    flops=stages * b * (450.0 * f + 150.0 * n))
    h = 64
    flops = 2.0 * n * (16 * h + h * h) + 2.0 * n * (h * h + h * 16)
    flops += 6 * (2.0 * e * (144 * h + h * h) + 2.0 * n * (128 * h + h * h))
    moved = n * 32 * 4 + 6 * (2 * n * h * 4 + e * (16 * 4 + 8))
    return dict(bytes=moved * (2 if case["kind"] == "train" else 1), flops=flops * (3 if case["kind"] == "train" else 1))


# ---------------------------------------------------------------------------
# the same results in 64 bits with plain torch
# ---------------------------------------------------------------------------

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
LATTICE = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)] + \
          [(a, b, c) for a in (1, -1) for b in (1, -1) for c in (1, -1)]


def f64(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEV)


class Flow:
    """Least-squares gradients, local-equilibrium fluxes and the four-stage update over the whole mesh at once."""

    def __init__(self, geo, n, p, patches, bpatch, lattice_dt=None):
        self.n, self.p = n, p
        self.own = torch.as_tensor(geo["owner"], device=DEV).long()
        nbr = torch.as_tensor(geo["nbr"], device=DEV).long()
        F, ni = len(self.own), int((geo["nbr"] < n).sum())
        self.ni = ni
        x = torch.stack([f64(geo[k]) for k in ("cx", "cy", "cz")], 1)
        self.x, self.vol, fc, self.fn, self.area = x, f64(geo["vol"]), f64(geo["fc"]), f64(geo["fn"]), f64(geo["area"])
        self.fdt = f64(geo["dt"]) if lattice_dt is None else lattice_dt
        self.nb = nbr[:ni]
        self.ro = x[self.own] - fc
        self.rn = x[nbr] - fc
        # patch values per boundary face
        q = torch.as_tensor(np.asarray(bpatch), device=DEV).long()
        col = lambda k: f64([P[k] for P in patches])[q]  # noqa: E731
        self.rt, self.vt = col("rho_type").long(), col("vel_type").long()
        assert all(P["rho_type"] in (1, 2, 3) and P["vel_type"] in (1, 2, 3) for P in patches)
        self.pv = torch.stack([col(k) for k in ("rho", "u", "v", "w")], 1)
        self.bo = self.own[ni:]
        self.dmag = (x[nbr[ni:]] - x[self.bo]).square().sum(1).sqrt()
        self.partner = self.bo.clone()
        move = f64([P["per_translate"] for P in patches])[q]
        for k in torch.nonzero((self.rt == 3) | (self.vt == 3))[:, 0].split(256):
            self.partner[k] = torch.cdist(x[self.bo[k]] + move[k], x[:n], compute_mode="donot_use_mm_for_euclid_dist").argmin(1)
        # least squares: weights of every (cell, other) pair
        cell, other = torch.cat([self.own, self.nb]), torch.cat([nbr, self.own[:ni]])
        face = torch.cat([torch.arange(F, device=DEV), torch.arange(ni, device=DEV)])
        sign = torch.cat([torch.ones(F, device=DEV, dtype=torch.float64), -torch.ones(ni, device=DEV, dtype=torch.float64)])
        d, nrm, sa = x[other] - x[cell], self.fn[face], self.area[face]
        dist = d.square().sum(1).sqrt()
        w = (2 * ((fc[face] - x[cell]) * nrm).sum(1) / (d * nrm).sum(1)) ** 2 * sa / dist
        most = lambda v: torch.zeros(n, dtype=torch.float64, device=DEV).scatter_reduce(0, cell, v, "amax")  # noqa: E731
        beta = torch.ones(n, dtype=torch.float64, device=DEV)
        if p["gradient_type"] == 1:
            beta = torch.clamp(2 / (2 * most(dist) * most(sa) / self.vol), max=1.0)
        elif p["gradient_type"] == 2:
            beta.zero_()
        bc = beta[cell, None]
        A = torch.zeros(n, 9, dtype=torch.float64, device=DEV)
        A.index_add_(0, cell, (bc[:, :, None] * w[:, None, None] * d[:, :, None] * d[:, None, :]).reshape(-1, 9))
        A[:, [0, 4, 8]] += (2 * (1 - beta) * self.vol)[:, None]
        rhs = bc * w[:, None] * d + (1 - bc) * nrm * (sign * sa)[:, None]
        a, b, c, dd, e, f, g, h, k = A.unbind(1)
        if p["lsq_exact_det"]:
            det = a * (e * k - f * h) - b * (dd * k - f * g) + c * (dd * h - e * g)
        else:  # the reference's expression
            det = a * (e * k - f * h) + b * (dd * k - f - g) + c * (dd * h - e * g)
        inv = torch.stack([e * k - f * h, c * h - b * k, b * f - c * e, f * g - dd * k, a * k - c * g, c * dd - a * f,
                           dd * h - e * g, b * g - a * h, a * e - b * dd], 1) / det[:, None]
        W = (inv.reshape(n, 3, 3)[cell] * rhs[:, None, :]).sum(2)
        self.Wo, self.Wn = W[:F], W[F:]
        # half the summed projected face areas of each cell
        self.cfl = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, cell, (nrm * sa[:, None]).abs().sum(1) / 2)
        # which side each lattice direction takes its values from
        self.side = [((e0 * self.fn[:, 0] + e1 * self.fn[:, 1] + e2 * self.fn[:, 2]) < 0)[:, None] for e0, e1, e2 in LATTICE]
        self.ceff = p["max_velocity"] * math.sqrt(1 - p["gamma"] + (p["gamma"] / math.sqrt(3) / p["max_velocity"]) ** 2)

    def by_type(self, r, v):
        """rho column from r[type], velocity columns from v[type]"""
        out = v[2].clone()
        for t in (1, 3):
            out = torch.where((self.vt == t).reshape(-1, *[1] * (out.dim() - 1)), v[t], out)
            r[2] = torch.where((self.rt == t).reshape(-1, *[1] * (r[2].dim() - 1)), r[t], r[2])
        out[:, 0] = r[2][:, 0]
        return out

    def ghosts(self, P, G=None):
        po, pp = P[self.bo], P[self.partner]
        if G is None:
            kinds = {1: 2 * self.pv - po, 2: po, 3: pp}
        else:
            nb, go = self.fn[self.ni:], G[self.bo]
            kinds = {1: (2 * (self.pv - po) / self.dmag[:, None])[:, :, None] * nb[:, None, :],
                     2: go * (1 - nb)[:, None, :], 3: G[self.partner]}
        return self.by_type(dict(kinds), kinds)

    def residual(self, P, visc, dt):
        n, ni, gam = self.n, self.ni, self.p["gamma"]
        other = torch.cat([P[self.nb], self.ghosts(P)])
        diff = other - P[self.own]
        G = torch.zeros(n, 12, dtype=torch.float64, device=DEV)
        G.index_add_(0, self.own, (diff[:, :, None] * self.Wo[:, None, :]).reshape(-1, 12))
        G.index_add_(0, self.nb, (-diff[:ni, :, None] * self.Wn[:, None, :]).reshape(-1, 12))
        G = G.reshape(n, 4, 3)
        go, gn = G[self.own], torch.cat([G[self.nb], self.ghosts(P, G)])
        pi = P[self.own] - (go * self.ro[:, None, :]).sum(2)
        pn = other - (gn * self.rn[:, None, :]).sum(2)
        p0 = 0.5 * (pi + pn)
        # boundary faces after the first: the patch's value, or the owner's taken to the face by the ghost's gradient
        b = slice(ni + 1, None)
        out = P[self.bo] - (gn[ni:] * self.ro[ni:, None, :]).sum(2)
        kinds = {1: self.pv, 2: out, 3: out}
        val = self.by_type(dict(kinds), kinds)[1:]
        pi[b] = val
        pn[b] = val
        p0[b] = val
        S = torch.zeros(len(self.own), 10, dtype=torch.float64, device=DEV)
        for k, e in enumerate(LATTICE):
            wk = 2.0 / 9.0 if k == 0 else 1.0 / 9.0 if k < 7 else 1.0 / 72.0
            if k == 0:
                q = p0
            else:
                along = lambda g: e[0] * g[:, :, 0] + e[1] * g[:, :, 1] + e[2] * g[:, :, 2]  # noqa: B023,E731
                q = torch.where(self.side[k], pn - along(gn) * dt[:, None], pi - along(go) * dt[:, None])
            eu = e[0] * q[:, 1] + e[1] * q[:, 2] + e[2] * q[:, 3]
            feq = wk * q[:, 0] * (1 + 3 * eu + (4.5 * eu * eu - 1.5 * (q[:, 1:] ** 2).sum(1)) / gam)
            for col, m in enumerate((1, *e, e[0] * e[0], e[1] * e[1], e[2] * e[2], e[0] * e[1], e[0] * e[2], e[1] * e[2])):
                if m:
                    S[:, col] += m * feq
        tau, rho = 3 * visc / gam / dt, S[:, 0]
        u = S[:, 1:4] / rho[:, None]
        M = (1 - tau)[:, None, None] * rho[:, None, None] * (torch.eye(3, dtype=torch.float64, device=DEV) / 3
                                                              + u[:, :, None] * u[:, None, :] / gam)
        M = M + tau[:, None, None] * S[:, [4, 7, 8, 7, 5, 9, 8, 9, 6]].reshape(-1, 3, 3)
        nA = self.fn * self.area[:, None]
        flux = torch.cat([(S[:, 1:4] * nA).sum(1, keepdim=True), (M * nA[:, None, :]).sum(2)], 1)
        R = torch.zeros(n, 4, dtype=torch.float64, device=DEV)
        R.index_add_(0, self.own, -flux)
        R.index_add_(0, self.nb, flux[:ni])
        return R / self.vol[:, None]

    def time_step(self, visc, rho, u):
        eig = (u.abs() + self.ceff) * self.cfl / self.p["gamma"]
        eig = eig + 4 * (2 * visc / self.p["gamma"] / rho / self.vol) * self.cfl ** 2
        dt = self.p["cfl"] * self.vol / eig
        return torch.full_like(dt, float(dt.min())) if self.p["time_stepping"] == 2 else dt

    def advance(self, state, ibm, visc, steps, face_dt):
        P = torch.stack([f64(a) for a in state], 1)
        Q, dt, hist = P.clone(), self.time_step(visc, P[:, 0], P[:, 1]), []
        body = Body(ibm, self.x[: self.n], self.vol) if ibm else None
        for _ in range(steps):
            force = body.step(P) if body else None
            T = Q.clone()
            for al, be in ((1.0, 1 / 6), (0.5, 1 / 3), (0.5, 1 / 3), (1.0, 1 / 6)):
                R = self.residual(P, visc, face_dt)
                if force is not None:
                    R[:, 1:] += force
                K = R.clone()
                K[:, 1] += self.p["force"]
                T = T + be * dt[:, None] * K
                P = Q + al * dt[:, None] * K
                P = torch.cat([P[:, :1], P[:, 1:] / P[:, :1]], 1)
            Q = T
            P = torch.cat([T[:, :1], T[:, 1:] / T[:, :1]], 1)
            dt = self.time_step(visc, P[:, 0], P[:, 1])
            r = (R.square().sum(0) / self.n).sqrt()
            r[0] /= self.p["ref_rho"]
            r[1:] /= self.p["ref_rho"] * self.p["max_velocity"]
            hist.append(r)
        return P, torch.stack(hist), body


class Body:
    """Immersed nodes: 4-point Peskin kernel, moved with the flow and pulled back by springs."""

    def __init__(self, a, x, vol):
        self.ref, self.x0, self.x, self.vol, self.a = f64(a["x_ref"]), f64(a["x"]), x, vol, a
        lo, hi = self.ref.min(0).values - 3.5, self.ref.max(0).values + 3.5
        near = torch.nonzero(((x > lo) & (x < hi)).all(1))[:, 0]
        node, cell = [], []
        for k in torch.arange(len(self.ref), device=DEV).split(64):
            hit = torch.nonzero(((x[near][None] - self.ref[k][:, None]).abs() < 3.0).all(2))
            node.append(k[hit[:, 0]])
            cell.append(near[hit[:, 1]])
        self.node, self.cell = torch.cat(node), torch.cat(cell)
        self.weights()

    def weights(self):
        r = (self.x[self.cell] - self.x0[self.node]).abs()
        one = (3 - 2 * r + torch.clamp(1 + 4 * r - 4 * r * r, min=0).sqrt()) / 8
        two = (5 - 2 * r - torch.clamp(-7 + 12 * r - 4 * r * r, min=0).sqrt()) / 8
        self.d = torch.where(r <= 1, one, torch.where(r <= 2, two, torch.zeros_like(r))).prod(1)
        wv = self.d * self.vol[self.cell]
        self.s = torch.zeros(len(self.ref), dtype=torch.float64, device=DEV).index_add_(0, self.node, wv)
        return wv

    def step(self, P):
        wv = self.weights()
        U = torch.zeros_like(self.ref).index_add_(0, self.node, wv[:, None] * P[self.cell, 1:])
        self.vel = U / self.s[:, None]
        self.x0 = self.x0 + self.vel * self.a["dt"]
        self.force = -self.a["stiffness"] * self.a["node_area"] * (self.x0 - self.ref)
        self.weights()
        f = torch.zeros(len(self.vol), 3, dtype=torch.float64, device=DEV)
        return f.index_add_(0, self.cell, self.force[self.node] * (self.d / self.s[self.node])[:, None])


def net_exact(c, d, geo, n):
    src, dst, ef, _ = mpnn.graph_from_geometry(geo, n)
    src, dst, ef = torch.as_tensor(src, device=DEV).long(), torch.as_tensor(dst, device=DEV).long(), f64(ef)
    train = c["kind"] == "train"
    w = f64(ws.load_params()).requires_grad_(train)
    parts, at = [], 0
    for _, k, o in mpnn.mlp_shapes():
        for shape in ((k, 64), (64,), (64, o), (o,)):
            parts.append(w[at:at + int(np.prod(shape))].reshape(shape))
            at += int(np.prod(shape))

    def mlp(q, z):
        w1, b1, w2, b2 = parts[4 * q:4 * q + 4]
        return torch.nn.functional.silu(z @ w1 + b1) @ w2 + b2

    deg = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, dst, torch.ones_like(dst, dtype=torch.float64))
    with torch.set_grad_enabled(train):
        h = mlp(0, f64(d["x"]))
        for layer in range(6):
            m = mlp(1 + 2 * layer, torch.cat([h[dst], h[src], ef], 1))
            a = torch.zeros_like(h).index_add(0, dst, m) / deg.clamp(min=1)[:, None]
            h = h + mlp(2 + 2 * layer, torch.cat([h, a], 1))
        y = mlp(13, h)
        if not train:
            return y
        loss = (((y - f64(d["target"])) * f64(d["mask"])) ** 2).sum() / float(d["mask"].sum())
        loss.backward()
    return dict(loss=float(loss.detach()), grads=w.grad)


def exact(case, seed):
    # about 20 seconds of torch at most
    if case["kind"] in ("solve", "batch") and sizes(case)[0] * case["steps"] * case.get("cases", 1) > 6e7:
        return None
    pm, hm, geo = mesh_of(case)
    n = pm.n_cells
    d = inputs(case, seed)
    if case["kind"] in ("infer", "train"):
        return net_exact(case, d, geo, n)
    p = d["case"].params
    flow = Flow(geo, n, p, d["case"].patches_for(pm.patch_names), hm.bface_patch())
    if case["kind"] == "solve":
        P, hist, body = flow.advance(d["state"], d["ibm"], p["visc"], case["steps"], flow.fdt)
        out = dict(fields=list(P.T), hist=hist, steps=None, rc=None)
        if body:
            out["nodes"] = [body.x0, body.vel, body.force]
        return out
    fields, last = [], []
    for e in d["each"]:
        face_dt = flow.fdt
        if p["fneq_min"]:
            face_dt = torch.clamp(0.5 * flow.area.sqrt(), max=3 * e["visc"] / p["gamma"] / p["fneq_min"])
        P, hist, _ = flow.advance(e["state"], e["ibm"], e["visc"], case["steps"], face_dt)
        fields.append(P.T)
        last.append(hist[-1])
    return dict(fields=torch.stack(fields), residual=torch.stack(last), rc=None, status=None)
