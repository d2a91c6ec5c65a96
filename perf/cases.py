"""Workloads whose speed is followed: what a program that uses this framework
has it do, through the public Python entry points, from the smallest call to
the largest.

A case is a dict of plain values:

  kind "force"  one handle (GLSTForce): clear, one force step, results back in
                the caller's atom order, as an MD program does every step;
  kind "batch"  many independent boxes in one GLSTBatch, as an ensemble does;
  kind "serve"  requests of mixed sizes handed to a GLSTServer and drained, as
                a client of the serving loop does.

ct "double" is the plain FP64 path; its results stay FP64.  ct "float" is the
mixed path, whose pair sums and phases are FP32: a program that chooses it
keeps its forces and energies in FP32, so those cases end with that
conversion.

Inputs are the rigid-water boxes of the benchmark (uniform centres, random
orientations, optional Na+/Cl- pairs) or, for boxes that are not cubic,
charges of +-1 on a jittered lattice as in the parity tests.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(
    os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
    "gauss-legendre-spherical-t_amd"))
import glst_amd as glst  # noqa: E402

WATER_DENSITY = 0.0334  # molecules per cubic Angstrom
SPACING = 2.6           # lattice spacing of the +-1 charges, Angstrom


def water_edge(nwater):
    return (nwater / WATER_DENSITY) ** (1.0 / 3.0)


def force(name, ct, nwater, tol, rcut, box=0.0, nion=0, stages=False,
          graph=0):
    """box 0: the cube that holds nwater molecules at liquid density."""
    c = dict(kind="force", ct=ct, nwater=nwater, nion=nion,
             box=float(box or water_edge(nwater)), rcut=float(rcut), tol=tol,
             stages=stages, graph=graph)
    return dict(c, name=name) if name else c


def lattice(name, ct, box, tol, rcut, stages=False):
    c = dict(kind="force", ct=ct, nwater=0, nion=0, lx=float(box[0]),
             ly=float(box[1]), lz=float(box[2]), rcut=float(rcut), tol=tol,
             stages=stages, graph=0)
    return dict(c, name=name) if name else c


def ensemble(name, kind, ct, nsys, smallest, largest, sizes, tol, rcut=9.0):
    """nsys boxes, waters log-uniform in [smallest, largest]; `sizes` seeds
    the sizes (they belong to the case, the positions to the run's seed)."""
    c = dict(kind=kind, ct=ct, nsys=nsys, smallest=smallest, largest=largest,
             sizes=sizes, tol=tol, rcut=float(rcut))
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest useful call: 300 charges on a 2^3 grid, where no cell
        # has a far field and launches are all there is
        force("near_only_300", "float", 100, 2e-5, 9),
        # a 1,000-water box (the driver's small configuration), both paths
        force("water_1000_mixed", "float", 1000, 1e-5, 9, box=31.04),
        force("water_1000_double", "double", 1000, 1e-5, 9, box=31.04),
        # a box with three different edges, driven stage by stage as the
        # reference's driver does, on the FP64 path
        lattice("slab_stages_double", "double", (52.0, 28.0, 70.0), 1e-5, 9,
                stages=True),
        # an MD loop on one mid-sized box: the captured step is replayed
        force("water_10000_graph", "float", 10000, 2e-5, 9, graph=1),
        # tight tolerance: many cubature nodes per atom, FP64
        force("water_3300_tight_double", "double", 3300, 1e-6, 9),
        # the headline box, 288,000 charges, both paths
        force("water_288k_mixed", "float", 96000, 1e-4, 10, box=142.0),
        force("water_288k_double", "double", 96000, 1e-4, 10, box=142.0),
        # the largest single system: 1.0M charges with ions
        force("water_ions_1m_mixed", "float", 333000, 1e-5, 12, box=215.0,
              nion=898),
        # ensembles of 100 to 10,000 waters, log-uniform, in one batch
        ensemble("batch_64_mixed", "batch", "float", 64, 100, 10000, 4, 2e-5),
        ensemble("batch_12_double", "batch", "double", 12, 100, 4000, 5,
                 2e-5),
        # a burst of served requests of the same kind of sizes
        ensemble("serve_16_mixed", "serve", "float", 16, 100, 10000, 6, 2e-5),
    ]


def log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    ct = rng.choice(("float", "double"))
    if pick < 0.4:      # boxes of up to 10,000 waters at the tight settings
        nw = log_between(rng, 100, 10000)
        return force(None, ct, nw, rng.choice((2e-5, 1e-5, 1e-6)),
                     rng.choice((8.0, 9.0, 10.0)),
                     nion=rng.choice((0, 0, 7)), stages=rng.random() < 0.25,
                     graph=int(rng.random() < 0.25))
    if pick < 0.6:      # large boxes
        top = 200000 if ct == "float" else 96000
        nw = log_between(rng, 10000, top)
        return force(None, ct, nw, 1e-4, 10.0, nion=rng.choice((0, 101)))
    if pick < 0.75:     # boxes that are not cubic
        box = [round(rng.uniform(25.0, 75.0), 2) for _ in range(3)]
        return lattice(None, ct, box, rng.choice((2e-5, 1e-5)), 9.0,
                       stages=rng.random() < 0.5)
    kind = rng.choice(("batch", "serve"))
    top = 12 if ct == "double" else 16 if kind == "serve" else 48
    return ensemble(None, kind, ct, log_between(rng, 1, top), 100,
                    10000 if ct == "float" else 4000, rng.randrange(1 << 20),
                    2e-5)


# ---- inputs ------------------------------------------------------------------

def on_gpu(arrays):
    return [torch.as_tensor(a, dtype=torch.float64, device="cuda")
            for a in arrays]


def lattice_charges(box, seed):
    """Neutral +-1 charges on a jittered lattice filling the box, the minimum
    of every coordinate at 0."""
    rng = np.random.default_rng(seed)
    axes = [np.arange(SPACING / 2, b, SPACING) for b in box]
    p = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    p = p + rng.uniform(-0.3, 0.3, p.shape)
    p -= p.min(axis=0)
    q = np.where(np.arange(len(p)) % 2 == 0, 1.0, -1.0)
    rng.shuffle(q)
    return [np.ascontiguousarray(p[:, d]) for d in range(3)] + [q]


def box_of(case):
    return ((case["lx"], case["ly"], case["lz"]) if "lx" in case
            else (case["box"],) * 3)


def systems(case, seed):
    """[(box edges, (x, y, z, q))] of the case, on the host."""
    if case["kind"] == "force":
        box = box_of(case)
        if "lx" in case:
            return [(box, lattice_charges(box, seed))]
        return [(box, glst.make_water_box(case["nwater"], case["box"],
                                          seed=seed + 1, nion=case["nion"]))]
    out = []
    for s, nw in enumerate(waters_of(case)):
        edge = water_edge(nw)
        out.append(((edge,) * 3, glst.make_water_box(
            nw, edge, seed=1000 * (seed + 1) + s)))
    return out


def waters_of(case):
    rng = np.random.default_rng(case["sizes"])
    lo, hi = math.log(case["smallest"]), math.log(case["largest"])
    return [int(round(math.exp(v))) for v in
            rng.uniform(lo, hi, case["nsys"])]


def prepare(case, seed):
    sets = systems(case, seed)
    state = dict(case=case)
    if case["kind"] == "force":
        box, arrays = sets[0]
        n = len(arrays[0])
        f = glst.GLSTForce(n, case["tol"], box, rcut=case["rcut"],
                           ct=case["ct"])
        f.set_option("graph", case["graph"])
        state.update(handle=f, inputs=on_gpu(arrays),
                     out=torch.empty(4, n, dtype=torch.float64,
                                     device="cuda"))
    elif case["kind"] == "batch":
        natoms = [len(a[0]) for _, a in sets]
        b = glst.GLSTBatch(natoms, [box for box, _ in sets], case["rcut"],
                           case["tol"], ct=case["ct"])
        packed = [np.concatenate([a[d] for _, a in sets]) for d in range(4)]
        state.update(handle=b, inputs=on_gpu(packed))
    else:
        srv = glst.GLSTServer(case["tol"], 16 << 30, max_batch=8,
                              ct=case["ct"])
        requests = []
        for box, arrays in sets:
            d = on_gpu(arrays)
            requests.append((box, d, [torch.empty_like(d[0])
                                      for _ in range(4)]))
        state.update(handle=srv, requests=requests)
    return state


# ---- one pass ----------------------------------------------------------------

def results(case, arrays):
    """The mixed path's results are kept in FP32 (see the top)."""
    if case["ct"] == "float":
        arrays = [a.float() for a in arrays]
    return tuple(arrays)


def run(state):
    case, h = state["case"], state["handle"]
    if case["kind"] == "serve":
        for box, d, o in state["requests"]:
            h.submit(box, case["rcut"], *d, *o)
        while h.pending():
            h.step()
        h.completed()
        return [results(case, o) for _, _, o in state["requests"]]
    h.zero_ef()
    if case["kind"] == "force" and case["stages"]:
        h.assign_atoms(*state["inputs"])
        h.calc_sf()
        h.sum_rmt_sf()
        h.calc_lr_ef()
        h.calc_sr_ef()
        h.comm_ef()
    else:
        h.calc_ener_force(*state["inputs"])
    if case["kind"] == "batch":
        return results(case, h.get_ef())
    h.get_ef(out=list(state["out"].unbind(0)))
    return tuple(results(case, [state["out"]])[0].unbind(0))


# ---- what a pass cannot do without -------------------------------------------

def node_count(ct, box, rcut, tol):
    """(cells, cubature nodes) of one system."""
    n = glst.grid_dims(1 if ct == "float" else 0, *box, rcut)
    cells = n[0] * n[1] * n[2]
    if min(n) <= 2:
        return cells, 0
    g = glst.alpha_groups(*n, rcut, rcut, rcut, tol)
    nodes = 0
    for r, a, z in zip(g["rmax"], g["alpha"], g["zcut"]):
        order = glst.select_gl_order(tol, r, a, z)
        _, dirs = glst.select_spherical_degree(order, tol, r, a, z)
        nodes += order // 2 * dirs
    return cells, nodes


def sizes_of(case):
    if case["kind"] != "force":
        return [((water_edge(nw),) * 3, 3 * nw) for nw in waters_of(case)]
    box = box_of(case)
    if "lx" in case:
        n = math.prod(len(np.arange(SPACING / 2, b, SPACING)) for b in box)
    else:
        n = 3 * case["nwater"] + 2 * case["nion"]
    return [(box, n)]


def work(case):
    """Bytes: x, y, z, q in, forces and energy out.  Operations: 20 for each
    pair of atoms in neighbouring cells, once, and for each (cell, cubature
    node) one complex multiply-add into the sums and one out of them."""
    out = 4 if case["ct"] == "float" else 8
    nbytes = flops = 0.0
    for box, n in sizes_of(case):
        cells, nodes = node_count(case["ct"], box, case["rcut"], case["tol"])
        nbytes += n * 4 * (8 + out)
        flops += 10.0 * n * n * 27.0 / max(cells, 27) + 16.0 * cells * nodes
    return {"bytes": nbytes, "flops": flops}


# ---- the same results from all pairs in FP64 ---------------------------------

def all_pairs(x, y, z, q):
    """en_i = sum_j q_i q_j / r_ij, F_i = sum_j q_i q_j (r_i - r_j) / r_ij^3."""
    n = x.numel()
    out = [torch.empty_like(x) for _ in range(4)]
    step = max(1, min(n, (1 << 27) // n))
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [c[a:b, None] - c[None, :] for c in (x, y, z)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        i = torch.arange(a, b, device=x.device)
        r2[i - a, i] = math.inf
        w = q[None, :] * r2.rsqrt()
        out[3][a:b] = q[a:b] * w.sum(1)
        w /= r2
        for k in range(3):
            out[k][a:b] = q[a:b] * d[k].mul_(w).sum(1)
    return out


def exact(case, seed):
    """The sums that the method approximates within its tolerance; none for
    the largest box, whose 10^12 pairs take too long."""
    sizes = [n for _, n in sizes_of(case)]
    if sum(n * n for n in sizes) > 2e11:
        return None
    each = [tuple(all_pairs(*on_gpu(a))) for _, a in systems(case, seed)]
    if case["kind"] == "serve":
        return each
    return tuple(torch.cat([e[k] for e in each]) for k in range(4))
