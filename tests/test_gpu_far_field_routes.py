"""Which far field a handle takes, and that every route gives the same fields:
grids with one long edge, captured and eager; dilute systems; global tables;
the matrix-core shell sums of expanded grids with unequal edges; most azimuths.

lr_blocks cuts the direct sums' back-projection into other partial sums and
has no effect on the expansion, so "the same bits under another lr_blocks"
tells which ran.  Bars are those of the mixed path, 2e-6 of the fields' norm.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def lattice(box, spacing, seed):
    rng = np.random.default_rng(seed)
    axes = [np.arange(spacing / 2, b, spacing) for b in box]
    p = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    p = p + rng.uniform(-0.3, 0.3, p.shape)
    q = rng.uniform(-1.0, 1.0, len(p))
    return [np.ascontiguousarray(p[:, d]) for d in range(3)] + [q]


def handle(g, torch, h, box, tol, ct="float", rcut=9.0, **options):
    f = g.GLSTForce(h[0].size, tol, box, rcut=rcut, ct=ct)
    for k, v in options.items():
        f.set_option(k, v)
    d = [torch.as_tensor(a, dtype=torch.float64, device="cuda") for a in h]
    return f, d


def step(f, d):
    f.zero_ef()
    f.calc_ener_force(*d)
    return [t.cpu().numpy() for t in f.get_ef()]


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def expands(f, d):
    """Whether this handle's steps expand the far field."""
    keep, a = f.get_option("lr_blocks"), step(f, d)
    f.set_option("lr_blocks", 1)
    b = step(f, d)
    f.set_option("lr_blocks", keep)
    return same(a, b)


@pytest.mark.parametrize("nz,want", [(24, True), (38, False)])
def test_long_grids_captured_and_eager(cuda, nz, want):
    """16 x 16 cells and a long third edge: at 24 cells the expansion's shell
    sums run on LDS tables, at 38 only the direct sums' fields fit a kernel in
    LDS.  A captured step, from the first call on, gives the eager step's bits
    and allocates nothing."""
    import torch
    import glst_amd as g
    box, tol = (144.0, 144.0, 9.0 * nz), 1e-4
    h = lattice(box, 3.0, 3)
    f, d = handle(g, torch, h, box, tol, graph=1)
    assert tuple(f.info().ncell) == (16, 16, nz)
    before = f.info().device_bytes
    captured = [step(f, d) for _ in range(3)]
    assert f.info().device_bytes == before
    f.close()
    f, d = handle(g, torch, h, box, tol)
    eager = step(f, d)
    assert expands(f, d) == want
    f.close()
    for c in captured:
        assert same(c, eager)
    f, d = handle(g, torch, h, box, tol, ct="double")
    ref = step(f, d)
    f.close()
    assert rel_err(eager[:3], ref[:3]) < 2e-6
    assert rel_err(eager[3:], ref[3:]) < 2e-6


@pytest.mark.parametrize("ct,n,spacing,tol,want", [
    ("float", 12, 3.0, 1e-4, True), ("float", 12, 4.0, 1e-4, False),
    ("float", 8, 4.0, 1e-5, True),
    ("double", 8, 3.0, 1e-5, True), ("double", 8, 4.0, 1e-5, False)])
def test_dilute_systems_keep_direct_sums(cuda, ct, n, spacing, tol, want):
    """Atoms per cell of n^3 grids: 27 (spacing 3) and 11.4 (spacing 4)."""
    import torch
    import glst_amd as g
    box = (9.0 * n - 0.5,) * 3
    h = lattice(box, spacing, 5)
    f, d = handle(g, torch, h, box, tol, ct=ct)
    assert f.info().ncell_total == n ** 3
    assert expands(f, d) == want
    f.close()


@pytest.mark.parametrize("ct,bar", [("double", 1e-11), ("float", 2e-6)])
def test_global_tables_on_node_major_fields(cuda, ct, bar):
    """17 x 18 x 31 cells, whose shell-sum tables fit no LDS (nor do the
    matrix-core slices): the expansion through the tables in global memory,
    tiles of 16 cells in z with a remainder, against the FP64 direct sums."""
    import torch
    import glst_amd as g
    box, tol = (152.0, 161.0, 278.0), 1e-4
    h = lattice(box, 2.95, 9)
    f, d = handle(g, torch, h, box, tol, ct=ct)
    assert tuple(f.info().ncell) == (17, 18, 31)
    assert expands(f, d)
    f.assign_atoms(*d)
    f.calc_sf()
    f.sum_rmt_sf()
    r = f.rmt()
    ef = step(f, d)
    f.close()
    f, d = handle(g, torch, h, box, tol, ct="double", lr_atom_groups=0)
    f.assign_atoms(*d)
    f.calc_sf()
    f.sum_rmt_sf()
    r0 = f.rmt()
    ef0 = step(f, d)
    f.close()
    scale = max(np.abs(a).max() for a in r0)
    assert max(np.abs(a - b).max() for a, b in zip(r, r0)) < \
        (1e-11 if ct == "double" else 1e-5) * scale
    assert rel_err(ef[:3], ef0[:3]) < bar
    assert rel_err(ef[3:], ef0[3:]) < bar


def fields(f, d):
    f.assign_atoms(*d)
    f.calc_sf()
    s = f.sf()
    f.sum_rmt_sf()
    r = f.rmt()
    return s, r, step(f, d)


def off(a, b):
    return max(np.abs(x - y).max() for x, y in zip(a, b)) / \
        max(np.abs(y).max() for y in b)


# 12 x 13 x 15 cells: matrix-core shell sums whose x and z axes differ, and
# 2,340 workgroups of the evaluation, which takes four waves from 2,048 on.
# 6^3 cells at tol 3e-7: the most azimuths (59 half azimuths) and, mixed, the
# most degrees (40) the kernels take.
# FP64 terms left out stay under 1e-15 of a wave and sums of up to 56 terms of
# a recurrence round under 1e-13; 1e-12 leaves room for the cancellation of a
# neutral system.  Mixed: the bars of the path.
@pytest.mark.parametrize("box,spacing,tol,ncell", [
    ((107.5, 116.5, 134.5), 3.0, 1e-4, (12, 13, 15)),
    ((46.2, 46.2, 46.2), 2.3, 3e-7, (6, 6, 6))])
def test_expansion_matches_direct_sums(cuda, box, spacing, tol, ncell):
    import torch
    import glst_amd as g
    h = lattice(box, spacing, 17)
    f, d = handle(g, torch, h, box, tol, ct="double", lr_atom_groups=0)
    s0, r0, ef0 = fields(f, d)
    f.close()
    for ct, sbar, bar in (("double", 1e-12, 1e-12), ("float", 1e-5, 2e-6)):
        f, d = handle(g, torch, h, box, tol, ct=ct)
        assert tuple(f.info().ncell) == ncell
        assert expands(f, d)
        s, r, ef = fields(f, d)
        f.close()
        assert off(s, s0) < sbar, ct
        assert off(r, r0) < sbar, ct
        assert rel_err(ef[:3], ef0[:3]) < bar, ct
        assert rel_err(ef[3:], ef0[3:]) < bar, ct
        # the same system in a batch beside a small one
        small = lattice((31.0, 40.0, 36.0), 2.6, 3)
        n = [h[0].size, small[0].size]
        b = g.GLSTBatch(n, [box, (31.0, 40.0, 36.0)], 9.0, tol, ct=ct)
        packed = [torch.as_tensor(np.concatenate([x, y]), dtype=torch.float64,
                                  device="cuda") for x, y in zip(h, small)]
        b.zero_ef()
        b.calc_ener_force(*packed)
        got = [t.cpu().numpy()[:n[0]] for t in b.get_ef()]
        b.close()
        assert rel_err(got[:3], ef0[:3]) < bar, ct
        assert rel_err(got[3:], ef0[3:]) < bar, ct


@pytest.mark.parametrize("ct,bar", [("double", 1e-12), ("float", 2e-6)])
@pytest.mark.parametrize("tol,crowd", [(2e-5, 3), (2e-5, 1000), (1e-5, 70)])
def test_atoms_outside_their_ball(cuda, ct, bar, tol, crowd):
    """Atoms beyond a corner of the box, which the binning puts into the corner
    cell but whose plane waves its expansion does not hold: 3 and 70 of them
    with the nodes shared out to workgroups (one or two lists of 64), 1,000 in one
    cell that one workgroup takes; and one across the opposite corner."""
    import torch
    import glst_amd as g
    box = (53.0, 49.0, 62.0)
    h = lattice(box, 2.6, 21)
    rng = np.random.default_rng(4)
    out = rng.uniform(-3.5, -0.5, (crowd, 3))
    out = np.concatenate([out, [[54.5, 54.5, 63.5]]])
    q = rng.uniform(-1.0, 1.0, len(out))
    h = [np.concatenate([a, b]) for a, b in zip(h, [*out.T, q])]
    f, d = handle(g, torch, h, box, tol, ct="double", lr_atom_groups=0)
    f.assign_atoms(*d)
    f.calc_sf()
    f.sum_rmt_sf()
    f.zero_ef()
    f.calc_lr_ef()
    far0 = [t.cpu().numpy() for t in f.get_ef()]
    f.close()
    f, d = handle(g, torch, h, box, tol, ct=ct)
    assert expands(f, d)
    for _ in range(2):
        f.assign_atoms(*d)
        f.calc_sf()
        f.sum_rmt_sf()
        f.zero_ef()
        f.calc_lr_ef()
        far = [t.cpu().numpy() for t in f.get_ef()]
        n = crowd + 1  # these atoms alone, then all
        assert rel_err([a[-n:] for a in far[:3]],
                       [a[-n:] for a in far0[:3]]) < bar
        assert rel_err([far[3][-n:]], [far0[3][-n:]]) < bar
        assert rel_err(far[:3], far0[:3]) < bar
        assert rel_err(far[3:], far0[3:]) < bar
    f.close()


@pytest.mark.parametrize("ct", ["double", "float"])
def test_captured_expanded_steps_replay(cuda, ct):
    """A handle and a batch (two expanded systems on their own streams beside a
    small one) captured: every replay gives the eager step's bits, with eager
    work of the same handle type in between."""
    import torch
    import glst_amd as g
    boxes = [(53.0, 49.0, 62.0), (46.2, 46.2, 46.2), (31.0, 40.0, 36.0)]
    tol = 2e-5
    sets = [lattice(b, 2.4, 30 + i) for i, b in enumerate(boxes)]
    f, d = handle(g, torch, sets[0], boxes[0], tol, ct=ct)
    assert expands(f, d)
    eager = step(f, d)
    e, _ = handle(g, torch, sets[0], boxes[0], tol, ct=ct, graph=1)
    for _ in range(3):
        assert same(step(e, d), eager)
        assert same(step(f, d), eager)
    e.close()
    f.close()
    n = [h[0].size for h in sets]
    packed = [torch.as_tensor(np.concatenate([h[k] for h in sets]),
                              dtype=torch.float64, device="cuda")
              for k in range(4)]
    out = {}
    batches = {v: g.GLSTBatch(n, boxes, 9.0, tol, ct=ct) for v in (0, 1)}
    batches[1].set_option("graph", 1)
    for _ in range(3):
        for v, b in batches.items():
            got = step(b, packed)
            assert same(got, out.setdefault(v, got))
    assert same(out[0], out[1])
    for b in batches.values():
        b.close()
