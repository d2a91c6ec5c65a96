"""Which far field a handle takes, and that every route gives the same fields:
grids with one long edge, captured and eager; dilute systems.

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
