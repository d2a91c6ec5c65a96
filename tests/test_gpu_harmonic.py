"""The far field through spherical harmonics (harmonic.hpp) against the direct
FP64 sums, where its kernels can go wrong: grids whose cell count is no
multiple of the eight cells of a tile, unequal edges, empty cells, a cell of
several passes (more than 128 atoms), atoms outside their cell's ball, one
system on each side of every ring, azimuth and degree step the tolerances
reach, and both widths of the evaluation (under and over 512 workgroups).

Bars, against the direct sums in FP64.  FP64: the terms left out stay under
1e-15 of a wave and the recurrences' rounding under 1e-13, so 1e-11 of the
fields' norm.  Mixed: the bars of the mixed path, 1e-5 of the largest S(k)
and 2e-6 of the fields' norm.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _system(box, spacing, seed):
    rng = np.random.default_rng(seed)
    axes = [np.arange(spacing / 2, b, spacing) for b in box]
    p = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    p = p + rng.uniform(-0.3, 0.3, p.shape)
    p = np.clip(p, 0.0, None)
    # empty cells: a corner and its neighbour
    p = p[~((p[:, 0] < 18) & (p[:, 1] < 9) & (p[:, 2] < 9))]
    # one crowded cell, and atoms 3 A outside the box
    p = np.concatenate([p, rng.uniform(18.1, 26.9, (150, 3))])
    p[::997, 0] = -3.0
    q = rng.uniform(-1.0, 1.0, len(p))
    return [np.ascontiguousarray(a) for a in (p[:, 0], p[:, 1], p[:, 2], q)]


def _far(h, box, tol, ct, direct, torch, g):
    d = [torch.as_tensor(a, dtype=torch.float64, device="cuda") for a in h]
    f = g.GLSTForce(h[0].size, tol, box, rcut=9.0, ct=ct)
    if direct:
        f.set_option("lr_atom_groups", 0)
    f.assign_atoms(*d)
    f.calc_sf()
    if not direct:
        f.set_option("sf_cheb", 0)  # the later stages follow the S at hand
    s = f.sf()
    f.sum_rmt_sf()
    f.calc_lr_ef()
    ef = [t.cpu().numpy() for t in f.get_ef()]
    f.close()
    return s, ef


@pytest.mark.parametrize("box,spacing,tol", [
    ((53.0, 40.0, 62.0), 2.6, 1e-6),
    ((53.0, 40.0, 62.0), 2.6, 1e-5),
    ((44.0, 44.0, 44.0), 2.2, 2e-5),
    ((80.0, 71.0, 89.0), 3.0, 1e-4)])
def test_far_field_matches_direct_sums(cuda, box, spacing, tol):
    import torch
    import glst_amd as g
    h = _system(box, spacing, 7)
    s0, ef0 = _far(h, box, tol, "double", True, torch, g)
    scale = max(np.abs(a).max() for a in s0)
    for ct, sbar, bar in (("double", 1e-11, 1e-11), ("float", 1e-5, 2e-6)):
        s, ef = _far(h, box, tol, ct, False, torch, g)
        err = max(np.abs(a - b).max() for a, b in zip(s, s0)) / scale
        assert err < sbar, (ct, err)
        assert rel_err(ef[:3], ef0[:3]) < bar, ct
        assert rel_err(ef[3:], ef0[3:]) < bar, ct
