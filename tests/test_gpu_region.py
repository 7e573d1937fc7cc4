"""The region voxel kernels (8 x 8 x 8 voxels per workgroup, 4 x 4 x 4 per
subtile) where they can go wrong: grids one voxel short of and one beyond a
subtile or region, voxels so coarse that a region spans more link cells
than its table holds (the per-voxel walk takes over at one voxel per lattice
parameter), fine ones, and atom sets dense enough for several passes of staged
candidates and several chunks of records.

Against the oracle: members and nearest ranges exact (they are evaluated with
the reference's FP64 expression), phase factors to 1e-12 and densities to
1e-14, the bounds of the field tests of test_gpu_parity.py.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from simulated_tem_amd import synth

pytestmark = pytest.mark.gpu

NTH = min(16, os.cpu_count() or 1)
A0 = 3.1652

# (voxels wanted along x, y, z; voxels per lattice parameter; copies of the
# crystal laid over each other, each shifted)
GRIDS = {
    "smallest": ((1, 1, 1), 4, 1),
    "below_edges": ((3, 7, 15), 4, 1),
    "above_edges": ((5, 9, 17), 4, 1),
    "coarse_walk": ((19, 17, 19), 1, 1),
    "coarse_region": ((17, 16, 9), 2, 1),
    "fine": ((13, 19, 21), 8, 1),
    "dense_passes": ((17, 12, 16), 4, 6),
}


def condition(grid, density):
    voxels, M, copies = GRIDS[grid]
    cfg = synth.scaled("c0", cells=(7, 7, 7))
    cfg.update(M=M, density=density, sg=[0.01], d=tuple(max(v, 0.75) * A0 / M for v in voxels))
    x, box = synth.make_atoms(cfg)
    rng = np.random.default_rng(11)
    x = np.concatenate([x] + [(x + rng.uniform(0.3, 1.2, 3)) % box for _ in range(copies - 1)])
    x, conds = synth.conditions(cfg, x, box)
    return x, conds[0][0]


@pytest.mark.parametrize("density", [False, True])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_fp64_field(grid, density):
    x, im = condition(grid, density)
    ph, rho, cnt, r2m = im.field(x, "fp64")
    oph, orho, ocnt, or2m = orc.Condition(im.rec, x).field(nthreads=NTH)
    print("[region fp64] %s voxels %s members <= %d max|dx| %.2e" % (grid, ph.shape, ocnt.max(), np.abs(ph - oph).max()), flush=True)
    assert np.array_equal(cnt, ocnt)
    assert np.array_equal(r2m, or2m)
    assert np.max(np.abs(ph - oph)) < 1e-12
    assert np.max(np.abs(rho - orho)) < 1e-14


@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 5000])
def test_linkcells_counts(n):
    """Binning at the edges of its workgroups (256 atoms), and of the scans:
    the link cells of 5000 atoms in a box of 40 x 40 x 36 cells are more than
    one workgroup scans alone (16,384), those of the small box fewer.  Cells,
    order inside each, offsets and g.r bit for bit, and a crowded cell (every
    atom of the last 60 within one) ranked by point number."""
    for voxels in ((24, 20, 18), (240, 240, 216)):
        cfg = synth.scaled("c0", cells=(7, 7, 7))
        cfg.update(sg=[0.01], d=tuple(v * A0 / 4 for v in voxels))
        box = np.array([v * A0 / 4 for v in voxels])
        x = np.random.default_rng(n).random((n, 3)) * box
        x[-60:] = 0.4 * box + 0.02 * (x[-60:] - x[-60:].mean(axis=0) if n else x[-60:])
        x, conds = synth.conditions(cfg, x, box)
        im = conds[0][0]
        cs, ids, frac, gd = im.linkcells(x)
        oc = orc.Condition(im.rec, x)
        ocs, oids, ofrac = oc.cells()
        assert np.array_equal(cs, ocs) and np.array_equal(ids, oids) and np.array_equal(frac, ofrac)
        assert np.array_equal(gd, oc.gdotr())
