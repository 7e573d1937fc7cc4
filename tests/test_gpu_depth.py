"""Deep columns whose RK4 steps are not norm-preserving.

The reference scales a column's amplitudes to unit length after every step.  A
march that divides by the length at the end only has to keep the amplitudes in
range on the way: past 2 dz 2 pi |s_g| = 2.83 a double step amplifies the
diffracted amplitude, and near 2.45 it halves it, over hundreds of steps.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from simulated_tem_amd import synth

pytestmark = pytest.mark.gpu

NTH = min(16, os.cpu_count() or 1)
A0 = 3.1652


def deep(sg, M, slices, xi0=103.9, density=False, columns=(10, 9)):
    """A foil of that many slices; g = (1, 0, 1) of a cell of 1 / |sg| A has
    about that deviation along the beam (sg = 0: g = (1, 0, 0))."""
    d = (columns[0] * A0 / M, columns[1] * A0 / M, slices * A0 / M)
    cells = tuple(int(np.ceil(v / A0)) + 2 for v in d[:2]) + (int(np.ceil(d[2] / A0)),)
    cfg = synth.scaled("c0", cells=cells)
    cfg.update(M=M, density=density, sg=[0.0], d=d, n_centres=4, n_voids=1)
    x, box = synth.make_atoms(cfg)
    x, conds = synth.conditions(cfg, x, box)
    im = conds[0][0]
    im.setSupercellTilt(np.eye(3), np.eye(3))
    im.rec.g = type(im.rec.g)(1.0, 0.0, 1.0 if sg else 0.0)
    im.setConventionalUnitCell((1 / sg if sg else A0) * np.eye(3))
    im.setExtinctionDistances(xi0, 207.5)
    return x, im


@pytest.mark.parametrize("sg,M,slices,xi0", [(0.40, 4, 900, 103.9), (0.35, 3, 401, 103.9), (0.246, 4, 1400, 103.9),
                                             (0.0, 4, 1300, 2.03), (0.0, 4, 2600, 103.9)])
@pytest.mark.parametrize("density", [False, True])
def test_large_deviation_fp64(sg, M, slices, xi0, density):
    x, im = deep(sg, M, slices, xi0, density)
    for n in (1, 2, 3, 5, 8, 13, 33):
        oc = orc.Condition(im.rec, x, 0.005, n)
        ref = oc.image(nthreads=NTH)
        assert np.all(np.isfinite(ref))
        e = np.max(np.abs(im.computeD2BI_img(x, 0.005, n, mode="fp64") - ref))
        print("[depth] s_g %.3f M=%d %d slices n=%d max|dI| %.2e of %.3f" % (oc.plan.aa[0] / 6.2832, M, slices, n, e, ref.max()), flush=True)
        assert e <= 1e-10, n


def test_large_deviation_fp64_many_columns():
    """One wave per column and no split: against the oracle on a window."""
    x, im = deep(0.40, 4, 900, columns=(136, 136))
    for n in (1, 4, 16, 32):
        ref = orc.Condition(im.rec, x, 0.005, n).image(window=(60, 64, 70, 72), nthreads=NTH)
        e = np.max(np.abs(im.computeD2BI_img(x, 0.005, n, mode="fp64")[70:72, 60:64] - ref))
        print("[depth] 136 x 136 n=%d max|dI| %.2e" % (n, e), flush=True)
        assert e <= 1e-10, n
