"""Column integration over precession points: every kernel instance (points per
pass) and the splits into passes, with and without the density field, an even
and an odd number of slices, on images whose columns fill no whole workgroup.

FP64 images against the oracle at the contract's 1e-10, FAST at 1e-4.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from simulated_tem_amd import synth

pytestmark = pytest.mark.gpu

NTH = min(16, os.cpu_count() or 1)
TOL = {"fp64": 1e-10, "fast": 1e-4}


def condition(density, slices):
    cfg = synth.scaled("c0", cells=(7, 6, 6))
    cfg.update(density=density, sg=[0.01], d=(19 * 3.1652 / 4, 13 * 3.1652 / 4, slices * 3.1652 / 4))
    x, box = synth.make_atoms(cfg)
    x, conds = synth.conditions(cfg, x, box)
    return x, conds[0][0]


@pytest.mark.parametrize("mode", ["fp64", "fast"])
@pytest.mark.parametrize("density,slices", [(False, 22), (True, 23)])
def test_precession_points(mode, density, slices):
    x, im = condition(density, slices)
    for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 16, 17, 20, 24, 25, 28, 31, 32, 33, 45, 64):
        ref = orc.Condition(im.rec, x, 0.005, n).image(nthreads=NTH)
        e = float(np.max(np.abs(im.computeD2BI_img(x, 0.005, n, mode=mode) - ref)))
        print("[precession] %s n=%d max|dI| %.2e" % (mode, n, e), flush=True)
        assert e <= TOL[mode], n


@pytest.mark.parametrize("columns", [(403, 397), (810, 790)])
@pytest.mark.parametrize("density", [False, True])
def test_fast_points_per_wave(columns, density):
    """Large images march more points per wave, a small one splits a column's
    points over waves; 160,000 and 640,000 columns take the instances the small
    images above don't (several points per wave, the shared step matrix alone
    and split).  Against the FP64 image, which is held to the oracle above."""
    cfg = synth.scaled("c0", cells=(102, 100, 3))
    cfg.update(density=density, sg=[0.01], d=(columns[0] * 3.1652 / 4, columns[1] * 3.1652 / 4, 13 * 3.1652 / 4))
    x, box = synth.make_atoms(cfg)
    x, conds = synth.conditions(cfg, x, box)
    im = conds[0][0]
    for n in (1, 2, 3, 4, 5, 6, 7, 8, 13, 16, 24, 32, 40):
        ref = im.computeD2BI_img(x, 0.005, n, mode="fp64")
        e = float(np.max(np.abs(im.computeD2BI_img(x, 0.005, n, mode="fast") - ref)))
        print("[per wave] %s n=%d max|dI| %.2e of %.2e" % (columns, n, e, ref.max()), flush=True)
        assert e <= TOL["fast"] * min(1.0, 10 * ref.max()), n
