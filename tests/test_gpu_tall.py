"""FAST images of voxels that are not cubes.

The row kernels split a weight into factors whose exponents grow with the
tile's extent in sigma: a tile that would take them out of FP32's range has to
give way to a smaller one, and the guard band has to cover their rounding.
Members are exact then, so the field is the oracle's to the bound of the other
FAST field tests, 1e-5.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from simulated_tem_amd import abi, imaging, synth

pytestmark = pytest.mark.gpu

NTH = min(16, os.cpu_count() or 1)
A0 = 3.1652
SIGMA = A0 / 2

# voxel sides in sigma
SIDES = [(0.5, 0.5, 2.87), (1.4, 1.4, 2.7), (1.0, 1.0, 2.8), (0.5, 0.5, 4.0), (0.5, 0.5, 8.0), (0.5, 0.5, 30.0),
         (0.5, 2.9, 2.9), (0.5, 9.0, 0.5), (7.0, 1.0, 1.0), (9.0, 0.5, 0.5)]


def boxes(sides, n=(18, 17, 19), density=False):
    h = np.array(sides) * SIGMA
    d = h * n
    cfg = synth.scaled("c0", cells=tuple(int(np.ceil(v / A0)) + 1 for v in np.maximum(d, 4 * A0)))
    cfg.update(sg=[0.01], d=tuple(np.maximum(d, A0)), density=density)
    x, box = synth.make_atoms(cfg)
    x, conds = synth.conditions(cfg, x, box)
    im = conds[0][0]
    for a in range(3):
        im.rec.gk_n[a] = n[a]
        im.rec.gk_a[4 * a] = h[a]
    return x, im


@pytest.mark.parametrize("sides", SIDES)
@pytest.mark.parametrize("density", [False, True])
def test_voxel_sides(sides, density, monkeypatch):
    x, im = boxes(sides, density=density)
    oph, orho, ocnt, _ = orc.Condition(im.rec, x).field(nthreads=NTH)
    for variant in ("0", "1", "2", "3", None):
        if variant is None:
            monkeypatch.delenv("D2BI_FAST_VARIANT")
        else:
            monkeypatch.setenv("D2BI_FAST_VARIANT", variant)
        ph, rho, _, _ = im.field(x, "fast", diag=False)
        err = np.abs(ph - oph).max()
        print("[tall] %s v%s members <= %d max|dx| %.2e" % (sides, variant, ocnt.max(), err), flush=True)
        assert err < 1e-5, variant
        assert np.max(np.abs(rho - orho)) < 1e-5, variant
    cnt = im.field(x, "fast")[2]
    assert np.array_equal(cnt, ocnt)


@pytest.mark.parametrize("sides", [(1.4, 1.4, 2.7), (0.5, 0.5, 8.0)])
def test_voxel_sides_aperture(sides, monkeypatch):
    """Several aperture points: the shared pass and a pass per point, which take
    the same tile."""
    x, im = boxes(sides)
    ref = orc.compute_img_aperture(im.rec, x, 0.005, 2, 0.002, 5, nthreads=NTH)
    got = im.computeD2BI_img(x, 0.005, 2, apertureAngle=0.002, nAperturePoints=5)
    assert np.max(np.abs(got - ref)) <= 1e-4
    monkeypatch.setenv("D2BI_APERTURE_SHARED", "0")
    assert np.array_equal(got, im.computeD2BI_img(x, 0.005, 2, apertureAngle=0.002, nAperturePoints=5))


def test_voxel_sides_batch():
    """A batch of cubes and of voxels too tall for the FAST tiles gives each
    condition's own image, launched and replayed."""
    todo = []
    for sides in ((0.5, 0.5, 0.5), (0.5, 0.5, 8.0), (1.4, 1.4, 2.7)):
        x, im = boxes(sides)
        todo.append((im, imaging.Atoms(x), 0.005, 3))
    alone = [im.computeD2BI_img(at, pa, n, mode="fast") for im, at, pa, n in todo]
    for _ in range(3):
        for got, want in zip(imaging.computeD2BI_img_batch(todo, mode="fast"), alone):
            assert np.array_equal(got, want)


@pytest.mark.parametrize("side", [3.5, 5.0])
def test_coarse_cubes_stay_refused(side):
    """Cubes beyond 3 sigma have a link cell each, more to a tile than its table
    holds: FAST says so, also where their weights would not fit its tiles; FP64
    images them."""
    x, im = boxes((side, side, side), n=(9, 9, 9))
    at = imaging.Atoms(x)
    for call in (lambda: im.computeD2BI_img(x, mode="fast"), lambda: im.field(x, "fast"),
                 lambda: im.computeD2BI_img(x, 0.005, 2, apertureAngle=0.002, nAperturePoints=2),
                 lambda: imaging.computeD2BI_img_batch([(im, at, 0.0, 1)] * 2, mode="fast")):
        with pytest.raises(abi.D2biError, match="spans 2[0-9][0-9] link cells"):
            call()
    assert np.max(np.abs(im.computeD2BI_img(x, mode="fp64") - orc.compute_img(im.rec, x, nthreads=NTH))) <= 1e-10
