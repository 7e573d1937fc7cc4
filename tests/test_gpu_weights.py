"""The FP64 region kernel's weights: voxels taller than the Gaussian, and their
rounding.

The weight of a point factorises over the axes.  Its factors have to stay in
range whatever the voxels' sides (a record may hold voxels several sigma tall),
and their product has to be as near the exact weight as one exponential of the
range is.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from simulated_tem_amd import synth

pytestmark = pytest.mark.gpu

NTH = min(16, os.cpu_count() or 1)
A0 = 3.1652
SIGMA = A0 / 2
U = 2.0 ** -53


def imaging_of(x, box, d, M, hz=None, sg=0.01):
    """The condition of atoms x in a periodic box, imaged over d; hz: voxel
    height along z (the box's z side must hold a whole number of them)."""
    cfg = synth.scaled("c0", cells=(7, 7, 7))
    cfg.update(M=M, sg=[sg], d=tuple(d))
    x, conds = synth.conditions(cfg, x, np.asarray(box))
    im = conds[0][0]
    if hz is not None:
        n = int(round(d[2] / hz))
        im.rec.gk_n[2] = n
        im.rec.gk_a[8] = d[2] / n
    return x, im


@pytest.mark.parametrize("height", [3.0, 5.3, 8.0])
@pytest.mark.parametrize("density", [False, True])
def test_tall_voxels(height, density):
    """Voxels a quarter of a lattice parameter wide and `height` sigma tall."""
    nz = 16
    hz = height * SIGMA
    cfg = synth.scaled("c0", cells=(7, 7, int(nz * hz / A0) + 1))
    x, box = synth.make_atoms(cfg)
    x, im = imaging_of(x, box, (17 * A0 / 4, 16 * A0 / 4, nz * hz), 4, hz)
    im.setUseDensityField(density)
    oc = orc.Condition(im.rec, x, 0.005, 3)
    oph, orho, ocnt, or2m = oc.field(nthreads=NTH)
    ph, rho, cnt, r2m = im.field(x, "fp64")
    print("[tall] %.1f sigma %s members %d..%d max|dx| %.2e" % (height, ph.shape, ocnt.min(), ocnt.max(), np.abs(ph - oph).max()), flush=True)
    assert np.array_equal(cnt, ocnt) and np.array_equal(r2m, or2m)
    assert np.max(np.abs(ph - oph)) < 1e-12
    assert np.max(np.abs(rho - orho)) < 1e-14
    assert np.max(np.abs(im.computeD2BI_img(x, 0.005, 3, mode="fp64") - oc.image(nthreads=NTH))) <= 1e-10


@pytest.mark.parametrize("M", [1, 2, 3, 4, 6])
def test_weight_rounding(M):
    """x = S / |S| against extended precision over the device's own FP64 offsets
    and g.r (exact values otherwise): with few members to a voxel the error of S
    is that of its weights.  Bound of |dS| / sum w, in units of u = 2^-53:
    exponent 4.5 times 3 roundings of the offsets' products (relative to its
    own value), three exponentials 2 each, their products 2, the phases' cos
    and sin 2, and 2 per addition of at most n members; 4 for S / |S|.  The
    offsets themselves are the reference's FP64 expression."""
    rng = np.random.default_rng(M)
    n = 24 if M == 1 else 26
    d = np.array([n, n - 1, 16]) * A0 / M
    box = d + 2 * A0
    x = rng.random((int(0.006 * np.prod(box)), 3)) * box
    x, im = imaging_of(x, box, d, M)
    p = im.plan(len(x))
    cs, ids, frac, gd = im.linkcells(x)
    ph, _, cnt, _ = im.field(x, "fp64")
    L = np.longdouble
    cell_of, zi = [], []
    for a in range(3):
        i = np.arange((p.Mx, p.My, p.Mz)[a])
        z = p.ia_col[4 * a] * (im.rec.gk_a[4 * a] * i - p.lc_delta[a])
        c = (np.floor(z).astype(int) + 16 * (p.Ex, p.Ey, p.Ez)[a]) % (p.Ex, p.Ey, p.Ez)[a]
        cell_of.append(c)
        zi.append(z - c)
    g = gd[ids - 1]
    cosg, sing = np.cos(L(g)), np.sin(L(g))
    E = (p.Ex, p.Ey, p.Ez)
    worst = 0.0
    for vz, vy, vx in np.ndindex(p.Mz, p.My, p.Mx):
        v = (vx, vy, vz)
        S, W, m = [L(0), L(0)], L(0), 0
        for kz in (-1, 0, 1):
            for ky in (-1, 0, 1):
                for kx in (-1, 0, 1):
                    k = (kx, ky, kz)
                    c = [(cell_of[a][v[a]] + E[a] + k[a]) % E[a] for a in range(3)]
                    j = c[0] + E[0] * (c[1] + E[1] * c[2])
                    for s in range(cs[j], cs[j + 1]):
                        q = [p.a_col[4 * a] * (frac[s, a] + (k[a] - zi[a][v[a]])) for a in range(3)]
                        if (q[0] * q[0] + q[1] * q[1]) + q[2] * q[2] <= p.rc2:
                            w = np.exp(-sum(L(t) * L(t) for t in q) * L(p.i2s2))
                            S[0] += w * cosg[s]
                            S[1] += w * sing[s]
                            W += w
                            m += 1
        assert m == cnt[vz, vy, vx]
        r = np.sqrt(S[0] * S[0] + S[1] * S[1])
        if m == 0 or r < 0.05 * W:
            continue
        e = max(abs(L(ph[vz, vy, vx].real) - S[0] / r), abs(L(ph[vz, vy, vx].imag) - S[1] / r))
        bound = ((3 * 4.5 + 6 + 2 + 2 + 2 * m) * W / r + 4) * U
        worst = max(worst, float(e / bound))
    print("[weights] M=%d members <= %d worst error / bound %.2f" % (M, cnt.max(), worst), flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("height", [90.0, 1000.0, 1733.0, 3000.0])
def test_members_at_the_rim(height):
    """Points a hair inside 3 sigma above and below voxels many sigma tall: a
    position is then larger than FP32 resolves the rim at, and every one of them
    still counts."""
    nz, hz = 16, height * SIGMA
    d = np.array([8 * A0 / 4, 8 * A0 / 4, nz * hz])
    cfg = synth.scaled("c0", cells=(7, 7, 7))
    cfg.update(d=tuple(d), sg=[0.0])
    _, conds = synth.conditions(cfg, np.zeros((1, 3)), np.array([40.0, 40.0, nz * hz]))
    im = conds[0][0]
    im.setSupercellTilt(np.eye(3), np.eye(3))
    im.rec.gk_n[2] = nz
    im.rec.gk_a[8] = d[2] / nz
    side = np.array([im.rec.gk_a[0], im.rec.gk_a[4], im.rec.gk_a[8]])
    rim = 3 * SIGMA * (1 - 1e-7)
    v = np.array([(iz % 8, (3 * iz) % 8, iz) for iz in range(nz)])
    up = np.array([0.0, 0.0, rim])
    x = np.concatenate([v * side + up, v * side - up]) - np.array(im.rec.delta)
    ph, _, cnt, r2m = im.field(x, "fp64")
    oph, _, ocnt, or2m = orc.Condition(im.rec, x).field(nthreads=NTH)
    print("[rim] %.0f sigma members %d of %d" % (height, cnt.sum(), ocnt.sum()), flush=True)
    assert ocnt.sum() >= 2 * nz - 2
    assert np.array_equal(cnt, ocnt) and np.array_equal(r2m, or2m)
