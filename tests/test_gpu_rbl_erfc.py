"""The analytic erfc of random-batch lists at values of sqrt(alpha) rc on both
sides of the line where the radial table is left for erfc itself, and far
beyond it.  No LJ, so that the Coulomb terms stand alone: a term's relative
error is that of erfc and exp, 2 x^2 u of the argument's rounding (x at most 6
for the pairs that count, u = 1.1e-16) and a few u of the functions, 1e-14; an
atom's terms alternate in sign and cancel to a tenth at most, so 1e-12 holds
with room.

The sums are formed here with scipy's erfc over the oracle's lists: the oracle
follows the reference's 1 - erf, which keeps 1e-16 of 1, not of a tail."""
import dataclasses
import math

import numpy as np
import pytest
from scipy.special import erfc

from tests.systems import rel_err, salt, salt_run, water, water_run
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu
QQR2E = {"LJ": 1.0, "REAL": 332.06371}


def shell_step(s, r):
    """every how many shell atoms one is kept (ExecutionMD.cpp:582-592)"""
    rho = s.n_atoms / np.prod(s.box)
    k = round(1.0 + (0.05 / rho - 0.05))
    count = [int(k * rho * math.ceil(4.0 / 3.0 * float(np.float32(math.pi)) * d ** 3)) + 1 for d in (r.r_core, r.cut_off)]
    return math.ceil((count[1] - count[0]) / r.neighbor_sample_num)


def g_of(alpha, d):
    b = math.sqrt(alpha)
    return erfc(b * d) / d ** 2 + 2 * b * np.exp(-alpha * d * d) / (math.sqrt(math.pi) * d)


def nearest(s, d):
    return d - s.box * np.round(d / s.box)


def forces(s, r, ids, off, num):
    """the corrected force, its mean removed"""
    f = np.zeros_like(s.x)
    core, kept = num[0::2], num[1::2]
    for i in range(s.n_atoms):
        slots = np.nonzero(ids[i] >= 0)[0]
        assert len(slots) == core[i] + kept[i]
        scale = np.where(np.arange(len(slots)) < core[i], 1.0, float(shell_step(s, r)))
        j = ids[i][slots]
        d = nearest(s, s.x[j] - off[i][slots] - s.x[i])
        dist = np.sqrt((d * d).sum(1))
        if r.special_bonds:
            scale = np.where((np.arange(len(slots)) >= core[i]) & (dist ** 2 <= r.r_core ** 2), 0.0, scale)
        c = -s.charge[i] * s.charge[j] * g_of(r.alpha, dist) / dist * scale * (dist < r.cut_off) * (dist > 0.01)
        f[i] = QQR2E[r.unit] * (c[:, None] * d).sum(0)
    return f - f.mean(0)


def energies(s, r):
    e = np.zeros(s.n_atoms)
    for i in range(s.n_atoms):
        d = nearest(s, s.x - s.x[i])
        dist = np.sqrt((d * d).sum(1))
        j = np.nonzero((r.cut_off ** 2 - dist ** 2 > 1e-4) & (dist ** 2 > 1e-4))[0]
        w = np.ones(len(j))
        if r.special_bonds:
            for k in range(s.special_offsets[i], s.special_offsets[i + 1]):
                w[j == s.special_ids[k]] = s.special_weights[k]
        e[i] = (s.charge[i] * s.charge[j] / (2 * dist[j]) * (erfc(math.sqrt(r.alpha) * dist[j]) - (1 - w))).sum()
    return QQR2E[r.unit] * e


@pytest.mark.parametrize("weighted", [False, True], ids=["plain", "weighted"])
@pytest.mark.parametrize("reach", [3.98, 4.02, 8.0, 20.0])
def test_forces_and_energies(ctx, reach, weighted):
    if weighted:
        s, r = water(nmol=600, seed=5), water_run(neighbor_type="RBL", r_core=5.0, neighbor_sample_num=100,
                                                  alpha=(reach / 10.0) ** 2)
    else:
        s, r = salt(n=2002, seed=7), salt_run(neighbor_type="RBL", r_core=2.0, neighbor_sample_num=40,
                                              alpha=(reach / 4.0) ** 2)
    s = dataclasses.replace(s, eps=np.zeros_like(s.eps))
    g, o = pair(ctx, s, r)
    gl, ol = g.neighbors(900), o.neighbors(900)
    for a, b in zip(gl, ol):
        assert np.array_equal(a, b)
    gf, _, _, gc = g.force_real()
    assert rel_err(gf, forces(s, r, *ol)) < 1e-12
    want = energies(s, r)
    assert np.abs(gc - want).max() <= 1e-12 * np.abs(want).max()
