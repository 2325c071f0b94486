"""The grid Ewald kernels (separable phases, half grid, matrix tiles) against
the direct sum over every k vector in numpy, at the edges of their tiles: atom
counts around 4, 16, 64 and 128, grids with a zero edge, one, two and three or
more column tiles (kz up to 7, 15, 23), unequal edges, and the batched plan of
the small workspace.

Tolerances: the phases carry |m| 2^-53 turns of rounding an axis, about
2 pi x 25 x 3 x 1.1e-16 = 5e-14 radian, and the sums over at most 1,500 atoms
and 5,000 vectors add sqrt(1e7) x 1.1e-16 = 4e-13 of the RMS term: 1e-11
relative to the largest force, energies 1e-11.
"""
import math

import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem, Pack
from tests.systems import salt_run
from rbmd_amd import make_salt

pytestmark = pytest.mark.gpu


def direct(s, alpha, kmax):
    m = np.stack(np.meshgrid(*[np.arange(-k, k + 1) for k in kmax], indexing="ij"), -1).reshape(-1, 3)
    m = m[np.any(m != 0, axis=1)]
    k = 2 * np.pi * m / s.box
    k2 = (k * k).sum(1)
    w = np.exp(-k2 / (4 * alpha)) / k2
    t = (s.x / s.box) @ m.T
    t = 2 * np.pi * (t - np.round(t))
    c, n = np.cos(t), np.sin(t)
    re, im = s.charge @ c, s.charge @ n
    g = -4 * np.pi * s.charge[:, None] * (c * (w * im) - n * (w * re)) / s.volume
    f = g @ k
    vir = np.stack([s.x[:, a] * f[:, b] + s.x[:, b] * f[:, a] for a, b in
                    ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))], 1)
    return f, vir, 2 * np.pi / s.volume * float((w * (re * re + im * im)).sum())


def box_of(n):
    s = make_salt(n_ions=n, seed=11)
    s.hi = s.hi * np.array([1.0, 1.1, 0.9])
    s.x = np.mod(s.x, s.hi)
    return s


@pytest.mark.parametrize("n", [2, 16, 66, 126, 130, 1500])
@pytest.mark.parametrize("kmax", [[1, 0, 0], [0, 0, 2], [2, 3, 4], [3, 2, 7], [4, 4, 8], [2, 1, 16], [0, 3, 24]])
def test_ewald_grid_matches_direct_sum(ctx, n, kmax):
    s, r = box_of(n), salt_run()
    g = GpuSystem(ctx, s, r)
    f, vir, e = g.ewald_force(kmax)
    of, ovir, oe = direct(s, r.alpha, kmax)
    assert np.abs(f - of).max() <= 1e-11 * max(np.abs(of).max(), 1e-3)
    assert np.abs(vir - ovir).max() <= 1e-11 * max(np.abs(ovir).max(), 1e-3)
    assert abs(e - oe) <= 1e-11 * abs(oe)
    g.close()


def test_ewald_energy_in_batches(ctx):
    """30,000 ions and 9,260 k vectors: the no-alloc plan runs several batches
    of atoms; the same energy as the whole-system call to the order of its sums"""
    s = make_salt(n_ions=30000, seed=4)
    g = GpuSystem(ctx, s, salt_run(kmax=[10, 10, 10]))
    g.md_init()
    g.md_energy_noalloc()
    a = g.thermo()["e_long"]
    _, _, e = g.ewald_force([10, 10, 10])
    self = -math.sqrt(0.64 / math.pi) * float((s.charge ** 2).sum())
    assert abs(a - (e + self) / s.n_atoms) <= 1e-11 * abs(a)
    g.close()


@pytest.mark.parametrize("kmax", [[3, 3, 3], [2, 3, 9], [1, 1, 20]])
def test_ewald_pack_equals_alone(ctx, kmax):
    inputs = [(make_salt(n_ions=n, seed=n), salt_run(coulomb_type="EWALD", kmax=kmax)) for n in (200, 514, 1000)]
    alone = [GpuSystem(ctx, *i) for i in inputs]
    packed = [GpuSystem(ctx, *i) for i in inputs]
    for g in alone + packed:
        g.md_init()
    p = Pack(ctx, packed)
    p.step(4)
    p.enqueue(4)
    p.wait()
    for g, h in zip(alone, packed):
        g.md_step(8)
        for u, v in zip(g.state(), h.state()):
            assert np.array_equal(u, v)
        assert g.thermo()["pressure"] == h.thermo()["pressure"]
    p.close()
