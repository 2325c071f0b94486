"""The no-alloc grid energy of long flat grids, whose separable plan does not fit
the scratch: taken as before, to the bits of the allocating call, and the sum
of the separable form (sums of 3e4 atoms and 4e4 vectors in other orders:
sqrt(1.2e9) x 1.1e-16 = 4e-12 of the terms, 1e-11 with room)."""
import math

import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import GpuSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kmax", [(30000, [100, 100, 0]), (30000, [100, 0, 100]), (2000, [0, 0, 40000]),
                                    (30000, [10000, 0, 0]), (2000, [100, 100, 0])])
def test_flat_grid(ctx, n, kmax):
    s = make_salt(n_ions=n, seed=4)
    g = GpuSystem(ctx, s, salt_config(kmax=kmax))
    g.md_init()
    g.md_energy_noalloc()
    a = g.thermo()["e_long"]
    g.md_energy()
    assert g.thermo()["e_long"] == a
    _, _, e = g.ewald_force(kmax)
    self = -math.sqrt(0.64 / math.pi) * float((s.charge ** 2).sum())
    assert abs(a - (e + self) / n) <= 1e-11 * abs(a)
    g.close()
