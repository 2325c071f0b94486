"""Random-batch lists, forces and energies against the oracle at the edges of
their kernels: stencils of 125, 343 and 729 cells (one and several tables
of 128), groups of four atoms that do and do not fill, boxes a few cells wide,
both erfc modes.  Lists are bit-exact; forces, energies and virials within
1e-10, the bar of the RBL parity tests."""
import numpy as np
import pytest

from tests.systems import rel_err, salt, salt_run, water, water_run
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["analytic", "table"])
@pytest.mark.parametrize("n", [514, 2002])
@pytest.mark.parametrize("r_core,samples", [(3.0, 30), (2.0, 40), (1.5, 25), (1.1, 7)])
def test_rbl_stencils(ctx, r_core, samples, n, mode):
    s = salt(n=n, seed=n)
    r = salt_run(neighbor_type="RBL", r_core=r_core, neighbor_sample_num=samples, erfc_mode=mode)
    g, o = pair(ctx, s, r)
    cap = 700
    gi, go, gn = g.neighbors(cap)
    oi, oo, on = o.neighbors(cap)
    assert np.array_equal(gn, on)
    assert np.array_equal(gi, oi)
    assert np.array_equal(go, oo)
    gf, gv, ge, gc = g.force_real()
    of, ov, oe, oc = o.force_real()
    assert rel_err(gf, of) < 1e-10
    assert rel_err(gv, ov) < 1e-9
    assert np.abs(ge - oe).max() <= 1e-10 * np.abs(oe).max()
    assert np.abs(gc - oc).max() <= 1e-10 * np.abs(oc).max()


@pytest.mark.parametrize("nmol", [601, 1400])
def test_rbl_water_steps(ctx, nmol):
    s, r = water(nmol=nmol, seed=8), water_run(neighbor_type="RBL", r_core=5.0, neighbor_sample_num=100)
    g, o = pair(ctx, s, r)
    g.md_init()
    assert o.md_init() == 0
    g.md_step(6)
    assert o.md_step(6) == 0
    assert rel_err(g.state()[2], o.state()[2]) < 1e-8
    tg, to = g.thermo(), o.thermo()
    for k in ("temperature", "pressure", "e_lj", "e_coul"):
        assert abs(tg[k] - to[k]) <= 1e-8 * max(1.0, abs(to[k])), k
