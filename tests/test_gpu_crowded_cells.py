"""Cells beyond what the cell sort holds (4,096 atoms) and beyond the work items
a cell can have (16,384): the call is refused with the capacity error, reads
nothing out of range on the way, and the system is as new after md_init on a
configuration that fits.  No LJ, so that crowded atoms give finite forces."""
import dataclasses

import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import GpuSystem, RbmdError

pytestmark = pytest.mark.gpu
RBL = dict(neighbor_type="RBL", cut_off=5.0, r_core=2.5, neighbor_sample_num=50)


@pytest.mark.parametrize("n,crowd", [(6000, 4200), (20000, 17000)])
@pytest.mark.parametrize("kw", [{}, {"precision": "mixed"}, {"pair_path": "cells"}, RBL], ids=["lists", "mixed", "cells", "rbl"])
def test_refused_and_recovers(ctx, n, crowd, kw):
    s = make_salt(n_ions=n, seed=3)
    s = dataclasses.replace(s, eps=np.zeros_like(s.eps))
    x = s.x.copy()
    x[:crowd] = 0.01 * s.box + np.random.default_rng(3).uniform(0, 1.2, (crowd, 3))
    r = salt_config(**kw)
    g = GpuSystem(ctx, s, r)
    g.set_state(x)
    print(f"[case] n={n} crowd={crowd} {kw} path={g.md_path()}", flush=True)
    with pytest.raises(RbmdError):
        g.md_init()
    g.set_state(s.x, s.v)
    g.md_init()
    g.md_step(3)
    fresh = GpuSystem(ctx, s, r)
    fresh.md_init()
    fresh.md_step(3)
    for a, b in zip(g.state()[:3], fresh.state()[:3]):
        assert np.array_equal(a, b)
    g.close()
    fresh.close()
