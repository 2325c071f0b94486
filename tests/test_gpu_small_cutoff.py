"""Cutoffs near the distance of 0.01 below which two atoms are taken for one:
lists and steps as the oracle has them, down to cutoffs that list no pair."""
import dataclasses

import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import GpuSystem
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 600])
@pytest.mark.parametrize("rc", [0.005, 0.01, 0.0102, 0.012, 0.0141, 0.0141421356, 0.0142, 0.015, 0.02, 0.05])
def test_lists_and_steps(ctx, n, rc):
    s = make_salt(n_ions=n, density=0.5, seed=3)
    f = 4.2 * rc / (s.hi - s.lo)[0]  # four cells an axis
    s = dataclasses.replace(s, x=s.x * f, lo=s.lo * f, hi=s.hi * f, v=s.v * f, sigma=np.asarray(s.sigma) * 1e-3 * f)
    r = salt_config(cut_off=rc, r_core=rc, force_field="LJ/CUT", coulomb_type="NONE")
    g, o = pair(ctx, s, r)
    for a, b in zip(g.neighbors(200 if n == 64 else 700), o.neighbors(200 if n == 64 else 700)):
        assert np.array_equal(a, b)
    out = []
    for calls in ([2], [1, 1]):
        h = GpuSystem(ctx, s, r)
        h.md_init()
        for k in calls:
            h.md_step(k)
        out.append(h.state())
        h.close()
    for u, v in zip(*out):
        assert np.array_equal(u, v)
