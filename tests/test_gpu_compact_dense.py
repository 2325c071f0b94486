"""The stencil pair kernel where an atom's neighbours overflow a wavefront's LDS
list, so that the stream is walked in rounds, in each of its four splits of the
work; and at the largest size it takes.  A call of two steps forms the first
step's forces by the stencil kernel, two calls of one by the lists: the same
bits.  No LJ, so that the crowded atoms stay where they are."""
import dataclasses

import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import GpuSystem

pytestmark = pytest.mark.gpu


def crowded(n, density, crowd):
    """the first `crowd` atoms within one cell's corner (diagonal below the cutoff of 4)"""
    s = make_salt(n_ions=n, density=density, seed=12)
    x = s.x.copy()
    if crowd:
        x[:crowd] = 0.02 * s.box + np.random.default_rng(12).uniform(0, 1.9, (crowd, 3))
    return dataclasses.replace(s, x=x, eps=np.zeros_like(s.eps))


def two_ways(ctx, s, r):
    out = []
    for calls in ([2], [1, 1]):
        g = GpuSystem(ctx, s, r)
        assert g.md_path() == "compact"
        g.md_init()
        for k in calls:
            g.md_step(k)
        out.append(g.state())
        g.close()
    for u, v in zip(*out):
        assert np.isfinite(u).all() and np.array_equal(u, v)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,density,crowd,longest", [
    (600, 8.1, 0, 2048),     # one atom over four wavefronts: 4 lists of 512 entries
    (1000, 13.5, 0, 2048),
    (2400, 32.4, 0, 2048),   # two atoms over four wavefronts
    (2000, 0.5, 600, 512),   # four atoms over four wavefronts, lists of 256: a wavefront's share of the
                             # stream is 320 at most, so one lies whole in the crowd of 600
    (4000, 0.5, 400, 256),   # four atoms a wavefront, lists of 256
])
def test_lists_that_overflow(ctx, n, density, crowd, longest, precision):
    s, r = crowded(n, density, crowd), salt_config(precision=precision, dt=1e-5)
    g = GpuSystem(ctx, s, r)
    assert g.neighbors(0)[2].max() > longest
    g.close()
    two_ways(ctx, s, r)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [7998, 8000])
def test_largest(ctx, n, precision):
    two_ways(ctx, make_salt(n_ions=n, seed=6), salt_config(precision=precision))
