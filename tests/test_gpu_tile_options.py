"""Every pair-lane and k-wavefront option on systems that run over lists: the
same forces to the order of their sums.  Pair sums hold at most 430 terms and
k-space sums 200, each below ten times the largest force: 630 x 10 x 1.1e-16 =
7e-13.  Mixed precision rounds each term to 32 bits before the same FP64 sums,
so the bound is the same."""
import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem
from tests.systems import salt, salt_run, water, water_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["salt", "water"])
def test_tile_options_of_listed_systems(ctx, kind, precision):
    s, run = (salt(n=9002, seed=4), salt_run) if kind == "salt" else (water(nmol=1667, seed=4), water_run)
    ref = None
    for lanes in (4, 8, 16):
        for waves in (2, 4, 8):
            g = GpuSystem(ctx, s, run(precision=precision, tiles="default", pair_lanes=lanes, kforce_lanes=waves))
            assert g.md_path() == "lists"
            g.md_init()
            f = g.state()[2]
            g.close()
            ref = f if ref is None else ref
            assert np.abs(f - ref).max() <= 7e-13 * np.abs(ref).max()
