"""VERLET lists at the sizes where the build can go wrong: cells of fewer and
of more atoms than a wavefront's or a workgroup's share, candidate windows that
end inside a batch, one to three cells an axis, atoms at the cutoff to the last
bits (the FP64 decision of the FP32 test), overlapping atoms, and rows filled to
and past their capacity.  Lists are compared entry by entry with the oracle's."""
import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem, RbmdError
from tests.test_gpu_parity import pair
from rbmd_amd import make_salt, salt_config

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from rbmd_amd.lib import Context

    return Context(0)


def same_lists(g, o, cap):
    gi, go, gn = g.neighbors(cap)
    oi, oo, on = o.neighbors(cap)
    assert np.array_equal(gn, on)
    assert np.array_equal(gi, oi)
    assert np.array_equal(go, oo)
    return gn


# boxes of one to ten cells an axis, 4 to 140 atoms a cell
@pytest.mark.parametrize("n", [64, 130, 216, 258, 512, 1000, 4096, 9826])
@pytest.mark.parametrize("rc,density", [(2.0, 0.5), (2.6, 0.5), (2.0, 4.0), (3.0, 4.0)])
def test_lists_equal_the_oracle(ctx, n, rc, density):
    s = make_salt(n_ions=n, density=density, seed=n)
    if 2 * rc > s.hi[0] - s.lo[0]:
        pytest.skip("cutoff beyond half the box")
    g, o = pair(ctx, s, salt_config(cut_off=rc, r_core=rc))
    same_lists(g, o, 700)


def test_crowded_cell(ctx):
    """one cell of 400 atoms among nearly empty ones"""
    rng = np.random.default_rng(5)
    s = make_salt(n_ions=1000, seed=5)
    x = np.array(s.x)
    box = np.asarray(s.hi)
    x[:400] = 0.02 * box + rng.uniform(0, 1.9, (400, 3))
    s = type(s)(**{**s.__dict__, "x": x})
    g, o = pair(ctx, s, salt_config(cut_off=2.0, r_core=2.0))
    same_lists(g, o, 900)


def test_cutoff_to_the_last_bits(ctx):
    """pairs at distances around sqrt(rc^2 - 1e-4), ulp by ulp, and at 0.01"""
    rc = 2.0
    s = make_salt(n_ions=512, seed=9)
    x = np.array(s.x)
    edge = np.sqrt(rc * rc - 1e-4)
    for k in range(60):
        d = edge
        for _ in range(abs(k - 30)):
            d = np.nextafter(d, 9.0 if k > 30 else 0.0)
        x[2 * k + 1] = x[2 * k] + np.roll([d, 0.0, 0.0], k % 3)
    x[130:160] = x[100:130] + [0.01, 0.0, 0.0]
    x[160] = x[161]
    box = np.asarray(s.hi)
    x = np.mod(x, box)
    s = type(s)(**{**s.__dict__, "x": x})
    g, o = pair(ctx, s, salt_config(cut_off=rc, r_core=rc))
    same_lists(g, o, 700)


def test_export_width(ctx):
    """a width one below the longest list is refused, the longest is not"""
    s = make_salt(n_ions=1000, seed=3)
    g, o = pair(ctx, s, salt_config(cut_off=2.6, r_core=2.6))
    longest = int(same_lists(g, o, 400).max())
    assert same_lists(g, o, longest).max() == longest
    with pytest.raises(RbmdError):
        g.neighbors(longest - 1)


def test_wide_rows(ctx):
    """an export width beyond all candidates there are, and one near 2^28"""
    s = make_salt(n_ions=64, seed=3)
    g, o = pair(ctx, s, salt_config(cut_off=2.0, r_core=2.0))
    same_lists(g, o, 27 * 64 + 100)
    g.build_neighbors(1 << 28)
    near = g.neighbor_entries()
    g.build_neighbors(0)
    assert near == g.neighbor_entries() > 0
