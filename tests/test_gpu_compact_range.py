"""Which systems take the stencil pair kernel: dense ones of up to a few thousand
atoms.  Where the lists were measured faster (sparse cells, more atoms) a
system keeps them, and a large empty box builds no table of its cells."""
import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import GpuSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,density,cut,path", [
    (600, 0.5, 4.0, "compact"), (4000, 0.5, 4.0, "compact"), (8000, 0.5, 4.0, "compact"),  # 8, 125, 216 cells
    (8002, 0.5, 4.0, "lists"), (9000, 0.5, 4.0, "lists"),
    (4000, 0.8, 2.5, "compact"), (2000, 0.5, 2.5, "compact"),                               # 216 cells
    (1000, 0.05, 2.5, "lists"), (4000, 0.02, 2.5, "lists"),                                 # 1,000 and 12,167 cells
    (14000, 0.2, 2.5, "lists"), (20000, 0.5, 2.5, "lists"),                                 # 4,096 and 2,197 cells
])
def test_path_by_size_and_density(ctx, n, density, cut, path):
    g = GpuSystem(ctx, make_salt(n_ions=n, density=density, seed=2), salt_config(cut_off=cut, r_core=cut))
    assert g.md_path() == path
    g.close()


def test_empty_box_holds_little(ctx):
    """1,000 ions in 64,000 cells: no more than the lists and the cells"""
    s, r = make_salt(n_ions=1000, density=0.001, seed=2), salt_config(cut_off=2.5, r_core=2.5)
    g = GpuSystem(ctx, s, r)
    assert g.footprint() < 20e6
    g.md_init()
    g.md_step(3)
    assert np.isfinite(g.state()[2]).all()
    g.close()


@pytest.mark.parametrize("n,density,cut,away", [
    (200, 0.8, 4.0, [(2, 0, 0), (-2, 0, 0), (0, -2, 0), (0, 0, -2), (0, 0, 2), (-3, 2, -2), (3, 3, -3)]),
    (600, 0.5, 4.0, [(2, 0, 0), (0, 2, 2), (3, 3, 3)]),  # (of two cells, those below the box are refused)
], ids=["one cell", "two cells"])
def test_atoms_boxes_away(ctx, n, density, cut, away):
    """atoms two and three box lengths outside (a step wraps one): their stencils
    hold image shifts of up to three boxes.  A step by the stencil kernel and
    one by the lists are two by the lists, to the bit."""
    s, r = make_salt(n_ions=n, density=density, seed=9), salt_config(cut_off=cut, r_core=cut)
    x = s.x.copy()
    for atom, boxes in enumerate(away):
        x[10 * atom] += np.array(boxes) * s.box
    out = []
    for calls in ([2], [1, 1]):
        g = GpuSystem(ctx, s, r)
        g.md_init()
        g.set_state(x)
        assert g.md_path() == "compact"
        for k in calls:
            g.md_step(k)
        out.append(g.state())
        g.close()
    for u, v in zip(*out):
        assert np.array_equal(u, v)


@pytest.mark.parametrize("lanes,path", [(0, "compact"), (4, "lists"), (8, "lists"), (16, "compact")])
def test_pair_lanes_asked_for(ctx, lanes, path):
    """4 and 8 lanes are the lists'; the forces differ by the order of at most 140
    terms, 140 x 1.1e-16 of the largest sum of magnitudes, which stays below ten
    times the largest force: 2e-13"""
    s = make_salt(n_ions=2000, seed=2)
    ref = GpuSystem(ctx, s, salt_config(tiles="default"))
    g = GpuSystem(ctx, s, salt_config(tiles="default", pair_lanes=lanes))
    assert ref.md_path() == "compact" and g.md_path() == path
    for k in (ref, g):
        k.md_init()
    a, b = ref.state()[2], g.state()[2]
    assert np.abs(a - b).max() <= 2e-13 * np.abs(a).max()
    assert np.array_equal(a, b) == (path == "compact")  # lanes of another number sum in another order
    for k in (ref, g):
        k.md_step(3)
    a, b = ref.state()[0], g.state()[0]
    assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
    ref.close()
    g.close()
