"""Lists built at other widths: packs follow their members' rows, and calls that
need a list keep the rows there are."""
import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem, Pack, RbmdError
from tests.systems import salt, salt_run, water, water_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_pack_follows_a_member_list_of_another_width(ctx, graph):
    """a member's list built wider (new rows, the old ones freed) between packed
    steps: the same bits as a pack that was left alone"""
    out = []
    for wider in (False, True):
        gs = [GpuSystem(ctx, salt(n=n, seed=20 + n), salt_run()) for n in (600, 1000)]
        for g in gs:
            g.md_init()
        p = Pack(ctx, gs)
        go = (lambda k: (p.enqueue(k), p.wait())) if graph else p.step
        go(3)
        if wider:
            before = gs[0].footprint()
            gs[0].neighbors(600)
            assert gs[0].footprint() != before
        go(4)
        out.append([g.state() for g in gs])
        p.close()
        for g in gs:
            g.close()
    for a, b in zip(*out):
        for u, v in zip(a, b):
            assert np.array_equal(u, v)


@pytest.mark.parametrize("make", [lambda: (salt(n=600, seed=3), salt_run()), lambda: (water(nmol=200, seed=5), water_run()),
                                  lambda: (salt(n=2000, seed=3),
                                           salt_run(neighbor_type="RBL", cut_off=5.0, r_core=2.5, neighbor_sample_num=50))],
                         ids=["salt", "water", "rbl"])
def test_real_force_keeps_the_rows(ctx, make):
    """force_real without a list builds one in the rows there are: neither the
    rows nor the memory held grow over new configurations"""
    s, r = make()
    g = GpuSystem(ctx, s, r)
    g.md_init()
    held, ref = g.footprint(), None
    for _ in range(3):
        g.set_state(s.x)
        f = g.force_real()[0]
        assert g.footprint() == held
        ref = f if ref is None else ref
        assert np.array_equal(f, ref)
    g.md_step(2)
    assert g.footprint() == held
    g.close()


def test_a_width_that_does_not_fit_leaves_the_system_usable(ctx):
    """rows wider than the card's memory are refused, and the steps that follow
    are those of a system that was never asked"""
    s = salt(n=70000, seed=4)  # rows of 27 n entries: 529 GB
    out = []
    for asked in (False, True):
        g = GpuSystem(ctx, s, salt_run())
        g.md_init()
        held = g.footprint()
        if asked:
            with pytest.raises(RbmdError, match="hipMalloc"):
                g.build_neighbors(2_000_000)
            assert g.footprint() == held
        g.md_step(2)
        out.append(g.state())
        g.close()
    for u, v in zip(*out):
        assert np.array_equal(u, v)
