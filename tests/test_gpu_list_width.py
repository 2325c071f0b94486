"""Lists built at other widths: packs follow their members' rows, and calls that
need a list keep the rows there are."""
import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem, Pack
from tests.systems import salt, salt_run

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
