"""Compact systems (few atoms): the stencil pair kernel and the fused launches of
their steps without thermo sums.

Against the stored lists of the same system: a call of n steps forms its pair
forces by the stencil kernel on all but the last step, n one-step calls by
the lists on every step, and the two agree to the bit.

Against the list path of a system that is not compact (17 atom types with
equal coefficients: the stencil kernel keeps the type tables of at most 16 in
LDS): the k-space sums differ in order, about 1,000 FP64 terms a force whose
absolute sum is below 1e3 times its RMS value, so 1e3 x 1e3 x 1.1e-16 = 1e-10
at most over 3 steps.

Sizes sit at the edges of the kernel's choices: a pair of ions, partial and
full groups of atoms, the sizes where stencil_choice changes, the largest of
the range, and boxes of one, two and more cells per axis.
"""
import dataclasses

import numpy as np
import pytest

from rbmd_amd.lib import GpuSystem
from rbmd_amd import make_salt, make_water, salt_config, water_config

pytestmark = pytest.mark.gpu
TOL = 1e-10


def listed_twin(s):
    """the same system with 17 types: the stored-list path"""
    k = 17 - len(s.eps)
    return dataclasses.replace(s, eps=np.concatenate([s.eps, np.zeros(k)]), sigma=np.concatenate([s.sigma, np.ones(k)]))


SIZES = [("salt", 2), ("salt", 62), ("salt", 130), ("salt", 600), ("salt", 3000), ("salt", 3002), ("salt", 9000),
         ("water", 3), ("water", 66), ("water", 999), ("water", 1002), ("water", 2400), ("water", 2403)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,n", SIZES)
def test_compact_steps_equal_listed_steps(ctx, kind, n, precision):
    if kind == "salt":
        s, r = make_salt(n_ions=n, seed=6), salt_config(precision=precision)
    else:
        s, r = make_water(n_mol=n // 3, seed=6), water_config(precision=precision)
    a, b = GpuSystem(ctx, s, r), GpuSystem(ctx, s, r)
    for g in (a, b):
        g.md_init()
    a.md_step(5)
    for _ in range(5):
        b.md_step(1)
    for u, v in zip(a.state(), b.state()):
        assert np.array_equal(u, v)
    assert a.neighbor_entries() == b.neighbor_entries()
    a.close()
    b.close()


@pytest.mark.parametrize("kind,n", SIZES)
def test_compact_equals_stored_lists(ctx, kind, n):
    if kind == "salt":
        s, r = make_salt(n_ions=n, seed=5), salt_config()
    else:
        s, r = make_water(n_mol=n // 3, seed=5), water_config()
    a, b = GpuSystem(ctx, s, r), GpuSystem(ctx, listed_twin(s), r)
    for g in (a, b):
        g.md_init()
    rms = np.sqrt(np.mean(b.state()[2] ** 2)) or 1.0
    assert np.abs(a.state()[2] - b.state()[2]).max() <= TOL * max(rms, np.abs(b.state()[2]).max())
    for g in (a, b):
        g.md_step(3)
    for u, v in zip(a.state(), b.state()):
        assert np.abs(u - v).max() <= TOL * max(1.0, np.abs(v).max())
    ta, tb = a.thermo(), b.thermo()
    for k in ("temperature", "pressure", "e_lj", "e_coul"):
        assert abs(ta[k] - tb[k]) <= TOL * max(abs(tb[k]), 1e-3 * np.abs(tb["virial"]).max())
    assert np.abs(np.array(ta["virial"]) - tb["virial"]).max() <= TOL * np.abs(tb["virial"]).max()
    assert ta["misfit_atoms"] == tb["misfit_atoms"] and ta["list_builds"] == tb["list_builds"]
    assert a.neighbor_entries() == b.neighbor_entries()
    a.close()
    b.close()
