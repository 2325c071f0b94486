"""The caller's arrays to the device and back at the sizes where the staging
splits them: one atom pair, one part filled to the last atom, one atom more,
several parts with a short last one.  Every value must come back bit for bit."""
import ctypes as C

import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from rbmd_amd.lib import Context, GpuSystem

pytestmark = pytest.mark.gpu

PART = (1 << 20) // (8 * 12)  # atoms of a state (x, v, f, image) in one part


def ptr(a, t=C.c_double):
    return a.ctypes.data_as(C.POINTER(t))


@pytest.mark.parametrize("n", [64, PART // 2 * 2, PART // 2 * 2 + 2, 3 * PART // 2 * 2 + 14])
def test_state_round_trip(n):
    g = GpuSystem(Context(0), make_salt(n_ions=n, seed=1), salt_config())
    rng = np.random.default_rng(n)
    x, v = rng.standard_normal((n, 3)), rng.standard_normal((n, 3))
    x[0], v[-1] = [-0.0, 5e-324, np.inf], [np.nan, -np.inf, 1e308]
    image = rng.integers(-2 ** 31, 2 ** 31, (n, 3)).astype(np.int32)
    assert g.L.rbmd_sys_upload_state(g.h, ptr(x), ptr(v), ptr(image, C.c_int32)) == 0
    gx, gv, _, gi = g.state()
    assert gx.tobytes() == x.tobytes()
    assert gv.tobytes() == v.tobytes()
    assert np.array_equal(gi, image)
    # one array alone: more atoms to a part
    x2 = rng.standard_normal((n, 3))
    assert g.L.rbmd_sys_upload_state(g.h, ptr(x2), None, None) == 0
    out = np.zeros((n, 3))
    assert g.L.rbmd_sys_download_state(g.h, ptr(out), None, None, None) == 0
    assert out.tobytes() == x2.tobytes()
    assert g.state()[1].tobytes() == v.tobytes()


@pytest.mark.parametrize("n", [PART // 2 * 2 + 2, 3 * PART // 2 * 2 + 14])
def test_real_space_results_in_parts(n):
    """forces, virials and energies of a call in several parts: the force sums
    to zero over the atoms and each atom's values equal those of the same call
    with only one of the arrays asked for"""
    g = GpuSystem(Context(0), make_salt(n_ions=n, seed=2), salt_config())
    f, vir, elj, ec = g.force_real()
    assert np.abs(f.sum(0)).max() < 1e-9 * np.abs(f).sum()
    for k, a in enumerate((f, vir, elj, ec)):
        out = np.zeros_like(a)
        args = [None] * 4
        args[k] = ptr(out)
        assert g.L.rbmd_force_real(g.h, *args) == 0
        assert out.tobytes() == a.tobytes()
