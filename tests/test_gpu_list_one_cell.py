"""VERLET lists in boxes narrower than two cutoffs, one cell an axis, where the
cell is visited through several images: entry by entry the oracle's."""
import numpy as np
import pytest

from rbmd_amd import make_salt, salt_config
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 64, 130, 512])
@pytest.mark.parametrize("cells", [0.55, 0.9, 1.01, 1.7])  # box edge over rc
def test_lists_equal_the_oracle(ctx, n, cells):
    s = make_salt(n_ions=n, density=0.5, seed=n)
    rc = float((s.hi - s.lo)[0]) / cells
    g, o = pair(ctx, s, salt_config(cut_off=rc, r_core=rc))
    assert g.geometry()[0].max() == 1
    for a, b in zip(g.neighbors(27 * n), o.neighbors(27 * n)):
        assert np.array_equal(a, b)
