"""The row-count scan at the counts where its form changes: one segment of 4096
rows, the four up to which a workgroup sums the counts before its own, and the
4096 up to which it sums the segments' sums; against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import assert_same_surface

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nz", [(64, 64), (17, 241), (128, 128), (127, 131), (128, 256), (4096, 4096), (4099, 4097)])
@pytest.mark.parametrize("dup", [True, False])
def test_row_counts(ny, nz, dup):
    # 4096, 4097, 16384, 16637, 32768, 4096 segments, more: some rows busy, the last among them
    rng = np.random.default_rng(ny)
    v = np.zeros((nz, ny, 2), np.uint8)
    v.reshape(-1)[rng.integers(0, v.size, 3000)] = 9
    v[-1, -1] = 9
    got = kmc.extract(v, 4.5, kmc.POLYGON_NORMAL, dup)
    assert_same_surface(got, oracle.extract(v, 4.5, kmc.POLYGON_NORMAL, dup), f"{v.shape} dup={dup}")
