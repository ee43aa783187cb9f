"""Classification by rows and by runs of 16 chunks, at the row lengths, level counts and
row numbers where one gives way to the other, against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import assert_same_surface

pytestmark = pytest.mark.gpu

SHAPES = [(64, 128), (91, 91)]          # 8192 rows (by rows) and 8281


@pytest.mark.parametrize("dtype,chunks", [(np.uint16, (2, 3, 4, 5, 6, 7, 8, 9)), (np.float32, (2, 3, 4, 5, 6, 7, 12, 13)),
                                          (np.float64, (2, 3, 4, 5, 6))])
@pytest.mark.parametrize("levels", [1, 2, 3, 4, 5, 8])
def test_forms(dtype, chunks, levels):
    for nz, ny in SHAPES:
        for c in chunks:
            nx = 64 * c - (c % 3) * 2 - 1            # odd: 16-bit rows are not whole dwords
            rng = np.random.default_rng(c)
            v = np.zeros((nz, ny, nx), dtype)
            at = rng.integers(0, v.size, 400)
            v.reshape(-1)[at] = rng.integers(1, 60, 400).astype(dtype)
            v[-1, -1, -1] = v[0, 0, 0] = 60
            iso = [0.5 + 7 * k for k in range(levels)]
            for s, l in zip(kmc.extract_levels(v, iso, kmc.POLYGON_NORMAL, True), iso):
                assert_same_surface(s, oracle.extract(v, l, kmc.POLYGON_NORMAL, True), f"{v.shape} {v.dtype} {levels} {l}")
