"""The min/max pass at the sizes where its number of parts changes (one, one more
than a merging thread's first, the most there are) against the serial scan."""

import numpy as np
import pytest

from kvs_amd import kmc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts", [1, 2, 256, 257, 2047, 2048, 2049])
@pytest.mark.parametrize("dtype", [np.uint8, np.float32, np.float64])
def test_parts(parts, dtype):
    per = 256 * 16 // np.dtype(dtype).itemsize
    for n in (parts * per, parts * per - per + 2):
        rng = np.random.default_rng(n)
        v = (100 + rng.random(n) * 50).astype(dtype)
        v[min(per, n - 2)] = 200    # the greatest opens the second part, the last value is the least
        v[-1] = 3
        assert kmc.min_max(v.reshape(n // 2, 1, 2)) == (3.0, 200.0), (parts, dtype, n)
