"""The slice's triangles where a wave's 64 lie in few rows, in rows of several
slices and in more than 64 rows (most of them without a triangle), and colour maps
around the size kept in LDS; against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import bits_equal

pytestmark = pytest.mark.gpu


def check(shape, coef, res):
    rng = np.random.default_rng(res)
    v = rng.standard_normal(shape).astype(np.float32)
    table = rng.integers(0, 256, (res, 3)).astype(np.uint8)
    label = f"{shape} {coef} {res}"
    print("case", label, flush=True)
    got, want = kmc.slice_plane(v, coef, table), oracle.slice_plane(v, coef, table)
    assert got["n_triangles"] == want["normals"].size // 3 > 0, label
    assert bits_equal(got["coords"], want["coords"]) and bits_equal(got["normals"], want["normals"]), label
    assert np.array_equal(got["colors"], want["colors"]), label


@pytest.mark.parametrize("shape,coef", [
    ((40, 300, 20), [0.1, 1.0, 0.0, -2.5]),       # three busy rows of 299 a slice
    ((40, 300, 3), [0.1, 1.0, 0.001, -2.5]),
    ((90, 2, 8), [1.0, 0.5, 0.05, -5.0]),         # one cell row a slice
    ((60, 5, 7), [1.0, 0.1, -0.02, -3.0]),        # four: a unit spans many slices
    ((12, 65, 9), [-1.0, 0.03, 0.02, 3.5]),       # 64 and 65 cell rows a slice
    ((12, 66, 9), [1.0, 0.03, -0.02, -4.5]),
    ((5, 4, 6), [0.0, 0.4, 1.0, -2.25]),          # constant along x; fewer than 64
])
def test_rows_of_a_unit(shape, coef):
    check(shape, coef, 256)


@pytest.mark.parametrize("res", [1, 2, 1024, 1025])
def test_color_map_sizes(res):
    check((20, 30, 40), [0.3, -0.5, 0.8, -3.0], res)
