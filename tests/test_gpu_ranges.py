"""Ranges of unstructured volumes found with the count pass, and the ordered
passes behind them where NaN or a negative zero makes the order matter."""
import numpy as np
import pytest

import oracle
from kvs_amd import datasets, kmc
from tests.conftest import bits_equal

pytestmark = pytest.mark.gpu


def check(v, c, k, cell, label):
    print("case", label, flush=True)
    got = kmc.extract_unstructured(v, c, k, cell, 0.5)
    want = oracle.unstructured_isosurface(v, c, k, cell, 0.5)
    assert got["n_triangles"] == want["n_triangles"], label
    assert bits_equal(got["coords"], want["coords"]) and bits_equal(got["normals"], want["normals"]), label
    mn, mx = oracle.unstructured_min_max(v, k)
    assert bits_equal(np.float64([got["min_value"], got["max_value"]]), np.float64([mn, mx])), label
    lo, hi = oracle.unstructured_min_max_coords(c, k)
    assert bits_equal(np.float32(got["min_coord"] + got["max_coord"]), np.float32(list(lo) + list(hi))), label


@pytest.mark.parametrize("cell", [kmc.TETRAHEDRA, kmc.HEXAHEDRA, kmc.PYRAMID, kmc.PRISM])
@pytest.mark.parametrize("dims", [(2, 2, 2), (5, 4, 3), (40, 41, 37)])
def test_plain_ranges(cell, dims):
    v, c, k = datasets.unstructured_mesh(dims, cell, seed=3)
    check(v, c, k, cell, f"{cell} {dims}")
    check(v.astype(np.float64), c, k, cell, f"{cell} {dims} double")
    v0 = v.copy()
    v0[0] = 77.0   # the first value counts even where no cell uses it
    check(v0, c, k, cell, f"{cell} {dims} first")


@pytest.mark.parametrize("where", ["value nan", "first nan", "value -0", "coord nan", "coord -0"])
def test_order_matters(where):
    v, c, k = datasets.unstructured_mesh((9, 8, 7), kmc.TETRAHEDRA, seed=4)
    v, c = v.copy(), c.copy()
    if where == "value nan":
        v[k[100]] = np.nan
    elif where == "first nan":
        v[0] = np.nan
    elif where == "value -0":
        v -= v.min()
        v[k[50]], v[k[300]] = -0.0, 0.0
    elif where == "coord nan":
        c[k[77], 1] = np.nan
    else:
        c[k[10], 2], c[k[400], 2] = -0.0, 0.0
    check(v, c, k, kmc.TETRAHEDRA, where)
