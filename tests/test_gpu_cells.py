"""The emit of cells, one triangle a lane, around the 64 cells a wave lists and with
the four cells a lane of large meshes; against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle
from kvs_amd import datasets, kmc
from tests.conftest import bits_equal

pytestmark = pytest.mark.gpu


NODES = {kmc.TETRAHEDRA: 4, kmc.HEXAHEDRA: 8, kmc.PYRAMID: 5, kmc.PRISM: 6}


def check(v, c, k, cell, label):
    print("case", label, flush=True)
    got, want = kmc.extract_unstructured(v, c, k, cell, 0.5), oracle.unstructured_isosurface(v, c, k, cell, 0.5)
    assert got["n_triangles"] == want["n_triangles"], label
    assert bits_equal(got["coords"], want["coords"]) and bits_equal(got["normals"], want["normals"]), label
    table = np.random.default_rng(1).integers(0, 256, (256, 3)).astype(np.uint8)
    coef = [0.31, -0.52, 0.79, -0.2]
    got = kmc.slice_plane_unstructured(v, c, k, cell, coef, table)
    want = oracle.unstructured_slice_plane(v, c, k, cell, coef, table)
    assert bits_equal(got["coords"], want["coords"]) and bits_equal(got["normals"], want["normals"]), label
    assert np.array_equal(got["colors"], want["colors"]), label


@pytest.mark.parametrize("cell", [kmc.TETRAHEDRA, kmc.HEXAHEDRA, kmc.PYRAMID, kmc.PRISM])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1000])
def test_cell_counts(cell, n):
    v, c, k = datasets.unstructured_mesh((12, 11, 10), cell, seed=5)
    rng = np.random.default_rng(n)
    v = rng.random(v.size).astype(np.float32)    # noise: most cells hold triangles, up to the most there are
    check(v, c, k.reshape(-1)[: n * NODES[cell]], cell, f"{cell} {n}")


@pytest.mark.parametrize("cell,dims", [(kmc.TETRAHEDRA, (72, 72, 71)), (kmc.HEXAHEDRA, (130, 130, 129))])
@pytest.mark.parametrize("noise", [False, True])
def test_large_meshes(cell, dims, noise):
    v, c, k = datasets.unstructured_mesh(dims, cell, seed=6)
    if noise:
        v = v.copy()
        v[: v.size // 50] = np.random.default_rng(2).random(v.size // 50)
    check(v, c, k, cell, f"{cell} {dims} noise={noise}")
