"""Surfaces that fall to few of the emit's units -- planes of one coordinate, small
ones in large volumes, rows of more than 64 chunks -- against the oracle."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import assert_same_surface

pytestmark = pytest.mark.gpu

MODES = [(kmc.POLYGON_NORMAL, True), (kmc.POLYGON_NORMAL, False), (kmc.VERTEX_NORMAL, False)]


def _planes(shape):
    nz, ny, nx = shape
    v = np.zeros(shape, np.uint8)
    v[nz // 2:, : ny // 2] = 9
    v[:, 1: ny // 3] = 9
    v[: nz // 3, :, nx // 2: nx // 2 + 3] = 9
    return v


@pytest.mark.parametrize("shape", [(33, 257, 513), (64, 64, 4096), (40, 33, 1100), (9, 50, 2049), (9, 20, 4161), (5, 7, 9000), (3, 2, 20000), (260, 130, 2),
                                   (70, 1, 64), (1, 70, 65)])
@pytest.mark.parametrize("normal,dup", MODES)
def test_planes(shape, normal, dup):
    v = _planes(shape)
    got = kmc.extract(v, 4.5, normal, dup)
    assert_same_surface(got, oracle.extract(v, 4.5, normal, dup), f"{shape}")


@pytest.mark.parametrize("normal,dup", MODES)
def test_speck_in_a_large_volume(normal, dup):
    # 2^22 chunks: a unit's pieces lie far apart for a speck, side by side for a plane (below)
    v = np.zeros((512, 512, 1024), np.uint8)
    v[300:303, 200:203, 511:514] = 9
    got = kmc.extract(v, 4.5, normal, dup)
    small = oracle.extract(v[298:306, 198:206, 508:518].copy(), 4.5, normal, dup)
    assert got["n_triangles"] == small["n_triangles"]
    assert np.array_equal(got["connections"], small["connections"])
    assert np.array_equal(got["coords"].reshape(-1, 3) - np.float32([508, 198, 298]), small["coords"].reshape(-1, 3))
    assert np.array_equal(got["normals"], small["normals"])


@pytest.mark.parametrize("normal,dup", MODES)
def test_plane_in_a_large_volume(normal, dup):
    v = np.zeros((512, 512, 1024), np.uint8)
    v[256:] = 9
    got = kmc.extract(v, 4.5, normal, dup)
    slab = oracle.extract(v[254:258].copy(), 4.5, normal, dup)
    assert got["n_triangles"] == slab["n_triangles"] == 2 * 1023 * 511
    assert np.array_equal(got["connections"], slab["connections"])
    assert np.array_equal(got["coords"].reshape(-1, 3) - np.float32([0, 0, 254]), slab["coords"].reshape(-1, 3))
    assert np.array_equal(got["normals"], slab["normals"])
