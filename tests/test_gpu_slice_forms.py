"""The slice's two device paths -- thresholds of node rows, classification of every
node -- where rows end near a 64-node chunk or hold more than 64 chunks, and with
colour maps around and above the size kept in LDS; against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import bits_equal

pytestmark = pytest.mark.gpu


def check(monkeypatch, shape, coef, res):
    rng = np.random.default_rng(res)
    v = rng.standard_normal(shape).astype(np.float32)
    table = rng.integers(0, 256, (res, 3)).astype(np.uint8)
    want = oracle.slice_plane(v, coef, table)
    for path in ("thresholds", "classify"):
        if path == "classify":
            monkeypatch.setenv("KMC_SLICE", "classify")
        else:
            monkeypatch.delenv("KMC_SLICE", raising=False)
        label = f"{shape} {coef} {res} {path}"
        print("case", label, flush=True)
        got = kmc.slice_plane(v, coef, table)
        assert got["n_triangles"] == want["normals"].size // 3 > 0, label
        assert bits_equal(got["coords"], want["coords"]) and bits_equal(got["normals"], want["normals"]), label
        assert np.array_equal(got["colors"], want["colors"]), label


@pytest.mark.parametrize("nx", [2, 63, 64, 65, 129, 1025, 4096, 4097, 8200])
def test_row_ends(monkeypatch, nx):
    x = float(nx) - 1.5                              # through the last cells of a row, and along it
    check(monkeypatch, (7, 9, nx), [1.0, 0.01, -0.02, -x], 256)
    check(monkeypatch, (7, 9, nx), [0.002, 1.0, 0.3, -4.0], 256)


@pytest.mark.parametrize("res", [1, 2, 1024, 1025, 4000])
def test_color_maps(monkeypatch, res):
    check(monkeypatch, (20, 30, 40), [0.3, -0.5, 0.8, -3.0], res)


def test_plane_beyond_the_float_range(monkeypatch):
    # infinite at the volume's corners: the classification path by itself
    check(monkeypatch, (29, 33, 70), [float(np.float32(c)) for c in (3e38, 3e38, 0.0, -3e38)], 256)
