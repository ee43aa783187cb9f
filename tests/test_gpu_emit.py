"""The emit at the sizes where its lists and chunks split, against the oracle,
bit for bit: rows around the 64-node chunk and past 64 chunks, every cell
active, several levels, clamp ranges that move the crossings and values that
are not finite."""

import numpy as np
import pytest

import oracle
from kvs_amd import kmc
from tests.conftest import assert_same_surface

pytestmark = pytest.mark.gpu

MODES = [(kmc.POLYGON_NORMAL, True), (kmc.POLYGON_NORMAL, False), (kmc.VERTEX_NORMAL, False)]


def check(v, iso, normal, dup, **kw):
    label = f"{v.dtype} {v.shape} iso={iso!r} normal={normal} dup={dup} {kw}"
    print("case", label, flush=True)
    want = oracle.extract(v, iso, normal, dup, min_max_values=kw.get("min_max"), coords=kw.get("coords"))
    assert_same_surface(kmc.extract(v, iso, normal, dup, **kw), want, label)


@pytest.mark.parametrize("nx", [2, 63, 64, 65, 127, 129, 257, 4096, 4097, 4160])
@pytest.mark.parametrize("normal,dup", MODES)
def test_row_lengths(nx, normal, dup):
    rng = np.random.default_rng(nx)
    for ny, nz in ((2, 2), (3, 5), (70, 2)) if nx < 1000 else ((2, 3),):
        check(rng.standard_normal((nz, ny, nx)).astype(np.float32), 0.1, normal, dup)


@pytest.mark.parametrize("dtype", [np.uint8, np.int16, np.float32, np.float64])
@pytest.mark.parametrize("normal,dup", MODES)
def test_every_cell_active(dtype, normal, dup):
    # a checkerboard makes every cell active with the most crossings, noise every case
    z, y, x = np.indices((9, 40, 131))
    check(((x + y + z) % 2 * 10 + 1).astype(dtype), 5.5, normal, dup)
    rng = np.random.default_rng(5)
    check(rng.integers(0, 120, (17, 33, 130)).astype(dtype), 60.25, normal, dup)


@pytest.mark.parametrize("normal,dup", MODES)
@pytest.mark.parametrize("min_max", [(0.25, 0.5), (0.1, 0.9), (-3.0, 3.0), (0.4, 0.2), (0.5, 0.5000001)])
def test_clamp_ranges(normal, dup, min_max):
    # crossings outside the edge (r > 1), 0 / 0 and x / 0, ends that are no floats, an inverted range
    rng = np.random.default_rng(11)
    v = rng.standard_normal((8, 9, 70)).astype(np.float32)
    check(v, 0.3, normal, dup, min_max=min_max, coords=((-1.5, 0.25, 3.0), (2.0, 9.0, 3.5)))
    check((v * 50).astype(np.int8), 3.0, normal, dup, min_max=(min_max[0] * 10, min_max[1] * 10))


@pytest.mark.parametrize("normal,dup", MODES)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_not_finite(normal, dup, dtype):
    rng = np.random.default_rng(12)
    v = rng.standard_normal((6, 10, 66)).astype(dtype)
    flat = v.reshape(-1)
    flat[rng.integers(1, flat.size, 40)] = np.nan
    flat[rng.integers(1, flat.size, 20)] = np.inf
    flat[rng.integers(1, flat.size, 20)] = -np.inf
    flat[rng.integers(1, flat.size, 40)] = -0.0
    check(v, 0.0, normal, dup, min_max=(-2.0, 2.0))
    check(v, 0.2, normal, dup)


@pytest.mark.parametrize("normal,dup", MODES)
def test_levels_with_and_without_surfaces(normal, dup):
    rng = np.random.default_rng(13)
    v = rng.standard_normal((20, 30, 150)).astype(np.float32)
    levels = [-0.5, 50.0, 0.0, 0.4, -60.0, 0.1, 0.2, 0.3, 0.6]
    got = kmc.extract_levels(v, levels, normal, dup)
    for iso, g in zip(levels, got):
        print("case level", iso, flush=True)
        assert_same_surface(g, oracle.extract(v, iso, normal, dup), f"level {iso}")
