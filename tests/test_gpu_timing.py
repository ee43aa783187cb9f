"""Device times of a call's kernels: the emit is its three parts, and there is no compaction."""
import ctypes

import pytest

from kvs_amd import datasets, kmc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normal,dup", [(kmc.POLYGON_NORMAL, True), (kmc.POLYGON_NORMAL, False), (kmc.VERTEX_NORMAL, False)])
def test_emit_is_its_parts(normal, dup):
    lib = kmc.load()
    v = datasets.blobs(48, seed=5)
    lib.kmc_set_timing(1)
    try:
        assert kmc.extract(v, 0.5, normal, dup)["n_triangles"] > 0
        t = kmc.Timing()
        assert lib.kmc_last_timing(ctypes.byref(t)) == kmc.OK
    finally:
        lib.kmc_set_timing(0)
    assert t.passes == 1 and t.emit_ms > 0 and t.triangles_ms > 0
    assert t.compact_ms == 0
    assert abs(t.vertices_ms + t.triangles_ms + t.vertex_normals_ms - t.emit_ms) < 1e-3
