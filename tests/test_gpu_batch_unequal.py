"""Batches of very unequal volumes -- one large among many small ones, of one node row
among them, with several levels and both classification forms -- against the
oracle, bit for bit."""

import numpy as np
import pytest
import torch

import oracle
from kvs_amd import kmc
from tests.conftest import assert_same_surface

pytestmark = pytest.mark.gpu


def _volume(dims, seed, dtype):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*(np.linspace(0, 3, n) for n in (nz, ny, nx)), indexing="ij")
    f = np.sin(2 * x + seed) + np.cos(3 * y) + np.sin(z * 2 + x) + 0.05 * rng.random((nz, ny, nx))
    return f.astype(np.float32) if dtype == np.float32 else ((f + 3) * 40).astype(dtype)


@pytest.mark.parametrize("normal,dup", [(kmc.POLYGON_NORMAL, True), (kmc.POLYGON_NORMAL, False), (kmc.VERTEX_NORMAL, False)])
@pytest.mark.parametrize("large_at,small", [(0, 300), (40, 40)])
def test_one_large_volume(normal, dup, large_at, small):
    specs = []
    for i in range(small + 1):
        dtype = np.uint8 if i % 5 == 3 else np.float32
        if i == large_at:
            dims, dtype = (300, 170, 130), np.float32
        else:
            dims = [(5, 6, 7), (8, 3, 2), (2, 2, 2), (65, 4, 3), (4, 1, 9), (16, 8, 4)][i % 6]
        levels = [0.3, -0.2] if i % 4 == 1 else [0.3]
        specs.append((_volume(dims, i, dtype), [120.5 + 20 * l for l in levels] if dtype == np.uint8 else levels, normal, dup))
    got = kmc.batch_extract(specs)
    for (v, levels, _, _), surfaces in zip(specs, got):
        for l, s in zip(levels, surfaces):
            assert_same_surface(s, oracle.extract(v, l, normal, dup), f"{v.shape} {v.dtype} {l}")


def test_autotuned_plan_runs_on_another_stream():
    # planned on one stream, its tables on the device before a run on a second
    made, used = torch.cuda.Stream(), torch.cuda.Stream()
    vols = [_volume((40 + i, 33, 20), i, np.float32) for i in range(12)]
    dev = [torch.from_numpy(v).cuda() for v in vols]
    torch.cuda.synchronize()
    specs = [(kmc.make_volume(t.data_ptr(), dims=v.shape[::-1], memory=kmc.MEMORY_DEVICE, dtype=np.float32,
                              min_max=(float(v.min()), float(v.max()))), [0.3], kmc.POLYGON_NORMAL, True)
             for t, v in zip(dev, vols)]
    b = kmc.Batch(specs, autotune=True, stream=made.cuda_stream)
    try:
        b.run(stream=used.cuda_stream)
        for v, s in zip(vols, b.surfaces()):
            assert_same_surface(kmc.device_surface_to_numpy(s), oracle.extract(v, 0.3, kmc.POLYGON_NORMAL, True), f"{v.shape}")
    finally:
        b.close()
