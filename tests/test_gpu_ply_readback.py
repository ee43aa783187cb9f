"""PLY files of surfaces with connections read back by a reader that knows the format
only -- what the header declares -- in both file types."""

import numpy as np
import pytest

from kvs_amd import datasets, kmc
from tests.conftest import bits_equal

pytestmark = pytest.mark.gpu

SCALAR = {"char": "i1", "uchar": "u1", "short": "<i2", "ushort": "<u2", "int": "<i4", "uint": "<u4", "float": "<f4", "double": "<f8"}


def read_ply(path):
    """{element: {property: array}} of a little-endian or ascii PLY file; a list property gives an array a row."""
    raw = open(path, "rb").read()
    head, body = raw.split(b"end_header\n", 1)
    lines = head.decode().splitlines()
    assert lines[0] == "ply"
    form = next(l.split()[1] for l in lines if l.startswith("format"))
    elements = []
    for l in (x.split() for x in lines):
        if l[0] == "element":
            elements.append((l[1], int(l[2]), []))
        elif l[0] == "property":
            elements[-1][2].append((l[-1], l[1:-1]))
    tokens = iter(body.split()) if form == "ascii" else None
    at = 0

    def take(kind):
        nonlocal at
        if tokens is not None:
            return np.dtype(SCALAR[kind]).type(next(tokens))
        d = np.dtype(SCALAR[kind])
        at += d.itemsize
        return np.frombuffer(body, d, 1, at - d.itemsize)[0]

    out = {}
    for name, count, props in elements:
        cols = {p: [] for p, _ in props}
        for _ in range(count):
            for p, kind in props:
                cols[p].append([take(kind[2]) for _ in range(take(kind[1]))] if kind[0] == "list" else take(kind[0]))
        out[name] = {p: np.array(c) for p, c in cols.items()}
    assert at == len(body) if tokens is None else next(tokens, None) is None
    return out


@pytest.mark.parametrize("normal", [kmc.POLYGON_NORMAL, kmc.VERTEX_NORMAL])
@pytest.mark.parametrize("binary", [True, False])
def test_surface_comes_back(tmp_path, normal, binary):
    d = kmc.extract(datasets.blobs(10, seed=7, nblobs=2), 0.4, normal, False)
    kmc.export_ply(d, normal, tmp_path / "s.ply", binary=binary, color=(10, 200, 30))
    back = read_ply(tmp_path / "s.ply")
    v, f = back["vertex"], back["face"]
    coords = np.stack([v["x"], v["y"], v["z"]], 1).astype(np.float32).reshape(-1)
    if binary:
        assert bits_equal(coords, d["coords"])
    else:
        assert np.allclose(coords, d["coords"], rtol=5e-6, atol=0)     # six significant digits
    assert np.array_equal(f["vertex_indices"].reshape(-1), d["connections"].astype(np.int64))
    assert (np.stack([v["red"], v["green"], v["blue"]], 1) == (10, 200, 30)).all()
