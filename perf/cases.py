"""Performance cases of the isosurface library: what users of libkmc.so have it do.

Each case is one call (or one batch, or one burst of requests) through the
public C ABI as kvs_amd.kmc binds it.  Volumes that a program holds on the GPU
are torch tensors; surfaces come back as views of the library's own arrays,
released at the next call, as a viewer that replaces its mesh would.

kinds: "extract" (kmc_extract / kmc_extract_levels), "noalloc"
(kmc_extract_noalloc into the caller's arrays), "batch" (kmc_batch_*),
"serve" (kmc_server_*), "slice" (kmc_slice_plane), "mesh"
(kmc_extract_unstructured), "meshslice" (kmc_slice_plane_unstructured).
"""
import ctypes
import math
import zlib

import numpy as np
import torch

from kvs_amd import kmc

DEV = "cuda"
TORCH = {"f32": torch.float32, "f64": torch.float64, "u8": torch.uint8, "i16": torch.int16, "u16": torch.uint16}
NUMPY = {"f32": np.float32, "f64": np.float64, "u8": np.uint8, "i16": np.int16, "u16": np.uint16}
SIZE = {"f32": 4, "f64": 8, "u8": 1, "i16": 2, "u16": 2}
CELL = {"tet": kmc.TETRAHEDRA, "hex": kmc.HEXAHEDRA, "prism": kmc.PRISM}
CELLS_PER_CUBE = {"tet": 6, "hex": 1, "prism": 2}


def listed():
    return [
        # the drop-in's ordinary small call: a host volume as an interactive program loads it, the
        # reference's default mode (PolygonNormal, duplicated vertices), min/max not known yet
        {"name": "host 64 f32 dup", "kind": "extract", "nx": 64, "ny": 64, "nz": 64, "dtype": "f32", "field": "blobs",
         "levels": 1, "normal": "polygon", "dup": True, "cached": False, "host": True},
        # the smallest calls on resident data: an interactive isolevel slider over a small ragged volume
        {"name": "small ragged u16 vn", "kind": "extract", "nx": 101, "ny": 87, "nz": 73, "dtype": "u16", "field": "ct",
         "levels": 1, "normal": "vertex", "dup": False, "cached": True, "host": False},
        # an ordinary simulation field on the GPU, default mode
        {"name": "device 256 f32 dup", "kind": "extract", "nx": 256, "ny": 256, "nz": 256, "dtype": "f32",
         "field": "blobs", "levels": 1, "normal": "polygon", "dup": True, "cached": True, "host": False},
        # a new double-precision time step: min/max computed by the call, odd sizes, two levels, shared vertices
        {"name": "ragged f64 x2 shared", "kind": "extract", "nx": 301, "ny": 257, "nz": 199, "dtype": "f64",
         "field": "turbulence", "levels": 2, "normal": "polygon", "dup": False, "cached": False, "host": False},
        # a CT scan: 512^3 uint8, one level, vertex normals (benchmark configuration)
        {"name": "ct 512 u8 vn", "kind": "extract", "nx": 512, "ny": 512, "nz": 512, "dtype": "u8", "field": "ct",
         "levels": 1, "normal": "vertex", "dup": False, "cached": True, "host": False},
        # the headline benchmark: 1024^3 float32 turbulence, three levels, vertex normals
        {"name": "turbulence 1024 f32 x3 vn", "kind": "extract", "nx": 1024, "ny": 1024, "nz": 1024, "dtype": "f32",
         "field": "turbulence", "levels": 3, "normal": "vertex", "dup": False, "cached": True, "host": False},
        # the drop-in on a medium host scan: upload, extraction and download of the surface
        {"name": "host 320x288x256 i16 shared", "kind": "extract", "nx": 320, "ny": 288, "nz": 256, "dtype": "i16",
         "field": "ct", "levels": 1, "normal": "polygon", "dup": False, "cached": True, "host": True},
        # a planned batch of uneven volumes (32..256 per axis, 1..4 levels), duplicated vertices
        {"name": "batch of 14", "kind": "batch", "volumes": 14, "edge": 256, "shape": 3000, "surfaces": 30},
        # requests that arrive together over resident volumes of three types and both normal types
        {"name": "serve 20 requests", "kind": "serve", "volumes": 6, "edge": 256, "shape": 4000, "requests": 20},
        # a cutting plane through a resident volume
        {"name": "slice 640x704x768 f32", "kind": "slice", "nx": 640, "ny": 704, "nz": 768, "dtype": "f32",
         "field": "turbulence"},
        # an unstructured simulation mesh: 3.07 M tetrahedra, ranges not known yet
        {"name": "tetrahedra 3.07M", "kind": "mesh", "nx": 81, "ny": 81, "nz": 81, "cell": "tet"},
        # a caller that owns its buffers and may not allocate
        {"name": "noalloc 256x240x224 u16 vn", "kind": "noalloc", "nx": 256, "ny": 240, "nz": 224, "dtype": "u16",
         "field": "ct", "normal": "vertex", "dup": False},
    ]


def _edges(rng, lo, hi, most):
    """Three edge lengths, log-uniform in [lo, hi] around a common size, at most `most` nodes."""
    while True:
        base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        e = [max(lo // 2, int(round(base * math.exp(rng.uniform(-0.4, 0.4))))) for _ in range(3)]
        if e[0] * e[1] * e[2] <= most:
            return e


def draw(rng):
    kind = rng.choice(["extract"] * 5 + ["batch", "serve", "slice", "mesh", "meshslice", "noalloc"])
    if kind == "extract":
        host = rng.random() < 0.2
        nx, ny, nz = _edges(rng, 32, 256 if host else 800, 3 * 10 ** 8)
        mode = rng.choice(["dup", "shared", "vertex"])
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "dtype": rng.choice(["f32", "f32", "u8", "u16", "i16", "f64"]),
                "field": rng.choice(["blobs", "ct", "turbulence"]), "levels": rng.choice([1, 1, 2, 3, 5]),
                "normal": "vertex" if mode == "vertex" else "polygon", "dup": mode == "dup",
                "cached": rng.random() < 0.7, "host": host}
    if kind == "noalloc":
        nx, ny, nz = _edges(rng, 32, 200, 10 ** 7)
        mode = rng.choice(["dup", "shared", "vertex"])
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "dtype": rng.choice(["f32", "u8", "u16", "i16", "f64"]),
                "field": rng.choice(["blobs", "ct"]), "normal": "vertex" if mode == "vertex" else "polygon",
                "dup": mode == "dup"}
    if kind == "batch":
        return {"kind": kind, "volumes": rng.randint(4, 14), "edge": rng.choice([64, 128, 192, 256]),
                "shape": rng.randint(1, 10 ** 6), "surfaces": rng.randint(16, 30)}
    if kind == "serve":
        return {"kind": kind, "volumes": rng.randint(2, 8), "edge": rng.choice([96, 160, 256]),
                "shape": rng.randint(1, 10 ** 6), "requests": rng.randint(4, 20)}
    if kind == "slice":
        nx, ny, nz = _edges(rng, 48, 900, 4 * 10 ** 8)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "dtype": rng.choice(["f32", "u8", "i16"]),
                "field": "blobs"}
    nx, ny, nz = _edges(rng, 12, 100, 10 ** 6)
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "cell": rng.choice(["tet", "hex", "prism"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _blobs(nx, ny, nz, g, count=3, noise=0.01):
    """Gaussian blobs (peak 1, centres U[0.2, 0.8], sigma U[0.08, 0.2] of the box) plus uniform noise, in [0, ~1.5]."""
    c = torch.rand(count, 3, device=DEV, generator=g) * 0.6 + 0.2
    s = torch.rand(count, 1, device=DEV, generator=g) * 0.12 + 0.08
    ax = [torch.exp(-((torch.linspace(0, 1, n, device=DEV)[None, :] - c[:, k:k + 1]) ** 2) / (2 * s * s))
          for k, n in enumerate((nx, ny, nz))]
    f = torch.zeros(nz, ny, nx, device=DEV)
    for m in range(count):
        f += ax[2][m][:, None, None] * ax[1][m][None, :, None] * ax[0][m][None, None, :]
    f += (torch.rand(nz, ny, nx, device=DEV, generator=g) * 2 - 1) * noise
    return f


def _turbulence(nx, ny, nz, g, modes=64):
    """64 random-phase Fourier modes, |k| U[1, 64] per box, amplitude |k|^(-5/3), normalised to [-1, 1]."""
    u = torch.rand(modes, 4, device=DEV, generator=g)
    mag = 1 + 63 * u[:, 0]
    cz = 2 * u[:, 1] - 1
    r = torch.sqrt(1 - cz * cz)
    k = torch.stack([mag * r * torch.cos(2 * math.pi * u[:, 2]), mag * r * torch.sin(2 * math.pi * u[:, 2]), mag * cz], 1)
    w = 2 * math.pi / max(nx, ny, nz)
    px, py, pz = (w * k[:, i:i + 1] * torch.arange(n, device=DEV)[None, :] for i, n in enumerate((nx, ny, nz)))
    pz = pz + 2 * math.pi * u[:, 3:4]
    right = torch.cat([torch.cos(px), -torch.sin(px)], 0)
    amp = (mag ** (-5.0 / 3.0))[:, None, None]
    f = torch.empty(nz, ny, nx, device=DEV)
    step = max(1, (1 << 20) // ny)
    for z in range(0, nz, step):
        p = pz[:, z:z + step, None] + py[:, None, :]
        left = torch.cat([amp * torch.cos(p), amp * torch.sin(p)], 0).reshape(2 * modes, -1)
        f[z:z + step] = (left.t() @ right).reshape(-1, ny, nx)
    lo, hi = f.min(), f.max()
    f -= lo
    f *= 2.0 / (hi - lo)
    f -= 1.0
    return f


def _ct(nx, ny, nz, g, ellipsoids=20):
    """Value noise on a 32^3 lattice, trilinearly upsampled, with constant ellipsoids, scaled to [0, 1]."""
    lat = torch.rand(1, 1, 33, 33, 33, device=DEV, generator=g)
    f = torch.nn.functional.interpolate(lat, size=(nz, ny, nx), mode="trilinear", align_corners=True)[0, 0]
    p = torch.rand(ellipsoids, 7, device=DEV, generator=g).cpu()
    for e in p.tolist():
        c, a, value = [0.1 + 0.8 * t for t in e[:3]], [0.03 + 0.12 * t for t in e[3:6]], (60 + 160 * e[6]) / 255
        lo = [max(0, int((c[k] - a[k]) * n)) for k, n in enumerate((nx, ny, nz))]
        hi = [min(n, int((c[k] + a[k]) * n) + 2) for k, n in enumerate((nx, ny, nz))]
        d = [((torch.arange(lo[k], hi[k], device=DEV) / max(1, n - 1) - c[k]) / a[k]) ** 2
             for k, n in enumerate((nx, ny, nz))]
        box = f[lo[2]:hi[2], lo[1]:hi[1], lo[0]:hi[0]]
        box.masked_fill_(d[2][:, None, None] + d[1][None, :, None] + d[0][None, None, :] <= 1, value)
    lo, hi = f.min(), f.max()
    return (f - lo) / (hi - lo)


def _place(case):
    """Where the case's surfaces run: a generator of its own for each case, the same for every seed."""
    return _gen(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))


def _values(f, levels, g, integer=False):
    """The field of the next time step or patient: every value moved by a random amount of at most 2 % of the range
    and never across an isolevel, so that the case keeps its surfaces' sizes."""
    span = 0.02 * float(f.max() - f.min())
    step = max(1, (1 << 27) // max(1, f[0].numel()))
    for k in range(0, f.shape[0], step):
        v = f[k:k + step]
        d = torch.full_like(v, 2 * span)
        for l in levels:
            d = torch.minimum(d, (v - l).abs())
        w = v + d * (torch.rand(v.shape, device=DEV, generator=g) - 0.5)
        w = torch.round(w) if integer else w
        for l in levels:
            w = torch.where((w > l) == (v > l), w, v)
        f[k:k + step] = w
    return f


def _volume(case, seed, levels=None):
    """(device tensor [z][y][x], isolevels): integer types span their range; `levels` in units of the field's own
    range, default the field's usual ones."""
    nx, ny, nz, field, dtype = case["nx"], case["ny"], case["nz"], case["field"], case["dtype"]
    f = {"blobs": _blobs, "ct": _ct, "turbulence": _turbulence}[field](nx, ny, nz, _place(case))
    if levels is None:
        levels = {"blobs": (0.5, 0.35, 0.65, 0.25, 0.75), "ct": (0.4, 0.55, 0.7, 0.3, 0.8),
                  "turbulence": (0.0, -0.3, 0.3, 0.15, -0.15)}[field][:case.get("levels", 1)]
    offset, scale = 0.0, 1.0
    if dtype in ("u8", "i16", "u16"):
        lo, hi = {"blobs": (-0.02, 2.0), "ct": (0.0, 1.0), "turbulence": (-1.0, 1.0)}[field]
        first, last = {"u8": (0, 255), "i16": (-1024, 3071), "u16": (0, 4095)}[dtype]
        scale = (last - first) / (hi - lo)
        offset = first - lo * scale
        f = torch.round((f.clamp_(lo, hi) - lo) * scale).add_(first)
    iso = [float(np.float32(offset + scale * l)) for l in levels]
    f = _values(f, iso, _gen(seed), integer=scale != 1.0)
    if scale != 1.0:
        f = f.clamp_(first, last)
        f = f.to(torch.uint8) if dtype == "u8" else f.to(torch.int32).to(TORCH[dtype])
    elif dtype == "f64":
        f = f.double()
    return f.contiguous(), iso


def _mesh(case, seed):
    """Nodes of a jittered grid cut into cells; values a blob field at the nodes."""
    nx, ny, nz, cell = case["nx"], case["ny"], case["nz"], case["cell"]
    g = _place(case)
    z, y, x = torch.meshgrid(*(torch.arange(n, device=DEV) for n in (nz, ny, nx)), indexing="ij")
    pos = torch.stack([x, y, z], -1).reshape(-1, 3).float()
    pos = pos + (torch.rand(pos.shape, device=DEV, generator=g) - 0.5) * 0.2
    n0 = ((z[:-1, :-1, :-1] * ny + y[:-1, :-1, :-1]) * nx + x[:-1, :-1, :-1]).reshape(-1)
    corner = torch.stack([n0 + (c * ny + b) * nx + a for a, b, c in
                          ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))], 1)
    parts = {"tet": [0, 1, 2, 6, 0, 2, 3, 6, 0, 3, 7, 6, 0, 7, 4, 6, 0, 4, 5, 6, 0, 5, 1, 6],
             "hex": [4, 5, 6, 7, 0, 1, 2, 3], "prism": [0, 1, 2, 4, 5, 6, 0, 2, 3, 4, 6, 7]}[cell]
    conn = corner[:, parts].reshape(-1).to(torch.int32).contiguous()
    values = _values(_blobs(nx, ny, nz, g, count=4, noise=0.0), [0.5], _gen(seed))
    return values.reshape(-1).contiguous(), pos.contiguous(), conn


def _jobs(case):
    """The batch's shapes: (nx, ny, nz, blobs, levels), fixed by the case; levels add up to at most `surfaces`."""
    rng = np.random.RandomState(case["shape"] % (1 << 31))
    left, out = case["surfaces"], []
    for i in range(case["volumes"]):
        dims = tuple(int(v) for v in rng.randint(32, case["edge"] + 1, 3))
        most = min(4, left - (case["volumes"] - 1 - i))
        n = int(rng.randint(1, most + 1)) if i + 1 < case["volumes"] else most
        out.append(dims + (int(rng.randint(1, 17)), [float(np.float32(v)) for v in rng.uniform(0.2, 0.8, n)]))
        left -= n
    return out


def _residents(case):
    """The server's volumes and requests, fixed by the case."""
    rng = np.random.RandomState(case["shape"] % (1 << 31))
    vols = []
    for i in range(case["volumes"]):
        dtype = ("f32", "u16", "u8")[i % 3]
        e = int(rng.randint(2, case["edge"] // 32 + 1)) * 32
        vols.append({"nx": e, "ny": e, "nz": e, "dtype": dtype, "field": "turbulence" if dtype == "f32" else "ct"})
    reqs = [(int(rng.randint(0, len(vols))), float(rng.uniform(0.3, 0.7)), int(rng.randint(0, 2)), bool(rng.randint(0, 2)))
            for _ in range(case["requests"])]
    return vols, reqs


# ---------------------------------------------------------------------------
# state and calls
# ---------------------------------------------------------------------------

class _State:
    """What the program holds: its volume, plan or server, and the surfaces of its last call."""

    def __init__(self, kind):
        self.kind, self.lib, self.outs, self.close = kind, kmc.load(), [], None

    def release(self):
        for s in self.outs:
            self.lib.kmc_surface_release(ctypes.byref(s))
        self.outs = []

    def __del__(self):
        try:
            self.release()
            if self.close:
                self.close()
        except Exception:
            pass


class _View:
    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _device(ptr, n, typestr, dtype):
    if not n or not ptr:
        return torch.empty(0, dtype=dtype, device=DEV)
    return torch.as_tensor(_View(ctypes.cast(ptr, ctypes.c_void_p).value, n, typestr), device=DEV)


def _arrays(s):
    """A surface's arrays, where they lie."""
    nv, nc, nn, nl = int(s.n_vertices), int(s.n_connections), int(s.n_normals), int(s.n_colors)
    if s.memory == kmc.MEMORY_HOST:
        out = {"coords": np.ctypeslib.as_array(s.coords, (3 * nv,)) if nv else np.zeros(0, np.float32),
               "normals": np.ctypeslib.as_array(s.normals, (3 * nn,)) if nn else np.zeros(0, np.float32)}
        if nc:
            out["connections"] = np.ctypeslib.as_array(s.connections, (nc,)).view(np.int32)
        return out
    out = {"coords": _device(s.coords, 3 * nv, "<f4", torch.float32),
           "normals": _device(s.normals, 3 * nn, "<f4", torch.float32)}
    if nc:
        out["connections"] = _device(s.connections, nc, "<i4", torch.int32)
    if nl and s.colors:
        out["colors"] = _device(s.colors, 3 * nl, "|u1", torch.uint8)
    return out


def _struct(t, dtype, minmax=None):
    """kmc_volume over a device tensor."""
    nz, ny, nx = t.shape
    return kmc.make_volume(t.data_ptr(), dims=(nx, ny, nz), memory=kmc.MEMORY_DEVICE, dtype=NUMPY[dtype], min_max=minmax)


def _minmax(t, dtype):
    if dtype == "u16":
        t = t.view(torch.int16)   # 12-bit data: the same values
    return float(t.min()), float(t.max())


def _check(status):
    if status != kmc.OK:
        raise kmc.KmcError(status)


def prepare(case, seed):
    kind = case["kind"]
    st = _State(kind)
    if kind in ("extract", "noalloc", "slice"):
        t, iso = _volume(case, seed)
        mm = _minmax(t, case["dtype"]) if case.get("cached", True) else None
        if case.get("host"):
            st.volume = kmc.make_volume(t.cpu().numpy(), min_max=mm)
        else:
            st.tensor, st.volume = t, _struct(t, case["dtype"], mm)
        st.normal = kmc.VERTEX_NORMAL if case.get("normal") == "vertex" else kmc.POLYGON_NORMAL
        st.dup = int(case.get("dup", True))
        st.memory = kmc.MEMORY_HOST if case.get("host") else kmc.MEMORY_DEVICE
        if kind == "slice":
            st.plane = _plane(case)
            st.table = kmc.colormap_table(kmc.COLORMAP_DEFAULT)
        else:
            st.levels = (ctypes.c_double * len(iso))(*iso)
        if kind == "noalloc":
            nt = 2 * int(_triangles(case)) + 200000
            st.coords = torch.empty(9 * nt if st.dup else 3 * nt, device=DEV)
            st.normals = torch.empty(3 * nt, device=DEV)
            st.connections = torch.empty(3 * nt, dtype=torch.int32, device=DEV)
    elif kind in ("mesh", "meshslice"):
        st.values, st.coords, st.connections = _mesh(case, seed)
        v = kmc.UnstructuredVolume()
        v.values, v.coords, v.connections = (a.data_ptr() for a in (st.values, st.coords, st.connections))
        v.memory, v.type, v.veclen, v.cell_type = kmc.MEMORY_DEVICE, kmc.REAL32, 1, CELL[case["cell"]]
        v.n_nodes = st.values.numel()
        v.n_cells = st.connections.numel() // kmc.CELL_NODES[CELL[case["cell"]]]
        st.volume = v
        if kind == "meshslice":
            st.plane = _plane(case)
            st.table = kmc.colormap_table(kmc.COLORMAP_DEFAULT)
    elif kind == "batch":
        st.tensors, specs = [], []
        for i, (nx, ny, nz, nb, levels) in enumerate(_jobs(case)):
            t = _values(_blobs(nx, ny, nz, _gen(case["shape"] * 64 + i), count=nb), levels, _gen(seed * 64 + i))
            st.tensors.append(t)
            specs.append((_struct(t, "f32", _minmax(t, "f32")), levels, kmc.POLYGON_NORMAL, True))
        st.batch = kmc.Batch(specs)
        st.close = st.batch.close
    else:
        vols, reqs = _residents(case)
        st.server = kmc.Server(out_memory=kmc.MEMORY_DEVICE)
        st.close = st.server.close
        st.tensors, st.requests = [], [None] * len(reqs)
        for i, v in enumerate(vols):
            mine = [k for k, r in enumerate(reqs) if r[0] == i]
            unit = (lambda u: 2 * u - 1) if v["field"] == "turbulence" else (lambda u: u)
            t, iso = _volume(dict(v, place=case["shape"] * 64 + i), seed * 64 + i, [unit(reqs[k][1]) for k in mine])
            st.tensors.append(t)
            torch.cuda.synchronize()
            vid = st.server.register(_struct(t, v["dtype"], _minmax(t, v["dtype"])))
            for k, level in zip(mine, iso):
                st.requests[k] = (vid, level, reqs[k][2], reqs[k][3])
    return st


def _plane(case):
    """Through the centre, normal (1, 2, 3) / sqrt(14)."""
    n = [k / math.sqrt(14) for k in (1, 2, 3)]
    c = [(case[k] - 1) / 2 for k in ("nx", "ny", "nz")]
    return (ctypes.c_float * 4)(*n, -sum(a * b for a, b in zip(n, c)))


def run(st):
    lib, kind = st.lib, st.kind
    st.release()
    if kind == "extract":
        n = len(st.levels)
        outs = (kmc.Surface * n)()
        if n == 1:
            _check(lib.kmc_extract(ctypes.byref(st.volume), st.levels[0], st.normal, st.dup, st.memory, None, outs))
        else:
            _check(lib.kmc_extract_levels(ctypes.byref(st.volume), st.levels, n, st.normal, st.dup, st.memory, None, outs))
        st.outs = list(outs)
        return [_arrays(s) for s in outs]
    if kind == "noalloc":
        s = kmc.Surface()
        _check(lib.kmc_extract_noalloc(ctypes.byref(st.volume), st.levels[0], st.normal, st.dup, None,
                                       st.coords.data_ptr(), st.coords.numel(), st.connections.data_ptr(),
                                       st.connections.numel(), st.normals.data_ptr(), st.normals.numel(),
                                       ctypes.byref(s)))
        return {"coords": st.coords[:3 * s.n_vertices], "normals": st.normals[:3 * s.n_normals],
                "connections": st.connections[:s.n_connections]}
    if kind == "batch":
        st.batch.run()
        return [_arrays(s) for s in st.batch.surfaces()]
    if kind == "serve":
        rids = [st.server.submit(*r) for r in st.requests]
        out = []
        for r in rids:
            s = kmc.Surface()
            _check(lib.kmc_server_wait(st.server.handle, r, -1, ctypes.byref(s)))
            st.outs.append(s)
            out.append(_arrays(s))
        return out
    s = kmc.Surface()
    if kind == "mesh":
        _check(lib.kmc_extract_unstructured(ctypes.byref(st.volume), 0.5, kmc.POLYGON_NORMAL, 1, kmc.MEMORY_DEVICE,
                                            None, ctypes.byref(s)))
    else:
        call = lib.kmc_slice_plane if kind == "slice" else lib.kmc_slice_plane_unstructured
        _check(call(ctypes.byref(st.volume), st.plane, st.table.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)),
                    st.table.size // 3, None, kmc.MEMORY_DEVICE, None, ctypes.byref(s)))
    st.outs = [s]
    return _arrays(s)


# ---------------------------------------------------------------------------
# work and 64-bit values
# ---------------------------------------------------------------------------

def _triangles(case):
    """Expected triangles per level: the fields' surfaces scale with the box's faces, at most one per node (volumes
    near the CT noise's 32-cell lattice)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return min({"blobs": 2.2, "turbulence": 8.7, "ct": 77.0}[case["field"]] * (nx * ny + ny * nz + nx * nz) / 3,
               1.0 * nx * ny * nz)


def _surface_bytes(triangles, dup, vertex):
    return triangles * (48 if dup else 12 + 6 + (6 if vertex else 12))


def work(case):
    kind = case["kind"]
    if kind in ("extract", "noalloc"):
        nt = _triangles(case) * case.get("levels", 1)
        out = _surface_bytes(nt, case["dup"], case["normal"] == "vertex")
        return {"bytes": case["nx"] * case["ny"] * case["nz"] * SIZE[case["dtype"]] + out, "flops": 30.0 * nt}
    if kind == "slice":
        nt = 4.0 * (case["nx"] * case["ny"] + case["ny"] * case["nz"] + case["nx"] * case["nz"]) / 3
        return {"bytes": nt * (57 + SIZE[case["dtype"]]), "flops": 60.0 * nt}
    if kind in ("mesh", "meshslice"):
        cubes = (case["nx"] - 1) * (case["ny"] - 1) * (case["nz"] - 1)
        cells, nodes = CELLS_PER_CUBE[case["cell"]], kmc.CELL_NODES[CELL[case["cell"]]]
        faces = cubes ** (2 / 3)
        return {"bytes": cubes * (cells * nodes * 4 + 16) + 6 * faces * 48, "flops": 10.0 * cubes * cells}
    if kind == "batch":
        jobs = _jobs(case)
        vol = sum(4 * j[0] * j[1] * j[2] for j in jobs)
        nt = sum(len(j[4]) * 4.0 * (j[0] * j[1] + j[1] * j[2] + j[0] * j[2]) / 3 for j in jobs)
        return {"bytes": vol + 48 * nt, "flops": 30.0 * nt}
    vols, reqs = _residents(case)
    total = 0.0
    for v, _, normal, dup in reqs:
        nt = _triangles(vols[v])
        total += vols[v]["nx"] ** 3 * SIZE[vols[v]["dtype"]] / 4 + _surface_bytes(nt, dup and normal, not normal)
    return {"bytes": total, "flops": 0.0}


def _edge_points(t, iso, mn, mx):
    """Crossing points of grid edges in node scan order, x / y / z edge of each node, in 64 bits."""
    nz, ny, nx = t.shape
    out = []
    slab = max(1, (1 << 26) // (nx * ny))
    for z0 in range(0, nz, slab):
        z1 = min(nz, z0 + slab)
        v = t[z0:min(nz, z1 + 1)].double()
        up = v > iso
        c = torch.zeros(z1 - z0, ny, nx, 3, dtype=torch.bool, device=t.device)
        m = z1 - z0
        c[:, :, :-1, 0] = up[:m, :, :-1] != up[:m, :, 1:]
        c[:, :-1, :, 1] = up[:m, :-1] != up[:m, 1:]
        k = v.shape[0] - 1
        c[:k, :, :, 2] = up[:k] != up[1:k + 1]
        z, y, x, axis = torch.nonzero(c, as_tuple=True)
        a = v[z, y, x].clamp(mn, mx)
        b = v[z + (axis == 2), y + (axis == 1), x + (axis == 0)].clamp(mn, mx)
        r = ((iso - a) / (b - a)).abs()
        p = torch.stack([x, y, z + z0], 1).double()
        q = p + torch.nn.functional.one_hot(axis, 3).double()
        out.append(((1 - r[:, None]) * p + r[:, None] * q).reshape(-1).cpu())
        del v, up, c
    return torch.cat(out).numpy()


def exact(case, seed):
    """Shared vertices are crossing points of grid edges, which need no case table; the other arrays follow from them
    by the table and have no value here."""
    if case["kind"] not in ("extract", "noalloc") or case["dup"]:
        return None
    t, levels = _volume(case, seed)
    if case["dtype"] == "u16":
        t = t.view(torch.int16)
    mn, mx = float(t.min()), float(t.max())
    pts = [{"coords": _edge_points(t, iso, mn, mx), "normals": None, "connections": None} for iso in levels]
    return pts[0] if case["kind"] == "noalloc" else pts
