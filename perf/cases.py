"""Performance cases of the isosurface, threshold and gradient paths.

A case is a plain dict; its "kind" names one way a program uses the package:

  contour    mc.forward: size, allocate and fill one isosurface (optionally
             with its interpolation records and a point field carried along)
  steady     mc.forward_into: the forward of a loop that keeps its buffers
  step       mc.forward_into + mc.backward_into: a differentiable step
  batch      mc.Batch forward + backward over many volumes of uneven size
  slice      mc.slice: a plane through a uniform grid
  tets       mc.tetrahedra on an unstructured grid
  hexes      mc.hexahedra on an unstructured grid
  threshold  topology.threshold on a uniform grid, then compact_point_field
  cells      topology.threshold on an unstructured hexahedral grid
  fields     cell_gradient, point_gradient and the per-cell classification

Fields are the benchmark's: Gaussian mixtures with noise, a Mandelbulb for the
dense surface, distances for the tetrahedra and the threshold.  exact() gives
a pass's floating outputs in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from daxtoolkit_amd import _lib, fields, mc, topology

DEV = "cuda"


# ---------------------------------------------------------------------------
# cases

def listed():
    return [
        # one small ragged volume, as an interactive tool extracts it: launches and read-backs
        {"name": "contour_small", "kind": "contour", "nx": 37, "ny": 29, "nz": 33, "interp": False,
         "h": 1.0},
        # an ordinary scan with odd extents and its own spacing; a second point field is carried
        # onto the surface
        {"name": "contour_ragged", "kind": "contour", "nx": 301, "ny": 257, "nz": 190,
         "interp": True, "h": 0.7},
        # the headline forward: 512^3 in a loop with kept buffers
        {"name": "steady_512", "kind": "steady", "nx": 512, "ny": 512, "nz": 512,
         "field": "mixture"},
        # the differentiable workload: forward and adjoint at 256^3
        {"name": "step_256", "kind": "step", "nx": 256, "ny": 256, "nz": 256, "field": "mixture"},
        # a dense, folded surface (Mandelbulb), forward and adjoint
        {"name": "step_bulb_640", "kind": "step", "nx": 640, "ny": 640, "nz": 640,
         "field": "bulb"},
        # many independent volumes (extents 32..160), forward and adjoint in one call each
        {"name": "batch_256", "kind": "batch", "volumes": 256, "lo": 32, "hi": 160},
        # a tilted plane through the benchmark grid
        {"name": "slice_512", "kind": "slice", "nx": 512, "ny": 512, "nz": 512, "h": 1.0},
        # the tetrahedral grid of the benchmark (12.3 M tetrahedra)
        {"name": "tets_128", "kind": "tets", "nx": 128, "ny": 128, "nz": 128},
        # the hexahedral grid of the benchmark (16.6 M hexahedra)
        {"name": "hexes_256", "kind": "hexes", "nx": 256, "ny": 256, "nz": 256},
        # the reference's threshold benchmark, the mask kept (the default)
        {"name": "threshold_512", "kind": "threshold", "nx": 512, "ny": 512, "nz": 512},
        # the same pipeline on an unstructured grid
        {"name": "cells_160", "kind": "cells", "nx": 160, "ny": 160, "nz": 160},
        # dense per-point and per-cell outputs of an odd-sized grid
        {"name": "fields_ragged", "kind": "fields", "nx": 253, "ny": 241, "nz": 230},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, lo, hi, most):
    """Three extents spread over the logarithm of [lo, hi], at most `most` points."""
    d = [_log_int(rng, lo, hi) for _ in range(3)]
    if rng.random() < 0.3:  # rows of whole 64-point words are common
        d[0] = max(64, min(hi, (d[0] + 32) // 64 * 64))
    while d[0] * d[1] * d[2] > most:
        a = d.index(max(d[1:]), 1)
        d[a] = max(lo, d[a] * 3 // 4)
    return {"nx": d[0], "ny": d[1], "nz": d[2]}


def draw(rng):
    kind = rng.choice(["contour", "steady", "step", "batch", "slice", "tets", "hexes", "threshold",
                       "cells", "fields"])
    if kind == "contour":
        return {"kind": kind, **_extents(rng, 12, 512, 1 << 26), "interp": rng.random() < 0.5,
                "h": rng.choice([1.0, 0.5, 0.7])}
    if kind in ("steady", "step"):
        return {"kind": kind, **_extents(rng, 24, 640, 1 << 27),
                "field": "mixture"}
    if kind == "batch":
        lo = _log_int(rng, 12, 64)
        return {"kind": kind, "volumes": _log_int(rng, 4, 256), "lo": lo,
                "hi": rng.randint(lo + 4, max(lo + 8, min(160, 4 * lo)))}
    if kind == "slice":
        return {"kind": kind, **_extents(rng, 24, 640, 1 << 27), "h": rng.choice([1.0, 0.5, 2.0])}
    if kind == "tets":
        return {"kind": kind, **_extents(rng, 12, 160, 1 << 21)}
    if kind == "hexes":
        return {"kind": kind, **_extents(rng, 16, 288, 1 << 24)}
    if kind == "threshold":
        return {"kind": kind, **_extents(rng, 24, 640, 1 << 27)}
    if kind == "cells":
        return {"kind": kind, **_extents(rng, 16, 192, 1 << 22)}
    return {"kind": kind, **_extents(rng, 16, 384, 1 << 24)}


# ---------------------------------------------------------------------------
# inputs

def _dims(case):
    return case["nx"], case["ny"], case["nz"]


# A case's output sizes are its own: a seed mirrors the field along its axes and stretches it about
# the isovalue (by 1 to 2, so no point changes sides), or moves a distance's centre by whole points.

def _case_seed(case):
    return case["nx"] + 641 * (case["ny"] + 641 * case["nz"])


def _vary(f, iso, rng):
    axes = [d for d in range(3) if rng.random() < 0.5]
    f = f.flip(axes) if axes else f
    return (f - iso).mul_(float(rng.uniform(1.0, 2.0))).add_(iso).contiguous()


def _field(case, seed):
    """The benchmark's Gaussian mixture (widths shrink with volumes too small for them), or the
    Mandelbulb."""
    d = _dims(case)
    if case.get("field") == "bulb":
        # with the mixtures' noise: without it the steps of the field have normals of length zero
        f = fields.mandelbulb_torch(d[0], device=DEV)
        g = torch.Generator(device=DEV)
        g.manual_seed(_case_seed(case))
        f += (torch.rand(f.shape, device=DEV, generator=g) - 0.5) * 0.02
    else:
        m = min(d)
        p = fields.gaussian_mixture_params(_case_seed(case), d,
                                           sigma=(min(20.0, 0.08 * m), min(60.0, 0.23 * m)))
        f = fields.gaussian_mixture_torch(d, p, DEV)
    return _vary(f, _iso(case), np.random.default_rng(seed))


def _distance(case, seed):
    """|p - c| from a point near the middle."""
    d = _dims(case)
    r = np.random.default_rng(seed)
    ax = []
    for n in d:
        s = max(min(d) // 12, 1)
        c = n // 2 + int(r.integers(-s, s + 1))
        ax.append((torch.arange(n, dtype=torch.float64, device=DEV) - c) + 0.3)
    nx, ny, nz = d
    out = torch.empty((nz, ny, nx), dtype=torch.float32, device=DEV)
    yx = ax[1][:, None] ** 2 + ax[0][None, :] ** 2
    for z0 in range(0, nz, 64):
        z = ax[2][z0:z0 + 64]
        out[z0:z0 + 64] = torch.sqrt(z[:, None, None] ** 2 + yx[None])
    return out


def _normal_like(n, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn((n, 3), dtype=torch.float32, device=DEV, generator=g)


def _plane(case, seed):
    """A tilted plane across the whole grid: slopes of whole 1/1024ths, which a seed mirrors, at a
    height that it moves by whole points."""
    nx, ny, nz = _dims(case)
    r = np.random.default_rng(seed)
    n = [float(r.choice([-1, 1]) * max(1, 200 * nz // m)) / 1024.0 for m in (nx, ny)] + [1.0]
    up = int(r.integers(-(nz // 5), nz // 5 + 1))
    # the surface of the reference's slice is dot(n, p) = 2 dot(n, o)
    c = [0.5 * (nx - 1), 0.5 * (ny - 1), 0.5 * (nz - 1) + up]
    return [0.5 * case["h"] * v for v in c], n


def _batch_inputs(case, seed):
    m = case["hi"]
    b = fields.volume_batch(case["volumes"], lo=case["lo"], hi=m,
                            seed=case["volumes"] + 257 * (case["lo"] + 161 * m),
                            sigma=(min(20.0, 0.15 * m), min(60.0, 0.4 * m)))
    flat, off = fields.volume_batch_torch(b, DEV), 0
    r = np.random.default_rng(seed)
    for d, iso in zip(b.dims, b.isos):
        v = flat[off:off + d[0] * d[1] * d[2]]
        v.copy_(_vary(v.reshape(d[2], d[1], d[0]), iso, r).reshape(-1))
        off += len(v)
    return b, flat


def _iso(case):
    if case["kind"] == "tets":
        return float(np.float32(0.3 * min(_dims(case))))
    # between two steps of the Mandelbulb
    return float(np.float32(0.45)) if case.get("field") == "bulb" else 0.5


def _range(case):
    if case["kind"] == "cells":
        return 0.0, float(np.float32(0.25 * min(_dims(case))))
    return 0.0, float(np.float32(0.2 * min(_dims(case))))


def _scratch(points):
    n = int(_lib.load().dax_hip_mc_backward_scratch_bytes(points))
    return torch.empty(n, dtype=torch.uint8, device=DEV)


def _clear(buffers):
    """A volume without a surface leaves its one-row buffers as they are: give them a value."""
    for t in buffers:
        if isinstance(t, torch.Tensor):
            t.zero_()


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "iso": _iso(case)}
    if kind == "batch":
        vb, flat = _batch_inputs(case, seed)
        b = mc.Batch(vb.dims, vb.isos)
        T, U = b.sizes(flat)
        bufs = b.alloc(U, T)
        _clear(bufs.values())
        st.update(batch=b, field=flat, bufs=bufs, dv=_normal_like(max(U, 1), seed + 1),
                  dn=_normal_like(max(U, 1), seed + 2),
                  scratch=_scratch(max(U, 1)), out=torch.empty_like(flat))
        return st
    dims = _dims(case)
    if kind == "slice":
        po, pn = _plane(case, seed)
        st.update(dims=dims, po=po, pn=pn, spacing=(case["h"],) * 3)
        return st
    if kind in ("threshold", "cells"):
        st["field"] = _distance(case, seed)
        st["lo"], st["hi"] = _range(case)
        if kind == "cells":
            st["cells"], st["points"] = fields.voxel_cells_torch(dims, "hexahedron", device=DEV)
            st["field"] = st["field"].reshape(-1)
        return st
    if kind in ("tets", "hexes"):
        f = _distance(case, seed) if kind == "tets" else _field(case, seed)
        shape = "tetrahedron" if kind == "tets" else "hexahedron"
        st["cells"], st["points"] = fields.voxel_cells_torch(dims, shape, device=DEV)
        st["field"] = f.reshape(-1)
        return st
    f = st["field"] = _field(case, seed)
    if kind == "contour":
        st.update(interp=case["interp"], spacing=(case["h"],) * 3)
        if case["interp"]:
            st["values"] = (f * 3.0 - 1.0).reshape(-1)
    elif kind in ("steady", "step"):
        _, cnt = mc.classify(f, st["iso"])
        T, U = mc.read_counts(cnt)
        st["buf"] = mc.ForwardBuffers(*dims, max(U, 1), max(T, 1), device=f.device,
                                      edges=kind == "step")
        _clear(vars(st["buf"]).values())
        if kind == "step":
            U = max(U, 1)
            st.update(dv=_normal_like(U, seed + 1), dn=_normal_like(U, seed + 2),
                      scratch=_scratch(U), out=torch.empty_like(f))
    return st


# ---------------------------------------------------------------------------
# one pass

def run(st):
    kind = st["kind"]
    if kind == "contour":
        c = mc.forward(st["field"], st["iso"], spacing=st["spacing"], interp=st["interp"])
        out = {"vertices": c.vertices, "normals": c.normals, "conn": c.connectivity}
        if st["interp"]:
            out.update(first=c.interp_first, second=c.interp_second, weight=c.interp_weight,
                       values=mc.interpolate_scalar(st["values"], c))
        return out
    if kind in ("steady", "step"):
        b = st["buf"]
        mc.forward_into(st["field"], st["iso"], b)
        out = {"vertices": b.vertices, "normals": b.normals, "conn": b.conn, "counts": b.counts}
        if kind == "step":
            mc.backward_into(st["field"], st["iso"], b, st["dv"], st["dn"], st["scratch"],
                             st["out"])
            out.update(edges=b.edges, grad=st["out"])
        return out
    if kind == "batch":
        b, bufs = st["batch"], st["bufs"]
        b.forward_into(st["field"], bufs)
        b.backward(st["field"], bufs, st["dv"], st["dn"], st["scratch"], st["out"])
        return {"vertices": bufs["vertices"], "normals": bufs["normals"], "conn": bufs["conn"],
                "edges": bufs["edges"], "counts": b.counts, "offsets": b.vol_offsets,
                "grad": st["out"]}
    if kind == "slice":
        c = mc.slice(st["dims"], st["po"], st["pn"], spacing=st["spacing"])
        return {"vertices": c.vertices, "conn": c.connectivity, "edges": c.edges}
    if kind in ("tets", "hexes"):
        fn = mc.tetrahedra if kind == "tets" else mc.hexahedra
        c = fn(st["cells"], st["field"], st["points"], st["iso"])
        return {"vertices": c.vertices, "conn": c.connectivity, "first": c.interp_first,
                "second": c.interp_second, "weight": c.interp_weight}
    if kind in ("threshold", "cells"):
        t = topology.threshold(st["field"], st["lo"], st["hi"], cells=st.get("cells"),
                               points=st.get("points"))
        v = t.compact_point_field(st["field"].reshape(-1))
        return {"counts": t.counts, "conn": t.connectivity, "points": t.points,
                "mask": t.point_mask, "values": v}
    f = st["field"]
    ws, cnt = mc.classify(f, st["iso"])
    cases, count, offs = mc.cell_outputs(f, ws)
    return {"cell_gradient": mc.cell_gradient(f), "point_gradient": mc.point_gradient(f),
            "cases": cases, "count": count, "offsets": offs, "totals": cnt}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _surface_points(case):
    """Surface points one expects of a case's inputs: the crossings of a surface of area a with
    the grid's edges are about 1.5 a."""
    d = _dims(case)
    m = min(d)
    if case["kind"] == "slice":
        return 1.5 * d[0] * d[1]
    if case["kind"] == "tets":  # seven edge directions, a sphere of radius 0.3 m
        return 5.0 * 4 * math.pi * (0.3 * m) ** 2 / 1.5
    if case.get("field") == "bulb":
        return 11.0 * m * m
    s = 0.5 * (min(20.0, 0.08 * m) + min(60.0, 0.23 * m))
    return min(16 * 1.5 * 4 * math.pi * (1.1 * s) ** 2, 1.8 * (d[0] * d[1] + d[1] * d[2] + d[0] * d[2]))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        mean = 0.5 * (case["lo"] + case["hi"])
        P, U = case["volumes"] * mean ** 3, case["volumes"] * 4.0 * mean * mean / 9.0
        return {"bytes": 4 * P * 2 + U * (24 + 4 + 24) + 24 * U, "flops": 0.0}
    nx, ny, nz = _dims(case)
    P, C = nx * ny * nz, (nx - 1) * (ny - 1) * (nz - 1)
    if kind == "fields":
        return {"bytes": 4 * P + 12 * P + 12 * C + 9 * C, "flops": 9.0 * P + 51.0 * C}
    if kind in ("threshold", "cells"):
        r = _range(case)[1]
        kept = 4.0 / 3.0 * math.pi * r ** 3
        ids = 32 * C if kind == "cells" else 0
        return {"bytes": 4 * P + ids + 4 * C + 4 * P + kept * (32 + 12 + 8), "flops": 0.0}
    U = _surface_points(case)
    T = 2 * U
    if kind == "tets":
        return {"bytes": 6 * C * 16 + 4 * P + U * 24 + T * 12, "flops": 0.0}
    if kind == "hexes":
        return {"bytes": C * 32 + 4 * P + U * 24 + T * 12, "flops": 0.0}
    if kind == "slice":
        return {"bytes": U * 16 + T * 12, "flops": 0.0}
    out = U * 24 + T * 12
    if kind == "contour" and case["interp"]:
        out += U * 16 + U * 12
    if kind == "step":
        return {"bytes": 4 * P + out + 4 * U + U * 24 + 4 * P, "flops": 0.0}
    return {"bytes": 4 * P + out, "flops": 0.0}


# ---------------------------------------------------------------------------
# the same results in 64 bits

def _active_edges(inside):
    """(lower point id, axis) of the sign-change edges, by point id, then axis."""
    nz, ny, nx = inside.shape
    act = torch.zeros((nz, ny, nx, 3), dtype=torch.bool, device=inside.device)
    act[:, :, :-1, 0] = inside[:, :, 1:] ^ inside[:, :, :-1]
    act[:, :-1, :, 1] = inside[:, 1:] ^ inside[:, :-1]
    act[:-1, :, :, 2] = inside[1:] ^ inside[:-1]
    e = act.reshape(-1).nonzero().reshape(-1)
    return e // 3, e % 3


class _Grid:
    """Points and stencils of a uniform grid in 64 bits."""

    def __init__(self, dims, spacing):
        self.n = dims
        self.h = [float(np.float32(v)) for v in spacing]
        self.step = (1, dims[0], dims[0] * dims[1])

    def ijk(self, p):
        nx, ny, _ = self.n
        return [p % nx, (p // nx) % ny, p // (nx * ny)]

    def stencil(self, p, d):
        """Flat ids of the two points of the difference along d and its divisor."""
        c = self.ijk(p)[d]
        lo, hi = (c > 0).long(), (c < self.n[d] - 1).long()
        return p - lo * self.step[d], p + hi * self.step[d], (lo + hi).clamp(min=1) * self.h[d]

    def gradient(self, f, p):
        cols = []
        for d in range(3):
            a, b, w = self.stencil(p, d)
            cols.append((f[b].double() - f[a].double()) / w)
        return torch.stack(cols, 1)


def _vertices(g, f, iso, A, axis):
    """Interpolation weight, coordinates, and normal data of the points on edges (A, axis)."""
    step = torch.tensor(g.step, device=A.device)
    B = A + step[axis]
    fa, fb = f[A].double(), f[B].double()
    t = (iso - fa) / (fb - fa)
    xyz = torch.stack([c.double() * h for c, h in zip(g.ijk(A), g.h)], 1)
    h = torch.tensor(g.h, dtype=torch.float64, device=A.device)
    xyz[torch.arange(len(A), device=A.device), axis] += t * h[axis]
    return B, fa, fb, t, xyz


def _contour64(f, iso, spacing):
    nz, ny, nx = f.shape
    g = _Grid((nx, ny, nz), spacing)
    A, axis = _active_edges(f > iso)
    flat = f.reshape(-1)
    B, fa, fb, t, xyz = _vertices(g, flat, iso, A, axis)
    ga, gb = g.gradient(flat, A), g.gradient(flat, B)
    m = ga + t[:, None] * (gb - ga)
    ln = m.norm(dim=1, keepdim=True)
    nrm = torch.where(ln > 0, m / ln.clamp(min=1e-300), torch.zeros_like(m))
    return g, A, B, axis, fa, fb, t, xyz, ga, gb, nrm, ln


def _adjoint64(f, iso, dv, dn):
    g, A, B, axis, fa, fb, t, xyz, ga, gb, nrm, ln = _contour64(f, iso, (1, 1, 1))
    n = len(A)
    dv, dn = dv[:n].double(), dn[:n].double()
    dm = torch.where(ln > 0, (dn - nrm * (nrm * dn).sum(1, keepdim=True)) / ln.clamp(min=1e-300),
                     torch.zeros_like(dn))
    h = torch.tensor(g.h, dtype=torch.float64, device=A.device)
    dt = dv[torch.arange(n, device=A.device), axis] * h[axis] + (dm * (gb - ga)).sum(1)
    out = torch.zeros(f.numel(), dtype=torch.float64, device=f.device)
    den = fb - fa
    out.index_add_(0, A, dt * (-(1 - t) / den))
    out.index_add_(0, B, dt * (-t / den))
    for p, w in ((A, 1 - t), (B, t)):
        for d in range(3):
            lo, hi, wd = g.stencil(p, d)
            v = w * dm[:, d] / wd
            out.index_add_(0, hi, v)
            out.index_add_(0, lo, -v)
    return out


_CELL_EDGES = {"tets": [(0, 1), (1, 2), (2, 0), (3, 0), (3, 1), (3, 2)],
               "hexes": [(0, 1), (1, 2), (3, 2), (0, 3), (4, 5), (5, 6), (7, 6), (4, 7), (0, 4),
                         (1, 5), (2, 6), (3, 7)]}


def _cells_contour64(case, seed):
    st = prepare(case, seed)
    f, pts, iso = st["field"], st["points"], st["iso"]
    ins, P = f > iso, f.numel()
    keys = []
    for a, b in _CELL_EDGES[case["kind"]]:
        ia, ib = st["cells"][:, a].long(), st["cells"][:, b].long()
        on = ins[ia] ^ ins[ib]
        ia, ib = ia[on], ib[on]
        keys.append(torch.minimum(ia, ib) * P + torch.maximum(ia, ib))
    k = torch.unique(torch.cat(keys))
    A, B = k // P, k % P
    fa, fb = f[A].double(), f[B].double()
    w = (iso - fa) / (fb - fa)
    pa, pb = pts[A].double(), pts[B].double()
    return {"vertices": pa + w[:, None] * (pb - pa), "conn": None, "first": None, "second": None,
            "weight": w}


def _slice64(case, seed):
    """The topology of the slice follows the float32 plane values; positions are the plane's."""
    po, pn = _plane(case, seed)
    f32 = np.float32
    h = f32(case["h"])
    iso = f32(f32(f32(pn[0]) * f32(po[0])) + f32(f32(pn[1]) * f32(po[1])))
    iso = f32(iso + f32(f32(pn[2]) * f32(po[2])))
    axes, axes64 = [], []
    for d, n in enumerate(_dims(case)):
        x = np.arange(n, dtype=f32)
        axes.append(torch.from_numpy(f32(pn[d]) * ((f32(0) + h * x) - f32(po[d]))).to(DEV))
        axes64.append(torch.from_numpy(pn[d] * (float(h) * np.arange(n) - po[d])).to(DEV))
    v = (axes[0][None, None, :] + axes[1][None, :, None]) + axes[2][:, None, None]
    A, axis = _active_edges(v > float(iso))
    g = _Grid(_dims(case), (case["h"],) * 3)
    step = torch.tensor(g.step, device=A.device)

    def at(p):
        i, j, k = g.ijk(p)
        return axes64[0][i] + axes64[1][j] + axes64[2][k]

    fa, fb = at(A), at(A + step[axis])
    t = (sum(a * b for a, b in zip(pn, po)) - fa) / (fb - fa)
    xyz = torch.stack([c.double() * s for c, s in zip(g.ijk(A), g.h)], 1)
    hh = torch.tensor(g.h, dtype=torch.float64, device=A.device)
    xyz[torch.arange(len(A), device=A.device), axis] += t * hh[axis]
    return {"vertices": xyz, "conn": None, "edges": None}


def _threshold64(case, seed):
    """Copies of inputs and whole numbers only; the used points' coordinates and values."""
    nx, ny, nz = _dims(case)
    f = _distance(case, seed)
    lo, hi = _range(case)
    ok = (f >= lo) & (f <= hi)
    c = ok[1:, 1:, 1:] & ok[1:, 1:, :-1] & ok[1:, :-1, 1:] & ok[1:, :-1, :-1]
    c &= ok[:-1, 1:, 1:] & ok[:-1, 1:, :-1] & ok[:-1, :-1, 1:] & ok[:-1, :-1, :-1]
    used = torch.zeros_like(ok)
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                used[dz:dz + nz - 1, dy:dy + ny - 1, dx:dx + nx - 1] |= c
    p = used.reshape(-1).nonzero().reshape(-1)
    xyz = torch.stack([p % nx, (p // nx) % ny, p // (nx * ny)], 1).double()
    return {"counts": None, "conn": None, "points": xyz, "mask": None,
            "values": f.reshape(-1)[p].double()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("tets", "hexes"):
        return _cells_contour64(case, seed)
    if kind == "slice":
        return _slice64(case, seed)
    if kind in ("threshold", "cells"):
        return _threshold64(case, seed)
    if kind == "batch":
        vb, flat = _batch_inputs(case, seed)
        xs, ns, grads, parts, off = [], [], [], [], 0
        for d, iso in zip(vb.dims, vb.isos):
            f = flat[off:off + d[0] * d[1] * d[2]].reshape(d[2], d[1], d[0])
            off += f.numel()
            r = _contour64(f, iso, (1, 1, 1))
            xs.append(r[7])
            ns.append(r[10])
            parts.append((f, iso, len(r[1])))
        U, u = sum(n for _, _, n in parts), 0
        dv, dn = _normal_like(max(U, 1), seed + 1), _normal_like(max(U, 1), seed + 2)
        for f, iso, n in parts:
            grads.append(_adjoint64(f, iso, dv[u:u + n], dn[u:u + n]))
            u += n
        return {"vertices": torch.cat(xs), "normals": torch.cat(ns), "conn": None, "edges": None,
                "counts": None, "offsets": None, "grad": torch.cat(grads)}
    f = _field(case, seed)
    if kind == "fields":
        g = _Grid(_dims(case), (1, 1, 1))
        pg = torch.cat([g.gradient(f.reshape(-1), p) for p in
                        torch.arange(f.numel(), device=f.device).split(1 << 24)])
        d = f.double()
        x = d[:, :, 1:] - d[:, :, :-1]
        y = d[:, 1:] - d[:, :-1]
        z = d[1:] - d[:-1]
        cg = torch.stack([
            (x[1:, 1:] + x[1:, :-1] + x[:-1, 1:] + x[:-1, :-1]).reshape(-1),
            (y[1:, :, 1:] + y[1:, :, :-1] + y[:-1, :, 1:] + y[:-1, :, :-1]).reshape(-1),
            (z[:, 1:, 1:] + z[:, 1:, :-1] + z[:, :-1, 1:] + z[:, :-1, :-1]).reshape(-1)], 1) / 4
        return {"cell_gradient": cg, "point_gradient": pg, "cases": None, "count": None,
                "offsets": None, "totals": None}
    iso = _iso(case)
    h = case.get("h", 1.0)
    r = _contour64(f, iso, (h,) * 3)
    A, B, t, xyz, nrm = r[1], r[2], r[6], r[7], r[10]
    out = {"vertices": xyz, "normals": nrm, "conn": None}
    if kind == "contour":
        if case["interp"]:
            v = (f * 3.0 - 1.0).reshape(-1)
            va, vb = v[A].double(), v[B].double()
            out.update(first=None, second=None, weight=t, values=va + t * (vb - va))
        return out
    out["counts"] = None
    if kind == "step":
        n = max(len(A), 1)
        del r
        out.update(edges=None,
                   grad=_adjoint64(f, iso, _normal_like(n, seed + 1),
                                   _normal_like(n, seed + 2)).reshape(f.shape))
    return out
