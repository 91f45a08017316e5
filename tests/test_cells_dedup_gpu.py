"""Edges numbered by tiles of 64 lower endpoints: tiles that hold up to 512
distinct edges, tiles of more that go through their endpoints in parts, and the
sort taken for more edges up from one point or very many corners of a tile.  All
give the oracle's numbering.  Cells at the edges of the 1024-cell blocks, and
connectivity off a 16-byte boundary."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import mc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _fan(n):
    """n tetrahedra around point 0, which alone is inside: every cell edge from
    it is active."""
    ring = np.arange(n, dtype=np.int32)
    cells = np.stack([np.zeros(n, np.int32), 3 + ring, 3 + (ring + 1) % n, 1 + ring % 2], 1)
    rng = np.random.default_rng(n)
    pts = rng.random((n + 3, 3)).astype(np.float32)
    f = rng.random(n + 3).astype(np.float32) * 0.4
    f[0] = 1.0
    return cells, f, pts


@pytest.mark.parametrize("n", [3, 14, 15, 16, 40, 509, 510, 511, 700, 1021, 1022, 1023, 1500,
                               9000])
@pytest.mark.parametrize("offset", [0, 1])
def test_fan_matches_oracle(n, offset):
    cells, f, pts = _fan(n)
    buf = torch.zeros(cells.size + offset, dtype=torch.int32, device="cuda")
    ct = buf[offset:].view(n, 4)
    ct.copy_(torch.from_numpy(cells))
    for dedup in (True, False):
        c = mc.tetrahedra(ct, torch.from_numpy(f).cuda(), torch.from_numpy(pts).cuda(), 0.5, dedup)
        r = orc.mt_generate(cells, f, pts, 0.5, dedup=dedup)
        assert np.array_equal(c.connectivity.cpu().numpy().reshape(-1), r["conn"])
        assert np.array_equal(c.interp_first.cpu().numpy(), r["first"])
        assert np.array_equal(c.interp_second.cpu().numpy(), r["second"])
        assert np.array_equal(c.vertices.cpu().numpy(), r["coords"])


@pytest.mark.parametrize("fans,n", [(16, 29), (16, 30), (16, 31), (25, 38), (25, 39), (26, 38),
                                    (63, 40), (65, 40), (200, 100), (5, 700), (66, 300),
                                    (300, 60)])
def test_many_fans_match_oracle(fans, n):
    """Tiles of up to 64 points with n + 2 edges up from each: around 512 edges,
    in halves, quarters and fewer points, and beyond 16384 corners."""
    parts = [_fan(n) for _ in range(fans)]
    step = n + 3
    # the inside points first, so that they are neighbours
    cells = np.concatenate([np.where(c == 0, i, fans + i * (step - 1) + c - 1)
                            for i, (c, _, _) in enumerate(parts)]).astype(np.int32)
    rng = np.random.default_rng(fans * n)
    f = np.concatenate([np.full(fans, 1.0), rng.random(fans * (step - 1)) * 0.4]).astype(np.float32)
    pts = rng.random((len(f), 3)).astype(np.float32)
    cells = np.ascontiguousarray(cells[rng.permutation(len(cells))])
    ct, ft, pt = (torch.from_numpy(a).cuda() for a in (cells, f, pts))
    c = mc.tetrahedra(ct, ft, pt, 0.5)
    r = orc.mt_generate(cells, f, pts, 0.5, dedup=True)
    assert np.array_equal(c.connectivity.cpu().numpy().reshape(-1), r["conn"])
    assert np.array_equal(c.interp_first.cpu().numpy(), r["first"])
    assert np.array_equal(c.interp_second.cpu().numpy(), r["second"])
    assert np.array_equal(c.vertices.cpu().numpy(), r["coords"])


def test_sorted_edges_take_no_longer():
    """200 000 cells around one point: finding out that its edges have to be
    sorted took 20 times as long as the cells' own work."""
    def best_of(cells, f, pts, n=5):
        args = [torch.from_numpy(a).cuda() for a in (cells, f, pts)]
        start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        mc.tetrahedra(*args, 0.5)
        best = float("inf")
        for _ in range(n):
            start.record()
            mc.tetrahedra(*args, 0.5)
            stop.record()
            stop.synchronize()
            best = min(best, start.elapsed_time(stop))
        return best

    n = 200_000
    cells, f, pts = _fan(n)
    apart = np.arange(4 * n, dtype=np.int32).reshape(n, 4)
    fa = np.zeros((n, 4), np.float32)
    fa[:, 0] = 1.0
    rng = np.random.default_rng(1)
    other = best_of(apart, fa.reshape(-1), rng.random((4 * n, 3)).astype(np.float32))
    assert best_of(cells, f, pts) < 4.0 * other


@pytest.mark.parametrize("tets", [1, 63, 64, 65, 1023, 1024, 1025, 4097, 300_000])
def test_disjoint_tetrahedra(tets):
    """Every tetrahedron its own four points, three of them lower endpoints."""
    cells = torch.arange(4 * tets, dtype=torch.int32, device="cuda").view(tets, 4)
    g = torch.Generator(device="cuda")
    g.manual_seed(tets)
    pts = torch.rand((4 * tets, 3), device="cuda", generator=g)
    f = torch.zeros((tets, 4), device="cuda")
    f[:, 3] = 1.0  # the highest id inside: edges (0,3), (1,3), (2,3)
    f += torch.rand((tets, 4), device="cuda", generator=g) * 0.4
    f = f.reshape(-1)
    c = mc.tetrahedra(cells, f, pts, 0.5)
    assert c.num_triangles == tets and c.num_points == 3 * tets
    base = 4 * torch.arange(tets, device="cuda")
    first = (base[:, None] + torch.arange(3, device="cuda")).reshape(-1)
    second = (base[:, None] + 3).expand(tets, 3).reshape(-1)
    assert torch.equal(c.interp_first.long(), first) and torch.equal(c.interp_second.long(), second)
    w = (0.5 - f[first]) / (f[second] - f[first])
    assert torch.equal(c.interp_weight, w)
    conn = c.connectivity.long()
    assert torch.equal(torch.sort(conn, 1).values, torch.arange(3 * tets, device="cuda").view(-1, 3))


def test_shuffled_hexahedra_match_the_count_and_offset_entries():
    """The entries that take a count and an offset per cell give the same grid."""
    import ctypes

    from daxtoolkit_amd import _lib
    dims = (23, 19, 21)
    hexes, pts = orc.voxel_hexes(dims)
    rng = np.random.default_rng(4)
    perm = rng.permutation(len(pts)).astype(np.int32)
    hexes = perm[hexes][rng.permutation(len(hexes))]
    f = rng.random(len(pts)).astype(np.float32)
    inv = np.empty_like(pts)
    inv[perm] = pts
    ct, ft, pt = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (hexes, f, inv))
    c = mc.hexahedra(ct, ft, pt, 0.5)
    C, P = len(hexes), len(pts)
    counts, offs = (torch.empty(C, dtype=torch.int32, device="cuda") for _ in range(2))
    t, u = ctypes.c_int64(), ctypes.c_int64()
    s = torch.cuda.current_stream().cuda_stream
    _lib.call("dax_hip_mc_hex_count", ct.data_ptr(), C, ft.data_ptr(), P, 0.5, counts.data_ptr(),
              offs.data_ptr(), ctypes.byref(t), s)
    n = 3 * t.value
    scratch = torch.empty(int(_lib.load().dax_hip_mc_hex_scratch_bytes(t.value)),
                          dtype=torch.uint8, device="cuda")
    v = torch.empty((n, 3), device="cuda")
    conn, a, b = (torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(3))
    w = torch.empty(n, device="cuda")
    _lib.call("dax_hip_mc_hex_generate", ct.data_ptr(), C, ft.data_ptr(), pt.data_ptr(), P, 0.5, 1,
              counts.data_ptr(), offs.data_ptr(), t.value, scratch.data_ptr(), scratch.numel(),
              v.data_ptr(), conn.data_ptr(), a.data_ptr(), b.data_ptr(), w.data_ptr(),
              ctypes.byref(u), s)
    assert t.value == c.num_triangles and u.value == c.num_points
    assert torch.equal(conn.view(-1, 3), c.connectivity) and torch.equal(v[:u.value], c.vertices)
    assert torch.equal(a[:u.value], c.interp_first) and torch.equal(w[:u.value], c.interp_weight)
