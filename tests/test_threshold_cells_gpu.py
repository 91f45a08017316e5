"""Threshold of unstructured grids by words of 64 cells and 64 points: sizes
at the edges of words and of tiles of 256 words, cells of every vertex count,
off 16-byte boundaries, counts given and found, against the oracle (and, for
counts above 1, the path that takes any counts)."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import _lib, topology
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _grid(C, P, V, seed, offset):
    rng = np.random.default_rng(seed)
    cells = rng.integers(0, P, (C, V)).astype(np.int32)
    pts = rng.random((P, 3)).astype(np.float32)
    f = rng.random(P).astype(np.float32)
    buf = torch.zeros(C * V + offset, dtype=torch.int32, device="cuda")
    cd = buf[offset:].view(C, V)
    cd.copy_(torch.from_numpy(cells))
    return cells, pts, f, cd, torch.from_numpy(pts).cuda(), torch.from_numpy(f).cuda()


def _check(out, ref, dedup):
    assert out.num_cells == ref["n_cells"]
    assert np.array_equal(out.counts.cpu().numpy(), ref["counts"])
    assert np.array_equal(out.connectivity.cpu().numpy(), ref["conn"])
    if dedup:
        assert out.num_points == ref["n_points"]
        assert np.array_equal(out.points.cpu().numpy(), ref["coords"])


@pytest.mark.parametrize("dedup", [True, False])
@pytest.mark.parametrize("V,offset", [(1, 0), (3, 0), (4, 0), (4, 1), (5, 0), (8, 0), (8, 2)])
@pytest.mark.parametrize("C,P", [(1, 1), (63, 64), (64, 65), (65, 1000), (16384, 16385),
                                 (16385, 300), (40000, 70000)])
def test_against_oracle(C, P, V, offset, dedup):
    print(f"[case] threshold cells C={C} P={P} V={V} offset={offset} dedup={dedup}", flush=True)
    cells, pts, f, cd, pd, fd = _grid(C, P, V, C + P + V, offset)
    lo, hi = 0.05, 0.9
    ref = orc.threshold(f, lo, hi, dedup=dedup, cells=cells, points=pts)
    out = topology.threshold(fd, lo, hi, cells=cd, points=pd, dedup=dedup)
    _check(out, ref, dedup)
    counts = topology.threshold_count(fd, lo, hi, cd)
    again = topology.generate_topology(counts, cells=cd, points=pd, dedup=dedup)
    _check(again, ref, dedup)
    if dedup:
        used = np.zeros(P, np.int32)
        used[cells[ref["counts"].astype(bool)].reshape(-1)] = 1
        for o in (out, again):
            assert np.array_equal(o.point_mask.cpu().numpy(), used)
            assert np.array_equal(o.compact_point_field(fd).cpu().numpy(), ref["field"])
    twice = topology.generate_topology(2 * counts, cells=cd, points=pd, dedup=dedup)
    assert np.array_equal(twice.connectivity.cpu().numpy(), np.repeat(ref["conn"], 2, axis=0))


@pytest.mark.parametrize("bad", [-1, 100, 2**31 - 1])
@pytest.mark.parametrize("V", [3, 4, 8])
def test_ids_out_of_range(V, bad):
    cells, pts, f, cd, pd, fd = _grid(200, 100, V, 1, 0)
    cd[150, V - 1] = bad
    with pytest.raises(_lib.ErrorControlBadValue, match="outside"):
        topology.threshold(fd, 2.0, 3.0, cells=cd, points=pd)  # also of a cell that is not kept
    counts = torch.ones(200, dtype=torch.int32, device="cuda")
    with pytest.raises(_lib.ErrorControlBadValue, match="kept cell"):
        topology.generate_topology(counts, cells=cd, points=pd)
    counts[150] = 0
    assert topology.generate_topology(counts, cells=cd, points=pd).num_cells == 199


@pytest.mark.parametrize("C", [2**17, 2**18])
@pytest.mark.parametrize("where", [0, -1])
def test_totals_of_many_counts(C, where):
    """Counts beyond one turn of the blocks that add them up: the sum is exact to
    the last cell, and a negative count is seen wherever it stands."""
    rng = np.random.default_rng(C)
    cells = torch.from_numpy(rng.integers(0, 99, (C, 8)).astype(np.int32)).cuda()
    points = torch.zeros((99, 3), device="cuda")
    counts = torch.full((C,), 2**28 // C, dtype=torch.int32, device="cuda")  # 2^31 ids
    with pytest.raises(_lib.ErrorControlBadValue):
        topology.generate_topology(counts, cells=cells, points=points)
    counts.zero_()
    counts[where] = -1
    counts[C // 2] = 2
    with pytest.raises(_lib.ErrorControlBadValue):
        topology.generate_topology(counts, cells=cells, points=points)
    counts[where] = 3
    out = topology.generate_topology(counts, cells=cells, points=points)
    kept = torch.repeat_interleave(torch.arange(C, device="cuda"), counts.long())
    used, ids = torch.unique(cells[kept], return_inverse=True)
    assert torch.equal(out.connectivity, ids.to(torch.int32))
    assert torch.equal(torch.nonzero(out.point_mask).reshape(-1), used.long())


def test_any_counts_take_no_longer_for_the_words():
    """Counts above 1 among 1.7 M cells, which are found while the cells' words
    are made: adding them up took as long as all the rest of the call."""
    cells, points = orc.voxel_hexes((121, 121, 121))
    cd, pd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (cells, points))
    counts = torch.zeros(len(cells), dtype=torch.int32, device="cuda")

    def best_of(above):
        counts[5::50] = above
        best = float("inf")
        start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        for _ in range(12):
            start.record()
            topology.generate_topology(counts, cells=cd, points=pd)
            stop.record()
            stop.synchronize()
            best = min(best, start.elapsed_time(stop))
        return best

    assert best_of(2) < 2.8 * best_of(1)
