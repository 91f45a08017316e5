"""The bit-word threshold pipeline at the edges of its words, tiles of 256
words and 16-byte stores: counts, mask, connectivity, coordinates and
CompactPointField equal the oracle's, from a field and from given counts."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import topology
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

DIMS = [(2, 2, 2), (3, 3, 2), (4, 5, 3), (5, 2, 9), (9, 33, 5), (63, 7, 6), (64, 9, 5), (65, 9, 5),
        (66, 17, 16), (67, 16, 18), (128, 33, 9), (129, 2, 2), (200, 30, 24), (513, 5, 7)]


def _check(out, ref, mask=True):
    assert out.num_cells == ref["n_cells"] and out.num_points == ref["n_points"]
    assert np.array_equal(out.counts.cpu().numpy(), ref["counts"])
    assert np.array_equal(out.connectivity.cpu().numpy(), ref["conn"])
    assert np.array_equal(out.points.cpu().numpy(), ref["coords"])


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("hi,offset", [(0.97, 0), (0.999, 1), (2.0, 3), (0.3, 2)])
def test_against_oracle(dims, hi, offset):
    rng = np.random.default_rng(sum(dims))
    f = rng.random(dims[::-1]).astype(np.float32)
    buf = torch.zeros(f.size + offset, device="cuda")
    ft = buf[offset:].view(*f.shape)  # off a 16-byte boundary
    ft.copy_(torch.from_numpy(f))
    ref = orc.threshold(f, 0.0, hi, origin=(1, 2, 3), spacing=(0.5, 0.25, 2.0))
    out = topology.threshold(ft, 0.0, hi, origin=(1, 2, 3), spacing=(0.5, 0.25, 2.0))
    _check(out, ref)
    mask = np.zeros(f.size, np.int32)
    P = np.arange(f.size).reshape(f.shape)
    keep = ref["counts"].reshape([d - 1 for d in f.shape]).astype(bool)
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                mask[P[dz:dz + f.shape[0] - 1, dy:dy + f.shape[1] - 1,
                       dx:dx + f.shape[2] - 1][keep]] = 1
    assert np.array_equal(out.point_mask.cpu().numpy(), mask)
    v3 = torch.from_numpy(np.stack([f, 2 * f, 3 * f], -1).reshape(-1, 3)).cuda()
    got = out.compact_point_field(v3).cpu().numpy()
    assert np.array_equal(got, v3.cpu().numpy()[mask.astype(bool)])
    again = topology.generate_topology(out.counts, dims=dims, origin=(1, 2, 3),
                                       spacing=(0.5, 0.25, 2.0))
    _check(again, ref)
    assert torch.equal(again.point_mask, out.point_mask)
    plain = topology.threshold(ft, 0.0, hi, dedup=False)
    assert np.array_equal(plain.connectivity.cpu().numpy(),
                          orc.threshold(f, 0.0, hi, dedup=False)["conn"])


def test_counts_above_one_keep_the_general_layout():
    dims = (66, 9, 8)
    rng = np.random.default_rng(2)
    n = 65 * 8 * 7
    counts = torch.from_numpy(rng.integers(0, 2, n).astype(np.int32)).cuda()
    one = topology.generate_topology(counts, dims=dims)
    counts[n - 1] = 3
    many = topology.generate_topology(counts, dims=dims)
    kept = int((counts[:n - 1] != 0).sum())
    assert many.num_cells == kept + 3
    # the extra cell adds points: compare by coordinates
    a = one.points[one.connectivity[:kept].long()]
    b = many.points[many.connectivity[:kept].long()]
    assert torch.equal(a, b)
