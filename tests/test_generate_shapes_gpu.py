"""The generate kernel's launch shapes picked by size (64-word tiles shared by
four, two or one waves; 256-word tiles; tiles of at least two wide rows) give
the output of 512-word tiles bit for bit, and at a small size the oracle's."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import mc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _scattered(dims, seed, share):
    """Scattered inside points: `share` of them above the isovalue 0.5."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    f = torch.rand(tuple(reversed(dims)), device="cuda", generator=g)
    return (f - (1.0 - share) + 0.5).contiguous()


def _outputs(f, dedup):
    c = mc.forward(f, 0.5, spacing=(0.5, 1.0, 0.7), dedup=dedup, edges=dedup, interp=True)
    return [t for t in (c.vertices, c.normals, c.connectivity, c.edges, c.interp_first,
                        c.interp_second, c.interp_weight) if t is not None]


@pytest.mark.parametrize("dims,share", [
    ((33, 512, 512), 0.005),    # 2^18 words: four waves per tile
    ((33, 513, 512), 0.005),    # just above: two
    ((20, 1024, 1024), 0.003),  # 2^20 words: two
    ((20, 1025, 1024), 0.003),  # just above: 256-word tiles
    ((2112, 9, 8), 0.4),        # rows of 33 words: 128-word tiles
    ((4200, 4, 5), 0.4),        # rows of 66 words: 256-word tiles
    ((65, 40, 31), 0.5),        # dense: every cell active
])
@pytest.mark.parametrize("dedup", [True, False])
def test_rule_matches_512_word_tiles(dims, share, dedup):
    f = _scattered(dims, 7, share)
    got = _outputs(f, dedup)
    saved = mc.get_tuning(dims)
    try:
        mc.set_tuning(dims, [4, 4, 8, 512, 0])
        want = _outputs(f, dedup)
        if dims[1] * dims[2] > 1 << 20:  # one wave per 64-word tile
            mc.set_tuning(dims, [4, 4, 4, 64, 0])
            got64 = _outputs(f, dedup)
            assert all(torch.equal(a, b) for a, b in zip(got64, want))
    finally:
        mc.set_tuning(dims, saved)
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dims", [(2, 2, 2), (64, 3, 3), (65, 5, 4), (127, 6, 9), (130, 17, 12)])
def test_dense_small_volumes_match_oracle(dims):
    f = _scattered(dims, sum(dims), 0.5)
    c = mc.forward(f, 0.5, edges=True, interp=True)
    r = orc.generate(f.cpu().numpy(), 0.5, dedup=True)
    assert np.array_equal(c.connectivity.cpu().numpy().reshape(-1), r["conn"])
    assert np.array_equal(c.vertices.cpu().numpy(), r["coords"])
    assert np.array_equal(c.interp_first.cpu().numpy(), r["first"])
