"""Batches with more tiles than one launch has room for at a block of 256
threads each: tiny volumes, all of one field, so that every volume's outputs are
the first one's."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 23) + 3, (1 << 24) + 3])
def test_more_tiles_than_a_launch(n):
    print(f"[case] batch of {n} volumes", flush=True)
    b = mc.Batch(np.full((n, 3), 2, np.int64), np.full(n, 0.5, np.float32))
    one = torch.tensor([1.0, 0.2, 0.1, 0.3, 0.25, 0.0, 0.05, 0.15], device="cuda")
    flat = one.repeat(n)
    bufs = b.alloc(3 * n, n, normals=False)
    b.forward_into(flat, bufs, normals=False)
    assert mc.read_counts(b.counts) == (n, 3 * n)
    first = mc.forward(one.view(2, 2, 2), 0.5, edges=True)
    assert first.num_triangles == 1 and first.num_points == 3
    assert bool((bufs["vertices"].view(n, 9) == first.vertices.view(1, 9)).all())
    assert bool((bufs["conn"] == first.connectivity).all())
    assert bool((bufs["edges"].view(n, 3) == first.edges).all())
    i = torch.arange(n, device="cuda")
    assert torch.equal(b.vol_offsets[:, 0], i) and torch.equal(b.vol_offsets[:, 1], 3 * i)
    g = torch.Generator().manual_seed(5)
    dx, dn = (torch.randn((3, 3), generator=g).cuda() for _ in range(2))
    scratch = torch.empty(b.scratch_bytes(3 * n), dtype=torch.uint8, device="cuda")
    got = torch.empty_like(flat)
    args = (flat, bufs, dx.repeat(n, 1), dn.repeat(n, 1), scratch, got)
    if n >= 1 << 24:
        with pytest.raises(RuntimeError, match="2\\^24"):
            b.backward(*args)
        return
    b.backward(*args)
    want = mc.backward(one.view(2, 2, 2), 0.5, first, dx, dn)
    assert bool((got.view(n, 8) == want.view(1, 8)).all())
