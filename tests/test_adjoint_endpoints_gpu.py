"""GPU adjoint over row words: sizes at the edges of words, waves (8, 32 or 64
words) and tiles (256 words), from no surface to a point in two an endpoint, bit
for bit against the oracle's FP32 restatement; an edge list cut below the
surface's vertices against the whole list with zero gradients from there on
(equal values: the vertices left out add exact zeros)."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import mc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _field(dims, seed, noise):
    nx, ny, nz = dims
    r = np.random.default_rng(seed)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    smooth = np.sin(x / 7.3) * np.cos(y / 5.1 + 0.3) + np.sin(z / 4.7 + 0.2)
    return (smooth + noise * r.standard_normal((nz, ny, nx))).astype(np.float32)


def _grads(U, seed):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn((U, 3), generator=gen, dtype=torch.float32),
            torch.randn((U, 3), generator=gen, dtype=torch.float32))


@pytest.mark.parametrize("noise", [0.0, 2.0])
@pytest.mark.parametrize("dims", [(2, 2, 2), (1, 9, 9), (63, 3, 5), (64, 17, 17), (65, 16, 8),
                                  (128, 8, 16), (130, 21, 19), (1000, 5, 3), (4, 64, 65)])
def test_endpoints_and_gather(dims, noise):
    print(f"[case] adjoint words {dims} noise {noise}", flush=True)
    f = _field(dims, 5, noise)
    sp = (0.5, 1.0, 1.5)
    field = torch.from_numpy(f).cuda()
    out = mc.forward(field, 0.1, edges=True, spacing=sp)
    U = out.num_points
    dx, dn = _grads(U, 7)
    got = mc.backward(field, 0.1, out, dx.cuda(), dn.cuda(), spacing=sp).cpu().numpy().reshape(-1)
    r = orc.generate(f, 0.1, spacing=sp)
    assert r["n_pts"] == U
    want = (orc.backward_f32(f, 0.1, r["first"], r["second"], dx.numpy(), dn.numpy(), spacing=sp)
            if U else np.zeros(f.size, np.float32))
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("dims", [(2, 256, 256), (2, 257, 256), (3, 512, 512), (2, 513, 512),
                                  (2, 2048, 2047), (2, 2049, 2048), (64, 2053, 2052)])
def test_many_row_words(dims):
    """Row words around 2^16, 2^18 (1024 tiles) and 2^22, where the words per
    wave and the way to the tiles' prefixes change, and more tiles than one
    block scans."""
    print(f"[case] adjoint words {dims}", flush=True)
    f = np.zeros((dims[2], dims[1], dims[0]), np.float32)
    r = np.random.default_rng(11)
    for k in (0, dims[2] // 2, dims[2] - 3):  # noise in three slabs
        f[k:k + 3, :, :] = r.random((3, dims[1], dims[0]), dtype=np.float32)
    field = torch.from_numpy(f).cuda()
    out = mc.forward(field, 0.4, edges=True)
    U = out.num_points
    dx, dn = _grads(U, 7)
    got = mc.backward(field, 0.4, out, dx.cuda(), dn.cuda()).cpu().numpy().reshape(-1)
    r = orc.generate(f, 0.4)
    assert r["n_pts"] == U
    want = orc.backward_f32(f, 0.4, r["first"], r["second"], dx.numpy(), dn.numpy())
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("n", [1, 40, 1025, 3000])
def test_batch_of_small_volumes(n):
    """Volumes that leave their tiles mostly empty, up to more of them than
    blocks add up the tiles before themselves; against each on its own."""
    print(f"[case] adjoint of {n} small volumes", flush=True)
    dims = [(5 + i % 3, 4 + i % 5, 3 + i % 4) for i in range(n)]
    r = np.random.default_rng(n)
    fs = [r.random((d[2], d[1], d[0]), dtype=np.float32) for d in dims]
    flat = torch.from_numpy(np.concatenate([f.reshape(-1) for f in fs])).cuda()
    b = mc.Batch(dims, [0.4] * n)
    T, U = b.sizes(flat)
    bufs = b.alloc(U, T)
    b.forward_into(flat, bufs)
    dx, dn = _grads(U, 3)
    scratch = torch.empty(b.scratch_bytes(U), dtype=torch.uint8, device="cuda")
    got = torch.empty_like(flat)
    b.backward(flat, bufs, dx.cuda(), dn.cuda(), scratch, got)
    got, at, u = got.cpu().numpy(), 0, 0
    for f in fs:
        ref = orc.generate(f, 0.4)
        m = ref["n_pts"]
        want = (orc.backward_f32(f, 0.4, ref["first"], ref["second"], dx[u:u + m].numpy(),
                                 dn[u:u + m].numpy()) if m else np.zeros(f.size, np.float32))
        assert np.array_equal(got[at:at + f.size].view(np.uint32),
                              np.asarray(want, np.float32).view(np.uint32))
        at += f.size
        u += m
    assert u == U


@pytest.mark.parametrize("cut", [0, 1, 2, 7, 100, 1000, -1])
def test_cut_edge_list(cut):
    dims = (70, 13, 11)
    print(f"[case] adjoint cut {cut}", flush=True)
    f = _field(dims, 3, 1.0)
    field = torch.from_numpy(f).cuda()
    out = mc.forward(field, 0.1, edges=True)
    U = out.num_points
    n = cut if cut >= 0 else U - 1
    assert n < U
    dx, dn = _grads(U, 9)
    dx[n:] = 0.0
    dn[n:] = 0.0
    whole = mc.backward(field, 0.1, out, dx.cuda(), dn.cuda())
    cut_out = mc.Contour(**{**out.__dict__, "vertices": out.vertices[:n]})
    assert cut_out.num_points == n
    got = mc.backward(field, 0.1, cut_out, dx[:n].contiguous().cuda(),
                      dn[:n].contiguous().cuda())
    assert torch.equal(got, whole)


def _batch(n_volumes):
    dims = [(9, 3, 5), (70, 13, 11), (64, 5, 6), (130, 9, 4)][:n_volumes]  # odd word offsets
    fs = [_field(d, 3 + i, 1.0).reshape(-1) for i, d in enumerate(dims)]
    flat = torch.from_numpy(np.concatenate(fs)).cuda()
    b = mc.Batch(dims, [0.1] * len(dims))
    T, U = b.sizes(flat)
    bufs = b.alloc(U, T)
    b.forward_into(flat, bufs)
    return b, flat, bufs, U


@pytest.mark.parametrize("cut", [1, 40, 2000, -1])
def test_batch_cut_edge_list(cut):
    print(f"[case] batch adjoint cut {cut}", flush=True)
    b, flat, bufs, U = _batch(4)
    n = cut if cut >= 0 else U - 1
    assert 0 < n < U
    dx, dn = (t.cuda() for t in _grads(U, 9))
    dx[n:] = 0.0
    dn[n:] = 0.0
    scratch = torch.empty(b.scratch_bytes(U), dtype=torch.uint8, device="cuda")
    whole, got = torch.empty_like(flat), torch.empty_like(flat)
    b.backward(flat, bufs, dx, dn, scratch, whole)
    b.backward(flat, dict(bufs, cap_points=n), dx, dn, scratch, got)
    assert torch.equal(got, whole)


def test_calls_write_the_same_workspace():
    """What a backward leaves in the workspace does not depend on how many of
    the edges it takes, so that calls that share one may overlap."""
    print("[case] adjoint workspace of whole and cut lists", flush=True)
    field = torch.from_numpy(_field((70, 13, 11), 3, 1.0)).cuda()
    out = mc.forward(field, 0.1, edges=True)
    U = out.num_points
    dx, dn = (t.cuda() for t in _grads(U, 9))
    mc.backward(field, 0.1, out, dx, dn)
    before = out.workspace.clone()
    for n in (1, 100, U // 2, U - 1):
        cut = mc.Contour(**{**out.__dict__, "vertices": out.vertices[:n]})
        mc.backward(field, 0.1, cut, dx[:n].contiguous(), dn[:n].contiguous())
        assert torch.equal(out.workspace, before), n

    b, flat, bufs, U = _batch(4)
    dx, dn = (t.cuda() for t in _grads(U, 9))
    scratch = torch.empty(b.scratch_bytes(U), dtype=torch.uint8, device="cuda")
    g = torch.empty_like(flat)
    b.backward(flat, bufs, dx, dn, scratch, g)
    before = b.workspace.clone()
    for n in (1, 100, U // 2, U - 1):
        b.backward(flat, dict(bufs, cap_points=n), dx, dn, scratch, g)
        assert torch.equal(b.workspace, before), n
