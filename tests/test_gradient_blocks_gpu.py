"""Point and cell gradients at the edges of their blocks of 256 (below, at and
above one and several; planes that fill their blocks and planes that do not),
with outputs on and off 16-byte boundaries, and the cells' cases, counts and
offsets (words with and without mixed cells), bit for bit against the oracle.
Grids of many small planes in the time of a cube of as many points, and with
more planes than a launch has room for at a block each."""
import ctypes

import numpy as np
import pytest
import torch

from daxtoolkit_amd import _lib, mc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 2, 2), (255, 1, 1), (257, 2, 2), (16, 16, 1),
                                  (17, 17, 17), (65, 5, 33), (64, 64, 9), (129, 3, 7), (1, 1, 700),
                                  (1, 5, 300), (7, 1, 90), (3, 4, 200), (13, 14, 30), (12, 16, 40),
                                  (14, 14, 21), (20, 15, 9), (33, 17, 5)])
def test_gradients(dims, offset):
    print(f"[case] gradients {dims} offset {offset}", flush=True)
    nx, ny, nz = dims
    f = np.random.default_rng(sum(dims)).standard_normal((nz, ny, nx)).astype(np.float32)
    field = torch.from_numpy(f).cuda()
    sp, org = (0.7, 1.5, 2.0), (1.0, -2.0, 3.0)
    C = (nx - 1) * (ny - 1) * (nz - 1)
    args = (ctypes.c_float * 3)(*sp)
    o3 = (ctypes.c_float * 3)(*org)
    stream = torch.cuda.current_stream().cuda_stream
    for n, ref, call in (
            (f.size, orc.point_gradient(f, spacing=sp),
             lambda o: _lib.call("dax_hip_point_gradient", field.data_ptr(), nx, ny, nz, args, o,
                                 stream)),
            (C, orc.cell_gradient(f, origin=org, spacing=sp) if C else None,
             lambda o: _lib.call("dax_hip_cell_gradient", field.data_ptr(), nx, ny, nz, o3, args,
                                 o, stream))):
        if n == 0:
            continue
        buf = torch.full((3 * n + offset + 4,), 7.0, device="cuda")
        call(buf[offset:].data_ptr())
        got = buf.cpu().numpy()
        assert np.array_equal(got[offset:offset + 3 * n].view(np.uint32),
                              np.asarray(ref, np.float32).reshape(-1).view(np.uint32))
        assert np.all(got[:offset] == 7.0) and np.all(got[offset + 3 * n:] == 7.0)


def _best_of(fn, n=5):
    start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    fn()
    best = float("inf")
    for _ in range(n):
        start.record()
        fn()
        stop.record()
        stop.synchronize()
        best = min(best, start.elapsed_time(stop))
    return best


@pytest.mark.parametrize("gradient", [mc.point_gradient, mc.cell_gradient])
@pytest.mark.parametrize("dims", [(2, 2, 4_000_000), (4, 4, 1_000_000), (8, 8, 250_000)])
def test_small_planes_take_no_longer(dims, gradient):
    """Lanes left idle by planes of a few points took 10 to 100 times as long."""
    print(f"[case] gradients of small planes {dims}", flush=True)
    nx, ny, nz = dims
    cube = torch.rand((252, 252, 252), device="cuda")
    thin = torch.rand((nz, ny, nx), device="cuda")
    assert thin.numel() <= cube.numel()
    assert _best_of(lambda: gradient(thin)) < 3.0 * _best_of(lambda: gradient(cube))


def test_more_planes_than_blocks_of_a_launch():
    n = (1 << 27) + 9  # eight planes a block of 256 threads would pass 2^32 threads
    print(f"[case] gradients of {n} planes", flush=True)
    f = (torch.arange(n, device="cuda", dtype=torch.int32) % 8191).float().view(n, 1, 1)
    g = mc.point_gradient(f)
    v = f.view(-1)
    assert torch.equal(g[1:-1, 2], (v[2:] - v[:-2]) * 0.5)
    assert float(g[0, 2]) == float(v[1] - v[0]) and float(g[-1, 2]) == float(v[-1] - v[-2])
    assert not bool(g[:, :2].any())
    del g, v, f
    m = (1 << 27) + 5
    f = (torch.arange(4 * m, device="cuda", dtype=torch.int32) % 8191).float().view(m, 2, 2)
    g = mc.cell_gradient(f)
    assert g.shape == (m - 1, 3)
    # exact in float32: sums of four whole numbers below 2^13, times a quarter; the
    # voxel's width is the difference of its float32 coordinates (0 or 2 from 2^24 on)
    q = f.view(m, 4)
    z = torch.arange(m, device="cuda", dtype=torch.int32).float()
    want = (q[1:].sum(1) - q[:-1].sum(1)) * 0.25 / (z[1:] - z[:-1])
    assert torch.equal(g[:, 2].nan_to_num(nan=-7.0, posinf=7e9, neginf=-7e9),
                       want.nan_to_num(nan=-7.0, posinf=7e9, neginf=-7e9))


@pytest.mark.parametrize("noise", [0.0, 0.2, 0.6, 1.0])
@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 70, 9), (66, 9, 7), (200, 12, 5), (600, 9, 9)])
def test_cell_outputs_quiet_and_mixed_words(dims, noise):
    """Groups of words of which few, some or all are mixed (noise: in how many
    of the rows)."""
    nx, ny, nz = dims
    f = np.zeros((nz, ny, nx), np.float32)
    f[:, :, nx // 2:] = 1.0          # whole words in and out
    f[nz // 2, ny // 2, 0] = 1.0     # and mixed ones
    rng = np.random.default_rng(nx)
    f = np.where(rng.random((nz, ny, 1)) < noise, rng.random(f.shape), f).astype(np.float32)
    field = torch.from_numpy(f).cuda()
    ws, _ = mc.classify(field, 0.5)
    C = (nx - 1) * (ny - 1) * (nz - 1)
    cases = torch.empty(C, dtype=torch.uint8, device="cuda")
    count = torch.empty(C, dtype=torch.int32, device="cuda")
    offs = torch.empty(C, dtype=torch.int32, device="cuda")
    _lib.call("dax_hip_mc_cell_outputs", nx, ny, nz, ws.data_ptr(), ws.numel(), cases.data_ptr(),
              count.data_ptr(), offs.data_ptr(), torch.cuda.current_stream().cuda_stream)
    m = (f > 0.5).astype(np.int64)
    c = np.zeros((nz - 1, ny - 1, nx - 1), np.int64)
    for v, (dx, dy, dz) in enumerate([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1),
                                      (1, 0, 1), (1, 1, 1), (0, 1, 1)]):
        c |= m[dz:nz - 1 + dz, dy:ny - 1 + dy, dx:nx - 1 + dx] << v
    assert np.array_equal(cases.cpu().numpy(), c.reshape(-1).astype(np.uint8))
    n = count.cpu().numpy()
    mixed = (c.reshape(-1) != 0) & (c.reshape(-1) != 255)
    assert np.array_equal(n > 0, mixed)
    assert np.array_equal(offs.cpu().numpy(), np.cumsum(n) - n)
