"""Inside-bits of rows that are not whole 64-point words and of fields off a
16-byte boundary (the flat-stream classify), against numpy."""
import numpy as np
import pytest
import torch

from daxtoolkit_amd import mc

pytestmark = pytest.mark.gpu


def _bits(field, iso):
    nz, ny, nx = field.shape
    ws, _ = mc.classify(field, iso)
    wpr = (nx + 63) // 64
    return ws.cpu().numpy()[:wpr * ny * nz * 8].view(np.uint64).reshape(nz, ny, wpr)


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("dims", [(1, 3, 5), (2, 2, 2), (5, 7, 9), (31, 17, 70), (32, 33, 16),
                                  (33, 5, 40), (63, 64, 3), (64, 9, 9), (65, 30, 8),
                                  (127, 3, 129), (128, 4, 4), (193, 11, 13), (700, 1, 2)])
def test_bits_match_numpy(dims, offset):
    nx, ny, nz = dims
    n = nx * ny * nz
    rng = np.random.default_rng(nx + offset)
    host = rng.uniform(-1, 1, size=n).astype(np.float32)
    host[rng.integers(0, n, size=n // 50)] = np.nan
    # the field ends where its allocation ends, and starts `offset` floats into it
    buf = torch.full((n + offset,), 9.0, dtype=torch.float32, device="cuda")
    field = buf[offset:].view(nz, ny, nx)
    field.copy_(torch.from_numpy(host).view(nz, ny, nx))
    for iso in (-0.25, 0.5):
        want = np.zeros((nz, ny, (nx + 63) // 64 * 64), dtype=np.uint8)
        want[:, :, :nx] = (host > np.float32(iso)).reshape(nz, ny, nx)
        want = np.packbits(want, axis=-1, bitorder="little").view(np.uint64)
        assert np.array_equal(_bits(field, iso), want.reshape(nz, ny, -1)), (dims, offset, iso)
