"""mc.forward and mc.slice generate from the classification they counted: the
count's launch shape travels in the workspace, and calls from several threads
and streams keep their sizes apart."""
import threading

import pytest
import torch

from daxtoolkit_amd import fields, mc

pytestmark = pytest.mark.gpu


def _field(dims, seed):
    m = min(dims)
    p = fields.gaussian_mixture_params(seed, dims, sigma=(0.1 * m, 0.3 * m))
    return fields.gaussian_mixture_torch(dims, p)


@pytest.mark.parametrize("count_sub,gen_sub", [(1, 8), (8, 1), (2, 4)])
def test_generate_under_another_tuning(count_sub, gen_sub):
    dims = (70, 61, 83)
    f = _field(dims, 3)
    want = mc.forward(f, 0.5, edges=True)
    buf = mc.ForwardBuffers(*dims, want.num_points, want.num_triangles, edges=True)
    saved = mc.get_tuning(dims)
    try:
        mc.set_tuning(dims, [4, 4, count_sub, 256, 0])
        mc.classify_into(f, 0.5, buf)
        mc.count_scan_into(buf)
        mc.set_tuning(dims, [4, 4, gen_sub, 128, 0])
        mc.generate_into(f, 0.5, buf)
    finally:
        mc.set_tuning(dims, saved)
    assert torch.equal(buf.vertices, want.vertices) and torch.equal(buf.conn, want.connectivity)
    assert torch.equal(buf.edges, want.edges) and torch.equal(buf.counts, want.counts)


def test_threads_and_streams():
    shapes = [(20 + 7 * i, 33, 40 - i) for i in range(8)]
    inputs = [_field(d, i) for i, d in enumerate(shapes)]
    want = [mc.forward(f, 0.5) for f in inputs]
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                c = mc.forward(inputs[i], 0.5)
                if not (torch.equal(c.vertices, want[i].vertices) and
                        torch.equal(c.connectivity, want[i].connectivity)):
                    bad.append(i)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(shapes))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_no_output():
    f = torch.zeros((5, 6, 70), device="cuda")
    c = mc.forward(f, 0.5, edges=True, interp=True)
    assert c.num_points == 0 and c.num_triangles == 0 and c.counts.tolist() == [0, 0]
    assert c.normals.shape == (0, 3) and c.edges.shape == (0,) and c.interp_weight.shape == (0,)
    g = torch.ones_like(f)
    e = torch.empty((0, 3), device="cuda")
    assert not mc.backward(f, 0.5, c, e, e, out=g).any()
