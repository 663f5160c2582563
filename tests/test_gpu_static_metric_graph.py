"""The cached metric (Context.set_static_metric) and graphs that the caller
captures: a replay takes the metric the caches hold at the replay, whatever the
comparison of the ghost metric with the neighbours' said when it was captured."""
import pytest

import grace_amd as ga
import grace_amd.workloads as W
from test_gpu_parity import dev_arrays

pytestmark = pytest.mark.gpu


def setup(dev):
    import torch
    wl = W.blast_ks(nb=(2, 2, 2), n=8)
    dt = torch.tensor([0.2 * wl.extra["dx"]], dtype=torch.float64, device=dev)
    return wl, dt, dev_arrays(wl, dev)


def restore(to, arrays):
    for a, b in zip((to[0], *to[1], to[2]), (arrays[0], *arrays[1], arrays[2])):
        a.copy_(b)


def changed_ghosts(wl, dev):
    """The workload with the lapse of one ghost cell beside block 1 a thousandth larger."""
    a = dev_arrays(wl, dev)
    g, n = wl.grid.ngz, wl.grid.nx
    a[0][0, ga.ALP, g + 2, g + 2, g + n] *= 1.001
    return a


def plain_steps(wl, arrays, dt, steps):
    import torch
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    for _ in range(steps):
        ctx.rk3_step(dt, *arrays)
    torch.cuda.synchronize()
    return arrays


def same(a, b):
    import torch
    return all(torch.equal(x, y) for x, y in zip((a[0], *a[1], a[2]), (b[0], *b[1], b[2])))


def test_gpu_captured_step_follows_the_cached_metric(dev):
    """A step captured while the ghost metric agrees; then a metric whose
    ghosts do not, cached again: the replays give that metric's steps."""
    import torch
    wl, dt, a = setup(dev)
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ctx.set_static_metric(a[0], stream=s.cuda_stream)
        ctx.rk3_step(dt, *a, stream=s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ctx.rk3_step(dt, *a, stream=s.cuda_stream)
    for arrays in (dev_arrays(wl, dev), changed_ghosts(wl, dev)):
        with torch.cuda.stream(s):
            restore(a, arrays)
            ctx.set_static_metric(a[0], stream=s.cuda_stream)
            for _ in range(3):
                g.replay()
        s.synchronize()
        assert same(a, plain_steps(wl, arrays, dt, 3))
    assert not same(plain_steps(wl, dev_arrays(wl, dev), dt, 3), a)     # the change is seen


def test_gpu_captured_metric_cache_is_not_compared(dev):
    """The caches refreshed by a replay, from a metric whose ghosts do not
    agree, after a call outside a capture had found that they do."""
    import torch
    wl, dt, a = setup(dev)
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ctx.set_static_metric(a[0], stream=s.cuda_stream)
        ctx.rk3_step(dt, *a, stream=s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ctx.set_static_metric(a[0], stream=s.cuda_stream)
    arrays = changed_ghosts(wl, dev)
    for graph in (False, True):
        with torch.cuda.stream(s):
            restore(a, dev_arrays(wl, dev))
            ctx.set_static_metric(a[0], stream=s.cuda_stream)
            restore(a, arrays)
            g.replay()
            for _ in range(2):
                ctx.rk3_step(dt, *a, stream=s.cuda_stream, graph=graph)
        s.synchronize()
        assert same(a, plain_steps(wl, changed_ghosts(wl, dev), dt, 2))
