"""The cached metric (Context.set_static_metric) and graphs that the caller
captures: a replay takes the metric the caches hold at the replay, whatever the
comparison of the ghost metric with the neighbours' said when it was captured."""
import numpy as np
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


def test_gpu_static_metric_comparison_decides(dev):
    """Ghosts that differ by a thousandth: the step with the cache is the one
    without, in the caller's order and in the context's graph.  Where they
    agree the later stages leave the ghost metric unread: a lapse that is
    changed behind the cache's back shows in a captured step, which shares
    nothing, and not in those stages of an eager one."""
    import torch
    wl, dt, _ = setup(dev)
    s = torch.cuda.Stream()
    for graph in (False, True):
        a = changed_ghosts(wl, dev)
        ctx = ga.Context(wl.params, wl.grid, wl.instances)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            ctx.set_static_metric(a[0], stream=s.cuda_stream)
            for _ in range(2):
                ctx.rk3_step(dt, *a, stream=s.cuda_stream, graph=graph)
        s.synchronize()
        assert same(a, plain_steps(wl, changed_ghosts(wl, dev), dt, 2))
    out = []
    for captured in (False, True):
        a = dev_arrays(wl, dev)
        ctx = ga.Context(wl.params, wl.grid, wl.instances)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            ctx.set_static_metric(a[0], stream=s.cuda_stream)
            ctx.rk3_step(dt, *a, stream=s.cuda_stream)
        s.synchronize()
        if captured:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                ctx.rk3_step(dt, *a, stream=s.cuda_stream)
        with torch.cuda.stream(s):
            restore(a, changed_ghosts(wl, dev))      # not cached again
            if captured:
                g.replay()
            else:
                ctx.rk3_step(dt, *a, stream=s.cuda_stream)
        s.synchronize()
        out.append(a)
    assert not same(*out)


@pytest.mark.parametrize("graph", [False, True])
def test_gpu_static_metric_shared_periodic_instances(dev, graph):
    """Two instances, one periodic in two dimensions, in a metric that is the
    same everywhere: with the cache (whose ghosts agree across every face) the
    bits of the steps without."""
    import torch
    n, ngz = 6, 3
    specs = [dict(nb=(2, 1, 2), q0=0, bc=(1, 1, 1, 1, 0, 0), idx=(16.0,) * 3, x0=(-0.4, -0.2, -0.4)),
             dict(nb=(1, 2, 1), q0=4, bc=(0,) * 6, idx=(16.0,) * 3, x0=(-0.2, -0.4, -0.2))]
    grid = ga.Grid(n, n, n, ngz, 6)
    state, B, aux = W.alloc(grid)
    state[:], aux[:] = 0.0, 0.0
    rng = np.random.default_rng(3)
    for v, x in ((ga.GXX, 1.1), (ga.GXX + 1, 0.05), (ga.GXX + 3, 1.05), (ga.GXX + 5, 0.95), (ga.ALP, 0.9),
                 (ga.ALP + 1, 0.05), (ga.ALP + 2, -0.02), (ga.ALP + 3, 0.03)):
        state[:, v] = x
    shape = state[:, ga.DENS].shape
    state[:, ga.DENS] = 1e-2 * (1.0 + 0.1 * rng.uniform(-1, 1, shape))
    state[:, ga.TAU] = 2e-2 * (1.0 + 0.2 * rng.uniform(0, 1, shape))
    for v in (ga.SX, ga.SY, ga.SZ):
        state[:, v] = 2e-3 * rng.uniform(-1, 1, shape)
    state[:, ga.ENTROPYSTAR] = state[:, ga.DENS]
    for d, b in enumerate(B):
        b[:] = 0.02 * (d + 1)
    params = ga.default_params(gamma=4.0 / 3.0, flat_metric=0)
    res = []
    s = torch.cuda.Stream()
    for cache in (False, True):
        ctx = ga.Context(params, grid, ga.make_instances(specs))
        st, Bg, ag = torch.from_numpy(state).to(dev), [torch.from_numpy(b).to(dev) for b in B], torch.from_numpy(aux).to(dev)
        ctx.fill_ghosts(st, Bg)
        ctx.compute_auxiliaries(st, Bg, ag)
        dt = torch.tensor([0.1 / 16.0], dtype=torch.float64, device=dev)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            if cache:
                ctx.set_static_metric(st, stream=s.cuda_stream)
            for _ in range(3):
                ctx.rk3_step(dt, st, Bg, ag, stream=s.cuda_stream, graph=graph)
        s.synchronize()
        assert torch.isfinite(st).all() and torch.isfinite(Bg[0]).all()
        res.append([st, *Bg, ag])
    for a, b in zip(*res):
        assert torch.equal(a, b)
