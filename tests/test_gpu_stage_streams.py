"""RK3 stages with a side stream (grids of 2^18 cells and more) against the
one-stream order, whose launches merge: the same bits; and the error fields,
which the first stage's inversion starts from zero."""
import pytest

import grace_amd as ga
import grace_amd.workloads as W
from test_gpu_parity import dev_arrays, small_blast

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    return torch.device("cuda:0")


def large(case):
    if case == "uct":
        return W.blast(nb=(4, 4, 4))
    if case == "gs":
        return W.blast(nb=(4, 4, 4), emf=ga.EMF_GS)
    if case == "curved":
        return W.blast_ks(nb=(4, 4, 4))
    return W.forest_wave(nb=(4, 4, 4), n=16, ngz=4, refined=[21], b_loop=0.2, p_in=3.0, r_in=0.3)


@pytest.mark.parametrize("case", ["uct", "gs", "curved", "forest"])
def test_gpu_side_stream_matches_one_stream(dev, case):
    import torch
    wl = large(case)
    assert wl.grid.nq * wl.grid.nx * wl.grid.ny * wl.grid.nz >= 1 << 18
    p1 = type(wl.params).from_buffer_copy(wl.params)
    p1.stage_streams = 0
    kw = dict(forest=wl.forest) if case == "forest" else {}
    dtd = torch.tensor([0.1 * wl.extra["dx"]], dtype=torch.float64, device=dev)
    out = []
    for params, graph in ((p1, False), (wl.params, False), (wl.params, True)):
        ctx = ga.Context(params, wl.grid, wl.instances, **kw)
        st, B, aux = dev_arrays(wl, dev)
        if case == "forest":
            ctx.fill_metric_ghosts(st)
        ctx.fill_ghosts(st, B)
        ctx.compute_auxiliaries(st, B, aux)
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        for _ in range(2):
            with torch.cuda.stream(s):
                ctx.rk3_step(dtd, st, B, aux, stream=s.cuda_stream, graph=graph)
        s.synchronize()
        out.append([st, *B, aux])
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("case", ["small", "uct"])
def test_gpu_step_clears_error_fields(dev, case):
    import torch
    wl = small_blast() if case == "small" else large("uct")
    dtd = torch.tensor([0.1 * wl.extra["dx"]], dtype=torch.float64, device=dev)
    out = []
    for junk in (0.0, 12345.0):
        ctx = ga.Context(wl.params, wl.grid, wl.instances)
        st, B, aux = dev_arrays(wl, dev)
        ctx.fill_ghosts(st, B)
        ctx.compute_auxiliaries(st, B, aux)
        aux[:, ga.C2P_ERR] = junk
        aux[:, ga.C2P_ERR - 1] = junk
        ctx.rk3_step(dtd, st, B, aux)
        torch.cuda.synchronize()
        out.append(aux)
    assert torch.equal(out[0], out[1])
