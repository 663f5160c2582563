"""The merged face-flux launch and the row layout of its outputs, at the block
extents where the face indexing can go wrong: odd and unequal extents, extents
equal to the ghost width, one cell across, each reconstruction and EMF; and the
reconstruction's form for values whose indicator products overflow."""
import numpy as np
import pytest

import grace_amd as ga
import grace_amd.workloads as W
from grace_amd.workloads import _p, lib
from test_gpu_parity import O, check_close, dev_arrays, linf_rel, run_rk3_pair, to_host

pytestmark = pytest.mark.gpu

_P, _O = ga.BC_PERIODIC, ga.BC_OUTFLOW


@pytest.fixture(scope="module")
def dev():
    import torch
    return torch.device("cuda:0")


def blast_of(nb, n, ngz, bc, recon, riemann, emf, thermo):
    """A blast in blocks of extents n: cells of spacing 1/16, centred on 0."""
    grid = ga.Grid(*n, ngz, nb[0] * nb[1] * nb[2])
    ext = np.array([nb[d] * n[d] / 16.0 for d in range(3)])
    spec = [dict(nb=nb, q0=0, bc=bc, idx=(16.0,) * 3, x0=tuple(-0.5 * ext))]
    state, B, aux = W.alloc(grid)
    lo, hi, Bv = -0.5 * ext, 0.5 * ext, np.array([0.1, 0.05, 0.02])
    rc = lib().grmhd_setup_blast(grid, ga.make_instances(spec), 1, 4.0 / 3.0, _p(lo), _p(hi), 1e-2, 1e-3, 0.1, 0.2,
                                 _p(Bv), 0.01, 7, _p(state), _p(B[0]), _p(B[1]), _p(B[2]), _p(aux))
    assert rc == 0
    params = ga.default_params(gamma=4.0 / 3.0, emf=emf, recon=recon, riemann=riemann, flat_metric=1)
    params.thermo_recon = thermo
    return W.Workload("blast", params, grid, spec, state, B, aux, zones=int(np.prod(n)) * grid.nq,
                      extra=dict(N=[nb[d] * n[d] for d in range(3)], dx=1.0 / 16.0))


@pytest.mark.parametrize("nb,n,ngz,bc,recon,riemann,emf,thermo", [
    ((2, 2, 1), (5, 9, 7), 3, (_O,) * 6, 0, 0, 0, 0),
    ((2, 1, 2), (3, 4, 3), 3, (_P, _P, _O, _O, _P, _P), 0, 1, 0, 1),
    ((1, 2, 2), (17, 4, 5), 4, (_P,) * 6, 0, 0, 1, 0),
    ((2, 2, 2), (4, 7, 4), 4, (_O,) * 6, 1, 1, 0, 0),
    ((1, 2, 1), (33, 6, 3), 3, (_P, _P, _P, _P, _O, _O), 2, 0, 0, 0),
    ((2, 1, 1), (13, 1, 1), 3, (_O,) * 6, 3, 1, 1, 1),
], ids=["odd_outflow", "ghost_wide_mixed", "gs_ngz4_periodic", "mc2_ngz4", "minmod_long_x", "donor_gs_line"])
def test_gpu_flux_faces_extents(dev, nb, n, ngz, bc, recon, riemann, emf, thermo):
    """Two RK3 steps against the oracle, at the bound of the cubic blocks."""
    wl = blast_of(nb, n, ngz, bc, recon, riemann, emf, thermo)
    ref, got, _ = run_rk3_pair(wl, dev, steps=2)
    check_close(wl, ref, got, 1e-12)
    assert np.array_equal(got[2][:, ga.C2P_ERR], ref[2][:, ga.C2P_ERR])


@pytest.mark.parametrize("where", ["everywhere", "beside small values"])
def test_gpu_flux_faces_overflowing_products(dev, where):
    """An advected scalar of 1e53: the products of the WENO-Z indicators
    overflow (the ratios themselves do not) and the face takes the form that
    divides each.  A few rounding errors of the largest value: 1e-12 as
    everywhere; the other variables keep theirs."""
    import torch
    wl = blast_of((2, 1, 1), (8, 8, 8), 3, (_O,) * 6, 0, 0, 0, 0)
    ye = wl.aux[:, ga.YE]
    big = 1e53 * (1.0 + 0.3 * np.sin(np.arange(ye.size).reshape(ye.shape)))
    ye[...] = big if where == "everywhere" else np.where(np.arange(ye.shape[-1]) % 14 < 7, big, 0.3)
    st, B, aux = wl.copy_arrays()
    dt = 0.25 * wl.extra["dx"]
    new_o, nB_o = st.copy(), [b.copy() for b in B]
    O.Stepper(wl).substep(dt, 1.0, new_o, st, nB_o, B, aux)
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    sg, Bg, ag = dev_arrays(wl, dev)
    ng, nBg = sg.clone(), [b.clone() for b in Bg]
    ctx.advance_substep(torch.tensor([dt], dtype=torch.float64, device=dev), 1.0, ng, sg, nBg, Bg, ag)
    torch.cuda.synchronize()
    gn = to_host(ng)
    assert np.max(np.abs(new_o[:, ga.YESTAR])) > 1e43 and np.all(np.isfinite(gn))
    assert linf_rel(gn[:, ga.YESTAR], new_o[:, ga.YESTAR]) < 1e-12
    for v in (ga.DENS, ga.TAU, ga.SX, ga.SY, ga.SZ, ga.ENTROPYSTAR):
        assert linf_rel(gn[:, v], new_o[:, v]) < 1e-12, v


@pytest.mark.parametrize("n,recon,riemann,thermo", [(5, 0, 0, 1), (6, 1, 1, 0), (7, 2, 1, 1), (16, 3, 0, 0)])
def test_gpu_flux_faces_gs_curved(dev, n, recon, riemann, thermo):
    """GS on a curved metric has a face kernel (and an inversion) of its own:
    two RK3 steps against the oracle."""
    wl = W.blast_ks(nb=(2, 2, 2), n=n, emf=ga.EMF_GS)
    wl.params.recon, wl.params.riemann, wl.params.thermo_recon = recon, riemann, thermo
    ref, got, _ = run_rk3_pair(wl, dev, steps=2)
    check_close(wl, ref, got, 1e-12)
    assert np.array_equal(got[2][:, ga.C2P_ERR], ref[2][:, ga.C2P_ERR])


@pytest.mark.parametrize("recon_field", ["everywhere", "beside small values"])
def test_gpu_edge_emfs_overflowing_products(dev, recon_field):
    """Face B of 1e27: the indicator products of the edge EMFs' transverse
    reconstructions overflow as well, and the edge takes its other form."""
    import torch
    wl = blast_of((2, 1, 2), (6, 7, 6), 3, (_O,) * 6, 0, 0, 0, 0)
    rng = np.random.default_rng(5)
    size = 1e27
    for d, b in enumerate(wl.B):
        b[...] = size * (0.5 + 0.3 * rng.uniform(-1, 1, b.shape))
        if recon_field == "beside small values":
            b[rng.uniform(size=b.shape) < 0.5] *= 1e-30
    O.Stepper(wl).ghosts(wl.state, wl.B)
    a = wl.aux
    a[:, ga.BX] = 0.5 * (wl.B[0][:, 0, :, :, :-1] + wl.B[0][:, 0, :, :, 1:])
    a[:, ga.BY] = 0.5 * (wl.B[1][:, 0, :, :-1] + wl.B[1][:, 0, :, 1:])
    a[:, ga.BZ] = 0.5 * (wl.B[2][:, 0, :-1] + wl.B[2][:, 0, 1:])
    for v in (ga.ZVECX, ga.ZVECY, ga.ZVECZ):
        a[:, v] = 0.3 * rng.uniform(-1, 1, a[:, v].shape)
    st, B, aux = wl.copy_arrays()
    dt = 0.25 * wl.extra["dx"]
    new_o, nB_o = st.copy(), [b.copy() for b in B]
    O.Stepper(wl).substep(dt, 1.0, new_o, st, nB_o, B, aux)
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    sg, Bg, ag = dev_arrays(wl, dev)
    ng, nBg = sg.clone(), [b.clone() for b in Bg]
    ctx.advance_substep(torch.tensor([dt], dtype=torch.float64, device=dev), 1.0, ng, sg, nBg, Bg, ag)
    torch.cuda.synchronize()
    for d in range(3):
        got = to_host(nBg[d])
        assert np.isfinite(got).all() and np.max(np.abs(nB_o[d] - B[d])) > 1e-3 * size
        assert linf_rel(got, nB_o[d]) < 1e-12, d
