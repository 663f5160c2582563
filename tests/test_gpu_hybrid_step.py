"""Substeps and RK3 steps with the hybrid EOS against the oracle, and its face
states at densities that the EOS clamps (a reconstruction may leave them at or
below zero): p and the sound speed come from the clamped density, the enthalpy
of the wave speeds from the reconstructed one."""
import numpy as np
import pytest

import grace_amd as ga
import grace_amd.workloads as W
from test_gpu_parity import O, check_close, dev_arrays, interior, linf_rel, run_rk3_pair, to_host

pytestmark = pytest.mark.gpu


def hybrid_blast(curved, recon=0, thermo=0, riemann=0, pieces=1):
    wl = W.blast_ks(nb=(2, 2, 2), n=8) if curved else W.blast(nb=(2, 2, 1), n=8, recon=recon)
    p = wl.params
    p.eos_kind, p.recon, p.thermo_recon, p.riemann = ga.EOS_HYBRID_PWPOLY, recon, thermo, riemann
    p.pwp_kappa0 = 0.05
    if pieces == 2:
        p.pwp_n, p.pwp_gamma[0], p.pwp_gamma[1], p.pwp_rho[0] = 2, 4.0 / 3.0, 2.0, 9e-3
    return wl


def consistent(wl):
    """Primitives of the workload's conserved under its own EOS, in place."""
    s = O.Stepper(wl)
    s.ghosts(wl.state, wl.B)
    s.aux(wl.state, wl.B, wl.aux)
    return s


@pytest.mark.parametrize("curved,recon,thermo,riemann,pieces", [
    (False, 0, 0, 0, 1), (False, 0, 1, 1, 2), (False, 1, 1, 0, 1), (True, 0, 0, 1, 2), (True, 0, 1, 0, 1)])
def test_gpu_hybrid_rk3(dev, curved, recon, thermo, riemann, pieces):
    wl = hybrid_blast(curved, recon, thermo, riemann, pieces)
    consistent(wl)
    ref, got, _ = run_rk3_pair(wl, dev, steps=2)
    check_close(wl, ref, got, 1e-12)


@pytest.mark.parametrize("riemann", [0, 1])
@pytest.mark.parametrize("curved", [False, True])
def test_gpu_hybrid_clamped_face_density(dev, curved, riemann):
    """Donor-cell faces of cells with zero and negative density."""
    import torch
    wl = hybrid_blast(curved, recon=3, riemann=riemann)
    s = consistent(wl)
    g = wl.grid.ngz
    rho = wl.aux[:, ga.RHO]
    rho[0, g + 2, g + 3, g + 4] = 0.0
    rho[1, g + 5, g + 2, g + 3] = -2e-3
    rho[0, g + 4, g + 6, g + 1] = -1e-8
    st, B, aux = wl.copy_arrays()
    dt = 0.1 * wl.extra["dx"]
    new_o, nB_o = st.copy(), [b.copy() for b in B]
    s.substep(dt, 1.0, new_o, st, nB_o, B, aux)
    ctx = ga.Context(wl.params, wl.grid, wl.instances)
    sg, Bg, ag = dev_arrays(wl, dev)
    new, nB = sg.clone(), [b.clone() for b in Bg]
    ctx.advance_substep(torch.tensor([dt], dtype=torch.float64, device=dev), 1.0, new, sg, nB, Bg, ag)
    torch.cuda.synchronize()
    a, b = interior(wl.grid, to_host(new)), interior(wl.grid, new_o)
    for v in range(7):
        assert np.isfinite(b[:, v]).all()
        assert linf_rel(a[:, v], b[:, v]) < 1e-12, v
    for d in range(3):
        assert linf_rel(to_host(nB[d]), nB_o[d]) < 1e-12, d
