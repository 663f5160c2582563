"""con2prim of conserved values whose quotients leave the range of a double
(or are infinite) against the oracle: the outcome, the error bits and the
limits that an infinite quotient runs into."""
import numpy as np
import pytest

import grace_amd as ga
import grace_amd.workloads as W
import _oracle as O
from test_gpu_parity import to_dev, to_host

pytestmark = pytest.mark.gpu


def run(dev, params, cons, met):
    import torch
    n = cons.shape[1]
    inst = ga.make_instances([dict(nb=(1, 1, 1), q0=0, bc=(0,) * 6, idx=(1.0, 1.0, 1.0))])
    ctx = ga.Context(params, ga.Grid(1, 1, 1, 3, 1), inst)
    c, m = to_dev(cons, dev), to_dev(met, dev)
    prims = torch.zeros((13, n), dtype=torch.float64, device=dev)
    err = torch.zeros(n, dtype=torch.int64, device=dev)
    fl = torch.zeros(n, dtype=torch.uint8, device=dev)
    ctx.c2p_batch(n, c, m, prims, err, fl)
    torch.cuda.synchronize()
    return to_host(prims), to_host(c), to_host(err).astype(np.uint64), to_host(fl)


@pytest.mark.parametrize("value", [1e300, -1e300, np.inf, -np.inf])
@pytest.mark.parametrize("var", [4, 5, 6], ids=["tau", "ye", "entropy"])
def test_gpu_c2p_infinite_quotients(dev, var, value):
    """One conserved of every second state is so large that its quotient by
    the density overflows: the limits of tau, Y_e and the entropy apply, as
    they do to an infinite value."""
    n = 256
    st = W.c2p_states(n, seed=5, rho=(1e-11, 1e-9), W=(1.0, 3.0), sigma=(1e-4, 1e-1))
    cons, met = st["cons"].copy(), st["met"]
    odd = np.arange(n) % 2 == 1
    cons[var, odd] = value
    pr, co, er, fl = run(dev, st["params"], cons, met)
    po, cc, eo, fo, _, _ = O.c2p_batch(st["params"], cons, met)
    assert np.array_equal(er, eo), [hex(int(x)) for x in (er ^ eo)[er != eo][:4]]
    assert np.array_equal(fl, fo)
    for got, ref in ((pr[:12], po[:12]), (co, cc)):
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(np.isinf(got), np.isinf(ref))


def test_gpu_c2p_magnetisation_out_of_range(dev):
    """B^2 / D beyond the largest double beside a density beyond the EOS: the
    density's own signal, fatal outside the lenient region, is raised."""
    n = 64
    st = W.c2p_states(n, seed=6)
    cons, met = st["cons"].copy(), st["met"]
    cons[0, 1::2] = 1e154
    cons[8, 1::2] = 1e300
    pr, co, er, fl = run(dev, st["params"], cons, met)
    po, cc, eo, fo, _, _ = O.c2p_batch(st["params"], cons, met)
    assert np.array_equal(er, eo), [hex(int(x)) for x in (er ^ eo)[er != eo][:4]]
    assert np.array_equal(fl, fo)
