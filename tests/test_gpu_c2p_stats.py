"""The statistics of a batch inversion against the per-state outputs: one
state, part of a wave and of a workgroup, the last size that one launch sums
up and the first one that takes two, and sizes that fill neither."""
import numpy as np
import pytest

import grace_amd as ga
import grace_amd.workloads as W
from test_gpu_parity import to_host

pytestmark = pytest.mark.gpu

ENT_BACKUP, ATMO_RESET = 19, 20   # bits of the error mask


@pytest.mark.parametrize("n", [1, 63, 257, 2048 * 256, 2048 * 256 + 1, 777_777])
def test_gpu_c2p_stats_sums(n):
    import torch
    dev = torch.device("cuda:0")
    st = W.c2p_states(5000, seed=3)
    pick = torch.arange(n, device=dev) % 5000
    cons = torch.from_numpy(st["cons"]).to(dev)[:, pick].contiguous()
    met = torch.from_numpy(st["met"]).to(dev)[:, pick].contiguous()
    cons[:, n // 2] *= 1e-12                # below the atmosphere threshold
    inst = ga.make_instances([dict(nb=(1, 1, 1), q0=0, bc=(0,) * 6, idx=(1.0, 1.0, 1.0))])
    st["params"].rho_fl = 1e-16
    ctx = ga.Context(st["params"], ga.Grid(1, 1, 1, 3, 1), inst)
    prims = torch.zeros((13, n), dtype=torch.float64, device=dev)
    err = torch.zeros(n, dtype=torch.int64, device=dev)
    fl = torch.zeros(n, dtype=torch.uint8, device=dev)
    counts = torch.zeros(n, dtype=torch.uint8, device=dev)
    ctx.set_c2p_eval_counts(counts)
    ctx.c2p_batch(n, cons, met, prims, err, fl)
    torch.cuda.synchronize()
    ctx.set_c2p_eval_counts(None)
    s = ctx.c2p_stats()
    e, c = to_host(err).astype(np.uint64), to_host(counts).astype(np.int64)
    assert c.max() < 255
    assert s["n_cells"] == n
    assert s["n_root_evals"] + s["n_bracket_evals"] == c.sum()
    assert s["n_ent_backup"] == int(np.sum((e >> np.uint64(ENT_BACKUP)) & np.uint64(1)))
    assert s["n_atmo_reset"] == int(np.sum((e >> np.uint64(ATMO_RESET)) & np.uint64(1))) >= 1
    assert s["max_root_evals"] <= c.max() and s["n_guess_used"] == 0


@pytest.mark.parametrize("n,at", [(1, 0), (257, 256), (777_777, 777_776), (777_777, 0), (2048 * 256 + 1, 2048 * 256),
                                  (2048 * 256 + 1, 131_071)])
def test_gpu_c2p_stats_maximum(n, at):
    """The largest number of root evaluations is that of the one state that
    takes more than the others, wherever it stands: alone, in the last, partly
    filled workgroup, in the first, and among records that two launches sum."""
    import torch
    dev = torch.device("cuda:0")
    st = W.c2p_states(4000, seed=3)
    inst = ga.make_instances([dict(nb=(1, 1, 1), q0=0, bc=(0,) * 6, idx=(1.0, 1.0, 1.0))])
    ctx = ga.Context(st["params"], ga.Grid(1, 1, 1, 3, 1), inst)
    cons0 = torch.from_numpy(st["cons"]).to(dev)
    met0 = torch.from_numpy(st["met"]).to(dev)

    def stats(pick):
        m = pick.numel()
        prims = torch.zeros((13, m), dtype=torch.float64, device=dev)
        err = torch.zeros(m, dtype=torch.int64, device=dev)
        fl = torch.zeros(m, dtype=torch.uint8, device=dev)
        ctx.c2p_batch(m, cons0[:, pick].contiguous(), met0[:, pick].contiguous(), prims, err, fl)
        torch.cuda.synchronize()
        return ctx.c2p_stats()

    one = [stats(torch.tensor([k], device=dev)) for k in range(40)]
    roots = [s["n_root_evals"] for s in one]
    assert all(s["max_root_evals"] == s["n_root_evals"] > 0 for s in one)
    few, many = int(np.argmin(roots)), int(np.argmax(roots))
    assert roots[many] > roots[few]
    pick = torch.full((n,), few, dtype=torch.int64, device=dev)
    pick[at] = many
    s = stats(pick)
    assert s["max_root_evals"] == roots[many]
    assert s["n_root_evals"] == roots[many] + (n - 1) * roots[few]
