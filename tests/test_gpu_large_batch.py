"""A batch of more evaluations than one launch's exchange rings are kept for (8 GiB, 77 of them at D = 64): its
device memory is bounded, and the results are the single calls' bits, also where the boundary solves of a launch
need several launches of their own (more than 16 of them at D = 64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rg():
    import rcmps_gpu
    return rcmps_gpu


def test_rings_of_a_large_batch_are_bounded(rg):
    import torch
    n, d = 110, 64
    print(f"case: batch of {n} at D={d}", flush=True)
    ip = rg.IntegratorParameters(n_quad=8, max_point=2.0, atol=1e-9, rtol=1e-9)
    arrays = [rg.random_state_arrays(d, scaling=0.2, seed=i) for i in range(n)]
    states = [rg.State(r, k, integrator_param=ip) for r, k in arrays]
    gs = [1.0 + 0.01 * i for i in range(n)]
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    energies, gradients = rg.fg_phi4_batch(states, gs)
    taken = free - torch.cuda.mem_get_info()[0]
    samples = 17 * 13 * d * d * 16 * n          # one evaluation's 13 channels at 17 points
    print(f"  taken {taken / 2**30:.2f} GiB, samples {samples / 2**30:.2f} GiB", flush=True)
    assert taken <= (8 << 30) + samples + (1 << 30)   # rings, samples, workspaces; with rings of all 12.6 GiB
    for i in (0, 20, 54, 55, n - 1):
        e, g = rg.fg_phi4(states[i], gs[i])
        assert e == energies[i]
        assert np.array_equal(g, gradients[i])
    for s in states:
        s.close()
