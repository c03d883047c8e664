"""The fused pullback (rc_pullback) where its instantiations and its streams of nodes change: tiles per
side, one node to a stream, node counts that do not divide; against the oracle's node sums.

The oracle integrates with the same controller and sums over the same nodes, so energies and gradients
agree up to rounding carried through the integration: 1e-10 of the energy and 1e-8 of the gradient's
largest entry (the bars of the route's other oracle tests are 1e-12 and 1e-10 on full windows)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rg():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import rcmps_gpu
    return rcmps_gpu


@pytest.mark.parametrize("d,n_quad", [(2, 8), (16, 150), (17, 9), (32, 64), (33, 8), (48, 50),
                                       (49, 11), (64, 8)])
def test_pullback_matches_oracle(rg, d, n_quad):
    print(f"case: pullback D={d} n_quad={n_quad}", flush=True)
    s = rg.State(*rg.random_state_arrays(d, scaling=0.2, seed=d))
    s.integrator_param = rg.IntegratorParameters(n_quad=n_quad, max_point=3.0, atol=1e-9, rtol=1e-8)
    e, g = rg.fg_phi4(s, 1.5)
    o = oracle.fg_phi4(s.R, s.Q, s.rho, 1.5, n_quad=n_quad, max_point=3.0, atol=1e-9, rtol=1e-8)
    err = np.abs(g - o["gradient"]).max() / np.abs(o["gradient"]).max()
    print(f"  energy {abs(e - o['energy']) / abs(o['energy']):.1e}, gradient {err:.1e}", flush=True)
    assert abs(e - o["energy"]) <= 1e-10 * abs(o["energy"])
    assert err <= 1e-8
    s.close()
