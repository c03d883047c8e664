"""Excitation actions and elements beyond 64 (Dp = 80 and 96), where no persistent launch and no fused node
sums serve them and a product has more than four k-tiles.

- D = 65: the :phi^4: part of F(W) against the oracle's (dense Poisson factors, SciPy's DOP853), both
  integrated to 1e-11 over a short window: within 1e-8 of |F|, the existing action test's 1e-9 at 1e-12
  scaled with the tolerance.
- D = 96: a Z2 state's parity blocks (three tiles each) skip only zeros, so the bits are those of every
  k-tile.
"""
import numpy as np
import pytest
import scipy.linalg as sla

from oracle import excitation as X

pytestmark = pytest.mark.gpu


def note(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def rg():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import rcmps_gpu
    return rcmps_gpu


def short_window(rg, tol=1e-11):
    return rg.IntegratorParameters(n_quad=8, max_point=2.0, atol=tol, rtol=tol)


def oracle_context(s, ip, p):
    """The oracle's context with the two Poisson factors an action needs (no Schur form of the transfer)."""
    xs = X.XState(s.R, s.Q, s.rho, n_quad=ip.n_quad, max_point=ip.max_point, atol=ip.atol, rtol=ip.rtol)
    a = np.outer(s.rho.ravel(), np.eye(s.D).ravel()) - X.transfer_matrix(s.Q, s.R)
    poisson = sla.lu_factor(a)
    a[np.diag_indices(len(a))] += 1j * p
    return X.Context(xs, p, None, None, None, poisson, sla.lu_factor(a, overwrite_a=True), None, 1e-10)


def test_phi4_action_matches_oracle(rg):
    d, p, g = 65, 0.3, 1.5
    note(f"case: :phi^4: action D={d} p={p}")
    from rcmps_gpu.excitation import ExcitationContext, ExcitationModel, action_batch
    s = rg.State(*rg.random_state_arrays(d, scaling=0.1, seed=3), steady_tol=1e-12)
    s.integrator_param = short_window(rg)
    rng = np.random.default_rng(1)
    w = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    ctx = ExcitationContext(s, p, dense_transfer=False)
    (f,) = action_batch(ctx, [w], ExcitationModel("phi4", g), 8, parts=2)
    terms = [t for t in X.phi4_terms(g) if not t[1].kinetic]
    ref = X.hamiltonian_action(oracle_context(s, s.integrator_param, p), w, terms)
    note(f"  rel {np.abs(f - ref).max() / np.abs(ref).max():.2e}")
    assert np.abs(f - ref).max() <= 1e-8 * np.abs(ref).max()
    ctx.close()
    s.close()


def test_z2_blocks_of_three_tiles_give_the_same_bits(rg):
    d = 96
    note(f"case: :phi^4: action of a Z2 state D={d}")
    from rcmps_gpu.excitation import ExcitationContext, ExcitationModel, action_batch
    s = rg.State(*rg.random_state_z2_arrays(d, scaling=0.1, seed=4), steady_tol=1e-12)
    s.integrator_param = short_window(rg, 1e-9)
    rng = np.random.default_rng(2)
    w = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    w[:d // 2, :d // 2] = 0
    w[d // 2:, d // 2:] = 0
    ctx = ExcitationContext(s, 0.3, dense_transfer=False)
    a, b = (action_batch(ctx, [w], ExcitationModel("phi4", 1.5), 8, parts=2, z2_blocks=z2)[0] for z2 in (True, False))
    assert np.isfinite(a).all() and np.abs(a).max() > 0
    assert np.array_equal(a, b)
    ctx.close()
    s.close()
