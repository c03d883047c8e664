"""Excitation actions and elements beyond 64 (Dp = 80 and 96), where no persistent launch and no fused node
sums serve them and a product has more than four k-tiles, and more Arnoldi bases than fit one launch.

- D = 65: the :phi^4: part of F(W) against the oracle's (dense Poisson factors, SciPy's DOP853), both
  integrated to 1e-11 over a short window: within 1e-8 of |F|, the existing action test's 1e-9 at 1e-12
  scaled with the tolerance.
- D = 65: the connected element's kinetic part against <u, F(w)>, whose products are other kernels (2e-8, as
  the existing element test), its :phi^4: part against the oracle's (1e-8, as above; <u, F(w)> has the
  quadrature error of its few nodes there, the element none).
- D = 64, five tangents: ten two-block bases, of which eight fit a launch of the persistent Arnoldi steps.
  The kinetic part of each against the tangent alone, 1e-8 of |F| with solves accepted at 1e-11 (as the
  existing batch test: a set's bases grow together, so alone they may be smaller).
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


def oracle_context(s, ip, p, bra=False):
    """The oracle's context with the Poisson factors an action needs, an element's third on request (no Schur
    form of the transfer)."""
    xs = X.XState(s.R, s.Q, s.rho, n_quad=ip.n_quad, max_point=ip.max_point, atol=ip.atol, rtol=ip.rtol)
    a = np.outer(s.rho.ravel(), np.eye(s.D).ravel()) - X.transfer_matrix(s.Q, s.R)
    factors = []
    for shift in (0.0, 1.0, -1.0) if bra else (0.0, 1.0):
        b = a.copy()
        b[np.diag_indices(len(b))] += 1j * shift * p
        factors.append(sla.lu_factor(b, overwrite_a=True))
    return X.Context(xs, p, None, None, None, factors[0], factors[1], factors[2] if bra else None, 1e-10)


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


def test_connected_element(rg):
    d, p, g = 65, 0.3, 1.5
    note(f"case: connected element D={d} p={p}")
    from rcmps_gpu.excitation import ExcitationContext, ExcitationModel, action_batch, excitation_element
    s = rg.State(*rg.random_state_arrays(d, scaling=0.1, seed=3), steady_tol=1e-12)
    s.integrator_param = short_window(rg)
    rng = np.random.default_rng(1)
    u, w = rng.standard_normal((2, d, d)) + 1j * rng.standard_normal((2, d, d))
    ctx, model = ExcitationContext(s, p, dense_transfer=False), ExcitationModel("phi4", g)
    (f,) = action_batch(ctx, [w], model, 32, parts=1)
    kin, pot = (excitation_element(ctx, [u], [w], model=model, kinetic_nodes=32, parts=parts)[0] for parts in (1, 2))
    ref = g * X.excitation_observable(X.pair(oracle_context(s, s.integrator_param, p, bra=True), u, w), X.monomial_spec(4))
    note(f"  kinetic {kin} vs {np.vdot(u, f)}; potential {pot} vs {ref}")
    assert abs(np.vdot(u, f) - kin) <= 2e-8 * max(1.0, abs(kin))
    assert abs(pot - ref) <= 1e-8 * max(1.0, abs(ref))
    ctx.close()
    s.close()


def test_more_bases_than_a_launch_holds(rg):
    d, n = 64, 5
    note(f"case: kinetic action D={d}, {n} tangents")
    from rcmps_gpu.excitation import ExcitationContext, ExcitationModel, action_batch
    s = rg.State(*rg.random_state_arrays(d, scaling=0.2, seed=7), steady_tol=1e-12)
    rng = np.random.default_rng(d)
    ws = [rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)) for _ in range(n)]
    ctxs = [ExcitationContext(s, 0.1 + 0.2 * i, dense_transfer=False) for i in range(n)]
    tight = rg.KineticKrylovOptions(tolerance=1e-11, fallback_tolerance=1e-11)
    model = ExcitationModel("phi4", 2.0)
    together = action_batch(ctxs, ws, model, 32, parts=1, krylov_options=tight)
    for c, w, f in zip(ctxs, ws, together):
        (alone,) = action_batch(c, [w], model, 32, parts=1, krylov_options=tight)
        note(f"  |together - alone| / |F| = {np.abs(f - alone).max() / np.abs(alone).max():.2e}")
        assert np.abs(f - alone).max() <= 1e-8 * np.abs(alone).max()
    for c in ctxs:
        c.close()
    s.close()
