"""The fused Krylov solve (rc_gmres: a whole restarted GMRES in one launch, Dp <= 64) at its tile edges.

rc_gmres serves the stationary state, the boundary environment and the Krylov Poisson solves of the
excitation action; D = 65 and the Schur form of the no-jump inverse take the sequence of launches.
Against plain numpy in double precision:

- rho0 solves L(rho) = 0 to 10 steady_tol, and the boundary environment -L^+(h) = a - tr(rho a) with
  tr(rho h) = 0 to the solver's bar, 20 tol max(1, |b|) (the residual it accepts, Frobenius);
- the Poisson solves of both directions and all three momentum shifts satisfy their equation to the
  excitation context's bar, 20 tol max(1, |b|) at tol = 1e-10, from non-Hermitian right-hand sides
  (src/excitation_environments.jl:75-85);
- the launch sequence on the same state (the Schur form forced) agrees to the sum of the two residuals
  times the inverse's norm, taken as 1e-9 relative (as the existing route test does);
- evaluations of one batch, whose boundary solves share a launch and whose trajectories lie on other
  XCDs than a single call's (several systems to an XCD, some on two, some spread), equal single calls
  bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [2, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65]


def note(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def rg():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import rcmps_gpu
    yield rcmps_gpu
    rcmps_gpu.nojump_threshold(1e6)


def lindblad(s, x, adjoint):
    if adjoint:
        return s.Q.conj().T @ x + x @ s.Q + s.R.conj().T @ x @ s.R
    return s.Q @ x + x @ s.Q.conj().T + s.R @ x @ s.R.conj().T


def random_matrix(d, seed, hermitian=False):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    return a + a.conj().T if hermitian else a


@pytest.mark.parametrize("d", SIZES)
def test_stationary_state_and_boundary(rg, d):
    note(f"case: fused solve D={d}")
    r, k = rg.random_state_arrays(d, scaling=0.2, seed=42)
    a = random_matrix(d, 3, True)
    out = {}
    for kappa in (1e6, 0.0):
        rg.nojump_threshold(kappa)
        try:
            s = rg.State(r, k, steady_tol=1e-12)
        finally:
            rg.nojump_threshold(1e6)
        h = rg.boundary_environment(s, a, tol=1e-12)
        form = s.nojump_form[0]
        res = np.linalg.norm(lindblad(s, s.rho, False))
        b = a - np.trace(s.rho @ a) * np.eye(d)
        bres = np.linalg.norm(lindblad(s, h, True) + b)
        note(f"  {form}: steps {s.steady_stats['krylov_matvecs']}, residuals {res:.2e} {bres:.2e}")
        assert res <= 1e-11
        assert bres <= 20e-12 * max(1.0, np.linalg.norm(b))
        assert abs(np.trace(s.rho @ h)) <= 20e-12 * max(1.0, np.linalg.norm(b))
        out[form] = (s.rho, h)
        s.close()
    assert ("schur" in out) == (d <= 64)   # larger states have the eigenbasis form only
    (r1, h1), (r0, h0) = out["eigen"], out.get("schur", out["eigen"])
    assert np.linalg.norm(r1 - r0) <= 1e-9
    assert np.linalg.norm(h1 - h0) <= 1e-9 * np.linalg.norm(h1)


@pytest.mark.parametrize("d", [2, 16, 17, 33, 64])
def test_excitation_poisson_equations(rg, d):
    note(f"case: fused Poisson solves D={d} p=0.7")
    from rcmps_gpu.excitation import ExcitationContext, action_dual_poisson, excitation_poisson
    r, k = rg.random_state_arrays(d, scaling=0.2, seed=7)
    s = rg.State(r, k, steady_tol=1e-12)
    assert s.nojump_form[0] == "eigen"
    ctx = ExcitationContext(s, 0.7, dense_transfer=False)
    b = random_matrix(d, 5)
    eye = np.eye(d)

    def check(x, adjoint, sigma, phi, psi):
        bb = b - np.trace(phi @ b) * psi
        res = np.linalg.norm(-lindblad(s, x, adjoint) + 1j * sigma * x - bb)
        note(f"  adjoint {adjoint} sigma {sigma}: residual {res:.2e}")
        assert res <= 20e-10 * max(1.0, np.linalg.norm(bb))
        assert abs(np.trace(phi @ x)) <= 20e-10 * max(1.0, np.linalg.norm(x))

    for shift in (-1, 0, 1):
        check(excitation_poisson(ctx, b, shift), False, 0.7 * shift, eye, s.rho)
    for shifted in (False, True):
        check(action_dual_poisson(ctx, b, shifted), True, -0.7 if shifted else 0.0, s.rho, eye)
    ctx.close()
    s.close()


@pytest.mark.parametrize("d", [5, 16, 17, 33, 48, 64])
def test_batched_boundary_solves_equal_single_ones(rg, d):
    note(f"case: batch of 3 at D={d}")
    states = [rg.State(*rg.random_state_arrays(d, scaling=0.2, seed=i)) for i in range(3)]
    single = [rg.fg_phi4(s, 1.5) for s in states]
    energies, gradients = rg.fg_phi4_batch(states, [1.5] * 3)
    for (e, g), be, bg in zip(single, energies, gradients):
        assert e == be
        assert np.array_equal(g, bg)
    for s in states:
        s.close()
