"""The persistent Arnoldi steps (rc_arnoldi) at tile edges and basis sizes, through the kinetic terms.

- kinetic1/kinetic2 (one-block bases of L and L*) from a basis grown in one call (up to 40 vectors in
  registers, later ones in memory) against one grown by doubling from 3, and against 300 steps asked for
  at once, which is beyond the kernel's sum records and takes the launch sequence; D = 65 takes that
  anyway.  The projected solves (rc_projected) meet one to eight rows a lane that way, and 600 vectors
  (D = 33) their host route.  Every solve is accepted at a true residual of 1e-12: values to 1e-11, gradients to 1e-8 of
  their largest entry (the bars of the route's oracle tests).
- the excitation action's kinetic part (two-block bases) against the dense resolvents of the same state,
  to 1e-8 of |F| with solves accepted at 1e-11 (as the route's batch test).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def note(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def rg():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import rcmps_gpu
    return rcmps_gpu


@pytest.mark.parametrize("d", [2, 15, 16, 17, 33, 49, 64, 65])
def test_basis_sizes_agree(rg, d):
    note(f"case: kinetic terms by basis growth, D={d}")
    r, k = rg.random_state_arrays(d, scaling=0.2, seed=11)
    s = rg.State(r, k, steady_tol=1e-12)
    out = []
    for initial in (3, min(100, d * d), min(300, d * d)) + ((600,) if d == 33 else ()):
        o = rg.KineticKrylovOptions(initialdim=initial, maxdim=max(512, initial))
        (v1, g1), st = rg.kinetic1(s, krylov_options=o, return_stats=True)
        v2, g2 = rg.kinetic2(s, krylov_options=o)
        note(f"  initial {initial}: basis {st['kinetic_basis']}, residual {st['kinetic_residual']:.2e}")
        assert st["kinetic_residual"] <= 1e-12
        out.append((v1 + v2, g1 + g2))
    for v, g in out[1:]:
        assert v == pytest.approx(out[0][0], rel=1e-11, abs=1e-11)
        assert np.abs(g - out[0][1]).max() <= 1e-8 * max(1.0, np.abs(g).max())
    s.close()


@pytest.mark.parametrize("d", [2, 16, 17, 32])
def test_two_block_bases_against_dense_resolvents(rg, d):
    note(f"case: action's kinetic part, Krylov vs dense resolvents, D={d}")
    from rcmps_gpu.excitation import ExcitationContext, ExcitationModel, action_batch
    r, k = rg.random_state_arrays(d, scaling=0.2, seed=7)
    s = rg.State(r, k, steady_tol=1e-12)
    model = ExcitationModel("phi4", 2.0)
    rng = np.random.default_rng(d)
    ws = [rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)) for _ in range(2)]
    tight = rg.KineticKrylovOptions(tolerance=1e-11, fallback_tolerance=1e-11)
    fs = {}
    for dense in (True, False):
        ctxs = [ExcitationContext(s, p, dense_transfer=dense) for p in (0.1, 0.6)]
        fs[dense] = action_batch(ctxs, ws, model, 48, parts=1, krylov_options=tight)
        for c in ctxs:
            c.close()
    for a, b in zip(fs[True], fs[False]):
        note(f"  |Krylov - dense| / |F| = {np.abs(a - b).max() / np.abs(a).max():.2e}")
        assert np.abs(a - b).max() <= 1e-8 * np.abs(a).max()
    s.close()
