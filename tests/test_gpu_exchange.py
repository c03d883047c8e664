"""The trajectory kernel's exchange rings and its instantiations against the oracle and against each
other, at the sizes where they change: one tile (stage input and P kept in LDS), the edges of two, three
and four tiles, steps rejected often enough that skipped events pass through the rings many times, and
launches that mix Z2-symmetric and general states."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rg():
    import rcmps_gpu
    return rcmps_gpu


@pytest.mark.parametrize("d,scaling", [(1, 0.3), (2, 0.5), (15, 0.2), (17, 0.2), (32, 0.2), (33, 0.15)])
def test_sizes_at_tile_edges_match_oracle(rg, d, scaling):
    """Energy, gradient and step sequences at the bars of the FP64 path (1e-12, 1e-10, equal steps)."""
    print(f"case: D={d}", flush=True)
    r, k = rg.random_state_arrays(d, scaling=scaling, seed=100 + d)
    s = rg.State(r, k)
    s.integrator_param.n_quad = 16
    e, g, st = rg.fg_phi4(s, 1.5, return_stats=True)
    ref = oracle.fg_phi4(s.R, s.Q, s.rho, 1.5, n_quad=16)
    assert abs(e - ref["energy"]) <= 1e-12 * max(1.0, abs(ref["energy"]))
    assert np.abs(g - ref["gradient"]).max() <= 1e-10 * max(1.0, np.abs(ref["gradient"]).max())
    assert list(st["accepted"]) == list(ref["stats"][:, 0])
    assert list(st["rejected"]) == list(ref["stats"][:, 1])
    # twelve right-hand sides an attempt... the FSAL one after acceptance, three for the dense output
    rhs = [1 + 11 * a + acc + 3 * dn for a, acc, dn in zip(st["attempts"], st["accepted"], st["dense_steps"])]
    assert list(st["rhs_calls"]) == rhs


@pytest.mark.parametrize("precision", ["fp64", "split"])
def test_mixed_z2_and_general_states_in_one_launch(rg, precision):
    """A launch skips the zero parity blocks only when all its states have them; the results are the
    single calls' bits either way."""
    states = []
    for d, z2, seed in [(32, True, 1), (32, False, 2), (31, False, 3), (64, True, 4), (64, True, 5)]:
        print(f"case: D={d} z2={z2}", flush=True)
        make = rg.random_state_z2_arrays if z2 else rg.random_state_arrays
        s = rg.State(*make(d, scaling=0.2, seed=seed))
        s.integrator_param.n_quad = 32
        states.append(s)
    gs = [0.7, 1.3, 2.0, 2.0, 3.1]
    E, G = rg.fg_phi4_batch(states, gs, precision=precision)
    for s, g, e, grad in zip(states, gs, E, G):
        e1, g1 = rg.fg_phi4(s, g, precision=precision)
        assert e == e1
        assert np.array_equal(grad, g1)
