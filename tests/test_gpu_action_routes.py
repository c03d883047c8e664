"""The persistent action ODE against the launch graphs where its instantiations and its grid change: one
tile per matrix, three tiles (D = 40), Z2 states of four tiles (half the workgroups, half the k-tiles),
more workgroups than CUs, and a call too large for the persistent launch.  The two routes add in the
same order, so they give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rg():
    import rcmps_gpu
    return rcmps_gpu


@pytest.mark.parametrize("d,z2,ntan", [(2, False, 1), (13, False, 20), (32, True, 1), (31, False, 8), (40, False, 1),
                                       (64, True, 1), (64, False, 1)])
def test_routes_give_the_same_bits(rg, d, z2, ntan):
    print(f"case: D={d} z2={z2} tangents={ntan}", flush=True)
    from rcmps_gpu.excitation import action_batch
    make = rg.random_state_z2_arrays if z2 else rg.random_state_arrays
    s = rg.State(*make(d, scaling=0.2, seed=d))
    s.integrator_param = rg.IntegratorParameters(n_quad=12, max_point=20.0, atol=1e-11, rtol=1e-10)
    model = rg.ExcitationModel("phi4", 1.5)
    ctxs = [rg.ExcitationContext(s, 0.2 * i, dense_transfer=d <= 16) for i in range(ntan)]
    rng = np.random.default_rng(d)
    ws = []
    for _ in range(ntan):
        w = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
        if z2:
            w[:d // 2, :d // 2] = 0
            w[d // 2:, d // 2:] = 0
        ws.append(w)
    out = {}
    for persistent in (True, False, None):
        out[persistent], st = action_batch(ctxs, ws, model, 8, parts=2, return_stats=True, persistent=persistent)
        if persistent is not False and not (d == 64 and not z2):
            assert st["phase_us"][4][3] > 0   # the persistent launch ran, and is the default
    for p in (True, None):
        for x, y in zip(out[p], out[False]):
            assert np.isfinite(x).all()
            assert np.array_equal(x, y)


def test_z2_samples_of_the_other_parity_are_zero(rg):
    """A Z2 state's tiles of the other parity have no workgroup in the persistent launch; their samples
    must be zero whatever the memory held, here the samples of a general state of the same size."""
    from rcmps_gpu.excitation import action_batch
    d = 32
    out = {}
    for persistent in (True, False):
        for z2 in (False, True):
            make = rg.random_state_z2_arrays if z2 else rg.random_state_arrays
            s = rg.State(*make(d, scaling=0.2, seed=d))
            s.integrator_param = rg.IntegratorParameters(n_quad=12, max_point=20.0, atol=1e-11, rtol=1e-10)
            w = np.random.default_rng(1).standard_normal((d, d)).astype(complex)
            if z2:
                w[:d // 2, :d // 2] = 0
                w[d // 2:, d // 2:] = 0
            ctx = rg.ExcitationContext(s, 0.3, dense_transfer=False)
            (f,) = action_batch(ctx, [w], rg.ExcitationModel("phi4", 1.5), 8, parts=2, persistent=persistent)
            out[persistent, z2] = f
            ctx.close()
            s.close()
    assert np.array_equal(out[True, True], out[False, True])
    assert np.array_equal(out[True, False], out[False, False])
