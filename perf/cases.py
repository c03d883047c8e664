"""The calls a user of rcmps_gpu makes, over the sizes and options they are made with, as cases that
can be timed one by one.

listed() gives named cases, draw(rng) another one of the same ranges, prepare(case, seed) what a
program holds before the call (states, momentum contexts, tangents), run(state) one pass through the
public entry points, work(case) the bytes and operations such a pass cannot do without, and
exact(case, seed) the same outputs from dense linear algebra and a fixed-step integration written
here, where that is quick enough.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rcmpscore.jl_amd")
if os.path.isdir(os.path.join(os.getcwd(), "rcmpscore.jl_amd")):
    _PKG = os.path.join(os.getcwd(), "rcmpscore.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import rcmps_gpu  # noqa: E402

SCALING = 0.2   # entries of R and K: iid complex normal times 0.2, the distribution of the benchmark states
DIMS = (8, 16, 24, 32, 48, 64)


def listed():
    return [
        # The boundary Poisson solve alone, on a small state: the shortest call the package has (a few
        # dozen Krylov steps of tiny products, all launches and latency).
        dict(name="boundary_d5", kind="boundary", D=5),
        # The default evaluation at the size first calculations are made with (128 nodes per half,
        # window 20, 1e-11/1e-10).
        dict(name="eval_d8", kind="eval", D=8, z2=False, g=2.0, n_quad=128, window=20.0, atol=1e-11, rtol=1e-10,
             precision="fp64", kinetic="ode"),
        # State(R, K): what every optimizer trial pays before it can evaluate (stationary density and
        # spectral data of Q).
        dict(name="state_d64", kind="state", D=64),
        # A Z2-symmetric ground-state evaluation, the symmetric states excitations are built on.
        dict(name="eval_d32_z2", kind="eval", D=32, z2=True, g=2.0, n_quad=256, window=20.0, atol=1e-11, rtol=1e-10,
             precision="fp64", kinetic="ode"),
        # The headline evaluation: D = 64, split precision.
        dict(name="eval_d64_split", kind="eval", D=64, z2=False, g=2.0, n_quad=256, window=20.0, atol=1e-11,
             rtol=1e-10, precision="split", kinetic="ode"),
        # A converged optimization's last evaluations: FP64 at the tight settings (window 30, 1e-13/1e-12).
        dict(name="eval_d64_tight", kind="eval", D=64, z2=False, g=2.0, n_quad=256, window=30.0, atol=1e-13,
             rtol=1e-12, precision="fp64", kinetic="ode"),
        # The infinite-line kinetic terms by Krylov bases, at a size that is no multiple of the tiles.
        dict(name="eval_d40_krylov", kind="eval", D=40, z2=False, g=2.0, n_quad=128, window=20.0, atol=1e-11,
             rtol=1e-10, precision="fp64", kinetic="krylov"),
        # One gradient step of a torch program: energy of (R, K) forward and backward, odd size.
        dict(name="grad_d27", kind="grad", D=27, g=1.0, n_quad=128),
        # A sweep over couplings and bond dimensions in one call, ragged sizes among them.
        dict(name="batch_48", kind="batch", count=48, mix=0, n_quad=128, precision="fp64"),
        # One excitation Hamiltonian action on a small symmetric state, as a Davidson search makes it.
        dict(name="action_d16", kind="action", D=16, z2=True, count=1, g=2.0, nodes=256, n_quad=128),
        # One round of a dispersion: nine momenta in lockstep on a D = 32 state.
        dict(name="dispersion_d32", kind="action", D=32, z2=True, count=9, g=2.0, nodes=256, n_quad=128),
        # The largest excitation action.
        dict(name="action_d64", kind="action", D=64, z2=True, count=1, g=2.7, nodes=128, n_quad=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["boundary", "eval", "eval", "eval", "state", "grad", "batch", "action", "action"])
    if kind in ("boundary", "state"):
        return dict(kind=kind, D=_log(rng, 3, 64))
    if kind == "eval":
        D, z2 = _log(rng, 4, 64), rng.random() < 0.25
        tight = rng.random() < 0.2
        return dict(kind=kind, D=D + D % 2 if z2 else D, z2=z2, g=rng.uniform(0.5, 4.0), n_quad=_log(rng, 64, 256),
                    window=30.0 if tight else 20.0, atol=1e-13 if tight else 1e-11, rtol=1e-12 if tight else 1e-10,
                    precision="fp64" if tight else rng.choice(["fp64", "fp64", "split"]),
                    kinetic=rng.choice(["ode", "ode", "ode", "krylov"]))
    if kind == "grad":
        return dict(kind=kind, D=_log(rng, 4, 64), g=rng.uniform(0.5, 4.0), n_quad=_log(rng, 64, 256))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(2, 40), mix=rng.randint(1, 10**6), n_quad=128,
                    precision=rng.choice(["fp64", "fp64", "split"]))
    D = 2 * _log(rng, 4, 32)
    return dict(kind="action", D=D, z2=rng.random() < 0.7, count=rng.randint(1, 9) if D <= 32 else 1,
                g=rng.uniform(0.5, 3.0), nodes=rng.choice([64, 128]), n_quad=_log(rng, 48, 128))


def _arrays(D, z2, seed):
    make = rcmps_gpu.random_state_z2_arrays if z2 else rcmps_gpu.random_state_arrays
    return make(D, scaling=SCALING, seed=seed)


def _batch(case, seed):
    """(dims, couplings, seeds): the sizes are the case's, the matrices and couplings the seed's."""
    pick = np.random.default_rng(case["mix"])
    dims = [int(d) for d in pick.choice(DIMS, size=case["count"])]
    dims = [d - int(pick.integers(1, 6)) if pick.random() < 0.25 else d for d in dims]
    rng = np.random.default_rng(seed)
    return dims, rng.uniform(0.5, 4.0, size=len(dims)), rng.integers(0, 2**31, size=len(dims))


def _integrator(case):
    return rcmps_gpu.IntegratorParameters(n_quad=case["n_quad"], max_point=case.get("window", 20.0),
                                          atol=case.get("atol", 1e-11), rtol=case.get("rtol", 1e-10))


def _tangents(case, seed):
    rng = np.random.default_rng([seed, 1])
    D = case["D"]
    ws = []
    for _ in range(case["count"]):
        w = rng.standard_normal((D, D)) + 1j * rng.standard_normal((D, D))
        if case["z2"]:   # the odd sector
            w[:D // 2, :D // 2] = 0
            w[D // 2:, D // 2:] = 0
        ws.append(w / np.linalg.norm(w))
    return ws


def _source_matrix(D, seed):
    a = np.random.default_rng([seed, 2]).standard_normal((2, D, D))
    a = a[0] + 1j * a[1]
    return (a + a.conj().T) / 2


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        dims, gs, seeds = _batch(case, seed)
        states = [rcmps_gpu.State(*_arrays(d, False, int(x)), integrator_param=_integrator(case))
                  for d, x in zip(dims, seeds)]
        return dict(case=case, states=states, gs=gs)
    R, K = _arrays(case["D"], case.get("z2", False), seed)
    if kind == "state":
        return dict(case=case, R=R, K=K)
    if kind == "grad":
        return dict(case=case, R=torch.from_numpy(R).cuda(), K=torch.from_numpy(K).cuda(), ip=_integrator(case))
    s = rcmps_gpu.State(R, K)
    if kind == "boundary":
        return dict(case=case, s=s, a=_source_matrix(case["D"], seed))
    s.integrator_param = _integrator(case)
    if kind == "eval":
        return dict(case=case, s=s)
    model = rcmps_gpu.ExcitationModel("phi4", case["g"])
    ctxs = [rcmps_gpu.ExcitationContext(s, 0.1 + 0.25 * i) for i in range(case["count"])]
    return dict(case=case, s=s, model=model, ctxs=ctxs, ws=_tangents(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "boundary":
        return [rcmps_gpu.boundary_environment(state["s"], state["a"])]
    if kind == "eval":
        e, grad = rcmps_gpu.fg_phi4(state["s"], case["g"], precision=case["precision"],
                                    kinetic_backend=case["kinetic"])
        return [e, grad]
    if kind == "state":
        s = rcmps_gpu.State(state["R"], state["K"])
        return [s.Q, s.rho]
    if kind == "grad":
        R = state["R"].clone().requires_grad_(True)
        K = state["K"].clone().requires_grad_(True)
        e = rcmps_gpu.phi4_energy(R, K, case["g"], integrator=state["ip"])
        e.backward()
        return [e.detach(), R.grad, K.grad]
    if kind == "batch":
        e, grads = rcmps_gpu.fg_phi4_batch(state["states"], state["gs"], precision=case["precision"])
        return [np.array(e)] + grads
    return rcmps_gpu.excitation_hamiltonian_action(state["ctxs"], state["ws"], model=state["model"],
                                                   kinetic_nodes=case["nodes"])


# --------------------------------------------------------------------------------------------------
# work: each input matrix read and each output written once; the operations of the algorithm (complex
# D x D products of 8 D^3 flops) at the usual number of steps of each integration
# --------------------------------------------------------------------------------------------------
def _eval_flops(D, n_quad, window=20.0, atol=1e-11, kinetic="ode"):
    # attempts of the six trajectories at 1e-11 on the window 20, fifteen right-hand sides each; the
    # products per right-hand side of each trajectory and per node of the pullback
    steps = np.array([118, 187, 147, 239, 120, 216]) * math.sqrt(window / 20.0) * (1e-11 / atol) ** 0.125
    products = np.array([4, 8, 4, 9, 12, 16])
    if kinetic == "krylov":
        return 8.0 * D**3 * (15 * float(steps[4:] @ products[4:]) + 2 * n_quad * 12 + 4 * 256 * 4)
    return 8.0 * D**3 * (15 * float(steps @ products) + 2 * n_quad * 21)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        dims, _, _ = _batch(case, 0)
        return dict(bytes=float(sum(16 * 4 * d * d for d in dims)),
                    flops=float(sum(_eval_flops(d, case["n_quad"]) for d in dims)))
    D = case["D"]
    if kind == "boundary":   # about 40 preconditioned Krylov steps of 8 products
        return dict(bytes=16.0 * 5 * D * D, flops=8.0 * D**3 * 8 * 40)
    if kind == "state":      # the eigenvectors of Q (about 40 D^3 complex operations) and 40 Krylov steps
        return dict(bytes=16.0 * 4 * D * D, flops=8.0 * D**3 * (40 + 8 * 40))
    if kind == "eval":
        return dict(bytes=16.0 * 4 * D * D,
                    flops=_eval_flops(D, case["n_quad"], case["window"], case["atol"], case["kinetic"]))
    if kind == "grad":
        return dict(bytes=16.0 * 4 * D * D, flops=_eval_flops(D, case["n_quad"]) + 8.0 * D**3 * 360)
    # actions: steps stop at every node; 17 products per right-hand side shared by the tangents, 27 for each
    n, rhs = case["count"], 12 * (2 * case["n_quad"] + 150)
    return dict(bytes=16.0 * (3 + 2 * n) * D * D, flops=8.0 * D**3 * (rhs * (17 + 27 * n) + case["nodes"] * 24 * n))


# --------------------------------------------------------------------------------------------------
# exact: dense 64-bit linear algebra, and a fixed-step integration with Richardson extrapolation
# differentiated by torch
# --------------------------------------------------------------------------------------------------
def _canonical_q(R, K):
    return -1j * (K + K.conj().T) / 2 - R.conj().T @ R / 2


def _transfer(R, Q):
    eye = np.eye(len(R))
    return np.kron(Q, eye) + np.kron(eye, Q.conj()) + np.kron(R, R.conj())


def _rho(R, Q):
    """Stationary density: (-L + |I><I| / D) x = I / D, one step of iterative refinement."""
    D = len(R)
    eye = np.eye(D).reshape(-1)
    A = -_transfer(R, Q) + np.outer(eye, eye) / D
    b = (eye / D).astype(complex)
    x = np.linalg.solve(A, np.stack([b], 1))[:, 0]
    rho = x.reshape(D, D)
    rho = (rho + rho.conj().T) / 2
    return rho / np.trace(rho)


def _source(t):
    """2|t| J(t^2), J(x) = K_{1/4}(x) / (2^{9/4} sqrt(pi) Gamma(5/4) x^{1/4}), the Bessel function from its
    integral of exp(-x cosh u) cosh(u / 4) by the trapezoidal rule."""
    a = abs(t)
    if a == 0:
        return 1 / math.sqrt(math.pi)
    x = a * a
    u = np.arange(0, 8000) * 0.0125
    u = u[u < math.log(1600 / x) + 1]
    f = np.exp(-x * np.cosh(u)) * np.cosh(u / 4)
    k = 0.0125 * (f.sum() - f[0] / 2)
    return 2 * a * k / (2**2.25 * math.sqrt(math.pi) * math.gamma(1.25) * x**0.25)


def _energy(R, K, g, window, n):
    """The finite-window energy of State(R, K) by n classical Runge-Kutta steps per half window (torch)."""
    D = R.shape[0]
    K = (K + K.mH) / 2
    Q = -1j * K - R.mH @ R / 2
    eye = torch.eye(D, dtype=torch.complex128)
    L = torch.kron(Q, eye) + torch.kron(eye, Q.conj()) + torch.kron(R, R.conj())
    v = eye.reshape(-1)
    rho = torch.linalg.solve(-L + torch.outer(v, v) / D, v / D).reshape(D, D)
    rho = (rho + rho.mH) / 2
    C = Q @ R - R @ Q
    s2 = math.sqrt(2.0)
    fixed = torch.stack([s2 * R @ rho, s2 * C @ rho, R @ rho + rho @ R.mH])
    Qh, Rh = Q.mH, R.mH
    O = torch.stack([R, C])

    def rhs(X, jac, src):
        d = jac * (Q @ X + X @ Qh + (R @ X) @ Rh)
        Y = R @ X[2:4]
        Y = (Y + X[2:4] @ Rh) * torch.tensor([2.0, 3.0], dtype=torch.float64).reshape(2, 1, 1)
        d = d + src * torch.cat([fixed, Y])
        kin = 2 * s2 * (X[:2] * O.conj()).real.sum()
        quartic = 8 * (R * X[4].mT).real.sum()
        return d, src * (kin + g * quartic)

    a = math.sqrt(window)
    X = torch.zeros((5, D, D), dtype=torch.complex128)
    E = torch.zeros((), dtype=torch.float64)
    h = a / n
    grid = [_source(h * i / 2) for i in range(2 * n + 1)]
    for half in (-1, 1):
        for i in range(n):
            # nodes counted from t = 0 outwards: the first half runs from -a to 0
            at = [2 * n - 2 * i, 2 * n - 2 * i - 1, 2 * n - 2 * i - 2] if half < 0 else [2 * i, 2 * i + 1, 2 * i + 2]
            j = [h * q for q in at]   # jac = 2|t|, t = q h / 2
            s = [grid[q] for q in at]
            k1, e1 = rhs(X, j[0], s[0])
            k2, e2 = rhs(X + h / 2 * k1, j[1], s[1])
            k3, e3 = rhs(X + h / 2 * k2, j[1], s[1])
            k4, e4 = rhs(X + h * k3, j[2], s[2])
            X = X + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
            E = E + h / 6 * (e1 + 2 * e2 + 2 * e3 + e4)
    return E


def _extrapolated(evaluate, n):
    """evaluate(n) -> list of arrays with error a n^-4 + b n^-5 + ...: n, 2n and 4n extrapolated."""
    v = [evaluate(n * k) for k in (1, 2, 4)]
    r = [[(16 * y - x) / 15 for x, y in zip(v[i], v[i + 1])] for i in (0, 1)]
    return [(32 * y - x) / 31 for x, y in zip(*r)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "state":
        R, K = _arrays(case["D"], False, seed)
        Q = _canonical_q(R, K)
        return [Q, _rho(R, Q)]
    if kind == "boundary" and case["D"] <= 48:
        D = case["D"]
        R, K = _arrays(D, False, seed)
        Q, a = _canonical_q(R, K), _source_matrix(D, seed)
        rho, eye = _rho(R, Q), np.eye(D)
        # (-L* + |I><rho|) H = a - tr(rho a) I; L* is the adjoint of L on row-major vectors
        A = -_transfer(R, Q).conj().T + np.outer(eye.reshape(-1), rho.conj().reshape(-1))
        b = a - np.trace(rho @ a) * eye
        return [np.linalg.solve(A, b.reshape(-1, 1)).reshape(D, D)]
    if kind in ("eval", "grad") and case["D"] <= 10 and case.get("kinetic", "ode") == "ode":
        R0, K0 = _arrays(case["D"], case.get("z2", False), seed)
        window = case.get("window", 20.0)
        reg = rcmps_gpu.ManifoldParameters().metric_reg

        def evaluate(n):
            if kind == "grad":
                R = torch.from_numpy(R0).requires_grad_(True)
                K = torch.from_numpy(K0).requires_grad_(True)
                e = _energy(R, K, case["g"], window, n)
                gR, gK = torch.autograd.grad(e, [R, K])
                return [e.detach().numpy(), gR.numpy(), gK.numpy()]
            # horizontal directions W: R + W, K + i (W^+ R - R^+ W) / 2; dE[W] = 2 Re tr(G^+ W (rho + reg))
            W = torch.zeros(R0.shape, dtype=torch.complex128, requires_grad=True)
            R, K = torch.from_numpy(R0), torch.from_numpy(K0)
            e = _energy(R + W, K + 0.5j * (W.mH @ R - R.mH @ W), case["g"], window, n)
            (gW,) = torch.autograd.grad(e, [W])
            rho = _rho(R0, _canonical_q(R0, K0))
            return [e.detach().numpy(), gW.numpy() @ np.linalg.inv(rho + reg * np.eye(len(R0))) / 2]

        e, *grads = _extrapolated(evaluate, 160)
        # the energy as run() returns it: a number, or for the gradient step a tensor
        return [float(e) if kind == "eval" else torch.tensor(float(e), dtype=torch.float64)] + grads
    # evaluations at larger sizes, the Krylov kinetic terms, batches and actions: minutes in dense form
    return None
