"""The complex64 adjoint forms every factor exp(c V), the predictor end and its
mean field in FP64: with a potential so large that an FP32 phase is off by
1e-5 rad, the gradient still follows from the engine's own complex64 states to
the roundings of the transforms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


def gradient_of_states(states, V, dt, a, target):
    """dL/dV of the split step in FP64 with the states at the step boundaries given."""
    shape = V.shape
    c = 0.5 * dt / 1j
    k = [2 * np.pi * np.fft.fftfreq(n) for n in shape]
    K = np.exp(c * (k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2] ** 2))
    kin = lambda p, f: np.fft.ifftn(f * np.fft.fftn(p))  # noqa: E731
    dg = 4 * np.pi * a
    g = lambda p: dg * np.abs(p) ** 2  # noqa: E731
    sens = lambda lam, y: 2 * np.real(np.conj(lam) * y * c)  # noqa: E731
    o = np.sum(np.conj(target) * states[-1])
    lam = -o * target / (np.sum(np.abs(target) ** 2) * np.sum(np.abs(states[0]) ** 2))
    grad = np.zeros(shape)
    for p0, p1 in zip(states[-2::-1], states[:0:-1]):
        V0 = V + g(p0)
        E0 = np.exp(c * V0)
        p3 = kin(p0 * E0, K) * E0
        W = np.exp(c * 0.5 * (V0 + V + g(p3)))
        vb1 = sens(lam, p1)
        lam = kin(np.conj(W) * lam, np.conj(K))
        vb1 += sens(lam, p0 * W)
        lam0 = np.conj(W) * lam
        grad += 0.5 * vb1
        l3 = 0.5 * vb1 * dg * p3
        vb0 = 0.5 * vb1 + sens(l3, p3)
        lam = kin(np.conj(E0) * l3, np.conj(K))
        vb0 += sens(lam, p0 * E0)
        grad += vb0
        lam = lam0 + np.conj(E0) * lam + dg * vb0 * p0
    return grad


# Two steps of three kinetic factors (six transforms of about 20 roundings of
# 2^-24 that add as a random walk) on states and an adjoint state kept in FP32:
# below 2e-6 as in the complex64 tests of the passes.  An FP32 phase c V = 250
# is off by up to half an ulp, 7.6e-6, and V itself by as much again.
@pytest.mark.parametrize("shape,variant", [((16, 16, 16), None), ((8, 12, 96), None), ((16, 32, 32), 32),
                                           ((12, 16, 24), 1)])
def test_large_phases_are_formed_in_fp64(shape, variant):
    print("[gpu-case] adjoint precision", shape, variant, flush=True)
    dt, a, nt = 0.05, 2.0, 2
    rng = np.random.default_rng(6)
    x = [2 * np.pi * np.arange(n) / n for n in shape]
    wave = sum(np.cos(v + p).reshape([-1 if i == j else 1 for j in range(3)]) for i, (v, p) in
               enumerate(zip(x, (0.3, 1.1, 2.0))))
    V = (1.0e4 + 10.0 * wave + rng.random(shape)).astype(np.float32).astype(np.float64)
    psi = ((1 + 0.1 * rng.random(shape)) * np.exp(1j * wave)).astype(np.complex64).astype(np.complex128)
    tgt = ((1 + 0.1 * rng.random(shape)) * np.exp(0.5j * wave)).astype(np.complex64).astype(np.complex128)

    def engine():
        g = E.Engine(shape, 1.0, 0.0, dt, 1.0, E.CONTACT, E.VARRAY, 0, E.C64)
        g.set_variant(0 if variant is None else variant)
        g.set_user_params([0.0, 0.0, 0.0, a])
        g.set_external_potential(V)
        g.set_psi(psi)
        return g

    g = engine()
    states = [g.get_psi()[0]]
    for _ in range(nt):
        g.evolve_qf(1)
        states.append(g.get_psi()[0])
    g.close()
    g = engine()
    g.adjoint_forward(nt, tgt)
    got = g.adjoint_backward()
    assert np.array_equal(g.get_psi()[0], states[-1])
    g.close()
    ref = gradient_of_states(states, V, dt, a, tgt)
    assert np.linalg.norm(got - ref) < 2e-6 * np.linalg.norm(ref)
