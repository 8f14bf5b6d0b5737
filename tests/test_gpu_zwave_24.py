"""z passes in wave registers at 24 points per lane (96 and 192 points): every
kind of pass they serve, complex64 against the complex128 engine in LDS tiles
(launcher variant bit 0), and complex128 on both sides of the size at which it
takes them, against the tiles; pencil counts that leave a remainder."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


def run(shape, mode, prec, variant):
    n = float(np.prod(shape))
    beta = 1.0 if mode in ("ite", "itev") else 0.0
    inter = E.DIPOLAR if mode == "dipolar" else E.UFG if mode in ("qf", "adjoint") else E.CONTACT
    vext = E.VARRAY if mode == "adjoint" else E.HARMONIC
    g = E.Engine(shape, 1.0 - beta, beta, 0.02, n, inter, vext, 0, prec)
    if variant is not None:
        g.set_variant(variant)
    g.set_user_params([0.05, 0.06, 0.02, 0.02, 0.015])
    rng = np.random.default_rng(7)
    psi = (1 + 0.2 * rng.random(shape)) * np.exp(0.3j * rng.standard_normal(shape))
    if mode == "adjoint":
        g.set_external_potential(0.1 * rng.random(shape))
    g.set_psi(psi)
    if mode == "adjoint":
        g.adjoint_forward(3, psi * np.exp(0.5j * rng.random(shape)))
        out = g.adjoint_backward()
    else:
        g.normalize_psi()
        if mode == "qf":
            g.set_quantum_friction_coeff(0.1)
        if mode == "itev":
            g.set_vortex(0.5, 0.5, 1)
        {"dipolar": g.evolve_dipolar, "itev": g.evolve_vortex}.get(mode, g.evolve_qf)(4)
        out = g.get_psi()[0] * g.energy()[1] if mode == "rte" else g.get_psi()[0]
    g.close()
    return out


MODES = ["rte", "ite", "itev", "qf", "dipolar", "adjoint"]


# four steps of about eight transforms, each ~20 roundings of 2^-24 that add as
# a random walk; the adjoint goes back over three with sums of signed terms
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("shape", [(8, 12, 96), (12, 8, 192)])
def test_complex64_follows_complex128_tiles(shape, mode):
    print("[gpu-case] 24 points per lane", shape, mode, flush=True)
    a, b = run(shape, mode, E.C64, None), run(shape, mode, E.C128, 1)
    assert np.linalg.norm(a - b) < (1e-5 if mode == "adjoint" else 2e-6) * np.linalg.norm(b)


# 64 pencils of 96 or 32 of 192 points per workgroup: 128 workgroups take the tiles on 256 CUs, 144 the waves
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("shape", [(128, 64, 96), (96, 96, 96), (64, 64, 192), (96, 48, 192)])
def test_complex128_waves_equal_tiles(shape, mode):
    print("[gpu-case] 24 points per lane, complex128", shape, mode, flush=True)
    a, b = run(shape, mode, E.C128, 0), run(shape, mode, E.C128, 1)
    assert np.linalg.norm(a - b) < (1e-10 if mode == "adjoint" else 1e-13) * np.linalg.norm(b)
