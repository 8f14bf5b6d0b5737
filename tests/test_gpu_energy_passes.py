"""The energy's passes (energy_t: one z pass that rescales, sums the potential
and interaction energies and the z part of the kinetic one, and a read-only y
and x pass) against plain numpy: every compiled length on each axis, tiles with
a remainder, z passes in wave registers and in LDS tiles, real and imaginary
time, both precisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402

SHAPES = [(8, 12, 16), (12, 8, 24), (16, 24, 32), (24, 16, 8), (32, 48, 12), (48, 32, 64), (64, 8, 48), (96, 12, 8),
          (12, 96, 96), (128, 8, 16), (8, 128, 12), (192, 8, 12), (8, 192, 192), (256, 8, 8), (8, 256, 8), (8, 8, 256),
          (512, 8, 12), (8, 512, 8), (8, 12, 512), (12, 8, 128)]


def expected(psi, params, npart, rescale):
    n = psi.size
    if rescale:
        psi = psi * np.sqrt(npart / np.sum(np.abs(psi) ** 2))
    rho = np.abs(psi) ** 2
    k = [2 * np.pi * np.fft.fftfreq(m) for m in psi.shape]
    k2 = k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2
    x = [np.arange(m) - m // 2 for m in psi.shape]
    v = sum(0.5 * (a * w) ** 2 for a, w in zip(np.ix_(*x), params))
    return (np.sum(k2 * np.abs(np.fft.fftn(psi)) ** 2) / (2 * n), np.sum(2 * np.pi * params[3] * rho ** 2),
            np.sum(rho * v), psi)


# each sum is of positive terms: a few roundings per term, none of them summed
# up coherently (2^-53 and 2^-24, times about thirty)
@pytest.mark.parametrize("prec,tol", [(E.C128, 4e-15), (E.C64, 2e-6)])
@pytest.mark.parametrize("shape", SHAPES)
def test_energy_of_every_length(shape, prec, tol):
    rng = np.random.default_rng(sum(shape))
    psi = (1 + 0.3 * rng.random(shape)) * np.exp(1j * rng.standard_normal(shape))
    params = [0.05, 0.06, 0.07, 0.02]
    npart = 0.7 * psi.size
    for beta, variant in ((0.0, None), (1.0, None), (0.0, 1)):
        print("[gpu-case] energy", shape, prec, beta, variant, flush=True)
        g = E.Engine(shape, 1.0 - beta, beta, 0.01, npart, E.CONTACT, E.HARMONIC, 0, prec)
        if variant is not None:
            g.set_variant(variant)
        g.set_user_params(params)
        g.set_psi(psi)
        _, ek, ei, ee = g.energy()
        got, _ = g.get_psi()
        g.close()
        wk, wi, we, want = expected(psi, params, npart, beta == 0.0)
        assert abs(ek - wk) < tol * wk and abs(ei - wi) < tol * wi and abs(ee - we) < tol * we
        assert np.max(np.abs(got - want)) < tol * np.max(np.abs(want))
