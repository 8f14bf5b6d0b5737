"""Vortex detection at the ends of its runs along x: lengths of 8 (one run), 12
(a run of 8 and a rest of 4) and more, with runs of 1 (small lattices) and 8, against the oracle bit for bit, and the
count alone, which takes no array."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


def state(shape, seed):
    """vortex lines along x, y and z, with noise that adds windings of both signs"""
    x, y, z = np.meshgrid(*[np.arange(n) for n in shape], indexing="ij")
    nx, ny, nz = shape
    a = ((x - 0.3 * nx) + 1j * (y - 0.6 * ny)) / nx
    b = ((y - 0.25 * ny) - 1j * (z - 0.55 * nz)) / ny
    c = ((z - 0.7 * nz) + 1j * (x - 0.8 * nx)) / nz
    rng = np.random.default_rng(seed)
    return a * b * c + 0.02 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))


@pytest.mark.parametrize("prec", [E.C128, E.C64])
@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 24, 16), (12, 8, 16), (12, 12, 12), (12, 64, 48), (16, 12, 8),
                                   (24, 16, 12), (48, 8, 8), (8, 512, 512), (12, 256, 512)])
def test_windings_and_count(oracle, shape, prec):
    print("[gpu-case] windings", shape, prec, flush=True)
    psi = state(shape, 5)
    if prec == E.C64:
        psi = psi.astype(np.complex64).astype(np.complex128)
    g = E.Engine(shape, 1.0, 0.0, 0.01, 100.0, precision=prec)
    g.set_psi(psi)
    ref = psi.astype(np.complex64) if prec == E.C64 else psi
    for rho_min in (0.0, 1e-3, 0.05):
        # the count alone first: no array has been made for the engine yet
        _, alone = g.detect_vortices(rho_min, False)
        w, count = g.detect_vortices(rho_min)
        wo, want = oracle.plaquette_windings(ref, rho_min)
        assert np.array_equal(w, wo)
        assert count == want == alone == np.count_nonzero(wo)
        assert want > 0 or rho_min > 0
    g.close()
