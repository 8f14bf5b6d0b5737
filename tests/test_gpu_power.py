"""The 2/3 power of the unitary gas over the range of densities (pow23): a
uniform state keeps its density, so one real-time step multiplies it by
exp(-2 i dt V) (gamma = 2) with V = 0.37 (3 pi^2 rho)^(2/3) / 2, rho = 2 |psi|^2
(orginal/gpe_user_defined.h:104-112), exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


# tolerances: about a dozen roundings of the two transforms and the phase
# factors (2^-53 and 2^-24 each), V entering with a phase of 0.4
@pytest.mark.parametrize("prec,amps,tol", [(E.C128, [1e-150, 1e-60, 1e-15, 0.03, 1.0, 7.0, 1e5, 1e100], 4e-15),
                                           (E.C64, [1e-15, 1e-6, 0.03, 1.0, 7.0, 1e5, 1e15], 2e-6)])
def test_uniform_unitary_gas_phase(prec, amps, tol):
    shape = (8, 8, 8)
    for amp in amps:
        print("[gpu-case] unitary gas", prec, amp, flush=True)
        a = float(np.float32(amp)) if prec == E.C64 else amp
        v = 0.37 * np.cbrt(3 * np.pi ** 2 * 2 * a * a) ** 2 / 2.0  # (a power of the rounded 2/3 is 1e-14 off here)
        g = E.Engine(shape, 1.0, 0.0, 0.2 / v, 1.0, E.UFG, E.HARMONIC, 0, prec)
        g.set_psi(np.full(shape, a, dtype=np.complex128))
        g.evolve_qf(1)
        psi, _ = g.get_psi()
        g.close()
        assert np.max(np.abs(psi / a - np.exp(-0.4j))) < tol, amp


@pytest.mark.parametrize("prec", [E.C128, E.C64])
def test_empty_lattice_stays_empty(prec):
    g = E.Engine((8, 8, 8), 1.0, 0.0, 0.1, 1.0, E.UFG, E.HARMONIC, 0, prec)
    g.set_user_params([0.3, 0.3, 0.3])
    g.set_psi(np.zeros((8, 8, 8), dtype=np.complex128))
    g.evolve_qf(2)
    psi, _ = g.get_psi()
    g.close()
    assert np.all(psi == 0)
