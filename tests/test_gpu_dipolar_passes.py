"""The dipolar step whose density and potential ride on the z passes
(evolve_dipolar_t): lengths and launcher variants whose z passes run in wave
registers and in LDS tiles, pencils that leave a remainder, and the user
hooks' potential, against the FP64 oracle; and the merged half steps of a
real-time block against one step per call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


def state(shape, seed):
    rng = np.random.default_rng(seed)
    return (1.0 + 0.2 * rng.random(shape)) * np.exp(0.4j * rng.standard_normal(shape))


def pair(oracle, shape, beta, vext, variant, prec):
    n = float(np.prod(shape))
    args = (shape, 1.0 - beta, beta, 0.02, 0.1 * n, E.DIPOLAR, vext, 0)
    g, o = E.Engine(*args, prec), oracle.OracleEngine(*args)
    g.set_variant(variant)
    for x in (g, o):
        # trap, a_con, a_dip (the hook potential reads the slots 4, 5 and 9: modulation and ramp)
        x.set_user_params([0.05, 0.06, 0.08, 0.03, 0.02, 1.7, 0.0, 0.0, 0.0, 0.05])
        x.set_psi(state(shape, 5), t=0.25)
        x.normalize_psi()
    return g, o


def rel_err(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("vext", [E.HARMONIC, E.WOODS_SAXON, E.USER])
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("shape,variant", [((8, 12, 96), 0), ((12, 8, 16), 1), ((12, 8, 16), 8), ((8, 8, 512), 0),
                                           ((24, 16, 8), 2)])
def test_dipolar_passes_match_oracle(oracle, shape, variant, beta, vext):
    print("[gpu-case] dipolar passes", shape, variant, beta, vext, flush=True)
    if vext == E.WOODS_SAXON and shape != (12, 8, 16):
        pytest.skip("the potential kind is covered by one shape")
    g, o = pair(oracle, shape, beta, vext, variant, E.C128)
    for nt in (1, 3):
        mg, mo = g.evolve_dipolar(nt, want_mu=True), o.evolve_dipolar(nt, want_mu=True)
        assert rel_err(g.get_psi()[0], o.get_psi()[0]) < 1e-12
        if beta:
            assert abs(mg - mo) < 1e-12 * abs(mo)
    for method in (1, 2):
        assert abs(g.energy_dipolar(method)[1] - o.energy_dipolar(method)[1]) < 1e-12 * abs(o.energy_dipolar(method)[1])
    g.close()


# a step is ~60 roundings of each amplitude, in steps that are rotations
@pytest.mark.parametrize("prec,tol", [(E.C128, 1e-13), (E.C64, 2e-5)])
def test_a_block_of_steps_is_its_single_steps(oracle, prec, tol):
    out = []
    for blocks in ([6], [1] * 6):
        g, o = pair(oracle, (16, 12, 24), 0.0, E.HARMONIC, 0, prec)
        for nt in blocks:
            g.evolve_dipolar(nt)
        out.append(g.get_psi()[0])
        g.close()
    assert rel_err(out[0], out[1]) < tol
