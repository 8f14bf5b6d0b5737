"""Runs of small lattices in one kernel on one XCD (gpe_xcd.hpp): bit for bit
the passes they stand for (the launcher variant a new engine of that size would
otherwise take, set by hand), at the edges of the sizes that take them, over
launches of up to 256 steps, with several engines at once, and under capture."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402

RTE, ITE = (1.0, 0.0), (0.0, 1.0)


def engine(shape, ab, prec, passes=False, inter=E.CONTACT, vext=E.COSINE, seed=3):
    n = float(np.prod(shape))
    g = E.Engine(shape, ab[0], ab[1], 0.02, n, inter, vext, 0, prec)
    if passes:  # half-width strided tiles, and planes where ny = nz = 32 or 48
        g.set_variant(34 if shape[1] == shape[2] and shape[1] in (32, 48) else 2)
    g.set_user_params([0.1, 2.0, 0.3, 0.02] if vext == E.COSINE else [0.05, 0.06, 0.07, 0.02])
    rng = np.random.default_rng(seed)
    g.set_psi((1 + 0.2 * rng.random(shape)) * np.exp(0.4j * rng.standard_normal(shape)))
    g.normalize_psi()
    return g


@pytest.mark.parametrize("prec", [E.C64, E.C128])
@pytest.mark.parametrize("ab", [RTE, ITE, (0.6, 0.3)])
@pytest.mark.parametrize("shape", [(8, 8, 8), (12, 24, 48), (16, 16, 16), (64, 8, 12), (8, 64, 64), (48, 16, 8),
                                   (24, 32, 32), (32, 32, 32), (48, 12, 64)])
def test_runs_equal_the_passes(shape, ab, prec):
    print("[gpu-case] xcd", shape, ab, prec, flush=True)
    a, b = engine(shape, ab, prec), engine(shape, ab, prec, passes=True)
    for nt in (1, 2, 7):
        mu = [g.evolve_qf(nt, want_mu=ab[1] != 0.0) for g in (a, b)]
        assert np.array_equal(a.get_psi()[0], b.get_psi()[0]), nt
        assert mu[0] == mu[1]
    assert a.energy() == b.energy() and a.get_norm() == b.get_norm()


@pytest.mark.parametrize("inter,vext", [(E.UFG, E.HARMONIC), (E.ETF, E.HARMONIC), (E.CONTACT, E.WOODS_SAXON),
                                        (E.CONTACT, E.VARRAY)])
@pytest.mark.parametrize("ab", [RTE, ITE])
def test_every_built_in_physics(inter, vext, ab):
    shape = (16, 24, 8)
    out = []
    for passes in (False, True):
        g = engine(shape, ab, E.C128, passes, inter, vext)
        if vext == E.VARRAY:
            g.set_external_potential(np.random.default_rng(1).random(shape))
        g.evolve_qf(5)
        out.append(g.get_psi()[0])
    assert np.array_equal(out[0], out[1])


def test_long_runs_are_several_launches():
    a, b = engine((8, 12, 16), RTE, E.C64), engine((8, 12, 16), RTE, E.C64, passes=True)
    for nt in (256, 257, 600):
        a.evolve_qf(nt)
        b.evolve_qf(nt)
        assert np.array_equal(a.get_psi()[0], b.get_psi()[0]), nt


def test_runs_not_covered_take_the_passes():
    """Pinning, friction, imaginary after real time, and back."""
    for setup in (lambda g: g.set_vortex(0.5, 0.5, 1), lambda g: g.set_quantum_friction_coeff(0.2)):
        out = []
        for passes in (False, True):
            g = engine((16, 12, 24), RTE, E.C128, passes)
            g.evolve_qf(3)
            setup(g)
            g.evolve_vortex(2) if setup.__code__.co_names[0] == "set_vortex" else g.evolve_qf(2)
            g.set_quantum_friction_coeff(0.0)
            g.set_ite_evolution()
            g.evolve_qf(4)
            g.set_rte_evolution()
            g.evolve_qf(3)
            out.append(g.get_psi()[0])
        assert np.array_equal(out[0], out[1])


def test_many_engines_at_once():
    """More engines than XCDs, their runs in flight together beside a large one's passes."""
    big = engine((128, 64, 64), RTE, E.C64)
    small = [engine((16, 24, 32), RTE, E.C64, seed=s) for s in range(11)]
    ref = [engine((16, 24, 32), RTE, E.C64, passes=True, seed=s) for s in range(11)]
    for _ in range(3):
        big.evolve_qf(20)
        for g in small:
            g.evolve_qf(30)
    for g in ref:
        g.evolve_qf(90)
    for g, r in zip(small, ref):
        assert np.array_equal(g.get_psi()[0], r.get_psi()[0])


def test_captured_runs_replay():
    """A run captured on the engine's stream is the passes, which replay."""
    a, b = engine((16, 16, 24), RTE, E.C64), engine((16, 16, 24), RTE, E.C64, passes=True)
    a.evolve_qf(2)  # a run on one XCD before the capture
    hip = E.lib()
    stream, graph, ex = ctypes.c_void_p(a.stream()), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    a.evolve_qf(3)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    b.evolve_qf(2)
    for _ in range(3):
        assert hip.hipGraphLaunch(ex, stream) == 0
        a.synchronize()
        b.evolve_qf(3)
        assert np.array_equal(a.get_psi()[0], b.get_psi()[0])
    a.evolve_qf(4)
    b.evolve_qf(4)
    assert np.array_equal(a.get_psi()[0], b.get_psi()[0])
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


def test_autotuned_engine_keeps_its_results():
    a, b = engine((16, 24, 32), RTE, E.C128), engine((16, 24, 32), RTE, E.C128, passes=True)
    a.autotune(3)
    a.evolve_qf(10)
    b.evolve_qf(10)
    pa, pb = a.get_psi()[0], b.get_psi()[0]
    assert np.max(np.abs(pa - pb)) < 1e-13 * np.max(np.abs(pb))  # ten steps of rotations, rounded differently
