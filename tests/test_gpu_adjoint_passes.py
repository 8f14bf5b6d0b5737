"""The adjoint's backward step on the z passes (gpe_adjoint.hpp): z lengths in
wave registers and in LDS tiles, pencil counts that leave a remainder, plane
and unsplit plans, segments with remainders, every interaction the adjoint
takes, against the FP64 oracle; and the run whose predictor ends do not fit
in memory."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from libcugpe_amd import engine as E  # noqa: E402


def inputs(shape, seed=4):
    rng = np.random.default_rng(seed)
    v = 0.2 * rng.random(shape)
    psi0 = (1 + 0.2 * rng.random(shape)) * np.exp(1j * rng.uniform(-0.5, 0.5, shape))
    psit = (1 + 0.2 * rng.random(shape)) * np.exp(1j * rng.uniform(-0.5, 0.5, shape))
    return v, psi0, psit


def engine(shape, inter, v, psi0, prec=E.C128, variant=None):
    g = E.Engine(shape, 1.0, 0.0, 0.05, 50.0, inter, E.VARRAY, 0, prec)
    if variant is not None:
        g.set_variant(variant)
    g.set_user_params([0.0, 0.0, 0.0, 0.05])
    g.set_external_potential(v)
    g.set_psi(psi0)
    return g


# the bounds of the oracle comparison of test_gpu_adjoint.py
@pytest.mark.parametrize("shape,variant,inter,nt,ckpt", [
    ((8, 12, 8), 0, E.UFG, 7, 3), ((8, 12, 8), 1, E.CONTACT, 7, 3), ((12, 8, 96), 0, E.UFG, 3, 0),
    ((8, 8, 512), 0, E.CONTACT, 2, 1), ((8, 32, 32), 32, E.UFG, 5, 2), ((16, 16, 16), 16, E.CONTACT, 4, 4),
    ((24, 8, 12), 8, E.UFG, 5, 9), ((16, 8, 24), 2, E.DIPOLAR, 4, 2), ((8, 24, 48), 0, E.UFG, 1, 0)])
def test_backward_passes_match_oracle(oracle, shape, variant, inter, nt, ckpt):
    print("[gpu-case] adjoint passes", shape, variant, inter, nt, ckpt, flush=True)
    v, psi0, psit = inputs(shape)
    g = engine(shape, inter, v, psi0, variant=variant)
    lg = g.adjoint_forward(nt, psit, ckpt)
    gg = g.adjoint_backward()
    o = oracle.OracleEngine(shape, 1.0, 0.0, 0.05, 50.0, inter, 3, 0)
    o.set_user_params([0.0, 0.0, 0.0, 0.05])
    o.set_vext_array(v)
    o.set_psi(psi0)
    lo, go = o.adjoint_overlap(nt, psit, ckpt)
    assert abs(lg - lo) < 1e-12
    assert np.max(np.abs(gg - go)) < 1e-10 * np.max(np.abs(go))
    pg, po = g.get_psi()[0], o.get_psi()[0]
    assert np.max(np.abs(pg - po)) < 1e-12 * np.max(np.abs(po))
    # a second gradient of the same engine, after its kinetic factors changed
    # and changed back, is the same one
    g.change_alpha_beta(0.5, 0.0)
    g.set_psi(psi0)
    g.adjoint_forward(nt, psit, ckpt)
    g.change_alpha_beta(1.0, 0.0)
    g.set_psi(psi0)
    g.adjoint_forward(nt, psit, ckpt)
    assert np.array_equal(g.adjoint_backward(), gg)
    g.close()
    o.close()


def test_predictor_ends_that_do_not_fit_are_computed_again():
    shape, nt = (128, 128, 128), 100
    v, psi0, psit = inputs(shape)
    state = 16 * 128 ** 3
    g = engine(shape, E.UFG, v, psi0)
    l0 = g.adjoint_forward(nt, psit, nt)
    g0 = g.adjoint_backward()
    g.close()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # room for the segment's states (101) and the engine's arrays (about 20
    # states), not for 100 predictor ends beside them
    g = engine(shape, E.UFG, v, psi0)
    free, _ = torch.cuda.mem_get_info()
    block = torch.empty(free - (101 + 20 + 60) * state, dtype=torch.uint8, device="cuda")
    l1 = g.adjoint_forward(nt, psit, nt)
    g1 = g.adjoint_backward()
    g.close()
    del block
    torch.cuda.empty_cache()
    assert abs(l1 - l0) < 1e-12
    assert np.max(np.abs(g1 - g0)) < 1e-10 * np.max(np.abs(g0))
