"""Imaginary and complex time over more steps than one launch of a run on one
XCD takes: the rescaling and the chemical potential at the launches' ends are
those of the passes, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_xcd import engine  # noqa: E402
from libcugpe_amd import engine as E  # noqa: E402


@pytest.mark.parametrize("prec", [E.C64, E.C128])
@pytest.mark.parametrize("ab", [(0.0, 1.0), (0.6, 0.3)])
def test_several_launches_of_imaginary_time(ab, prec):
    a, b = engine((8, 12, 16), ab, prec), engine((8, 12, 16), ab, prec, passes=True)
    for nt in (256, 257, 520):
        mu = [g.evolve_qf(nt, want_mu=True) for g in (a, b)]
        assert np.array_equal(a.get_psi()[0], b.get_psi()[0]), nt
        assert mu[0] == mu[1], nt
    assert a.get_norm() == b.get_norm()
