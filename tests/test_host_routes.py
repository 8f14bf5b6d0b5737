"""Which kernels serve a call, on the host runtime: the rules that choose
between forms of a pass, at both sides of their lines."""
import pytest

import host_runtime


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return host_runtime.build(tmp_path_factory.mktemp("host"))


ENGINE = """
def engine(shape, ab=(1.0, 0.0), prec=E.C64, inter=E.CONTACT, vext=E.HARMONIC):
    return E.Engine(shape, ab[0], ab[1], 0.01, 1.0, inter, vext, 0, prec)

RT, IT = (1.0, 0.0), (0.0, 1.0)
"""

ZWAVE = ENGINE + """
def z_passes(shape, ab, prec, inter, pinned=False, qf=0.0):
    "(in waves, in LDS tiles) of the z passes of a run of three steps"
    g = engine(shape, ab, prec, inter)
    if pinned:
        g.set_vortex(0.5, 0.5, 1)
    if qf:
        g.set_quantum_friction_coeff(qf)
    names = launched(g.evolve_vortex if pinned else g.evolve_qf, 3)
    g.close()
    t = "f" if prec == E.C64 else "d"
    waves = sum("zwave_kernelI%sLi%dE" % (t, shape[2]) in n for n in names)
    tiles = sum("fft_pass_kernelI%sLi%dELb1E" % (t, shape[2]) in n for n in names)
    return waves, tiles

# z passes of three steps: open, then two per step in real time, four in
# imaginary time (the last one's rescaling is not a z pass)
N = {RT: 7, IT: 12}
for ab in (RT, IT):
    n = N[ab]
    # contact: complex64 always, complex128 above 128 workgroups
    assert z_passes((8, 12, 96), ab, E.C64, E.CONTACT) == (n, 0)
    assert z_passes((64, 64, 192), ab, E.C128, E.CONTACT) == (0, n)
    assert z_passes((96, 48, 192), ab, E.C128, E.CONTACT) == (n, 0)
    # unitary gas: complex64 above 256, complex128 above 170; the passes
    # without its potential as the contact ones
    light = 1 if ab == RT else 3  # the last corrector end; every corrector end
    assert z_passes((128, 128, 96), ab, E.C64, E.UFG) == (light, n - light)
    assert z_passes((192, 96, 96), ab, E.C64, E.UFG) == (n, 0)
    assert z_passes((96, 96, 96), ab, E.C128, E.UFG) == (light, n - light)
    assert z_passes((128, 96, 96), ab, E.C128, E.UFG) == (n, 0)
    # extended Thomas-Fermi: where the last round of two workgroups per CU is full
    for shape, prec, waves in (((128, 128, 192), E.C128, True), ((128, 96, 192), E.C128, False),
                               ((96, 96, 192), E.C128, False), ((128, 128, 192), E.C64, True),
                               ((192, 192, 192), E.C64, False), ((8, 12, 96), E.C64, False)):
        assert z_passes(shape, ab, prec, E.ETF) == ((n, 0) if waves else (light, n - light)), (shape, prec)
    # pinned: only in complex128, there the same
    for shape, prec, waves in (((128, 128, 192), E.C128, True), ((128, 96, 192), E.C128, False),
                               ((128, 128, 192), E.C64, False), ((12, 8, 192), E.C64, False)):
        pin = n - (light + 3 if ab == RT else 6)  # open and corrector ends that open a step; openings and re-imprints
        got = z_passes(shape, ab, prec, E.CONTACT, pinned=True)
        assert got == ((n, 0) if waves else (n - pin, pin)), (shape, prec, got, pin)
# other lengths take waves whatever the pass
for shape, precs in (((12, 8, 128), (E.C64, E.C128)), ((24, 8, 256), (E.C64, E.C128)),
                     ((96, 96, 128), (E.C64, E.C128)), ((8, 12, 512), (E.C64,))):
    for prec in precs:
        for inter in (E.UFG, E.ETF, E.CONTACT):
            assert z_passes(shape, RT, prec, inter, pinned=True) == (7, 0)
"""


def test_z_passes_of_24_points_per_lane(runtime):
    host_runtime.run(runtime, ZWAVE)


XCD = ENGINE + """
def one_xcd(shape, ab, prec, nt, inter=E.CONTACT, prepare=None):
    g = engine(shape, ab, prec, inter, E.COSINE)
    if prepare:
        prepare(g)
    names = launched(g.evolve_qf, nt)
    g.close()
    on = any("xcd_" in n for n in names)
    assert on == all("xcd_" in n for n in names), names
    return on

# (points' sides of the lines: shape, time, precision, steps -> one XCD)
for shape, ab, prec, nt, want in [
        ((32, 32, 32), RT, E.C64, 1, True), ((64, 64, 8), RT, E.C64, 1, True), ((24, 24, 64), RT, E.C64, 20, False),
        ((24, 32, 32), RT, E.C64, 3, False), ((24, 32, 32), RT, E.C64, 4, True),
        ((16, 24, 32), RT, E.C128, 1, True), ((16, 32, 24), RT, E.C128, 3, True), ((12, 24, 64), RT, E.C128, 3, False),
        ((12, 24, 64), RT, E.C128, 4, True), ((16, 16, 16), RT, E.C128, 1, True), ((48, 12, 8), RT, E.C128, 3, False),
        ((48, 12, 8), RT, E.C128, 4, True), ((64, 64, 8), RT, E.C128, 4, True), ((24, 24, 64), RT, E.C128, 20, False),
        ((8, 32, 32), RT, E.C128, 1, True), ((12, 32, 32), RT, E.C128, 3, False), ((16, 32, 32), RT, E.C128, 4, True),
        ((24, 32, 32), RT, E.C128, 20, False), ((12, 48, 48), RT, E.C64, 20, False),
        ((32, 32, 32), IT, E.C128, 1, True), ((48, 24, 32), IT, E.C128, 20, False), ((48, 24, 32), IT, E.C64, 1, True),
        ((48, 48, 16), IT, E.C64, 20, False), ((48, 48, 16), (0.6, 0.3), E.C64, 20, False),
        ((32, 32, 32), (0.6, 0.3), E.C64, 1, True), ((96, 8, 8), RT, E.C64, 20, False)]:
    assert one_xcd(shape, ab, prec, nt) == want, (shape, ab, prec, nt)
for inter in (E.UFG, E.ETF):
    assert one_xcd((16, 16, 16), RT, E.C64, 5, inter)

# what keeps the passes, and what does not
SMALL = ((16, 24, 32), RT, E.C64, 20)
assert one_xcd(*SMALL)
assert not one_xcd(*SMALL, prepare=lambda g: g.set_variant(0))
assert not one_xcd(*SMALL, prepare=lambda g: g.set_quantum_friction_coeff(0.1))
H.hh_capture(1)
assert not one_xcd(*SMALL)
H.hh_capture(0)
# a partition of the card: fewer CUs, or another count, than eight XCDs of 32
for cus in (32, 64, 128, 255, 304):
    H.hh_cus(cus)
    assert not one_xcd(*SMALL), cus
    assert not one_xcd((32, 32, 32), IT, E.C128, 20), cus
H.hh_cus(256)
assert one_xcd(*SMALL)
"""


def test_runs_on_one_xcd(runtime):
    host_runtime.run(runtime, XCD)


AUTOTUNE = ENGINE + """
def on(g, n=20):
    return all("xcd_" in k for k in launched(g.evolve_qf, n))

def other(g, rt):
    g.set_ite_evolution() if not rt else g.set_rte_evolution()

H.hh_cost(b"xcd_", float(XCD_MS))
fast = XCD_MS < 0.1
for prec, shape in ((E.C64, (16, 24, 32)), (E.C128, (32, 32, 16))):
    # never set: imaginary time keeps its route, real time the faster one
    g = engine(shape, RT, prec)
    assert on(g)
    g.autotune(3)
    assert on(g) == fast
    g.set_ite_evolution()
    assert on(g)
    g.close()
    # set by hand: passes; a timing brings back real time, where it wins
    g = engine(shape, RT, prec)
    g.set_variant(2)
    g.set_ite_evolution()
    g.autotune(3)
    assert not on(g)
    g.set_rte_evolution()
    assert on(g) == fast
    g.close()
    # not timed: the route stays as it was
    for start in (None, 2):
        for busy, quiet in ((lambda g: g.set_quantum_friction_coeff(0.1), lambda g: g.set_quantum_friction_coeff(0.0)),
                            (lambda g: g.set_graph(True), lambda g: g.set_graph(False)),
                            (lambda g: g.profile(1), lambda g: g.profile(1, False))):
            g = engine(shape, RT, prec)
            if start is not None:
                g.set_variant(start)
            busy(g)
            g.autotune(3)
            quiet(g)
            assert on(g) == (start is None), (start, prec)
            g.close()
"""


@pytest.mark.parametrize("ms", [0.001, 1000.0])
def test_autotune_changes_a_route_only_by_a_timing(runtime, ms):
    host_runtime.run(runtime, "XCD_MS = %r\n" % ms + AUTOTUNE)


WINDINGS = ENGINE + """
for shape, run in (((8, 8, 8), 1), ((64, 64, 64), 1), ((128, 128, 64), 1), ((128, 128, 128), 8), ((12, 256, 512), 8)):
    for prec in (E.C64, E.C128):
        g = engine(shape, prec=prec)
        names = [n for n in launched(g.detect_vortices, 0.1, False) if "windings" in n]
        assert len(names) == 1 and "Lj%dE" % run in names[0], (shape, names)
        g.close()
"""


def test_vortex_detection_runs(runtime):
    host_runtime.run(runtime, WINDINGS)
