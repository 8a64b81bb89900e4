"""Resident solves whose waits are given up at the first poll that finds nothing (CNV_RESIDENT_POLLS=0; every
kernel still runs to its end): the solve is repeated as launches, so fields, counts and statistics are
those of a context whose named launch shape has no resident form."""
import ctypes as C

import numpy as np
import pytest

import cnv

pytestmark = pytest.mark.gpu
LAUNCHES = {64: (5, 8, 8), 257: (5, 8, 8), 600: (6, 8, 8), 1030: (5, 8, 8)}  # sides, and the sweeps a launch has there
NAMES = ("sweeps_per_launch", "tile_waves", "wave_rows")


@pytest.fixture
def no_polls(monkeypatch):
    return lambda: monkeypatch.setenv("CNV_RESIDENT_POLLS", "0")


def field(n, seed=3):
    x = np.arange(n) / n
    return np.sin(7 * x)[:, None] * np.cos(4 * x)[None, :] + 0.1 * np.random.default_rng(seed).standard_normal((n, n))


def same_fields(a, b):
    return all(np.array_equal(a[k], b[k]) for k in ("w", "psi", "u", "v"))


@pytest.mark.parametrize("graph", [0, 1], ids=["eager", "graph"])
@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
@pytest.mark.parametrize("n", sorted(LAUNCHES))
def test_step(n, precision, graph, no_polls):
    # the diagnostic and the speed that blowup_speed is held against are those of the solve's end
    kw = dict(precision=precision, Re=400.0, dt=1e-5, tol=1e-8, itmax=100000, diagnostics=1, blowup_speed=50.0)
    with cnv.Cavity(cnv.default_params(n, **kw, **dict(zip(NAMES, LAUNCHES[n])))) as cav:
        want, fields = cav.step(3), cav.get_state()
    no_polls()
    with cnv.Cavity(cnv.default_params(n, use_graph=graph, **kw)) as cav:
        got = cav.step(3)
        for g, w in zip(got, want):
            assert (g.status, g.k, g.sweeps, g.outer) == (w.status, w.k, w.sweeps, w.outer) and g.status == cnv.OK
            assert (g.cont_max, g.cont_min) == (w.cont_max, w.cont_min)
        assert same_fields(cav.get_state(), fields)


@pytest.mark.parametrize("ptype", [1, 2])
@pytest.mark.parametrize("n", sorted(LAUNCHES))
def test_solves(n, ptype, no_polls):
    kw = dict(tol=1e-3, itmax=3000, poisson_type=ptype, beta=1.6)
    f = field(n)
    with cnv.Cavity(cnv.default_params(n, **kw, **dict(zip(NAMES, LAUNCHES[n])))) as cav:
        rc, psi, k, e = cav.poisson(f)
    no_polls()
    with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
        for _ in range(2):
            rc2, psi2, k2, e2 = cav.poisson(f)
            assert (rc2, k2) == (rc, k) and abs(e2 - e) <= 1e-12 * e and np.array_equal(psi2, psi)
        if n <= 1024:
            cav.set_state(w=f)
            dw, du, kk, ee = C.c_void_p(), C.c_void_p(), C.c_int(), C.c_double()
            cnv._check(cnv.lib().cnv_device_state(cav.h, C.byref(dw), None, C.byref(du), None), cav.h)
            assert cnv.lib().cnv_poisson_device_noalloc(n, 1.0 / n, 1.0 / n, 1.6, 1e-3, 3000, ptype, dw, du, C.byref(kk),
                                                        C.byref(ee)) == rc
            assert kk.value == k and np.array_equal(cav.get_state()["u"], psi)


@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
def test_batch(precision, no_polls):
    ps = [cnv.default_params(n, Re=100.0 + 50 * i, dt=1e-4, tol=1e-6, itmax=200000, precision=precision, diagnostics=1,
                             inner_test_every=1, beta=cnv.reference_beta(n)) for i, n in enumerate([64, 97, 33, 256] * 3)]
    out = []
    for give_up in (False, True):
        if give_up:
            no_polls()
        with cnv.Batch(ps) as b:
            st = [[(s.status, s.k, s.sweeps, s.outer, s.cont_max, s.cont_min) for s in row] for row in b.step(3)]
            out.append((st, [b.get_state(i) for i in range(len(ps))]))
    assert out[0][0] == out[1][0]
    assert all(same_fields(a, b) for a, b in zip(out[0][1], out[1][1]))


@pytest.mark.parametrize("graph", [0, 1], ids=["eager", "graph"])
@pytest.mark.parametrize("n", [64, 257])
def test_speed_limit_is_held_against_the_end_of_the_solve(n, graph, no_polls):
    # over-relaxed short waves: the iterate that is given up has 1.5 times the solution's speed
    i, j = np.indices((n, n))
    w = 100 * np.sin(2 * np.pi * i / 8) * np.sin(2 * np.pi * j / 8)
    kw = dict(Re=1e6, dt=1e-12, tol=1e-9, itmax=100000, beta=1.95, u=[0.0] * 4, diagnostics=1)
    out = []
    for blowup in (None, 1.1):
        if blowup:
            no_polls()
            kw.update(blowup_speed=1.1 * max(np.abs(out[0][1][x]).max() for x in "uv"), use_graph=graph)
        else:
            kw.update(zip(NAMES, LAUNCHES[n]))
        with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
            cav.set_state(w=w, psi=0 * w, u=0 * w, v=0 * w)
            st = cav.step(2, check=False) if blowup else cav.step(2)
            out.append(([(s.status, s.k, s.cont_max, s.cont_min) for s in st], cav.get_state()))
        for name in NAMES:
            kw.pop(name, None)
    assert out[1][0] == out[0][0] and same_fields(out[1][1], out[0][1])


@pytest.mark.parametrize("polls", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
def test_whenever_a_wait_is_too_long(precision, polls, monkeypatch):
    # a few polls may or may not be enough, in the first kernel of a solve or a later one: solves of 12 000 sweeps and
    # more (plain relaxation), of which a kernel runs 9600 to 11 520
    n = 200
    kw = dict(precision=precision, Re=400.0, dt=1e-5, tol=1e-7, itmax=200000, beta=1.0, inner_test_every=1)
    with cnv.Cavity(cnv.default_params(n, **kw, **dict(zip(NAMES, (5, 8, 8))))) as cav:
        want, fields = cav.step(2), cav.get_state()
    assert want[0].sweeps > 12000
    monkeypatch.setenv("CNV_RESIDENT_POLLS", str(polls))
    for _ in range(3):
        with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
            got = cav.step(2)
            assert [(s.status, s.sweeps, s.outer) for s in got] == [(s.status, s.sweeps, s.outer) for s in want]
            assert same_fields(cav.get_state(), fields)
