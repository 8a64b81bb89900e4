"""Resident Poisson solves (csrc/hip/sor_resident.h) against the oracle and against the same solves as
launches: every tile shape at the edges of its range of grids, solves that end in the first
epoch, inside an epoch, on its last sweep, on a spent budget, and from so far out that the tiles kept
nothing to go back to; the refined form's inner solves; two solves at once from two threads."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import cnv
from oracle import orc

pytestmark = pytest.mark.gpu


def field(n, seed=3):
    x = np.arange(n) / n
    rng = np.random.default_rng(seed)
    return np.sin(7 * x)[:, None] * np.cos(4 * x)[None, :] + 0.1 * rng.standard_normal((n, n))


def check(n, f, beta, tol, itmax, ptype=2):
    """One solve against the oracle: the iterate bit for bit, k, and the update to rounding."""
    p = orc.make_params(n, tol=tol, itmax=itmax, ordering=orc.REDBLACK, beta_=beta, threads=8, poisson_type=ptype)
    want, st = orc.poisson(p, f)
    with cnv.Cavity(cnv.default_params(n, tol=tol, itmax=itmax, beta=beta, poisson_type=ptype)) as cav:
        rc, psi, k, e = cav.poisson(f)
    assert k == (st.k if rc == cnv.OK else itmax - 1), (n, k, st.k)  # the oracle logs no k for a failed solve
    assert abs(e - st.e) <= 1e-12 * abs(st.e)
    assert np.array_equal(psi, want)
    return rc, k


# sides around the largest grid of each tile shape (8 x 104, 12 x 108, 16 x 112, 24 x 104, 40 x 104,
# 44 x 108 owned points, at most 32 tiles on each of 8 XCDs; 76 x 108, 100 x 108, and 156 x 116,
# at most 255 in all), the smallest grid, and beyond the last
@pytest.mark.parametrize("n", [8, 9, 64, 97, 104, 105, 416, 417, 432, 512, 540, 541, 560, 672, 673, 728, 744, 745, 960, 1000,
                               1001, 1055, 1056, 1057, 1080, 1081, 1300, 1404, 1405, 1620, 1621, 1800, 2048, 2088,
                               2089])
def test_solves_equal_the_oracle(n):
    f = field(n)
    e = [orc.poisson(orc.make_params(n, tol=-1.0, itmax=s, ordering=orc.REDBLACK, beta_=0.9, threads=8), f)[1].e
         for s in (1, 17, 24)]
    for tol in (2 * e[0], e[1] * (1 + 1e-9), e[2] * (1 + 1e-9)):  # the first sweep, inside an epoch, and later
        assert check(n, f, 0.9, tol, 1000)[0] == cnv.OK
    assert check(n, f, 0.9, -1.0, 23)[0] == cnv.NOT_CONVERGED  # a budget that ends inside an epoch
    assert check(n, f, 1.0, e[1], 1000, ptype=1)[0] == cnv.OK


@pytest.mark.parametrize("n", [300, 600, 1024, 1250, 1501, 1700, 2048])
def test_solve_that_ends_from_far_out(n):
    # a short-wave source under weak relaxation: its update falls about twofold a sweep, so when it
    # crosses the tolerance the tiles held in device memory have kept no epoch's start
    i, j = np.indices((n, n))
    f = np.sin(2 * np.pi * i / 5) * np.sin(2 * np.pi * j / 5)
    e = {s: orc.poisson(orc.make_params(n, tol=-1.0, itmax=s, ordering=orc.REDBLACK, beta_=0.6, threads=8), f)[1].e
         for s in (4, 13, 15, 16, 17, 18, 20, 21)}
    assert e[4] > 50 * e[13]
    for s, v in e.items():
        assert check(n, f, 0.6, v * (1 + 1e-9), 1000)[1] == s - 1


@pytest.mark.parametrize("n,launches", [(64, (5, 8, 8)), (257, (5, 8, 8)), (600, (6, 8, 8)), (900, (6, 8, 8)),
                                        (1030, (5, 8, 8)), (1211, (5, 8, 8)), (1444, (5, 8, 8))])
def test_refined_equals_launches(n, launches):
    # the named shape is compiled for launches only; the sweeps and their order are the same
    kw = dict(precision=cnv.PREC_FP32_DC, Re=400.0, dt=1e-5, tol=1e-8, itmax=100000)
    out = []
    for shape in ({}, dict(zip(("sweeps_per_launch", "tile_waves", "wave_rows"), launches))):
        with cnv.Cavity(cnv.default_params(n, **kw, **shape)) as cav:
            st = cav.step(2)
            out.append(([(s.status, s.sweeps, s.outer) for s in st], cav.get_state()))
    assert out[0][0] == out[1][0]
    for name in ("w", "psi", "u", "v"):
        assert np.array_equal(out[0][1][name], out[1][1][name]), name


@pytest.mark.parametrize("n", [8, 65, 417, 600, 1001, 1024])
def test_noalloc_equals_context(n):
    f = field(n)
    with cnv.Cavity(cnv.default_params(n, tol=1e-3, itmax=100000, beta=1.5)) as cav:
        rc, psi, k, e = cav.poisson(f)
        cav.set_state(w=f)
        dw, du = C.c_void_p(), C.c_void_p()
        cnv._check(cnv.lib().cnv_device_state(cav.h, C.byref(dw), None, C.byref(du), None), cav.h)
        k2, e2 = C.c_int(), C.c_double()
        assert cnv.lib().cnv_poisson_device_noalloc(n, 1.0 / n, 1.0 / n, 1.5, 1e-3, 100000, 2, dw, du, C.byref(k2),
                                                    C.byref(e2)) == rc  # the larger grids run out of sweeps
        assert (k, e) == (k2.value, e2.value) and np.array_equal(cav.get_state()["u"], psi)


@pytest.mark.parametrize("n", [8, 65, 257, 600, 1024, 1444])
def test_fp64_solve_of_a_refined_context(n):
    # the context's resident memory is laid out for its FP32 inner solves
    f = field(n)
    kw = dict(Re=400.0, dt=1e-5, tol=1e-3, itmax=20000)
    with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
        want = cav.poisson(f)
    with cnv.Cavity(cnv.default_params(n, precision=cnv.PREC_FP32_DC, **kw)) as cav, \
            cnv.Cavity(cnv.default_params(n, precision=cnv.PREC_FP32_DC, **kw)) as plain:
        for _ in range(2):  # between steps of the refined form, which it leaves as they were
            rc, psi, k, e = cav.poisson(f)
            assert (rc, k) == (want[0], want[2]) and abs(e - want[3]) <= 1e-12 * want[3]
            assert np.array_equal(psi, want[1])
            assert [(s.status, s.sweeps, s.outer) for s in cav.step(1)] == \
                   [(s.status, s.sweeps, s.outer) for s in plain.step(1)]
        a, b = cav.get_state(), plain.get_state()
        for name in ("w", "psi", "u", "v"):
            assert np.array_equal(a[name], b[name]), name


def test_two_solves_at_once():
    n, f = 1024, field(1024)
    kw = dict(tol=1e-4, itmax=100000, beta=1.9)
    with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
        alone = cav.poisson(f)
    got = {}

    def work(name):
        with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
            got[name] = [cav.poisson(f) for _ in range(3)]

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for t in range(2):
        for rc, psi, k, e in got[t]:
            assert (rc, k) == (alone[0], alone[2]) and abs(e - alone[3]) <= 1e-12 * e
            assert np.array_equal(psi, alone[1])


def batch_equals_alone(ps, steps, states=None):
    """Each cavity of a batch as it is alone: fields and counts bit for bit, the FP64 update (summed
    per tile) to rounding; the FP32 solves add theirs in FP32 over a lane's rows, whose number differs."""
    states = states or [None] * len(ps)
    with cnv.Batch(ps) as b:
        for i, s in enumerate(states):
            if s:
                b.set_state(i, **s)
        st = b.step(steps)
        got = [b.get_state(i) for i in range(len(ps))]
    for i, p in enumerate(ps):
        if p.precision == cnv.PREC_FP32_DC:  # its solves test every fifth sweep, as the batch's do
            p.sweeps_per_launch, p.tile_waves, p.wave_rows = 5, 16, 4
        with cnv.Cavity(p) as cav:
            if states[i]:
                cav.set_state(**states[i])
            alone, state = cav.step(steps), cav.get_state()
        for t in range(steps):
            a, g = alone[t], st[t][i]
            assert (g.status, g.k, g.sweeps, g.outer) == (a.status, a.k, a.sweeps, a.outer), (i, t)
            assert p.precision != cnv.PREC_FP64 or abs(g.e - a.e) <= 1e-12 * abs(a.e)
        for name in ("w", "psi", "u", "v"):
            assert np.array_equal(got[i][name], state[name]), (i, name)
    return [s for row in st for s in row]


# few cavities (2 rows a wave), many (4; in FP32 8 where dx = dy), one that takes most of the GPU
@pytest.mark.parametrize("sides", [[8, 9, 97], [64, 104, 105, 33] * 4, [256, 255, 240, 100] * 8, [900, 40, 300, 41]],
                         ids=["few", "some", "many", "large"])
@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
@pytest.mark.parametrize("kind", ["square", "oblong", "gs"])
def test_batch_equals_alone(sides, precision, kind):
    ps = []
    for i, n in enumerate(sides):
        p = cnv.default_params(n, Re=100.0 + 50 * i, dt=1e-4 if n < 500 else 1e-5, tol=1e-6, itmax=200000,
                               precision=precision, inner_test_every=1, poisson_type=1 if kind == "gs" else 2,
                               beta=cnv.reference_beta(n), u=[0.0, 0.0, 0.0, 1.0 + 0.01 * i])
        if kind == "oblong":
            p.dy = 0.8 * p.dx
        if kind == "gs":
            p.itmax, p.tol = 400, 1e-3  # plain Gauss-Seidel sweeps; the larger sides run out of them
        ps.append(p)
    if kind == "gs":
        ps = [p for p in ps if p.n <= 105] or ps[:2]
    if kind == "gs" and precision == cnv.PREC_FP32_DC:
        for p in ps:
            p.itmax = 200000
    print(sides, precision, kind, flush=True)
    assert all(s.status == cnv.OK for s in batch_equals_alone(ps, 2)) or kind == "gs"


@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
def test_batch_solves_longer_than_a_kernel(precision):
    # beta = 1: 10^4 and more sweeps, which is more epochs than one resident kernel runs
    ps = [cnv.default_params(n, Re=100.0, dt=1e-4, tol=1e-9, itmax=200000, precision=precision, inner_test_every=1,
                             beta=1.0) for n in (33, 160, 64, 161)]
    st = batch_equals_alone(ps, 1)
    assert max(s.sweeps for s in st) > 1984 * 5


def test_batch_solves_that_end_from_far_out():
    # as test_solve_that_ends_from_far_out, each cavity of a batch ending at another sweep
    n, ends = 256, (4, 13, 15, 16, 17, 18, 20, 21) * 4
    i, j = np.indices((n, n))
    f = np.sin(2 * np.pi * i / 5) * np.sin(2 * np.pi * j / 5)
    e = {s: orc.poisson(orc.make_params(n, tol=-1.0, itmax=s, ordering=orc.REDBLACK, beta_=0.6, threads=8), f)[1].e
         for s in ends}
    ps = [cnv.default_params(n, Re=1e6, dt=1e-12, tol=e[s] * (1 + 1e-6), itmax=1000, beta=0.6) for s in ends]
    st = batch_equals_alone(ps, 1, [dict(w=f, psi=np.zeros((n, n))) for _ in ends])
    assert {s.k for s in st} == {s - 1 for s in ends}


# dx = dy a power of two: the update's short form, and values for which it does not hold
@pytest.mark.parametrize("n", [8, 64, 256, 512, 1024])
@pytest.mark.parametrize("scale", [1.0, 1e-40, 1e-70, 1e-250, 1e-290, 1e260, 1e285])
def test_scaled_update_equals_the_oracle(n, scale):
    f = scale * field(n, seed=n)
    for beta in (1.0 + 1 / 64, 1.9, 0.3, 1.001):  # the last one has a factor 1 - beta too small for it
        check(n, f, beta, -1.0, 29)
    f[:, n // 2:] = 0.0
    check(n, f, 1.7, -1.0, 29)
    spot = np.zeros((n, n))  # the front of a first iterate: subnormal numbers at its edge
    spot[n // 3, n // 2] = scale
    check(n, spot, 1.5, -1.0, min(n, 300))


@pytest.mark.parametrize("n", [64, 1024])
def test_diverging_solve_reports_as_launches(n):
    f = 1e200 * field(n)
    for beta in (3.5, 12.0):
        sums = []
        with cnv.Cavity(cnv.default_params(n, tol=-1.0, itmax=400, beta=beta)) as cav, \
                cnv.Cavity(cnv.default_params(n, tol=-1.0, itmax=400, beta=beta, sweeps_per_launch=5, tile_waves=8,
                                              wave_rows=8)) as launches:
            for c in (cav, launches):
                rc, _, k, _ = c.poisson(f)
                sums.append((rc, k))
        assert sums[0] == sums[1] and sums[0][0] == cnv.DIVERGED


# sides whose resident epochs are of 6, 4, 6, 5 and 3 sweeps, where a launch has 5 or 6; the slowest overflows in the
# second kernel of its solve
@pytest.mark.parametrize("n,beta", [(64, 3.5), (64, 2.05), (500, 3.5), (700, 12.0), (1024, 3.5), (2048, 12.0)])
def test_diverging_solve_ends_as_launches(n, beta):
    f = 1e200 * field(n) if beta > 3 else field(n)
    kw = dict(tol=-1.0, itmax=30000, beta=beta)
    with cnv.Cavity(cnv.default_params(n, **kw)) as cav:
        got = [cav.poisson(f), cav.poisson(f)]
        s = cav.sweeps_per_launch
    with cnv.Cavity(cnv.default_params(n, sweeps_per_launch=s, tile_waves=8, wave_rows=8, **kw)) as cav:
        rc, psi, k, e = cav.poisson(f)
    assert rc == cnv.DIVERGED and (beta > 3 or k > 1920 * 6)
    for g in got:
        assert (g[0], g[2]) == (rc, k)
        assert np.array_equal(g[1], psi, equal_nan=True) and np.array_equal(g[3], e, equal_nan=True)


@pytest.mark.parametrize("n", [64, 97, 256, 500, 700])
def test_adjoint_equals_launches(n):
    # its solves end with the last sweep of the epoch, or launch, in which the relative rule is met
    w0, out = cnv.gaussian_vorticity(n, count=12, seed=4), []
    with cnv.Cavity(cnv.default_params(n)) as cav:
        s = cav.sweeps_per_launch
    for shape in ({}, dict(sweeps_per_launch=s, tile_waves=8, wave_rows=8)):
        p = cnv.default_params(n, Re=400.0, dt=0.05 / n ** 2 * 400, tol=1e-8, itmax=200000, **shape)
        with cnv.Adjoint(p, checkpoint_every=2) as adj:
            E = adj.forward(w0, 1.0, 5)
            out.append((adj.backward(), E, adj.sweeps()))
    (g, dU), E, sweeps = out[0]
    assert (dU, E, sweeps) == (out[1][0][1],) + out[1][1:] and np.array_equal(g, out[1][0][0])


def test_warm_start_after_a_solve_of_two_kernels():
    # 12000 sweeps are more than one resident kernel runs; the next step starts from where they got to
    n, out = 256, []
    for graph in (0, 1):
        p = cnv.default_params(n, Re=400.0, dt=1e-5, tol=1e-3, itmax=12000, beta=1.0, warm_start=1, use_graph=graph)
        with cnv.Cavity(p) as cav:
            first = cav.step(1, check=False)
            rc, _, k, _ = cav.poisson(field(n))
            assert (rc, k) == (cnv.NOT_CONVERGED, 11999)
            st = first + cav.step(2, check=False)
            out.append(([(s.status, s.k, s.e) for s in st], cav.get_state()))
    assert out[0][0] == out[1][0]
    for name in ("w", "psi", "u", "v"):
        assert np.array_equal(out[0][1][name], out[1][1][name]), name


@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
@pytest.mark.parametrize("when", ["dropped", "back"])
def test_autotuned_batch_follows_its_live_cavities(precision, when):
    # the autotuner makes the workgroup maps anew after a cavity has been dropped or come back; the next
    # step's queues have to follow
    sides = (48, 64, 97)
    ps = [cnv.default_params(n, Re=100.0 + 50 * i, dt=1e-4, tol=1e-6, itmax=200000, precision=precision,
                             inner_test_every=1, beta=cnv.reference_beta(n)) for i, n in enumerate(sides)]
    ps[1].blowup_speed = 5.0
    good = {k: 1e-3 * field(64, seed) for seed, k in enumerate(("w", "u", "v"))}
    out = []
    for tune in (False, True):
        with cnv.Batch(ps) as b:
            b.step(4)
            b.set_state(1, w=1e5 * field(64))
            assert b.step(1, check=False)[0][1].status == cnv.DIVERGED
            dropped = b.get_state(1)
            if tune and when == "dropped":
                b.autotune(8)
            b.step(2, check=False)
            now = b.get_state(1)
            assert all(np.isfinite(now[k]).all() and np.array_equal(now[k], dropped[k]) for k in ("w", "u", "v"))
            b.set_state(1, psi=np.zeros((64, 64)), **good)
            if tune and when == "back":
                b.autotune(8)
            st = b.step(2)
            out.append(([(s.status, s.sweeps, s.outer) for row in st for s in row],
                        [b.get_state(i) for i in range(len(sides))], now["psi"]))
    if precision == cnv.PREC_FP64:  # the refined form's tests follow the launches' sweeps, which the tuner may choose anew
        assert out[0][0] == out[1][0]
        assert all(np.array_equal(x[k], y[k]) for x, y in zip(out[0][1], out[1][1]) for k in x)
    else:
        assert all(np.max(np.abs(x[k] - y[k])) <= 1e-6 * np.max(np.abs(x[k])) for x, y in zip(out[0][1], out[1][1]) for k in x)
    # (the tuner zeroes the live cavities' iterates only)
    assert np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("precision", [cnv.PREC_FP64, cnv.PREC_FP32_DC], ids=["fp64", "refined"])
def test_batch_of_more_solves_at_once_than_128(precision):
    # one tile each (two deciding workgroups on an XCD): those of unlike lengths take one another's places
    ps = [cnv.default_params(n, Re=100.0 + i, dt=1e-5, tol=1e-6 * 10.0 ** -(i % 4), itmax=200000, precision=precision,
                             inner_test_every=1, beta=cnv.reference_beta(n)) for i, n in enumerate([40, 33, 44] * 84)]
    assert all(s.status == cnv.OK for s in batch_equals_alone(ps, 2))


# uniform batches on either side of the line between resident solves and launches
@pytest.mark.parametrize("n,count,precision", [(256, 27, cnv.PREC_FP32_DC), (256, 28, cnv.PREC_FP32_DC),
                                               (800, 3, cnv.PREC_FP64), (800, 8, cnv.PREC_FP64)])
def test_batch_of_like_cavities(n, count, precision):
    ps = [cnv.default_params(n, Re=400.0, dt=1e-5, tol=1e-5, itmax=200000, precision=precision, inner_test_every=1,
                             beta=cnv.reference_beta(n), u=[0.0, 0.0, 0.0, 1.0 + 0.01 * i]) for i in range(count)]
    assert all(s.status == cnv.OK for s in batch_equals_alone(ps, 3))


@pytest.mark.parametrize("n", [64, 256, 1024])
def test_source_in_and_out_of_the_short_updates_range(n):
    # one context, sources of either kind in turn, solves of one kernel and of two: the form follows the source
    near, far = field(n), field(n, 5)
    far[:, : n // 3] *= 1e-80
    for itmax in (31, 11600 if n < 1000 else 43):
        want = {i: orc.poisson(orc.make_params(n, tol=-1.0, itmax=itmax, ordering=orc.REDBLACK, beta_=1.5, threads=8), f)
                for i, f in enumerate((near, far))}
        with cnv.Cavity(cnv.default_params(n, tol=-1.0, itmax=itmax, beta=1.5)) as cav:
            for i in (0, 1, 1, 0, 0, 1):
                rc, psi, k, e = cav.poisson((near, far)[i])
                assert rc == cnv.NOT_CONVERGED and np.array_equal(psi, want[i][0])
                assert abs(e - want[i][1].e) <= 1e-12 * want[i][1].e


@pytest.mark.parametrize("n,most", [(256, 1.12), (1024, 1.16)])
def test_far_front_costs_no_more_than_the_general_update(n, most):
    # a sweep of the general form against the short one: 1.03 at 256^2, 1.10 at 1024^2 by the kernels' own times;
    # the general form as an epoch of the short one's kernel: 1.22 and 1.23
    near, far = field(n), field(n)
    far[:, : n // 3] *= 1e-80
    dt = {0: [], 1: []}
    with cnv.Cavity(cnv.default_params(n, tol=-1.0, itmax=9000, beta=1.5)) as cav:
        for _ in range(6):
            for i, f in enumerate((near, far)):
                cav.poisson(f)
                t = time.perf_counter()
                cav.poisson(f)
                dt[i].append(time.perf_counter() - t)
    print(n, min(dt[1]) / min(dt[0]), flush=True)
    assert min(dt[1]) <= most * min(dt[0])
