"""The short form of the scaled SOR update (SorTile in csrc/hip/sor_rb.h) against the reference's
association, in numpy: the same bits over 12 half-sweeps from values that are 0 or of a magnitude in
[2^-200, 2^900), for every scale 2^-m and relaxation factor that the form is used with."""
import numpy as np
import pytest

N = 24


def draw(rng, lo, hi):
    """Signed values of random magnitude in [2^lo, 2^hi), a fifth of them 0 and some nearly cancelling."""
    x = np.ldexp(1.0 + rng.random((N, N)), rng.integers(lo, hi, (N, N)).astype(np.int64))
    x *= rng.choice((-1.0, 1.0), (N, N)) * (rng.random((N, N)) < 0.8)
    near = rng.random((N, N)) < 0.3
    x[1:][near[1:]] = -np.nextafter(x[:-1][near[1:]], 0.0)
    bad = (x != 0) & ((np.abs(x) < 2.0 ** lo) | (np.abs(x) >= 2.0 ** hi))
    x[bad] = 0.0
    return x


def half_sweep(u, colour, update):
    i, j = np.indices(u.shape)
    inner = (i > 0) & (i < N - 1) & (j > 0) & (j < N - 1)
    ns, ew = np.zeros_like(u), np.zeros_like(u)
    ns[1:-1] = u[2:] + u[:-2]
    ew[:, 1:-1] = u[:, 2:] + u[:, :-2]
    return np.where(inner & ((i + j) % 2 == colour), update(u, ns, ew), u)


@pytest.mark.parametrize("m", [0, 6, 20, 22, 61])
@pytest.mark.parametrize("beta", [0.0625, 0.5, 63 / 64, 65 / 64, 1.95, 15.9999])
@pytest.mark.parametrize("lo,hi", [(-200, -190), (-200, 900), (-30, 10), (880, 900)])
def test_short_update_has_the_same_bits(m, beta, lo, hi):
    rng = np.random.default_rng(m * 1000 + int(beta * 64))
    c1, omb = np.ldexp(1.0, -m), 1 - beta
    rB = 1 / (4 * c1)
    for _ in range(4):
        f1 = draw(rng, lo, hi)        # (c3*f)/c1
        c3f = c1 * f1
        a = b = draw(rng, lo, hi)
        for h in range(12):
            a = half_sweep(a, h & 1, lambda u, ns, ew: (((c1 * ns + c1 * ew) - c3f) * beta) * rB + omb * u)
            b = half_sweep(b, h & 1, lambda u, ns, ew: (((ns + ew) - f1) * beta) * 0.25 + omb * u)
            assert np.isfinite(a).all() and np.array_equal(a, b) and np.array_equal(np.signbit(a), np.signbit(b))
