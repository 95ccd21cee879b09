"""The kernels' division by a kept reciprocal against the IEEE quotient.

conservedToPrimitive divides five values of a cell by its density, and mass fractions by the run's
molar masses, so its results against numpy's IEEE division show the helper bit for bit: quotients that
lie as close to a rounding boundary as 53-bit operands allow, ordinary ones over 2^+-300, zeros of both
signs, infinities, NaN and zero divisors.  No tolerance: the values are equal or the test fails.  Divisors
whose reciprocal Newton's iteration does not round may round a quotient beside a boundary the other way,
and the ends of the exponent range follow rules of their own; both have a test.
Likewise the noise whose Box-Muller radius is zero, against the oracle's.
"""
from fractions import Fraction

import numpy as np
import pytest

from fhdex_amd import params as P

pytestmark = pytest.mark.gpu

N = (24, 16, 16)
CELLS = N[0] * N[1] * N[2]


def hard_pairs(count, divisors):
    """Operand pairs whose quotient is within 2^-53 of its last place of a rounding boundary: for odd b, a is
    +-1, +-3, ... times the inverse of 2^54 modulo b, kept where the quotient's 54th bit is set."""
    a, b = [], []
    while len(a) < count:
        d = next(divisors)
        inv = pow(2 ** 54, -1, d)
        for e in (1, -1, 3, -3):
            n = e * inv % d
            if 2 ** 52 <= n < d and ((n << 54) - e) // d % 2 == 1:
                a.append(float(n))
                b.append(float(d))
    return np.array(a[:count]), np.array(b[:count])


def random_divisors(rng):
    while True:
        yield int(rng.integers(2 ** 52, 2 ** 53)) | 1


def values(kind, rng):
    if kind == "hard":
        return hard_pairs(CELLS, random_divisors(rng))
    s = rng.choice([-1.0, 1.0], CELLS)
    if kind == "wide":
        return s * rng.uniform(1, 2, CELLS) * 2.0 ** rng.integers(-300, 300, CELLS), \
            rng.uniform(1, 2, CELLS) * 2.0 ** rng.integers(-300, 300, CELLS)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.5])
    return rng.choice(special, CELLS), rng.choice(special, CELLS)


@pytest.mark.parametrize("kind", ["hard", "wide", "special"])
def test_quotients_are_ieee(kind):
    import torch
    from fhdex_amd import compressible as fc
    from fhdex_amd import lib as L
    rng = np.random.default_rng(7)
    p = P.make_params(2, N, 8e-6, [39.948, 4.0026], [3.66e-8, 2.18e-8])
    ctx = L.Context(p)
    cons, prim = fc.MultiFab.cell(p, p.nvars), fc.MultiFab.cell(p, p.nprimvars)
    g = p.ngc
    v = (slice(None), slice(g, g + N[2]), slice(g, g + N[1]), slice(g, g + N[0]))
    a, b = values(kind, rng)
    c = np.empty((p.nvars, CELLS))
    c[0] = b
    for q in (1, 2, 3, 5, 6):
        c[q] = np.roll(a, q) if kind != "hard" else a * 2.0 ** (q - 3)
    c[4] = a
    cons.t[v] = torch.from_numpy(c.reshape(p.nvars, N[2], N[1], N[0])).cuda()
    fc.conservedToPrimitive(ctx, prim, cons)
    got = prim.t[v].cpu().numpy().reshape(p.nprimvars, CELLS)
    ctx.close()
    with np.errstate(all="ignore"):
        vel, Y = c[1:4] / b, c[5:7] / b
        molmix = 1.0 / ((0.0 + Y[0] / p.molmass[0]) + Y[1] / p.molmass[1])
        X = np.stack([Y[n] * molmix / p.molmass[n] for n in range(2)])
    np.testing.assert_array_equal(got[1:4], vel)
    np.testing.assert_array_equal(got[6:8], Y)
    np.testing.assert_array_equal(got[8:10], X)
    zero = np.concatenate([vel, Y]) == 0.0
    assert np.array_equal(np.signbit(got[[1, 2, 3, 6, 7]])[zero], np.signbit(np.concatenate([vel, Y]))[zero])


def divide(a, b):
    """a / b of conservedToPrimitive, three dividends (momenta) a cell."""
    import torch
    from fhdex_amd import compressible as fc
    from fhdex_amd import lib as L
    p = P.make_params(2, N, 8e-6, [39.948, 4.0026], [3.66e-8, 2.18e-8])
    ctx = L.Context(p)
    cons, prim = fc.MultiFab.cell(p, p.nvars), fc.MultiFab.cell(p, p.nprimvars)
    g = p.ngc
    v = (slice(None), slice(g, g + N[2]), slice(g, g + N[1]), slice(g, g + N[0]))
    c = np.full((p.nvars, CELLS), 1.0)
    c[0], c[1:4] = b, a
    cons.t[v] = torch.from_numpy(c.reshape(p.nvars, N[2], N[1], N[0])).cuda()
    fc.conservedToPrimitive(ctx, prim, cons)
    got = prim.t[v].cpu().numpy().reshape(p.nprimvars, CELLS)[1:4]
    ctx.close()
    return got


def end_divisors():
    """The odd significands from both ends of their range inwards, 2^53 - 1 and 2^52 + 1 first."""
    for q in range(1, 2 ** 51, 2):
        yield 2 ** 53 - q
        yield 2 ** 52 + q


def test_quotients_by_unrounded_reciprocals():
    """Divisors at the ends of the significand's range.  The reciprocal is within one last place of 1 / b, so
    the corrected quotient before its rounding is within 2^-50 last places of a / b: it is the IEEE one
    unless a rounding boundary lies that near, and then one of its two neighbours."""
    rng = np.random.default_rng(7)
    a, b = hard_pairs(CELLS // 2, end_divisors())
    few = np.array([2.0 ** 53 - q for q in range(1, 9)] + [2.0 ** 52 + q for q in range(8)])
    a = np.concatenate([a, rng.integers(2 ** 52, 2 ** 53, CELLS - len(a)).astype(float)])
    b = np.concatenate([b, rng.choice(few, CELLS - len(b))])
    got, want = divide(np.stack([a, 2.0 * a, 0.25 * a]), b), a / b
    other = np.flatnonzero(got[0] != want)
    print("quotients rounded the other way:", len(other), "of", CELLS, flush=True)
    for q in other:
        lo, hi = sorted((Fraction(float(got[0][q])), Fraction(float(want[q]))))
        assert float(hi) == np.nextafter(float(lo), np.inf)
        exact = Fraction(int(a[q]), int(b[q]))
        assert abs(exact - (lo + hi) / 2) <= (hi - lo) / 2 ** 50
    np.testing.assert_array_equal(got[1:], np.stack([2.0 * got[0], 0.25 * got[0]]))


def test_quotients_beyond_the_range():
    """Where the helper leaves out the compiler's scalings: dividends, divisors and quotients up to the
    ends of the double range.  A finite quotient is the IEEE one to its last place, except that a divisor
    below 2^-1024 may give an infinite one; nothing turns finite."""
    rng = np.random.default_rng(11)
    a = np.ldexp(rng.uniform(1, 2, (3, CELLS)), rng.integers(-1074, 1024, (3, CELLS)))
    b = np.ldexp(rng.uniform(1, 2, CELLS), rng.integers(-1074, 1024, CELLS))
    got = divide(a, b)
    with np.errstate(all="ignore"):
        want = a / b
        near = (got == want) | (got == np.nextafter(want, np.inf)) | (got == np.nextafter(want, -np.inf))
    tiny = np.broadcast_to(b < 2.0 ** -1024, want.shape)
    finite, large = np.isfinite(want), np.abs(a) >= 2.0 ** -968
    assert (got == want)[finite & large & ~tiny].all()
    assert near[finite & ~tiny].all()
    assert (near | np.isinf(got))[finite & tiny].all()
    assert np.isinf(got[~finite]).all()


# Counters whose Philox block has its first 53 bits all ones, solved for by running the rounds backwards:
# u1 then rounds to 1, its logarithm is +0 and the radius the root of -0.  (step, instance, direction,
# component, cell) at seed 9 in argon 16^3.
ZERO_RADIUS = [(0x91696f0562fab3, 0xd3e6bb24, 2, 4, (4, 15, 10)), (0xc71df094702bd4, 0x240e31da, 1, 2, (15, 9, 0))]


@pytest.mark.parametrize("step,instance,d,comp,cell", ZERO_RADIUS)
def test_noise_of_a_zero_radius(orc, step, instance, d, comp, cell):
    """The one zero a Box-Muller radius can be, -0: both values are the oracle's zeros, signs included."""
    from fhdex_amd import compressible as fc
    from fhdex_amd import lib as L
    p = P.argon_gas(16).params
    print(f"case zero radius, face direction {d}", flush=True)
    st = orc.HostState(p)
    orc.fill_noise(p, st, 9, step, instance)
    i, j, k = cell
    assert st.sA[d][comp, k, j, i] == 0.0 and st.sB[d][comp, k, j, i] == 0.0
    ctx = L.Context(p)
    nz = fc.NoiseSets(p)
    fc.fill_noise(ctx, nz, 9, step, instance)
    got = [(nz.A[q].t.cpu().numpy(), nz.B[q].t.cpu().numpy()) for q in range(3)]
    ctx.close()
    for q in range(3):
        for dev, host in zip(got[q], (st.sA[q], st.sB[q])):
            np.testing.assert_array_equal(dev, host)
            assert np.array_equal(np.signbit(dev), np.signbit(host))
