"""The kernels' division by a kept reciprocal gives the IEEE quotient.

conservedToPrimitive divides five values of a cell by its density, and mass fractions by the run's
molar masses, so its results against numpy's IEEE division show the helper bit for bit: quotients that
lie as close to a rounding boundary as 53-bit operands allow, ordinary ones over 2^+-300, zeros of both
signs, infinities, NaN and zero divisors.  No tolerance: the values are equal or the test fails.
Likewise the noise whose Box-Muller radius is zero, against the oracle's.
"""
import numpy as np
import pytest

from fhdex_amd import params as P

pytestmark = pytest.mark.gpu

N = (24, 16, 16)
CELLS = N[0] * N[1] * N[2]


def hard_pairs(count, rng):
    """Operand pairs whose quotient is within 2^-53 of its last place of a rounding boundary: for odd b, a is
    +-1, +-3, ... times the inverse of 2^54 modulo b, kept where the quotient's 54th bit is set."""
    a, b = [], []
    while len(a) < count:
        d = int(rng.integers(2 ** 52, 2 ** 53)) | 1
        inv = pow(2 ** 54, -1, d)
        for e in (1, -1, 3, -3):
            n = e * inv % d
            if 2 ** 52 <= n < d and ((n << 54) - e) // d % 2 == 1:
                a.append(float(n))
                b.append(float(d))
    return np.array(a[:count]), np.array(b[:count])


def values(kind, rng):
    if kind == "hard":
        return hard_pairs(CELLS, rng)
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
