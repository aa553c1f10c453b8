"""Time lines at the limits of what the loop measurements may invert: temporal links of a scale
whose lines leave the range of FP32, against the FP64 oracle.

A loop of T times is of the order f^2T: its error is measured against that times the largest
correlator at T = 0.  FP32: 5e-5, products of up to ~50 FP32 links.

And lines that are unitary but for the rounding of their links, which leans to one side as after
many updates without reunitarisation: a loop takes the T links that it has, not the X3 of its
lines.  The errors of single loops (a few roundings, 1e-16 and 6e-8) average out over the loops of
a volume, so the bars are a few roundings: FP64 4e-15 of the loops and 6e-15 of the largest
correlator, FP32 4e-8 and 1e-7.  The deviations of whole lines are 3e-14 and 5e-7.

And lines that a single time slice makes badly conditioned: through the inverses of such lines the
loops that do not touch the slice lose the condition number's square, 2e4 roundings in FP64 and 60
in FP32; multiplied out they have a few.  Bars: 1e-14 and 6e-8 of the largest correlator of each T."""
import numpy as np
import pytest

import sun_amd
from test_gpu_parity import BETAS, thermalised

pytestmark = pytest.mark.gpu


# f^-2(X3 - 1) is 1e57, 1e38 and 1e39
@pytest.mark.parametrize("scale,times", [(0.25, 48), (0.5, 64), (0.7, 128)])
@pytest.mark.parametrize("nc,family", [(2, 0), (3, 0), (3, 1)])
def test_correlator_of_lines_out_of_range(ctx, oracle, nc, family, scale, times):
    dims, r, mu, tmax = (2, 2, 2, times), 2, 1, 16
    U = thermalised(oracle, nc, dims, 18).copy()
    U[3] *= scale
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, 4) as lat:
        lat.from_host(U)
        U = lat.to_host()
        with sun_amd.WilsonLoopOps(lat, family, tmax) as ops:
            ops.fields(r, mu)
            ops.correlate(r, mu)
            got = ops.read()
    want = oracle.wlop_correlate(U, dims, oracle.wlop_fields(U, dims, family, r, mu), r, mu, tmax)
    bar = 5e-5 * np.abs(want[:, 0]).max() * scale ** (2.0 * np.arange(tmax + 1))
    assert (np.abs(got - want).max(0) <= bar).all()


def correlators(U, dims, fields, rs, tmax):
    """sum over the spatial directions of Tr(O_i t1 (t0 O_j(x + T))^+) / (3 N V), fields[mu][i] the operators
    of length rs[mu], in 80 bits (the oracle's running sums of values next to 1 are good to 2e-14)"""
    n, V = U.shape[-1], U.shape[1]
    lex = np.arange(V)
    x = np.stack([lex // int(np.prod(dims[:d])) % dims[d] for d in range(4)])
    order = np.argsort(x.sum(0) & 1, kind="stable")
    eo = np.empty(V, int)
    eo[order] = lex
    x = x[:, order]

    def moved(mu, d):
        y = x.copy()
        y[mu] = (y[mu] + d) % dims[mu]
        return eo[sum(y[k] * int(np.prod(dims[:k])) for k in range(4))]

    def mm(a, b):
        return sum(a[..., :, k, None] * b[..., k, None, :] for k in range(n))

    out = 0
    for mu in range(3):
        ops = fields[mu].astype(np.clongdouble)
        t = np.broadcast_to(np.eye(n, dtype=np.clongdouble), (V, n, n))
        w = []
        for T in range(tmax + 1):
            left = mm(ops, t[moved(mu, rs)]).reshape(len(ops), -1)
            right = mm(t, ops[:, moved(3, T)]).reshape(len(ops), -1)
            w.append(left.real @ right.real.T + left.imag @ right.imag.T)
            t = mm(t, U[3].astype(np.clongdouble)[moved(3, T)])
        out = out + np.stack([a.reshape(-1) for a in w], -1) / (3 * n * V)
    return out


def lines(oracle, U, dims, r):
    """the straight lines of r links, slot 0 of the operators"""
    if r == 0:
        return [np.broadcast_to(np.eye(U.shape[-1]), (1, *U.shape[1:])) for mu in range(3)]
    return [oracle.wlop_fields(U, dims, 0, r, mu)[:1] for mu in range(3)]


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (2, 4), (3, 4), (4, 4)])
def test_links_that_lean_to_one_side(ctx, oracle, nc, prec):
    dims = (4, 4, 6, 16 if prec == 8 else 8)
    U = thermalised(oracle, nc, dims, 18).copy()
    U[3] *= 1 + (1e-15 if prec == 8 else 4e-8)
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        lat.from_host(U)
        U = lat.to_host()
        got = lat.wilson_loops(2, 8)
        ops = [lat.wilson_loops_ops(2, 8, family) for family in (0, 1)]
    for r in range(3):
        want = correlators(U, dims, lines(oracle, U, dims, r), r, 8)[0]
        assert np.abs(got[r].real - want).max() <= (4e-15 if prec == 8 else 4e-8)
    for family in (0, 1):
        fields = [oracle.wlop_fields(U, dims, family, 2, mu) for mu in range(3)]
        want = correlators(U, dims, fields, 2, 8)
        assert np.abs(ops[family][0] - want).max() <= (6e-15 if prec == 8 else 1e-7) * np.abs(want).max()


def stretched(oracle, nc, dims, condition):
    """the links of the first time slice times a matrix of |m| |m^-1| / N = condition (not a diagonal one: what
    that costs, row by row, its inverse gives back)"""
    U = thermalised(oracle, nc, dims, 18).copy()
    a = np.roots([1, -(nc * condition - (nc - 2)), 1]).real.max() ** 0.5  # (a^2 + 1/a^2 + N - 2) / N
    first = np.arange(U.shape[1]) % (U.shape[1] // 2) < U.shape[1] // 2 // dims[3]
    rng = np.random.default_rng(1)
    left, right = (np.linalg.qr(rng.normal(size=(nc, nc)) + 1j * rng.normal(size=(nc, nc)))[0] for _ in range(2))
    U[3, first] = left @ np.diag([a, 1 / a, 1, 1][:nc]) @ right @ U[3, first]
    return U


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (2, 4), (3, 4)])
def test_badly_conditioned_lines(ctx, oracle, nc, prec):
    dims, tmax = (2, 2, 2, 16), 8
    U = stretched(oracle, nc, dims, 90 if prec == 8 else 3.8)
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        lat.from_host(U)
        U = lat.to_host()
        got = lat.wilson_loops(2, tmax).real
        ops = [lat.wilson_loops_ops(2, tmax, family)[0] for family in (0, 1)]
    bar = 1e-14 if prec == 8 else 6e-8
    want = np.array([correlators(U, dims, lines(oracle, U, dims, r), r, tmax)[0] for r in range(3)])
    assert (np.abs(got - want).max(0) <= bar * np.abs(want).max(0)).all()
    for family in (0, 1):
        want = correlators(U, dims, [oracle.wlop_fields(U, dims, family, 2, mu) for mu in range(3)], 2, tmax)
        assert (np.abs(ops[family] - want).max(0) <= bar * np.abs(want).max(0)).all()
