"""Loop measurements whose temporal links are not unitary, and the edges of the kernels that
move operators along time lines: temporal links scattered away from SU(N) (inverted lines),
a zero temporal link (lines that cannot be inverted: the kernels that multiply the links out
for every T take the call), more T and more times than one workgroup takes at once, and
spatial volumes below and above one wavefront of lines.  Against the FP64 oracle.

Tolerances, relative to the largest element: FP64 1e-11 (rounding 1e-16 of ~40 products,
times the square of the condition number of up to 100), FP32 5e-5 (products of up to ~40 FP32
links)."""
import numpy as np
import pytest

import sun_amd
from test_gpu_parity import BETAS, load_config, thermalised

pytestmark = pytest.mark.gpu

BAR = {8: 1e-11, 4: 5e-5}


def field(lat, oracle, nc, dims, kind, seed=3):
    U = thermalised(oracle, nc, dims, 18).copy()
    rng = np.random.default_rng(seed)
    if kind == "scattered":
        U[3] *= rng.uniform(0.7, 1.1, U.shape[1])[:, None, None]
        U[3] += 0.02 * (rng.normal(size=U[3].shape) + 1j * rng.normal(size=U[3].shape))
    elif kind == "singular":
        U[3, U.shape[1] // 3] = 0.0
    lat.from_host(U)
    return lat.to_host()


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (3, 4), (4, 8), (4, 4)])
@pytest.mark.parametrize("kind", ["scattered", "singular"])
@pytest.mark.parametrize("family", [0, 1], ids=["A0", "33"])
def test_correlator_of_non_unitary_lines(ctx, oracle, nc, prec, kind, family):
    dims, r, mu, tmax = (4, 2, 6, 8), 3, 2, 8
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        U = field(lat, oracle, nc, dims, kind)
        with sun_amd.WilsonLoopOps(lat, family, tmax) as ops:
            ops.fields(r, mu)
            ops.correlate(r, mu)
            got = ops.read()
    want = oracle.wlop_correlate(U, dims, oracle.wlop_fields(U, dims, family, r, mu), r, mu, tmax)
    assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max()


@pytest.mark.parametrize("dims,tmax", [((2, 2, 2, 2), 2), ((2, 4, 2, 34), 34), ((4, 4, 4, 70), 17), ((6, 6, 4, 20), 4),
                                       ((8, 8, 6, 6), 5)], ids=str)
@pytest.mark.parametrize("prec,family", [(8, 0), (8, 1), (4, 1)], ids=["f64-A0", "f64-33", "f32-33"])
def test_correlator_extents(ctx, oracle, dims, tmax, prec, family):
    r, mu = 2, 1
    with sun_amd.Lattice(ctx, 3, dims, 6.0, 18, prec) as lat:
        U = field(lat, oracle, 3, dims, "unitary")
        with sun_amd.WilsonLoopOps(lat, family, tmax) as ops:
            ops.fields(r, mu)
            ops.correlate(r, mu)
            ops.correlate(r, mu)  # adds to the accumulator
            got = ops.read()
    want = 2 * oracle.wlop_correlate(U, dims, oracle.wlop_fields(U, dims, family, r, mu), r, mu, tmax)
    assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max()


@pytest.mark.parametrize("nc,prec", [(2, 8), (2, 4), (3, 8), (3, 4), (4, 8), (4, 4)])
@pytest.mark.parametrize("kind", ["scattered", "singular"])
def test_wilson_loops_of_non_unitary_lines(ctx, oracle, nc, prec, kind):
    dims, rmax, tmax = (4, 2, 6, 8), 2, 8
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        U = field(lat, oracle, nc, dims, kind)
        got = lat.wilson_loops(rmax, tmax)
    want = oracle.wilson_loops(U, dims, rmax, tmax)
    assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max()


@pytest.mark.parametrize("dims,tmax", [((2, 2, 2, 2), 2), ((2, 4, 2, 34), 34), ((4, 4, 4, 70), 17), ((6, 6, 4, 20), 0),
                                       ((8, 6, 10, 6), 5), ((2, 2, 2, 516), 3)], ids=str)
@pytest.mark.parametrize("storage,prec", [(18, 8), (12, 4)], ids=["f64", "f32"])
def test_wilson_loops_extents(ctx, oracle, dims, tmax, storage, prec):
    with sun_amd.Lattice(ctx, 3, dims, 6.0, storage, prec) as lat:
        U = load_config(lat, thermalised(oracle, 3, dims, storage))
        rmax = min(dims[:3])
        got = lat.wilson_loops(rmax, tmax)
        assert np.array_equal(got, lat.wilson_loops(rmax, tmax))
    want = oracle.wilson_loops(U, dims, rmax, tmax)
    assert np.abs(got - want).max() <= BAR[prec]


@pytest.mark.parametrize("family,dims,rmax", [(0, (6, 6, 4, 10), 4), (1, (6, 6, 4, 10), 4), (0, (2, 2, 2, 6), 2),
                                              (1, (2, 2, 2, 6), 2)], ids=str)
@pytest.mark.parametrize("nc,storage,prec", [(2, 18, 8), (3, 18, 8), (3, 12, 4), (4, 18, 4)])
def test_operator_loops_of_ragged_volumes(ctx, oracle, family, dims, rmax, nc, storage, prec):
    """the fields from shared products: volumes that are no multiple of 64 or 256 sites, radii up
    to the extent, sides of eight links around extents of 2, 4 and 6"""
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], storage, prec) as lat:
        U = load_config(lat, thermalised(oracle, nc, dims, storage))
        got = lat.wilson_loops_ops(rmax, 5, family)
    want = oracle.wilson_loops_ops(U, dims, rmax, 5, family)
    assert np.abs(got - want).max() <= (1e-12 if prec == 8 else 2e-5)


# the numbers of T at which the matrix-core correlator takes one more column of tiles or workgroup
@pytest.mark.parametrize("tmax", [5, 6, 8, 9, 11, 12, 14, 15, 17, 18, 20])
@pytest.mark.parametrize("nc,prec,family,kind", [(3, 8, 0, "unitary"), (3, 8, 0, "scattered"), (2, 4, 0, "scattered"),
                                                 (3, 8, 1, "unitary"), (3, 4, 1, "scattered"), (4, 8, 1, "scattered")])
def test_correlator_tiles(ctx, oracle, nc, prec, family, kind, tmax):
    dims, r, mu = (2, 4, 2, 22), 1, 1
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        U = field(lat, oracle, nc, dims, kind)
        with sun_amd.WilsonLoopOps(lat, family, tmax) as ops:
            ops.fields(r, mu)
            ops.correlate(r, mu)
            got = ops.read()
    want = oracle.wlop_correlate(U, dims, oracle.wlop_fields(U, dims, family, r, mu), r, mu, tmax)
    assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max()
