"""Operator correlators on each side of the rules that choose a kernel and the layout of the operator
fields: few T (every link multiplied out, fields in planes or as matrices) and more, volumes below
and above the lines where row blocks give way to tiles and to staged operators, for lines that can be
inverted and lines that cannot.  Against the FP64 oracle: FP64 1e-12 (sums in another order), FP32
5e-5 (products of up to ~40 FP32 links) of the largest correlator."""
import numpy as np
import pytest

import sun_amd
from test_gpu_parity import BETAS

pytestmark = pytest.mark.gpu

BAR = {8: 1e-12, 4: 5e-5}


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (2, 4), (3, 4), (4, 4)])
@pytest.mark.parametrize("family,dims,tmaxs", [
    (0, (6, 4, 6, 10), (0, 3, 6, 7)), (0, (12, 10, 12, 10), (5, 6)), (0, (16, 16, 16, 18), (2, 4)),
    (1, (6, 4, 6, 10), (0, 1, 2, 5)), (1, (12, 12, 12, 12), (1, 3))], ids=str)
def test_routes(ctx, oracle, family, dims, tmaxs, nc, prec):
    r, mu = 2, 1
    big = int(np.prod(dims)) > 1 << 14
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        U = oracle.hot_start(nc, dims, 5, 18)
        for kind in ("unitary", "singular"):
            if kind == "singular":
                U[3, U.shape[1] // 3] = 0.0
            lat.from_host(U)
            U = lat.to_host()
            fields = oracle.wlop_fields(U, dims, family, r, mu)
            for tmax in tmaxs[-1:] if big else tmaxs:
                with sun_amd.WilsonLoopOps(lat, family, tmax) as ops:
                    ops.fields(r, mu)
                    got = ops.fields_to_host()
                    if prec == 8:
                        assert np.array_equal(got, fields)
                    else:
                        assert np.abs(got - fields).max() <= 5e-5
                    ops.correlate(r, mu)
                    got = ops.read()
                want = oracle.wlop_correlate(U, dims, fields, r, mu, tmax)
                assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max(), (kind, tmax)


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (4, 4)])
def test_shared_products_in_planes(ctx, oracle, nc, prec):
    """sun_wilson_loops_ops of few T: the A0 fields from shared products, written as planes; a ragged volume"""
    dims = (6, 6, 4, 10)
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        U = oracle.hot_start(nc, dims, 6, 18)
        lat.from_host(U)
        U = lat.to_host()
        got = lat.wilson_loops_ops(4, 2, 0)
    want = oracle.wilson_loops_ops(U, dims, 4, 2, 0)
    assert np.abs(got - want).max() <= BAR[prec] * np.abs(want).max()
