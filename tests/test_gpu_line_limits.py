"""Time lines at the limits of what the loop measurements may invert: temporal links of a scale
whose lines leave the range of FP32, against the FP64 oracle.

A loop of T times is of the order f^2T: its error is measured against that times the largest
correlator at T = 0.  FP32: 5e-5, products of up to ~50 FP32 links."""
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
