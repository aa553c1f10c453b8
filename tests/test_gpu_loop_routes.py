"""Wilson loops on both sides of the rule that chooses planes or multiplied-out links, and of the sizes
at which the latter keep two line fields: both entry points against the FP64 oracle and each other, bit
for bit, for lines that can be inverted, badly conditioned ones and lines that cannot be.
Bars: FP64 1e-13 (a few roundings of up to ~40 products), FP32 5e-5."""
import ctypes

import numpy as np
import pytest

import sun_amd
from test_gpu_line_limits import correlators, lines, stretched
from test_gpu_parity import BETAS, thermalised
from test_zz_no_alloc import noalloc_loops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (2, 4), (3, 4), (4, 4)])
@pytest.mark.parametrize("dims,loops", [((4, 6, 4, 8), ((0, 0), (1, 2), (4, 1), (4, 8))),
                                        ((6, 6, 4, 30), ((1, 30), (4, 9))), ((12, 12, 12, 14), ((1, 1), (5, 7)))], ids=str)
def test_routes(ctx, oracle, nc, prec, dims, loops):
    stream = sun_amd.new_stream()
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        for kind in ("unitary", "stretched", "singular"):
            U = oracle.hot_start(nc, dims, 7, 18)
            at = U.shape[1] // 3
            if kind == "stretched":
                U[3, at:at + 9] = np.diag([4, 0.25, 1, 1][:nc]) @ U[3, at:at + 9]
            elif kind == "singular":
                U[3, at] = 0.0
            lat.from_host(U)
            U = lat.to_host()
            for rmax, tmax in loops:
                got = lat.wilson_loops(rmax, tmax, stream)
                assert np.array_equal(got, noalloc_loops(lat, rmax, tmax, stream)), (kind, rmax, tmax)
                want = oracle.wilson_loops(U, dims, rmax, tmax)
                bar = (1e-13 if prec == 8 else 5e-5) * max(1.0, np.abs(want).max())
                assert np.abs(got - want).max() <= bar, (kind, rmax, tmax)
    sun_amd.lib().sun_stream_destroy(stream)


def launches(lat, rmax, tmax):
    """kernels of the call by either route: planes launch those of the other route besides"""
    hip, stream, graph, n = sun_amd.lib(), sun_amd.new_stream(), ctypes.c_void_p(), ctypes.c_size_t(0)
    out = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(out), ctypes.c_size_t(16 * (rmax + 1) * (tmax + 1))) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    lat.wilson_loops_noalloc(rmax, tmax, out.value, stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipFree(out) == 0
    sun_amd.lib().sun_stream_destroy(stream)
    return n.value


# extents at which a workgroup takes one site or several, threads without a time, T in one chunk and more
@pytest.mark.parametrize("dims,rmax,tmax", [((4, 4, 4, 70), 4, 17), ((2, 4, 2, 34), 2, 34), ((10, 10, 12, 10), 10, 10),
                                            ((6, 6, 6, 20), 6, 9), ((2, 2, 2, 200), 2, 199), ((18, 4, 6, 12), 4, 12)], ids=str)
@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (2, 4), (3, 4), (4, 4)])
def test_planes_at_their_edges(ctx, oracle, nc, prec, dims, rmax, tmax):
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        for kind in ("near", "scaled"):  # scaled: the inverses, of a condition that FP64 takes
            U = oracle.hot_start(nc, dims, 8, 18)
            if kind == "scaled":
                U[3] *= np.random.default_rng(3).uniform(0.8, 1.1, U.shape[1])[:, None, None]
            lat.from_host(U)
            U = lat.to_host()
            assert launches(lat, rmax, tmax) > rmax + 2
            got = lat.wilson_loops(rmax, tmax)
            want = oracle.wilson_loops(U, dims, rmax, tmax)
            bar = (1e-13 if prec == 8 else 5e-5) * max(1.0, np.abs(want).max())
            assert np.abs(got - want).max() <= bar, kind


@pytest.mark.parametrize("nc,prec", [(2, 8), (3, 8), (4, 8), (2, 4), (3, 4), (4, 4)])
def test_planes_keep_precision(ctx, oracle, nc, prec):
    """Links that lean to one side and a badly conditioned slice, as for the correlators (test_gpu_line_limits.py,
    with its bars): a call that goes by planes, unless the condition is too bad for FP64."""
    dims, rmax, tmax = (4, 4, 6, 16), 4, 16
    with sun_amd.Lattice(ctx, nc, dims, BETAS[nc], 18, prec) as lat:
        for kind in ("lean", "stretched", "badly stretched"):
            if kind == "lean":
                U = thermalised(oracle, nc, dims, 18).copy()
                U[3] *= 1 + (1e-15 if prec == 8 else 4e-8)
                bar = 4e-15 if prec == 8 else 4e-8
            else:
                U = stretched(oracle, nc, dims, (90 if prec == 8 else 3.8) if kind == "badly stretched" else 1.5)
                bar = 1e-14 if prec == 8 else 6e-8
            lat.from_host(U)
            U = lat.to_host()
            assert launches(lat, rmax, tmax) > rmax + 2
            got = lat.wilson_loops(rmax, tmax).real
            want = np.array([correlators(U, dims, lines(oracle, U, dims, r), r, tmax)[0] for r in range(rmax + 1)])
            scale = 1.0 if kind == "lean" else np.abs(want).max(0)
            assert (np.abs(got - want) <= bar * scale).all(), kind
