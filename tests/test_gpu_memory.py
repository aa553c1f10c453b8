"""Device memory of operator handles: no more than the parts that a handle uses, and, where the card has
no room for the parts that only make it faster, a handle without them."""
import ctypes

import numpy as np
import pytest

import sun_amd

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert sun_amd.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec,family,tmax,lines,aux", [(8, 1, 8, True, False), (8, 1, 1, False, False),
                                                        (4, 1, 8, True, True), (4, 1, 2, False, True),
                                                        (8, 0, 2, False, False), (4, 0, 10, True, False)])
def test_handles_hold_what_they_use(prec, family, tmax, lines, aux):
    dims = (16, 16, 16, 32)
    V, nop = int(np.prod(dims)), sun_amd.WLOP_NOPS[family]
    most = nop * V * 18 * prec + nop * nop * (tmax + 1) * (V // 256 + 1) * 8
    if lines:
        most += V // dims[3] * (2 * dims[3] + tmax) * 144
    if aux:
        most += 14 * V * 18 * prec
    with sun_amd.Context(0) as c, sun_amd.Lattice(c, 3, dims, 6.0, 18, prec) as lat:
        before = free_bytes()
        with sun_amd.WilsonLoopOps(lat, family, tmax):
            held = before - free_bytes()
    assert held <= most + (8 << 20)


def test_operators_where_memory_is_short():
    dims, r, mu, tmax = (32, 32, 32, 32), 3, 1, 8
    with sun_amd.Context(0) as c, sun_amd.Lattice(c, 3, dims, 6.0, 18, 4) as lat:
        lat.hot_start(3)
        lat.heatbath(3, 0)

        def measure():
            with sun_amd.WilsonLoopOps(lat, sun_amd.WLOP_33, tmax) as ops:
                ops.fields(r, mu)
                ops.correlate(r, mu)
                pairs = ops.read()
            return pairs, lat.wilson_loops(2, 4)  # with the handle's block idle or given back

        want, loops = measure()  # 3.5 GB: operators and sums 2.1, scratch 1.1, time lines 0.3
        filler = ctypes.c_void_p()
        size = ctypes.c_size_t(free_bytes() - 2_900_000_000)
        if sun_amd.lib().hipMalloc(ctypes.byref(filler), size) != 0:
            pytest.skip("the rest of the card cannot be taken in one piece")
        try:
            got, again = measure()
        finally:
            assert sun_amd.lib().hipFree(filler) == 0
    assert np.abs(got - want).max() <= 5e-5 * np.abs(want).max()
    assert np.abs(again - loops).max() <= 5e-5
