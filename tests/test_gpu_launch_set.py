"""A launch shape that the caller sets is the shape that runs, also where small lattices otherwise
run the kernel that shares a link's staple among waves: seen from the kernel node that an update
leaves in a captured graph."""
import ctypes

import pytest

import sun_amd

pytestmark = pytest.mark.gpu

DIMS = (8, 8, 8, 16)
VARIANTS = [(2, 18, 8, 448), (3, 18, 4, 448), (3, 12, 4, 448), (3, 8, 8, 448), (4, 18, 8, 256)]


class KernelNode(ctypes.Structure):
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def threads(lat, kernel):
    """threads of a workgroup of the lattice's heatbath (0) or overrelaxation (1) launch"""
    hip, stream, graph, n = sun_amd.lib(), sun_amd.new_stream(), ctypes.c_void_p(), ctypes.c_size_t(1)
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    if kernel:
        lat.overrelax_sub(0, 1, stream)
    else:
        lat.heatbath_sub(3, 0, 0, 1, stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    node, got = ctypes.c_void_p(), KernelNode()
    assert hip.hipGraphGetNodes(graph, ctypes.byref(node), ctypes.byref(n)) == 0 and n.value == 1
    assert hip.hipGraphKernelNodeGetParams(node, ctypes.byref(got)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    sun_amd.lib().sun_stream_destroy(stream)
    return got.block[0]


@pytest.mark.parametrize("nc,storage,prec,split", VARIANTS)
def test_set_shape_runs(ctx, nc, storage, prec, split):
    with sun_amd.Lattice(ctx, nc, DIMS, 6.0, storage, prec) as lat:
        for kernel in (0, 1):
            assert threads(lat, kernel) == split
            lat.set_launch(kernel, 128)
            assert threads(lat, kernel) == 128
            lat.set_launch(kernel, 0, (2, 1, 1))
            assert threads(lat, kernel) == 64


@pytest.mark.parametrize("nc,storage,prec,split", VARIANTS)
def test_context_shape_runs(nc, storage, prec, split):
    with sun_amd.Context(0) as c:
        c.set_launch(nc, DIMS, 6.0, storage, prec, 1, 192)
        with sun_amd.Lattice(c, nc, DIMS, 6.0, storage, prec) as lat:
            assert threads(lat, 0) == split and threads(lat, 1) == 192


def test_autotuner_keeps_shared_staples():
    with sun_amd.Context(0, 0, 1) as c, sun_amd.Lattice(c, 3, DIMS, 6.0, 12, 4) as lat:
        lat.cold_start()
        lat.overrelax()
        assert threads(lat, 0) == threads(lat, 1) == 448
