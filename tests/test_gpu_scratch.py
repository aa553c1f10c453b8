"""Measurements take their scratch from blocks that earlier calls gave back: the same results in
memory that calls of other sizes and kinds have written, and from several threads at once, each
with its own lattice and stream."""
import ctypes
import threading

import numpy as np
import pytest

import sun_amd

pytestmark = pytest.mark.gpu

KINDS = [((4, 4, 4, 8), 3, 12, 4), ((6, 4, 8, 4), 3, 18, 8), ((8, 8, 8, 8), 2, 18, 4), ((4, 6, 4, 8), 4, 18, 8)]


def chain(lat, stream=None):
    lat.generate(11, 2, n_or=1, stream=stream)
    links = [lat.to_host()]
    out = [lat.wilson_loops(3, 3, stream=stream)]
    lat.hyp_smear((0.75, 0.6, 0.3), 1, 4, stream=stream)
    out += [lat.wilson_loops(2, 2, stream=stream), lat.wilson_loops_ops(2, 2, 0, stream=stream)]
    lat.ape_smear(0.2, 3, 4, stream=stream)
    links.append(lat.to_host())
    lat.from_host(links[0])
    return out + [lat.wilson_loops(3, 3, stream=stream)] + links


def fresh(kind):
    with sun_amd.Context() as ctx, sun_amd.Lattice(ctx, kind[1], kind[0], 6.0, kind[2], kind[3]) as lat:
        lat.cold_start()
        return chain(lat)


@pytest.fixture(scope="module")
def want():
    return [fresh(kind) for kind in KINDS]


def same(got, want):
    assert all(np.array_equal(a, b) for a, b in zip(got, want))


def test_scratch_of_other_calls(want):
    with sun_amd.Context() as ctx:
        for order in ((0, 1, 2, 3), (2, 0, 3, 1, 1)):
            for i in order:
                dims, nc, storage, prec = KINDS[i]
                with sun_amd.Lattice(ctx, nc, dims, 6.0, storage, prec) as lat:
                    lat.cold_start()
                    same(chain(lat), want[i])


def test_scratch_of_several_threads(want):
    got = [None] * len(KINDS)
    with sun_amd.Context() as ctx:
        lats = [sun_amd.Lattice(ctx, k[1], k[0], 6.0, k[2], k[3]) for k in KINDS]
        streams = [ctypes.c_void_p() for _ in KINDS]
        for lat, st in zip(lats, streams):
            assert sun_amd.lib().sun_stream_create(ctypes.byref(st)) == 0
            lat.cold_start()
            lat.to_host()

        def work(i):
            got[i] = chain(lats[i], streams[i])

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(KINDS))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for g, w in zip(got, want):
            same(g, w)
        for lat, st in zip(lats, streams):
            lat.close()
            assert sun_amd.lib().sun_stream_destroy(st) == 0
