"""Long generation calls replay a captured iteration (shorter ones launch it): the same rows and
links as without a graph, for one lattice (with both kinds of iterations) and for a batch over
several streams, replayed in two calls with eager work between them."""
import numpy as np
import pytest

import sun_amd

pytestmark = pytest.mark.gpu

ITERS = 30


@pytest.mark.parametrize("nc,storage,prec", [(2, 18, 4), (3, 12, 4), (3, 18, 8)])
def test_long_calls_replay_a_graph(ctx, nc, storage, prec):
    beta = {2: 2.4, 3: 6.0}[nc]
    out = []
    for graph in (False, True):
        with sun_amd.Lattice(ctx, nc, (4, 6, 4, 8), beta, storage, prec) as lat:
            lat.cold_start()
            every = 1 if storage == 12 else 3
            rows = [lat.generate(7, ITERS, n_or=1, reunit_every=every, use_graph=graph)]
            lat.heatbath(7, 1000)
            rows.append(lat.generate(7, ITERS, n_or=1, reunit_every=every, first_sweep=ITERS, use_graph=graph))
            out.append((rows, lat.to_host()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_long_batch_calls_replay_a_graph(ctx):
    dims = [(4, 4, 4, 4), (6, 4, 4, 8), (8, 8, 8, 8), (4, 4, 6, 6)]
    out = []
    for graph in (False, True):
        lats = [sun_amd.Lattice(ctx, 3, d, 5.9, 12, 4) for d in dims]
        for lat in lats:
            lat.cold_start()
        batch = sun_amd.Batch(ctx, lats, [3, 4, 5, 6])
        rows = [batch.generate(0, ITERS, n_or=1, use_graph=graph)]
        batch.overrelax()
        rows.append(batch.generate(ITERS, ITERS, n_or=1, use_graph=graph))
        out.append((rows, [lat.to_host() for lat in lats]))
        batch.close()
        for lat in lats:
            lat.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))


# past the lattices whose updates share staples: bricks, linear order and the pipelined kernels of
# their default shapes, every storage
@pytest.mark.parametrize("nc,storage,prec,dims", [(2, 18, 4, (16, 16, 16, 18)), (3, 12, 4, (32, 16, 16, 40)),
                                                  (3, 8, 4, (16, 16, 16, 18)), (3, 18, 4, (32, 16, 16, 40)),
                                                  (3, 18, 8, (16, 16, 16, 10)), (3, 12, 8, (16, 16, 16, 10)),
                                                  (3, 8, 8, (16, 16, 16, 18)), (4, 18, 4, (12, 12, 12, 12))])
def test_large_lattices_replay_a_graph(ctx, nc, storage, prec, dims):
    out = []
    for graph in (False, True):
        with sun_amd.Lattice(ctx, nc, dims, {2: 2.4, 3: 6.0, 4: 10.8}[nc], storage, prec) as lat:
            lat.hot_start(3)
            rows = []
            for call in range(2):
                rows.append(lat.generate(7, 24, n_or=1, reunit_every=1 if storage == 8 else 5,
                                         first_sweep=24 * call, use_graph=graph))
                lat.overrelax()
            out.append((rows, lat.to_host()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("nc,storage,prec,count", [(3, 12, 4, 24), (3, 8, 4, 36), (4, 18, 4, 10)])
def test_chunks_on_several_streams_replay_a_graph(ctx, nc, storage, prec, count):
    """16^4 lattices of 300 MB together: more than three chunks of a third of the 256 MB cache, whose launches
    the captured iteration forks over the batch's streams"""
    assert sun_amd.lattice_bytes(nc, (16,) * 4, storage, prec) * count > 3 * (256 << 20) // 3
    out = []
    for graph in (False, True):
        lats = [sun_amd.Lattice(ctx, nc, (16,) * 4, {3: 5.9, 4: 10.8}[nc], storage, prec) for _ in range(count)]
        for i, lat in enumerate(lats):
            lat.hot_start(i)
        batch = sun_amd.Batch(ctx, lats, range(count))
        rows = []
        for call in range(2):
            rows.append(batch.generate(24 * call, 24, n_or=1, use_graph=graph))
            batch.overrelax()
        out.append((rows, [lat.plaquette() for lat in lats], lats[0].to_host(), lats[-1].to_host()))
        batch.close()
        for lat in lats:
            lat.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2]) and np.array_equal(out[0][3], out[1][3])


def test_many_chunks_in_flight_at_the_end_of_a_call(ctx):
    """Eleven chunks and iterations of 10 ms: a call has launched all its replays long before the first is done,
    and keeps their graph until the last is."""
    lats = [sun_amd.Lattice(ctx, 3, (16,) * 4, 5.9, 18, 8) for _ in range(24)]
    batch = sun_amd.Batch(ctx, lats, range(24))
    rows = []
    for graph in (False, True):
        for i, lat in enumerate(lats):
            lat.hot_start(i)
        rows.append([batch.generate(0, 24, n_or=3, use_graph=graph), batch.generate(24, 40, n_or=3, use_graph=graph)])
    assert all(np.array_equal(a, b) for a, b in zip(*rows))
    batch.close()
    for lat in lats:
        lat.close()
