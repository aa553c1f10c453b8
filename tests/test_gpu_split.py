"""Small lattices share a link's staple among waves: the links are those of the batched kernels,
which compute it in one, bit for bit, on both sides of the largest lattice that is shared."""
import numpy as np
import pytest

import sun_amd

pytestmark = pytest.mark.gpu

VARIANTS = [(2, 18, 8), (3, 18, 4), (3, 12, 4), (3, 8, 4), (3, 18, 8), (3, 12, 8), (3, 8, 8), (4, 18, 8)]
# fewer than 64 links of a parity, a ragged last workgroup, 256 workgroups and one more, 512 and more
DIMS = [(2, 2, 2, 2), (10, 6, 14, 8), (16, 16, 16, 8), (4, 258, 8, 4), (16, 16, 16, 16), (16, 16, 16, 18)]


@pytest.mark.parametrize("nc,storage,prec", VARIANTS)
@pytest.mark.parametrize("dims", DIMS)
def test_split_updates_equal_batched(ctx, nc, storage, prec, dims):
    beta = {2: 1.2, 3: 5.7, 4: 10.2}[nc]  # SU(2): many rejected first attempts, al <= 2 among them
    with sun_amd.Lattice(ctx, nc, dims, beta, storage, prec) as a, \
            sun_amd.Lattice(ctx, nc, dims, beta, storage, prec) as b:
        batch = sun_amd.Batch(ctx, [b], [9])
        a.hot_start(5)
        b.hot_start(5)
        for sweep in range(3):
            a.heatbath(9, sweep)
            batch.heatbath([sweep])
            a.overrelax()
            batch.overrelax()
        assert np.array_equal(a.to_host(), b.to_host())
        batch.close()
