"""The SU(N) projection of the smearing kernels at the ends of the number range: it does not
depend on the scale of the links (a power of two), also where the norms it takes the reciprocal
root of are below what the native instruction reads, and a zero matrix is left alone."""
import numpy as np
import pytest

import sun_amd

pytestmark = pytest.mark.gpu

DIMS = (4, 6, 4, 8)


def links(nc):
    rng = np.random.default_rng(17 + nc)
    v = int(np.prod(DIMS))
    u = np.eye(nc) + 0.3 * (rng.standard_normal((4, v, nc, nc)) + 1j * rng.standard_normal((4, v, nc, nc)))
    q, r = np.linalg.qr(u)
    q *= (np.einsum("...ii->...i", r) / np.abs(np.einsum("...ii->...i", r)))[..., None, :]
    return q / np.linalg.det(q)[..., None, None] ** (1 / nc)


# Without the staple (cubic in the scale): the links themselves are projected.  SU(3) starts from
# the identity: |r|^2 goes as the square of the scale, else as its fourth power.
# Bars: FP32 5e-5 and FP64 1e-12 per link, as for smearing against the oracle.
@pytest.mark.parametrize("nc,prec,power", [(2, 4, 5), (2, 4, 29), (3, 4, 20), (3, 4, 60), (4, 4, 29),
                                           (2, 8, 245), (3, 8, 40), (3, 8, 500), (4, 8, 245)])
def test_projection_does_not_see_the_scale(ctx, nc, prec, power):
    out = []
    for scale in (1.0, 2.0 ** -power):
        with sun_amd.Lattice(ctx, nc, DIMS, 6.0, 18, prec) as lat:
            u = links(nc)
            lat.from_host(np.ascontiguousarray(u * scale))
            lat.ape_smear(0.0, 1, 10)
            out.append(lat.to_host()[:3])
    got = out[1] if nc == 3 else out[1] / 2.0 ** -power
    assert np.abs(got - out[0]).max() <= (5e-5 if prec == 4 else 1e-12)


@pytest.mark.parametrize("nc,prec", [(2, 4), (3, 4), (3, 8), (4, 8)])
def test_projection_of_zero(ctx, nc, prec):
    with sun_amd.Lattice(ctx, nc, DIMS, 6.0, 18, prec) as lat:
        u = links(nc)
        u[:3] = 0
        lat.from_host(np.ascontiguousarray(u))
        lat.ape_smear(0.2, 1, 10)
        got = lat.to_host()[:3]
    assert np.array_equal(got, np.broadcast_to(np.eye(nc) if nc == 3 else np.zeros((nc, nc)), got.shape))


@pytest.mark.parametrize("nc", [2, 3, 4])
def test_fp32_projection_keeps_the_norm(ctx, nc):
    """Thirty and more reciprocal roots, one after another, none of them leaning to one side: the norm of a
    projected link is off by some 1e-6 at most, its mean over V x 3 links (2304) by a fiftieth of that, 2e-8
    (the native instruction alone is 7e-9 too small, links 4e-7 after ten hits)."""
    with sun_amd.Lattice(ctx, nc, DIMS, 6.0, 18, 4) as lat:
        lat.from_host(links(nc))
        lat.ape_smear(0.2, 1, 20)
        u = lat.to_host()[:3]
    assert abs((np.abs(u) ** 2).sum((2, 3)).mean() / nc - 1) <= 1e-7
