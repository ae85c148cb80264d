"""The kinetic flux's stencil on both of its paths and at both prefetch depths, bit for bit against
the oracle with the linear (P_N) ansatz, which involves no exponential: few blocks (four ordinates
in flight) and many (two), planes smaller than a wave and just over a block, ordinate counts that
leave a remainder of four, spacings that are and are not powers of two, theta 1 and others.  A
NaN, an infinity or a huge value in one cell takes the general path, whose treatment of them is
the reference's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _flux(P, O, dev, T, dims, alpha, d, theta):
    import torch
    nx, ny, nz = dims
    ref = np.zeros_like(alpha)
    O.lib().orc_flux_kinetic(nx, ny, nz, T.nm, T.nq, alpha, ref, O.C.byref(T.c), *d, theta, 1,
                             np.zeros(alpha.shape[0]), 0)
    ctx = P.Ctx(tables=T)
    fd = torch.zeros(alpha.shape, dtype=torch.float64, device=dev)
    ctx.flux_kinetic(nx, ny, nz, torch.from_numpy(alpha).to(dev), fd, *d, theta, 1)
    torch.cuda.synchronize()
    f = fd.cpu().numpy().reshape(nx + 4, ny + 4, nz + 4, -1)[2:-2, 2:-2, 2:-2]
    ctx.close()
    return f, ref.reshape(nx + 4, ny + 4, nz + 4, -1)[2:-2, 2:-2, 2:-2]


def _alpha(dims, nm):
    ng = (dims[0] + 4) * (dims[1] + 4) * (dims[2] + 4)
    rng = np.random.default_rng(7)
    return rng.normal(0, 1, (ng, nm)) * np.exp(rng.normal(0, 3, (ng, 1)))


@pytest.mark.parametrize("N", [1, 2, 3, 4])
@pytest.mark.parametrize("Q", [5, 6])
@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 3, 86), (260, 3, 5)])
@pytest.mark.parametrize("d,theta", [((0.25, 0.5, 0.125), 1.0), ((0.25, 0.5, 0.125), 1.5),
                                     ((0.3, 0.7, 0.06), 1.0), ((0.3, 0.7, 0.06), 2.0)])
def test_linear_flux_bit_exact(P, O, dev, N, Q, dims, d, theta):
    T = O.Tables(N, Q)
    f, ref = _flux(P, O, dev, T, dims, _alpha(dims, T.nm), d, theta)
    assert np.array_equal(f, ref)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1e300])
@pytest.mark.parametrize("theta", [1.0, 2.0])
def test_wild_values_take_the_general_path(P, O, dev, value, theta):
    T = O.Tables(2, 6)
    dims = (6, 5, 7)
    alpha = _alpha(dims, T.nm)
    # an interior cell of the middle
    alpha[(5 * 9 + 4) * 11 + 5, 0] = value
    with np.errstate(all="ignore"):
        f, ref = _flux(P, O, dev, T, dims, alpha, (0.3, 0.7, 0.06), theta)
    assert np.array_equal(f, ref, equal_nan=True)


@pytest.mark.parametrize("d,theta", [((1e-20, 0.5, 0.1), 1.0), ((0.3, 0.7, 0.1), 1e16)])
def test_unreasonable_spacing_and_theta(P, O, dev, d, theta):
    T = O.Tables(1, 6)
    dims = (3, 4, 5)
    f, ref = _flux(P, O, dev, T, dims, _alpha(dims, T.nm), d, theta)
    assert np.array_equal(f, ref, equal_nan=True)
