"""The kinetic flux of an ansatz with very small values, bit for bit against the oracle: fluxes near
the bottom of the exponent range, where the fast path's quotients and halved slopes would no longer
be the reference's, with both kinds of spacing, tiny and zero theta, tables with tiny weights, and
the reference-order mode's own exponentials."""
import numpy as np
import pytest

from test_gpu_flux_paths import _alpha, _flux

pytestmark = pytest.mark.gpu

DIMS = (6, 5, 7)
POW2, OTHER = (0.25, 0.5, 0.125), (0.3, 0.7, 0.06)


# 1e-190 is on the fast path, 1e-205 with power-of-two spacings only; the flux is a few orders lower
@pytest.mark.parametrize("scale", [1e-190, 1e-205, 1e-268, 1e-285, 1e-292, 1e-300, 1e-306, 1e-312])
@pytest.mark.parametrize("d", [POW2, OTHER])
@pytest.mark.parametrize("theta", [1.0, 2.0, 1.5e-15])
def test_small_values(P, O, dev, scale, d, theta):
    T = O.Tables(2, 6)
    f, ref = _flux(P, O, dev, T, DIMS, _alpha(DIMS, T.nm) * scale, d, theta)
    assert np.array_equal(f, ref)
    assert ref.any()


# one small cell among ordinary ones, and zeros, which are ordinary
@pytest.mark.parametrize("value", [0.0, 1e-295, 5e-324])
@pytest.mark.parametrize("d", [POW2, OTHER])
@pytest.mark.parametrize("theta", [1.0, 2.0])
def test_mixed_magnitudes(P, O, dev, value, d, theta):
    T = O.Tables(2, 6)
    alpha = _alpha(DIMS, T.nm)
    alpha[::3] *= value
    f, ref = _flux(P, O, dev, T, DIMS, alpha, d, theta)
    assert np.array_equal(f, ref)


@pytest.mark.parametrize("theta", [0.0, 1e-300, -1.0])
@pytest.mark.parametrize("d", [POW2, OTHER])
def test_unusual_theta(P, O, dev, d, theta):
    T = O.Tables(2, 6)
    f, ref = _flux(P, O, dev, T, DIMS, _alpha(DIMS, T.nm), d, theta)
    assert np.array_equal(f, ref)


def test_tiny_weights(P, O, dev):
    T = O.Tables(2, 6)
    T.w[:] *= 1e-307
    f, ref = _flux(P, O, dev, T, DIMS, _alpha(DIMS, T.nm), OTHER, 1.0)
    assert np.array_equal(f, ref)
    assert ref.any()


@pytest.mark.parametrize("a0", [-1580.0, -2390.0, -2480.0])
def test_reference_order_exponentials(P, O, dev, a0):
    import torch
    T = O.Tables(2, 6)
    nx, ny, nz = DIMS
    alpha = 0.3 * _alpha(DIMS, T.nm)
    alpha = np.clip(alpha, -2.0, 2.0)
    alpha[:, 0] += a0
    ref = np.zeros_like(alpha)
    with O.exp_mode(1):
        O.lib().orc_flux_kinetic(nx, ny, nz, T.nm, T.nq, alpha, ref, O.C.byref(T.c), *OTHER, 2.0,
                                 0, np.zeros(alpha.shape[0]), 0)
    ctx = P.Ctx(tables=T)
    ctx.set_precision(P.PREC_FP64_REFORDER)
    fd = torch.zeros(alpha.shape, dtype=torch.float64, device=dev)
    ctx.flux_kinetic(nx, ny, nz, torch.from_numpy(alpha).to(dev), fd, *OTHER, 2.0, 0)
    torch.cuda.synchronize()
    ctx.close()
    inner = (slice(2, -2),) * 3
    shape = (nx + 4, ny + 4, nz + 4, -1)
    assert np.array_equal(fd.cpu().numpy().reshape(shape)[inner], ref.reshape(shape)[inner])
    assert ref.any()
