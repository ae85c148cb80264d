"""The P_N step's fused stage kernel at the sizes where its tiling can go wrong -- planes smaller
than a wave, one cell more than a block, several strips of blocks -- and at every order, with
power-of-two spacings (reciprocals) and others (divisions): bit for bit against the oracle's
separate flux, Euler and average."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 3, 4])
@pytest.mark.parametrize("dims", [(2, 2, 2), (5, 3, 7), (3, 257, 1 + 16), (2, 1 + 64, 65), (9, 8, 32)])
@pytest.mark.parametrize("pow2", [True, False])
def test_moment_step_bit_exact(P, O, dev, N, dims, pow2):
    import torch
    T = O.Tables(N, 6)
    nx, ny, nz = dims
    u, sT, sS = O.init_grid(nx, ny, nz, T.nm, ic=1, sigma=0.3, floor=1e-3, noise=0.05, seed=5)
    rng = np.random.default_rng(5)
    u[:, 1:] = u[:, :1] * rng.uniform(-0.3, 0.3, (u.shape[0], T.nm - 1))
    sT = rng.uniform(0.5, 2, sT.shape)
    sS = sT * rng.uniform(0, 1, sT.shape)
    d = (0.25, 0.5, 0.125) if pow2 else (0.3, 0.25, 0.7)
    dt = 0.02
    ref, flux = u.copy(), np.zeros_like(u)
    ng = u.shape[0]
    O.lib().orc_flux_moment(nx, ny, nz, T.nm, u, flux, T.ops, *d, 0)
    O.lib().orc_update(nx, ny, nz, T.nm, T.nm2, T.nq, 0, 0, ref, u.copy(), np.zeros_like(u),
                       np.zeros_like(u), np.zeros(ng * T.nq), sT, sS, O.C.byref(T.c), T.ops,
                       O.C.byref(O.opts()), *d, 1.0, dt, None, 0)
    ctx = P.Ctx(tables=T)
    ud, fd = torch.from_numpy(u).to(dev), torch.zeros(u.shape, dtype=torch.float64, device=dev)
    ctx.flux_moment(nx, ny, nz, ud, fd, *d)
    ctx.update(nx, ny, nz, ud, None, torch.from_numpy(sT).to(dev), torch.from_numpy(sS).to(dev), *d,
               1.0, dt, solver=0)
    assert ctx.sync() == 0
    inner = (slice(2, -2),) * 3
    f = fd.cpu().numpy().reshape(nx + 4, ny + 4, nz + 4, -1)
    assert np.array_equal(f[inner], flux.reshape(f.shape)[inner])
    f[inner] = 0.0
    assert not f.any()  # the ghosts' flux is not written
    assert np.array_equal(ud.cpu().numpy(), ref)
    ctx.close()
