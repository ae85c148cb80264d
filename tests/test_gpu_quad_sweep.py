"""The four-cells-a-wave FP64 sweep at the edges of its layout: batches that fill a wave, a block
or neither, ordinate counts that leave a chunk partly padded, every order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,Q", [(1, 4), (2, 5), (2, 8), (3, 6), (4, 7)])
def test_hessian_batches_and_padding(P, dev, N, Q):
    T = P.tables_host(N, Q)
    nm, nq = T["M"].shape[1], T["M"].shape[0]
    M, w = T["M"], T["w"]
    ctx = P.Ctx(N, Q)
    rng = np.random.default_rng(100 * N + Q)
    for n in (1, 3, 4, 5, 15, 16, 17, 67):
        al = rng.normal(scale=1.5, size=(n, nm))
        H = torch.full((n, nm, nm), float("nan"), dtype=torch.float64, device=dev)
        ctx.hessian(torch.from_numpy(al).to(dev), H)
        assert ctx.sync() == 0
        x = al @ M.T
        e = np.exp(x) * w
        ref = np.einsum("cq,qi,qj->cij", e, M, M)
        # rounding: the exponent's nm-term sum moves e^x by nm eps max|alpha_i m_qi| a term, the
        # exp and the products by a few eps, the nq-term sum by nq eps of the terms' absolute sum
        mag = np.einsum("cq,qi,qj->cij", e, np.abs(M), np.abs(M))
        xs = np.max(np.abs(al) @ np.abs(M).T, axis=1)
        tol = np.finfo(np.float64).eps * (nq + nm * xs + 8)[:, None, None] * mag
        got = H.cpu().numpy()
        assert np.all(np.abs(got - ref) <= tol), (N, Q, n, np.max(np.abs(got - ref) / tol))
        assert np.array_equal(got, got.transpose(0, 2, 1))
    ctx.close()
