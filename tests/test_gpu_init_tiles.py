"""The closure's state set-up works on tiles of cells, small ones for small batches: a cell's
result does not depend on the batch it is in, over batch sizes around both tile sizes and around
the switch between them, both stopping rules, and cells with u0 <= 0, which are flagged and left."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unbatched", [False, True])
@pytest.mark.parametrize("N", [1, 2, 4])
def test_result_independent_of_the_batch(P, O, dev, N, unbatched):
    import torch
    T = O.Tables(N, 5)
    n = 64 * torch.cuda.get_device_properties(dev).multi_processor_count + 65
    _, ub, ab = O.closure_batch_input(T, 129, 0x711E, 0.5, 2.0)
    ub[[0, 17, 128], 0] = (0.0, -1.0, 0.0)
    u = np.ascontiguousarray(np.resize(ub, (n, T.nm)))
    a = np.ascontiguousarray(np.resize(ab, (n, T.nm)))
    opts = P.closure_opts(unbatched=unbatched, maxIter=20)
    ctx = P.Ctx(tables=T)
    got = {}
    for m in (1, 7, 8, 9, 129, n - 66, n - 65, n):
        ud, ad = torch.from_numpy(u[:m]).to(dev), torch.from_numpy(a[:m]).to(dev)
        st = P.alloc_stats(m, dev)
        ctx.closure(ud, ad, opts, stats=st)
        ctx.sync()
        torch.cuda.synchronize()
        got[m] = [ud.cpu().numpy(), ad.cpu().numpy(), P.stats_to_numpy(st)]
    ctx.close()
    for m, (x, y, s) in got.items():
        for r, (full, part) in enumerate(zip(got[n], (x, y, s))):
            assert full[:m].tobytes() == part.tobytes(), (m, r)
        k = min(m, 129)
        assert np.array_equal(x[:k][ub[:k, 0] <= 0], ub[:k][ub[:k, 0] <= 0])
        assert ((s["flags"][:k] != 0) | (ub[:k, 0] > 0)).all()
