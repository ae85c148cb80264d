"""The fused tail's line search, which settles many trials a round, against the bulk passes, which
take one each: the same bits through searches that accept late in a round, that carry over to the
next one and that give up.  A tolerance below what the gradient can reach makes every cell
end in such searches; Q = 5 and 9 give one chunk of ordinates and an odd count of them."""
import numpy as np
import pytest

from test_gpu_closure import _run_gpu_closure

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("tail", ["fused1", "fused"])
@pytest.mark.parametrize("N,Q", [(1, 5), (2, 9), (3, 9), (4, 9)])
def test_long_searches_equal_bulk(P, O, dev, N, Q, tail, mixed):
    T = O.Tables(N, Q)
    _, u, a0 = O.closure_batch_input(T, 37, 0x5EA2C4, 0.5, 9.0)
    opts = P.closure_opts(tol=1e-15, maxIter=12)
    prec = P.PREC_MIXED if mixed else P.PREC_FP64
    bulk = _run_gpu_closure(P, dev, T, u, a0, opts, prec, tail="bulk")
    fused = _run_gpu_closure(P, dev, T, u, a0, opts, prec, tail=tail)
    assert bulk[3] == fused[3]
    for x, y in zip(bulk[:2], fused[:2]):
        assert np.array_equal(x.view(np.int64), y.view(np.int64))
    assert bulk[2].tobytes() == fused[2].tobytes()
