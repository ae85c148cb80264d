"""The bulk step pass (rows of a cell over 4 or 16 lanes) against the fused kernel's state machine
(one element per lane): the same bits at batches that fill a wave, a block's appends or neither,
through converging cells, restarts, the ladder, and both stopping rules."""
import numpy as np
import pytest

from test_gpu_closure import _run_gpu_closure

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("unbatched", [False, True])
@pytest.mark.parametrize("N,Q", [(1, 6), (2, 8), (3, 12), (4, 10)])
def test_bulk_step_equals_fused(P, O, dev, N, Q, unbatched, mixed):
    T = O.Tables(N, Q)
    prec = P.PREC_MIXED if mixed else P.PREC_FP64
    for n, smax, cond in ((1, 4.0, 1e20), (3, 8.0, 1e20), (15, 8.0, 30.0), (16, 8.0, 1e20),
                          (17, 8.0, 300.0), (67, 8.0, 1e20), (333, 8.0, 1e4)):
        _, u, a0 = O.closure_batch_input(T, n, 0x57E9 + n, 0.5, smax)
        opts = P.closure_opts(unbatched=unbatched, condHMax=cond, maxIter=25)
        bulk = _run_gpu_closure(P, dev, T, u, a0, opts, prec, tail="bulk")
        fused = _run_gpu_closure(P, dev, T, u, a0, opts, prec, tail="fused1")
        assert bulk[3] == fused[3]
        for x, y in zip(bulk[:2], fused[:2]):
            assert np.array_equal(x.view(np.int64), y.view(np.int64)), (n, cond)
        assert bulk[2].tobytes() == fused[2].tobytes(), (n, cond)
