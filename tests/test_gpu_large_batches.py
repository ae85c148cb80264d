"""Batches large enough that every block of the set-up, sweep and step kernels takes several tiles
(LDS reused, appends flushed on the way and at the end): the batch repeats a short prefix, and
every repeat must get the prefix's bits.  Statistics are preset, so that a cell left out shows."""
import numpy as np
import pytest

from test_gpu_closure import _set_tail

pytestmark = pytest.mark.gpu


# (set-up: 4096 blocks of 64 cells on 256 CUs; step: as many of 16 cells, of four at nm = 25)
@pytest.mark.parametrize("N,Q,n,prec,tail", [
    (1, 4, 1310743, "FP64", None), (1, 4, 1310743, "MIXED", None),
    (1, 4, 1310743, "FP64", "bulk"), (1, 4, 1310743, "FP64_REFORDER", "bulk"),
    (2, 5, 300007, "MIXED", "bulk"), (3, 6, 150001, "FP64", "bulk"),
    (4, 6, 70001, "FP64", "bulk"), (4, 6, 70001, "MIXED", "bulk")])
def test_every_repeat_gets_the_prefix_bits(P, O, dev, N, Q, n, prec, tail):
    import torch
    T = O.Tables(N, Q)
    k = 131
    _, ub, ab = O.closure_batch_input(T, k, 0xB16 + N, 0.5, 3.0)
    reps = -(-n // k)
    ctx = P.Ctx(tables=T)
    ctx.set_precision(getattr(P, "PREC_" + prec))
    _set_tail(ctx, tail, n)
    u = torch.from_numpy(ub).to(dev).repeat(reps, 1)[:n].contiguous()
    a = torch.from_numpy(ab).to(dev).repeat(reps, 1)[:n].contiguous()
    st = P.alloc_stats(n, dev)
    st.fill_(0x5A)
    ctx.closure(u, a, P.closure_opts(maxIter=12), stats=st)
    ctx.sync()
    st = st.reshape(n, -1)
    for x in (u, a, st):
        b = x.view(torch.uint8).reshape(n, -1)
        full = (n // k) * k
        assert bool((b[:full].reshape(-1, k, b.shape[1]) == b[:k]).all())
        assert bool((b[full:] == b[:n - full]).all())
    s = P.stats_to_numpy(st[:k].contiguous().reshape(-1))
    assert (s["totalIter"] >= 1).all() and (s["totalIter"] <= 12 * 20).all()
    assert (s["regIndex"] >= 0).all() and (s["regIndex"] < 5).all()
    ctx.close()
