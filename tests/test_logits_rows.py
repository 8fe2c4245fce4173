"""Which rows llama_get_logits shows when a run brings none (llama.cpp:5734-5743 leaves the buffer as it was): the layers of the context are served by callbacks here, so no GPU is needed."""
import ctypes as C
import os

import numpy as np
import pytest

from pipeinfer_amd import lib as L, llama as LL, pipeline as P

MODEL = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "tiny_llama_q2_k.gguf")


class Served:
    """a context whose runs give rows of one value, `value`; start_rc: what starting a run returns"""

    def __init__(self, ctx):
        self.ctx, self.value, self.start_rc, self.seen, self.n = ctx, 0.0, 0, [], {}
        self.ops = P.RemoteOps(None, P.START_FN(self._start), P.POLL_FN(lambda user: 1), P.WAIT_FN(self._wait), P.CANCEL_FN(lambda user, batch: None))
        ctx.lib.pipeinfer_context_set_remote.argtypes = [C.c_void_p, C.c_void_p]
        ctx.lib.pipeinfer_context_set_remote.restype = None
        ctx.lib.pipeinfer_context_set_remote(ctx.h, C.byref(self.ops))

    def _start(self, user, run_seq, batch_id, n, meta, nbytes):
        self.n[run_seq] = n
        return self.start_rc

    def _wait(self, user, run_seq, logits, ids, vals, sums):
        n = self.n[run_seq]
        np.ctypeslib.as_array(C.cast(logits, C.POINTER(C.c_float)), shape=(n, self.ctx.n_vocab))[:] = self.value
        for p, k in ((ids, 8), (vals, 8), (sums, 1)):
            C.memset(p, 0, 4 * k * n)
        shown = self.ctx.lib.llama_get_logits(self.ctx.h)
        self.seen.append(float(shown[0]) if shown else None)
        return 1


@pytest.mark.parametrize("rows", ["many", "some", "few"])
def test_rows_stay_where_a_run_brings_none(rows):
    """rows that are many change hands with the run's buffer, few are copied: either way the rows of the last run that brought some are read until the next one brings its own — past a run that could not be
    started, through the next run's time in flight, and past a cancelled run, shorter or longer"""
    model = LL.Model(MODEL)
    n = {"many": (4 << 20) // (4 * model.n_vocab) + 1, "some": (3 << 16) // (4 * model.n_vocab) + 1, "few": 3}[rows]
    ctx = LL.Context(model, n_ctx=2 * n + 64, n_batch=2 * n, logits_all=True)
    s = Served(ctx)

    def batch(k):
        ctx.kv_clear()
        return [1] * k, list(range(k)), [[0]] * k

    s.value = 1.0
    assert np.all(ctx.decode(*batch(n)) == 1.0)
    s.start_rc = -1
    with pytest.raises(L.PipeInferError):
        ctx.decode(*batch(n))
    assert np.all(ctx.logits(n) == 1.0)
    s.start_rc, s.value = 0, 2.0
    ticket = ctx.start(*batch(n))
    assert np.all(ctx.logits(n) == 1.0)
    assert np.all(ctx.finish(ticket) == 2.0) and s.seen[-1] == 1.0
    ctx.cancel([9])
    for k in (1, n, 2 * n):
        assert np.all(ctx.finish(ctx.start(*batch(k), batch_id=9))[:min(k, n)] == 2.0)
        assert np.all(ctx.logits(n) == 2.0)
    s.value = 3.0
    assert np.all(ctx.decode(*batch(n)) == 3.0)
    assert np.all(ctx.decode(*batch(n), batch_id=9) == 3.0)
    s.value = 4.0
    assert np.all(ctx.decode(*batch(2)) == 4.0)
    ctx.free()
    model.free()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [2, 97, 400])
def test_rows_of_a_next_run_are_where_the_last_ones_were(rows):
    """a program that asked for the buffer once reads every later run's rows there, whether they are as many or fewer and whether or not the next run started before this one's rows were fetched - as long as they are below the 4 MB from
    which rows change hands with the run's buffer"""
    model = LL.Model(MODEL)
    assert 4 * rows * model.n_vocab < 4 << 20
    ctx = LL.Context(model, n_ctx=4 * rows + 64, n_batch=2 * rows, logits_all=True)

    def batch(token, n, seq=0):
        return [token] * n, list(range(n)), [[seq]] * n

    def shown():
        return np.ctypeslib.as_array(C.cast(ctx.lib.llama_get_logits(ctx.h), C.POINTER(C.c_float)), shape=(rows, model.n_vocab))

    own = ctx.decode(*batch(5, rows))
    kept = shown()
    assert np.array_equal(kept, own)
    for token, n in ((6, rows), (7, 1), (8, rows), (9, rows - 1)):
        ctx.kv_clear()
        own = ctx.decode(*batch(token, n))
        assert shown().ctypes.data == kept.ctypes.data and np.array_equal(kept[:n], own), (token, n)
    ctx.kv_clear()
    tickets = [ctx.start(*batch(10 + i, rows, i)) for i in range(2)]
    for t in tickets:
        own = ctx.finish(t)
        assert shown().ctypes.data == kept.ctypes.data and np.array_equal(kept, own)
    ctx.free()
    model.free()
