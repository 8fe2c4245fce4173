"""Norms in one launch with what comes ahead of them or behind them: the same bits as the operators one by one, at the edges of what the fused kernels take and beyond them."""
import ctypes as C

import numpy as np
import pytest

from pipeinfer_amd import lib as L
from tests import gpu_util as U

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return U.init()


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def upload(lib, w):
    w = bf16(w)
    return lib.pi_weight_upload(30, w.shape[1], w.shape[0], w.ctypes.data_as(C.c_void_p), None)


class Rows:
    """rows of n values, `pad` floats between them"""

    def __init__(self, values, pad=0):
        self.T, self.stride = values.shape
        self.n = self.stride - pad
        self.dev = U.Dev(values.astype(np.float32))
        self.ptr = self.dev.ptr

    def get(self):
        return self.dev.get(np.uint32, (self.T, self.stride))[:, :self.n]


@pytest.mark.parametrize("n", [8, 1000, 1024, 1028, 2048, 2056, 4096, 4104])
@pytest.mark.parametrize("T,E,top,exact,pad", [(1, 10, 2, 0, 0), (3, 1, 1, 1, 4), (65, 70, 3, 0, 0), (2, 5, 5, 0, 1)])
def test_norm_and_router_and_second_norm(lib, n, T, E, top, exact, pad):
    rng = np.random.default_rng(n + T)
    y, w, w2 = Rows(rng.standard_normal((T, n + pad)), pad), Rows(rng.standard_normal((1, n))), Rows(rng.standard_normal((1, n)))
    x = rng.standard_normal((T, n + pad))
    router, corr = upload(lib, rng.standard_normal((E, n)) * 0.1), U.Dev((rng.standard_normal(E) * 0.01).astype(np.float32))
    got = []
    for fused in (False, True):
        xs = Rows(x, pad)
        sel, sw, o2, h, h2 = U.Dev(nbytes=4 * T * top), U.Dev(nbytes=4 * T * top), Rows(np.zeros((T, n + pad)), pad), U.Dev(np.zeros((T, n), np.uint16)), U.Dev(np.zeros((T, n), np.uint16))

        def asked(buf, op):
            lib.pi_set_rounded_output(buf.ptr, n, 0, n, 0)
            L.check(op())
            return bool(lib.pi_rounded_output_written())

        if fused:
            a = asked(h, lambda: lib.pi_op_rms_scale_route(y.ptr, y.stride, w.ptr, 1.0, 1e-6, xs.ptr, xs.stride, 0.5, xs.ptr, xs.stride, router, corr.ptr, T, top, exact, sel.ptr, sw.ptr, None))
        else:
            a = asked(h, lambda: lib.pi_op_rms_scale(y.ptr, y.stride, w.ptr, 1.0, 1e-6, n, T, None, 0, xs.ptr, xs.stride, 0.5, xs.ptr, xs.stride, None, 0, None))
            L.check(lib.pi_op_moe_route(router, corr.ptr, xs.ptr, xs.stride, T, top, exact, sel.ptr, sw.ptr, None))
        first = xs.get()
        if fused:
            b = asked(h2, lambda: lib.pi_op_rms_scale_twice(y.ptr, y.stride, w.ptr, 0.0, 1e-6, n, T, xs.ptr, xs.stride, -2.0, xs.ptr, xs.stride, w2.ptr, 1.0, o2.ptr, o2.stride, None))
        else:
            L.check(lib.pi_op_rms_scale(y.ptr, y.stride, w.ptr, 0.0, 1e-6, n, T, None, 0, xs.ptr, xs.stride, -2.0, xs.ptr, xs.stride, None, 0, None))
            b = asked(h2, lambda: lib.pi_op_rms_scale(xs.ptr, xs.stride, w2.ptr, 1.0, 1e-6, n, T, None, 0, None, 0, 1.0, o2.ptr, o2.stride, None, 0, None))
        got.append([first, sel.get(np.int32, (T, top)), sw.get(np.uint32, (T, top)), xs.get(), o2.get(), np.array([a, b]), h.get(np.uint16, (T, n)), h2.get(np.uint16, (T, n))])
    for one, other in zip(*got):
        assert np.array_equal(one, other)


@pytest.mark.parametrize("width,T,second,pad", [(64, 32, False, 0), (1024, 33, True, 0), (1088, 40, True, 4), (2048, 70, False, 0), (4096, 32, True, 0), (4160, 32, True, 0), (128, 64, True, 1)])
def test_experts_of_a_prompt_and_the_norms_behind_them(lib, width, T, second, pad):
    rng = np.random.default_rng(width + T)
    n_exp, ff, top = 4, 64, 2
    up, dn = upload(lib, rng.standard_normal((n_exp * ff, width)) * 0.05), upload(lib, rng.standard_normal((n_exp * width, ff)) * 0.1)
    assert lib.pi_op_moe_rounded_ok(up, dn, n_exp, ff, width, T, top)
    x = rng.standard_normal((T, width + pad))
    xh, w, w2 = U.Dev(bf16(x[:, :width])), Rows(rng.standard_normal((1, width))), Rows(rng.standard_normal((1, width)))
    sel = rng.integers(0, n_exp + 2, (T, top)).astype(np.int32)                   # (experts and identities)
    sd, sw = U.Dev(sel), U.Dev(rng.random((T, top)).astype(np.float32))
    got = []
    for fused in (False, True):
        xs, o2, sums = Rows(x, pad), Rows(np.zeros((T, width))), Rows(np.zeros((T, width)))
        mid, out, idx = U.Dev(nbytes=2 * T * top * ff + 64), U.Dev(nbytes=4 * T * top * width), U.Dev(nbytes=4 * lib.pi_op_moe_grouped_index_ints(T, top, n_exp))
        args = (up, dn, n_exp, ff, xh.ptr, width, xs.ptr, xs.stride, sd.ptr, sw.ptr, T, top, mid.ptr, out.ptr, idx.ptr, sums.ptr, width)
        if fused:
            L.check(lib.pi_op_moe_experts_rounded_norm(*args, w.ptr, 1.0, 1e-6, xs.ptr, xs.stride, 0.5, xs.ptr, xs.stride, w2.ptr if second else None, 1.0, o2.ptr, width, None))
        else:
            L.check(lib.pi_op_moe_experts_rounded(*args, None))
            L.check(lib.pi_op_rms_scale(sums.ptr, width, w.ptr, 1.0, 1e-6, width, T, None, 0, xs.ptr, xs.stride, 0.5, xs.ptr, xs.stride, None, 0, None))
            if second:
                L.check(lib.pi_op_rms_scale(xs.ptr, xs.stride, w2.ptr, 1.0, 1e-6, width, T, None, 0, None, 0, 1.0, o2.ptr, width, None, 0, None))
        got.append([xs.get()] + ([o2.get()] if second else []))
    for one, other in zip(*got):
        assert np.array_equal(one, other)


@pytest.mark.parametrize("rank,T,n_kv,pad", [(256, 1, 40, 0), (512, 1, 700, 4), (512, 7, 96, 0), (256, 30, 100, 0), (256, 5, 64, 1), (64, 3, 50, 0), (512, 200, 200, 0), (1024, 2, 33, 0)])
def test_latents_into_their_cells_and_the_attention_over_them(lib, rank, T, n_kv, pad):
    rng = np.random.default_rng(rank + T)
    H, D, V = 4, 32, 64
    w_uk, w_uv = upload(lib, rng.standard_normal((H * D, rank)) * rank ** -0.5), upload(lib, rng.standard_normal((H * V, rank)) * rank ** -0.5)
    row = H * D + rank + pad
    p, w, sink = U.Dev(rng.standard_normal((T, row)).astype(np.float32)), Rows(rng.standard_normal((1, rank))), U.Dev(rng.standard_normal(H).astype(np.float32))
    old, vis = rng.standard_normal((n_kv, rank)).astype(np.float32), np.arange(n_kv)[None, :] <= np.arange(n_kv - T, n_kv)[:, None]
    mask = U.Dev(np.packbits(np.pad(vis, ((0, 0), (0, -n_kv % 32))), axis=1, bitorder="little").view(np.uint32))
    dyn = U.Dev(np.array([n_kv - T, n_kv, T, 0], np.int32))
    n_scr = lib.pi_op_latent_attention_scratch_floats(H, rank, T, n_kv)
    got = []
    for fused in (False, True):
        cache, scr, out = U.Dev(old), U.Dev(nbytes=4 * n_scr), U.Dev(nbytes=4 * T * H * V)
        latents = p.ptr + 4 * H * D
        tail = (mask.ptr, w_uk, w_uv, sink.ptr, D ** -0.5, H, D, V, rank, T, n_kv, scr.ptr, n_scr, out.ptr, H * V, dyn.ptr, None)
        if fused:
            L.check(lib.pi_op_latent_attention_tokens(latents, row, w.ptr, 1e-6, p.ptr, row, cache.ptr, *tail))
        else:
            L.check(lib.pi_op_rms_scale(latents, row, w.ptr, 0.0, 1e-6, rank, T, None, 0, None, 0, 1.0, cache.ptr, rank, dyn.ptr, 1, None))
            L.check(lib.pi_op_latent_attention(p.ptr, row, cache.ptr, *tail))
        got.append([cache.get(np.uint32, old.shape), out.get(np.uint32, (T, H * V))])
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert np.array_equal(got[1][0][:n_kv - T], old.view(np.uint32)[:n_kv - T])
