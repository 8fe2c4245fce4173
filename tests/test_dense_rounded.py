"""The products of bfloat16 activations (pi_op_dense_rounded) in every tile shape, at the edges of tiles, of K's stages and of segments, against the sums in 64 bits."""
import ctypes as C

import numpy as np
import pytest

from pipeinfer_amd import lib as L


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def wide(h):
    return (h.astype(np.uint32) << 16).view(np.float32)


# rows, K, tokens, segments, activation: one K step, fewer steps than stages, odd rows and tokens, each shape's first and last partial tile
CASES = [(40, 64, 33, 1, 0), (33, 128, 65, 1, 1), (512, 192, 100, 1, 0), (1000, 256, 257, 1, 2), (2048, 2048, 333, 1, 0), (2052, 512, 700, 1, 0), (4096, 1024, 1000, 1, 0), (12288, 512, 700, 1, 1), (32000, 128, 200, 1, 0),
         (32000, 128, 515, 1, 0), (1024 + 64, 320, 100, 5, 3), (2048 + 36, 256, 333, 3, 0), (16384, 192, 9, 1, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,T,segs,act", CASES)
def test_products_of_rounded_activations(rows, K, T, segs, act):
    from tests import gpu_util as U
    lib = U.init()
    rng = np.random.default_rng([rows, K, T])
    w = bf16(rng.standard_normal((rows, K)))
    pad = 16                                                    # a token's row is longer than what the product reads
    x = rng.standard_normal((T, segs * K + pad)).astype(np.float32)
    bias = rng.standard_normal(rows).astype(np.float32)
    seg_rows = rows // segs // 4 * 4 if segs > 1 else 0
    W = lib.pi_weight_upload(30, K, rows, w.ctypes.data_as(C.c_void_p), None)
    xd, bd = U.Dev(x), U.Dev(bias)
    xh, out = U.Dev(nbytes=2 * x.size), U.Dev(np.full((T, rows + 4), 7.0, np.float32))
    L.check(lib.pi_op_round_bf16(xd.ptr, x.shape[1], x.shape[1], T, xh.ptr, x.shape[1], None))
    assert np.array_equal(xh.get(np.uint16, x.shape), bf16(x))
    assert lib.pi_op_dense_rounded_ok(W, x.shape[1], T) == 1
    L.check(lib.pi_op_dense_rounded(W, bd.ptr, xh.ptr, x.shape[1], seg_rows, K, segs, T, out.ptr, rows + 4, act, rows // 2, 0, None))
    got = out.get(np.float32, (T, rows + 4))
    assert (got[:, rows:] == 7.0).all()                         # nothing past a row
    xr, wr = wide(bf16(x)).astype(np.float64), wide(w).astype(np.float64)
    want, size = np.empty((T, rows)), np.empty((T, rows))
    for g in range(segs):
        r0, r1 = g * seg_rows, rows if g == segs - 1 else (g + 1) * seg_rows
        want[:, r0:r1] = xr[:, g * K:(g + 1) * K] @ wr[r0:r1].T
        size[:, r0:r1] = np.abs(xr[:, g * K:(g + 1) * K]) @ np.abs(wr[r0:r1]).T
    want += bias
    half = rows // 2
    if act == 1:
        want[:, :half] = want[:, :half] / (1 + np.exp(-want[:, :half]))
    elif act == 2:
        want[:, :half] = 1 / (1 + np.exp(-want[:, :half]))
    elif act == 3:
        want[:, :half] = np.maximum(want[:, :half], 0) ** 2
    # fp32 sums of K exact products: an error of at most K roundings of the sum of magnitudes, in practice a few dozen; the activations' slopes are below 1.1, but of the square 2 |y|
    slope = 2 * np.sqrt(np.abs(want)).max() if act == 3 else 1.2
    assert (np.abs(got[:, :rows] - want) <= slope * (2.0 ** -24 * 16 * (size + 4) + 1e-6)).all()
    again = U.Dev(np.full((T, rows + 4), 7.0, np.float32))
    L.check(lib.pi_op_dense_rounded(W, bd.ptr, xh.ptr, x.shape[1], seg_rows, K, segs, T, again.ptr, rows + 4, act, rows // 2, 0, None))
    assert np.array_equal(again.get(np.float32, (T, rows + 4)), got)
    lib.pi_weight_free(W)


@pytest.mark.gpu
def test_what_the_rounded_products_refuse():
    from tests import gpu_util as U
    lib = U.init()
    w = np.zeros((64, 72), np.uint16)
    W = lib.pi_weight_upload(30, 72, 64, w.ctypes.data_as(C.c_void_p), None)
    x, out = U.Dev(nbytes=2 * 64 * 72), U.Dev(nbytes=4 * 64 * 64)
    assert lib.pi_op_dense_rounded_ok(W, 72, 64) == 0
    assert lib.pi_op_dense_rounded(W, None, x.ptr, 72, 0, 0, 1, 64, out.ptr, 64, 0, 64, 0, None) == -1
    lib.pi_weight_free(W)


def _asked(lib, U, op, out, from_, n, rows, only):
    """runs op() with its columns [from_, from_ + n) asked for in bfloat16 as well: (rounded values, whether the operator wrote them)"""
    h = U.Dev(np.full((rows, n + 8), 0x1234, np.uint16))
    lib.pi_set_rounded_output(h.ptr, n + 8, from_, n, only)
    L.check(op())
    met = lib.pi_rounded_output_written()
    got = h.get(np.uint16, (rows, n + 8))
    assert (got[:, n:] == 0x1234).all()
    return got[:, :n], met


@pytest.mark.gpu
@pytest.mark.parametrize("T,n", [(33, 64), (40, 1000), (35, 2048), (33, 4096)])
def test_rounded_outputs_are_the_fp32_ones_rounded(T, n):
    """norms, gates, shifts and embeddings: the rounded rows against the rounded fp32 result of the same call; asked for alone they leave the fp32 rows as they were, but for the operators whose fp32 rows something else reads as well"""
    from tests import gpu_util as U
    lib = U.init()
    rng = np.random.default_rng([T, n])
    x, y, g = (U.Dev(rng.standard_normal((T, n)).astype(np.float32)) for _ in range(3))
    w = U.Dev(1 + 0.1 * rng.standard_normal(n).astype(np.float32))
    two = U.Dev(rng.standard_normal((T, 2 * n)).astype(np.float32))
    mu, state, rec = U.Dev(rng.random((3, n)).astype(np.float32)), U.Dev(np.zeros((2, n), np.float32)), U.Dev(np.full(T, 1 << 30, np.int32))
    table = bf16(rng.standard_normal((50, n)))
    W = lib.pi_weight_upload(30, n, 50, table.ctypes.data_as(C.c_void_p), None)
    tok = U.Dev(rng.integers(0, 50, T).astype(np.int32))
    out = U.Dev(nbytes=4 * T * 3 * n)
    heads = n // 64 if n % 64 == 0 else n // 8
    ops = {
        "rms_scale": (n, lambda: lib.pi_op_rms_scale(x.ptr, n, w.ptr, 1.0, 1e-5, n, T, g.ptr, n, y.ptr, n, 0.5, out.ptr, n, None, 0, None)),
        "residual_norm": (n, lambda: lib.pi_op_residual_norm(x.ptr, y.ptr, n, None, w.ptr, 1e-5, n, T, None, out.ptr, n, None)),
        "rms_post": (n, lambda: lib.pi_op_rms_post(y.ptr, n, None, None, 0, None, 1.0, w.ptr, x.ptr, n, 2.0, w.ptr, 1e-5, n, T, out.ptr, n, None, None, 0, None)),
        "rms_post, next norm": (n, lambda: lib.pi_op_rms_post(y.ptr, n, w.ptr, g.ptr, n, w.ptr, 0.5, w.ptr, x.ptr, n, 2.0, w.ptr, 1e-5, n, T, two.ptr, 2 * n, w.ptr, out.ptr, n, None)),
        "head_norm_gate": (n, lambda: lib.pi_op_head_norm_gate(y.ptr, n, heads, n // heads, w.ptr, 1, g.ptr, n, 1, 1e-5, T, out.ptr, n, None)),
        "token_shift": (3 * n, lambda: lib.pi_op_token_shift(x.ptr, n, n, mu.ptr, 3, state.ptr, rec.ptr, T, out.ptr, 3 * n, None)),
        "glu_mul": (n, lambda: lib.pi_op_glu_mul(two.ptr, 2 * n, n, T, out.ptr, n, None)),
        "glu_mul_ex": (n, lambda: lib.pi_op_glu_mul_ex(two.ptr, 2 * n, n, 2, 7.0, -1, T, out.ptr, n, None)),
        "embed": (n, lambda: lib.pi_op_embed(W, tok.ptr, T, 0.7, out.ptr, None)),
        "embed_pair": (n, lambda: lib.pi_op_embed_pair(W, tok.ptr, T, 0.7, W, tok.ptr, out.ptr, None)),
    }
    for name, (width, op) in ops.items():
        got, met = _asked(lib, U, op, out, 0, width, T, 0)
        full = out.get(np.float32, (T, width), 0, T * width)
        assert met == 1, name
        assert np.array_equal(got, bf16(full)), name
        before = np.full(T * 3 * n, 777.0, np.float32)
        L.check(lib.pi_memcpy_h2d(out.ptr, before.ctypes.data_as(C.c_void_p), before.nbytes, None))
        L.check(lib.pi_stream_sync(None))
        alone, met = _asked(lib, U, op, out, 0, width, T, 1)
        assert met == 1 and np.array_equal(alone, got), name
        assert np.array_equal(out.get(np.float32, (T, width), 0, T * width), full if name in ("rms_post", "embed", "embed_pair") else before[:T * width].reshape(T, width)), name
        _, met = _asked(lib, U, op, out, 0, width - 8, T, 0)      # not the operator's rows: not met, and not left behind for the next one
        assert met == 0 and lib.pi_rounded_output_written() == 1, name
        assert np.array_equal(out.get(np.float32, (T, width), 0, T * width), full), name
    lib.pi_weight_free(W)


@pytest.mark.gpu
def test_a_products_columns_rounded_for_the_next():
    from tests import gpu_util as U
    lib = U.init()
    rng = np.random.default_rng(3)
    rows, K, T = 1000, 128, 77
    w = bf16(rng.standard_normal((rows, K)))
    W = lib.pi_weight_upload(30, K, rows, w.ctypes.data_as(C.c_void_p), None)
    xh, out = U.Dev(bf16(rng.standard_normal((T, K)))), U.Dev(nbytes=4 * T * rows)
    got, met = _asked(lib, U, lambda: lib.pi_op_dense_rounded(W, None, xh.ptr, K, 0, 0, 1, T, out.ptr, rows, 4, rows // 2, 0, None), out, 488, 64, T, 0)
    assert met == 1 and np.array_equal(got, bf16(out.get(np.float32, (T, rows))[:, 488:552]))
    odd = U.Dev(rng.standard_normal((T, 67)).astype(np.float32))      # rows that no 16-byte load can take
    h = U.Dev(nbytes=2 * T * 64)
    L.check(lib.pi_op_round_bf16(odd.ptr + 4, 67, 64, T, h.ptr, 64, None))
    assert np.array_equal(h.get(np.uint16, (T, 64)), bf16(odd.get(np.float32, (T, 67))[:, 1:65]))
    lib.pi_weight_free(W)


# tiles of 64 and 128 slots by every number of rows; one step of K and fewer than stages; an expert without tokens, identity experts, runs that end inside a tile
@pytest.mark.gpu
@pytest.mark.parametrize("E,I,ff,width,T,top", [(2, 1, 128, 192, 300, 2), (8, 2, 64, 3136, 200, 2), (8, 0, 64, 1536, 210, 2), (70, 3, 64, 64, 40, 6), (1, 0, 64, 64, 33, 1), (3, 0, 64, 128, 700, 2), (2, 0, 64, 8256, 1500, 2), (8, 0, 2048, 256, 3000, 2)])
def test_experts_of_rounded_inputs(E, I, ff, width, T, top):
    from tests import gpu_util as U
    lib = U.init()
    rng = np.random.default_rng([E, T])
    x = rng.standard_normal((T, width)).astype(np.float32)
    ups, downs = bf16(rng.standard_normal((E, ff, width)) * width ** -0.5), bf16(rng.standard_normal((E, width, ff)) * ff ** -0.5)
    sel = np.stack([rng.permutation(E + I)[:top] for _ in range(T)]).astype(np.int32)
    sel[sel == 1] = 0 if E > 3 else 1
    selw = rng.uniform(0.1, 1.0, (T, top)).astype(np.float32)
    ud = lib.pi_weight_upload(30, width, E * ff, ups.ctypes.data_as(C.c_void_p), None)
    dd = lib.pi_weight_upload(30, ff, E * width, downs.ctypes.data_as(C.c_void_p), None)
    xd, xh, sd, wd = U.Dev(x), U.Dev(bf16(x)), U.Dev(sel), U.Dev(selw)
    hd, nd, od = U.Dev(nbytes=2 * T * top * ff), U.Dev(nbytes=4 * T * top * width), U.Dev(nbytes=4 * T * width)
    idx = U.Dev(nbytes=4 * lib.pi_op_moe_grouped_index_ints(T, top, E))
    assert lib.pi_op_moe_rounded_ok(ud, dd, E, ff, width, T, top) == 1
    L.check(lib.pi_op_moe_experts_rounded(ud, dd, E, ff, xh.ptr, width, xd.ptr, width, sd.ptr, wd.ptr, T, top, hd.ptr, nd.ptr, idx.ptr, od.ptr, width, None))
    hidden, got = wide(hd.get(np.uint16, (T, top, ff))).astype(np.float64), od.get(np.float32, (T, width))
    xr = wide(bf16(x)).astype(np.float64)
    want = np.zeros((T, width))
    for e in range(E + I):
        for k in range(top):
            at = np.flatnonzero(sel[:, k] == e)
            if e >= E:
                want[at] += selw[at, k, None] * x[at]
                continue
            h = np.maximum(xr[at] @ wide(ups[e]).astype(np.float64).T, 0) ** 2
            # a hidden value is the fp32 one rounded to bfloat16: 2^-8 of it, and the fp32 sum's own error (squared)
            assert (np.abs(hidden[at, k] - h) <= 2.0 ** -8 * h + 1e-5).all()
            want[at] += selw[at, k, None] * (hidden[at, k] @ wide(downs[e]).astype(np.float64).T)
    assert np.sqrt(((got - want) ** 2).mean()) < 3e-6 * np.sqrt((want ** 2).mean())      # (fp32 sums of at most 8256 terms)
    for w in (ud, dd):
        lib.pi_weight_free(w)
