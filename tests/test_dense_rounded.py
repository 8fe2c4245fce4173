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
