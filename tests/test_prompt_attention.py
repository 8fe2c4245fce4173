"""Attention on the matrix cores.  Passes of many tokens (prompt_attention.hip): 32 tokens of a head at a time, keys and values of a latent written out first; few tokens over a latent (hybrid.hip).  Against the explicit fp64 sums that the per-token kernels are tested with."""
import numpy as np
import pytest

from pipeinfer_amd import lib as L
from tests import test_fasovik as fasovik
from tests.test_letevik import HALVES, NEIGHBOURS, SIGMOID, O, diff_attention_ref, gpu, latent_case, pack_mask, rel_rms, run_diff
from tests.test_rarevik import CHUNK


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,R,V,rank,T,n_kv", [(3, 8, 4, 12, 24, 9, 33), (32, 8, 4, 12, 24, 33, 33), (32, 64, 0, 64, 72, 32, 300), (8, 128, 64, 128, 512, 130, 200), (16, 64, 32, 64, 256, 50, 80), (11, 20, 36, 68, 136, 95, 161), (4, 64, 0, 64, 256, 300, 2500), (64, 4, 2, 4, 8, 70, 97)])
def test_latent_prompt(H, D, R, V, rank, T, n_kv):
    """tiles that are not full (tokens, cells, key and output values), both pairings, every kind of gate, with and without a sink; the long one takes two launches over the cells (its scratch memory holds the
    keys and values of 1600)"""
    U, lib = gpu()
    rng = np.random.default_rng(H * 100 + T)
    pos = np.arange(n_kv - T, n_kv)
    for pairing, width, sink in ((HALVES, V, True), (NEIGHBOURS, 1, False)) if n_kv > 1000 else ((HALVES, V, True), (NEIGHBOURS, V, False), (HALVES, 1, True), (HALVES, 0, False)):
        got, want = latent_case(U, lib, rng, H, D, R, V, rank, n_kv, pos, 500.0, pairing, width, rng.standard_normal(H) * 2 if sink else None, (D + R) ** -0.5)
        assert rel_rms(got, want) < 1e-5, (pairing, width, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,R,V,rank", [(16, 8, 64, 24, 512), (5, 20, 36, 17, 512), (3, 8, 0, 33, 256), (7, 4, 4, 8, 256)])
@pytest.mark.parametrize("T,n_kv", [(1, 33), (1, 700), (4, 64), (8, 130), (3, 4200)])
def test_latent_few_tokens(H, D, R, V, rank, T, n_kv):
    """sixteen rows (token, head) at a time over splits of 32 cells: rows and splits that are not full, more than 64 splits, a rotated part that ends inside a step"""
    U, lib = gpu()
    rng = np.random.default_rng(H * 100 + n_kv)
    pos = np.arange(n_kv - T, n_kv)
    for pairing, width, sink in ((HALVES, V, True), (NEIGHBOURS, 1, False)):
        got, want = latent_case(U, lib, rng, H, D, R, V, rank, n_kv, pos, 500.0, pairing, width, rng.standard_normal(H) * 2 if sink else None, (D + R) ** -0.5)
        assert rel_rms(got, want) < 1e-5, (pairing, width, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("H,R,rank", [(16, 64, 512), (17, 0, 512), (7, 8, 256), (32, 0, 256), (33, 4, 256), (64, 4, 512)])
@pytest.mark.parametrize("T,n_kv", [(9, 9), (16, 100), (17, 700), (31, 40), (32, 600), (33, 64)])
def test_latent_rows_and_tiles(H, R, rank, T, n_kv):
    """both sides of the line between splits of 32 cells and the tiles of a prompt (32 tokens; 512 rows of rank 512, 1024 of rank 256)"""
    U, lib = gpu()
    rng = np.random.default_rng(H + T)
    got, want = latent_case(U, lib, rng, H, 8, R, 12, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, NEIGHBOURS, 1, None, (8 + R) ** -0.5)
    assert rel_rms(got, want) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("H,rank,T", [(40, 256, 8), (33, 512, 8), (3, 512, 2), (8, 256, 32)])
@pytest.mark.parametrize("live", [40, 700, 9000])
def test_latent_context_that_holds_less_than_it_could(H, rank, T, live):
    """16384 cells of which a few are live (the operator learns how many on the device): workgroups that take several splits in turn, splits that nobody writes and nobody reads"""
    U, lib = gpu()
    rng = np.random.default_rng(H + live)
    D, V, cells, pos = 8, 12, 16384, np.arange(live - T, live)
    wk, wv = (O.bf16_round((rng.standard_normal((H * n, rank)) / np.sqrt(rank)).astype(np.float32)) for n in (D, V))
    cache = np.full((cells, rank), np.nan, np.float32)
    cache[:live] = rng.standard_normal((live, rank))
    q, vis = rng.standard_normal((T, H, D)).astype(np.float32), np.arange(cells)[None, :] <= pos[:, None]
    uk, uv = fasovik.upload_bf16(lib, wk), fasovik.upload_bf16(lib, wv)
    qd, cd, md, sd, dd, od = U.Dev(q), U.Dev(cache), U.Dev(pack_mask(vis, cells)), U.Dev(np.full(H, -30.0, np.float32)), U.Dev(np.array([0, live, T, 0], np.int32)), U.Dev(nbytes=4 * T * H * V)
    n = lib.pi_op_latent_attention_rot_scratch_floats(H, rank, 0, T, cells)
    scr = U.Dev(np.full(n, np.nan, np.float32))
    L.check(lib.pi_op_latent_attention(qd.ptr, H * D, cd.ptr, md.ptr, uk, uv, sd.ptr, 0.3, H, D, V, rank, T, cells, scr.ptr, n, od.ptr, H * V, dd.ptr, None))
    got, c = od.get(np.float32, (T, H, V)), cache[:live].astype(np.float64)
    for h in range(0, H, 7):
        s = (c @ wk.reshape(H, D, rank)[h].T.astype(np.float64)) @ q[:, h].T.astype(np.float64) * np.float32(0.3)
        w = np.where(vis[:, :live].T, np.exp(s), 0)
        want = (w / (w.sum(0) + np.exp(-30.0))).T @ (c @ wv.reshape(H, V, rank)[h].T.astype(np.float64))
        assert rel_rms(got[:, h], want) < 1e-5
    lib.pi_weight_free(uk)
    lib.pi_weight_free(uv)


@pytest.mark.gpu
@pytest.mark.parametrize("H,rank,T", [(8, 264, 9), (7, 264, 40), (2, 64, 20), (16, 512, 30)])
@pytest.mark.parametrize("live", [45, 7000, 8300, 8738, 8739, 11650, 11750, 16384])
def test_latent_both_sides_of_the_line_between_tiles_and_tokens(H, rank, T, live):
    """16384 cells: which kernels take a pass is decided on the device, by how many are live; the ones that do not take it leave nothing behind"""
    U, lib = gpu()
    rng = np.random.default_rng(H + live)
    D, V, cells, pos = 8, 12, 16384, np.arange(live - T, live)
    wk, wv = (O.bf16_round((rng.standard_normal((H * n, rank)) / np.sqrt(rank)).astype(np.float32)) for n in (D, V))
    cache = np.full((cells, rank), np.nan, np.float32)
    cache[:live] = rng.standard_normal((live, rank))
    q, vis = rng.standard_normal((T, H, D)).astype(np.float32), np.arange(cells)[None, :] <= pos[:, None]
    uk, uv = fasovik.upload_bf16(lib, wk), fasovik.upload_bf16(lib, wv)
    qd, cd, md, sd, dd, od = U.Dev(q), U.Dev(cache), U.Dev(pack_mask(vis, cells)), U.Dev(np.full(H, -30.0, np.float32)), U.Dev(np.array([0, live, T, 0], np.int32)), U.Dev(nbytes=4 * T * H * V)
    n = max(lib.pi_op_latent_attention_rot_scratch_floats(H, rank, 0, T, cells), 1 << 22)
    scr = U.Dev(np.full(n, np.nan, np.float32))
    L.check(lib.pi_op_latent_attention(qd.ptr, H * D, cd.ptr, md.ptr, uk, uv, sd.ptr, 0.3, H, D, V, rank, T, cells, scr.ptr, n, od.ptr, H * V, dd.ptr, None))
    got, c = od.get(np.float32, (T, H, V)), cache[:live].astype(np.float64)
    for h in range(H):
        s = (c @ wk.reshape(H, D, rank)[h].T.astype(np.float64)) @ q[:, h].T.astype(np.float64) * np.float32(0.3)
        w = np.where(vis[:, :live].T, np.exp(s), 0)
        want = (w / (w.sum(0) + np.exp(-30.0))).T @ (c @ wv.reshape(H, V, rank)[h].T.astype(np.float64))
        assert rel_rms(got[:, h], want) < 1e-5
    lib.pi_weight_free(uk)
    lib.pi_weight_free(uv)


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [40, 64, 256, 512, 768])
@pytest.mark.parametrize("T,n_kv", [(1, 2600), (2, 300), (3, 2600), (4, 4500), (7, 900)])
def test_latent_splits_are_merged(rank, T, n_kv):
    """one to four tokens of a tile, splits that groups of threads share out (all tokens at once, one after the other) and that one group takes, rounds of 64 splits that are not full"""
    U, lib = gpu()
    rng = np.random.default_rng(rank + T)
    got, want = latent_case(U, lib, rng, 5, 12, 0, 20, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, HALVES, 0, rng.standard_normal(5), 12 ** -0.5)
    assert rel_rms(got, want) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("H,rank,T,n_kv", [(6, 256, 5, 700), (16, 512, 4, 200), (1, 256, 1, 64), (5, 512, 8, 100)])
def test_latent_few_tokens_over_scattered_cells(H, rank, T, n_kv):
    """what a token sees is any set of cells; what lies behind the cells in use is no number"""
    fasovik.test_latent_attention_against_explicit_keys_and_values(H, 16, 24, rank, T, n_kv)


@pytest.mark.gpu
@pytest.mark.parametrize("H,R,rank,T,n_kv", [(6, 4, 256, 5, 70), (16, 0, 512, 3, 33), (3, 0, 256, 8, 200), (5, 64, 512, 4, 64), (6, 4, 64, 12, 90)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_latents_that_are_no_numbers(H, R, rank, T, n_kv, bad):
    """rows of several tokens share a tile, and some of them see a latent that is no number: it reaches those and no others"""
    U, lib = gpu()
    rng = np.random.default_rng(H * 100 + n_kv)
    cache = rng.standard_normal((n_kv, rank + R)).astype(np.float32)
    cache[n_kv - 2, 1] = bad
    with np.errstate(invalid="ignore"):
        got, want = latent_case(U, lib, rng, H, 8, R, 12, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, HALVES, 12, None, (8 + R) ** -0.5, cache=cache)
    assert rel_rms(got[:-2], want[:-2]) < 1e-5 and not np.isfinite(got[-2:]).any()


def scattered(rng, T, n_kv, n_ctx):
    """positions of cells in any order, tokens' positions, what the mask shows (a token sees at least itself)"""
    cpos = rng.permutation(n_ctx).astype(np.int32)
    pos = np.sort(rng.integers(n_kv // 3, n_kv, T)).astype(np.int32)
    near = [int(np.argmax(np.where(cpos[:n_kv] <= p, cpos[:n_kv], -1))) for p in pos]
    pos = cpos[near]
    vis = (cpos[None, :n_kv] <= pos[:, None]) & (rng.random((T, n_kv)) < 0.8)
    vis[np.arange(T), near] = True
    return cpos, pos, vis


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,size,keep,n_kv,T", [(2, 1, 4, 4, 3, 2, 40, 32), (8, 2, 64, 128, 256, 4, 700, 97), (3, 3, 36, 68, 0, 0, 130, 65), (4, 1, 128, 64, 9, 33, 333, 200), (16, 1, 64, 128, 256, 4, 700, 4), (6, 2, 128, 64, 9, 33, 333, 31), (5, 5, 64, 64, 0, 0, 1200, 1), (4, 2, 192, 128, 50, 0, 161, 40)])
@pytest.mark.parametrize("maps", [2, 1])
def test_window_prompt(H, G, D, V, size, keep, n_kv, T, maps):
    """plain and differential heads over windows with kept positions, cells in any order, garbage behind the live cells"""
    U, lib = gpu()
    rng = np.random.default_rng(D + T)
    kc, vc = (rng.standard_normal((n_kv + 13, G, maps, D)) * 1.5).astype(np.float32), rng.standard_normal((n_kv + 13, G, V)).astype(np.float32)
    kc[n_kv:], vc[n_kv:] = np.nan, np.nan
    cpos, pos, vis = scattered(rng, T, n_kv, n_kv + 13)
    q = (rng.standard_normal((T, H, maps, D)) * 2).astype(np.float32)
    args = (q, kc, vc, cpos, vis, pos, 0.6 * D ** -0.25, size, keep, maps, 0.45, 0.7, 1e-3, H, G)
    want = diff_attention_ref(*(a[:n_kv] if a is kc or a is vc or a is cpos else a for a in args))
    assert rel_rms(run_diff(U, lib, *args, True), want) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,size,keep,n_kv,T", [(2, 1, 64, 64, 60, 3, 9300, 33), (2, 2, 36, 68, 60, 0, 17001, 40), (3, 1, 64, 128, 60, 3, 9300, 5), (2, 2, 128, 64, 5000, 0, 70001, 2), (2, 1, 64, 64, 0, 0, 8225, 32), (32, 32, 64, 64, 0, 0, 700, 31)])
@pytest.mark.parametrize("maps", [2, 1])
def test_window_in_a_long_context(H, G, D, V, size, keep, n_kv, T, maps):
    """walks that look at 64 runs of 32 cells at a time and visit the ones with something to see (more than 8192 cells, 4096 of two maps; splits of more than 256): every run and few, cells in any order, the last run and the
    last 64 not full; an infinity that nobody sees stays out"""
    U, lib = gpu()
    rng = np.random.default_rng(n_kv + T)
    kc, vc = (rng.standard_normal((n_kv + 13, G, maps, D)) * 1.5).astype(np.float32), rng.standard_normal((n_kv + 13, G, V)).astype(np.float32)
    kc[n_kv:], vc[n_kv:] = np.nan, np.nan
    cpos, pos, vis = scattered(rng, T, n_kv, n_kv + 13)
    q = (rng.standard_normal((T, H, maps, D)) * 2).astype(np.float32)
    hidden = np.nonzero(~(vis & ((cpos[None, :n_kv] > pos[:, None] - size) | (cpos[None, :n_kv] < keep) | (size == 0))).any(0))[0][-1]
    vc[hidden] = np.inf                                                # (nobody sees it)
    args = (q, kc, vc, cpos, vis, pos, 0.6 * D ** -0.25, size, keep, maps, 0.45, 0.7, 1e-3, H, G)
    clean = vc.copy()
    clean[hidden] = 0
    want = diff_attention_ref(*(clean[:n_kv] if a is vc else a[:n_kv] if a is kc or a is cpos else a for a in args))
    assert rel_rms(run_diff(U, lib, *args, True), want) < 1e-5


@pytest.mark.gpu
def test_latent_prompt_in_a_long_context():
    """the walk of the mask alone (keys written out of a latent), in one launch and in several over the cells"""
    U, lib = gpu()
    rng = np.random.default_rng(5)
    for n_kv, rank in ((9300, 264), (30000, 128)):
        got, want = latent_case(U, lib, rng, 2, 12, 4, 12, rank, n_kv, np.arange(n_kv - 9, n_kv), 500.0, NEIGHBOURS, 1, None, 0.3)
        assert rel_rms(got, want) < 1e-5, n_kv


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,chunk,n_kv,T", [(2, 1, 16, 8, 32, 90, 33), (8, 2, 128, 128, 256, 600, 150), (40, 1, 8, 128, 9, 290, 32), (1, 1, 64, 64, 7, 65, 1), (32, 2, 128, 64, 64, 300, 4), (24, 8, 64, 128, 300, 1100, 31),
                                                   (30, 2, 128, 128, 700, 2100, 8)])
@pytest.mark.parametrize("softcap", [0.0, 3.0])
def test_weights_of_a_prompt(H, G, D, V, chunk, n_kv, T, softcap):
    """passes of many tokens, and of few over splits of the cells (sixteen query heads of a key head or fewer, a split of one round and of several, splits that show nothing): sigmoid weights, a soft-max and one with a sink, a bias and a gate per head, capped scores (of a soft-max); a token that sees nothing; values that are no numbers reach the tokens that see them and no others"""
    U, lib = gpu()
    rng = np.random.default_rng(n_kv + T)
    kc, vc = rng.standard_normal((n_kv, G, D)).astype(np.float32), rng.standard_normal((n_kv, G, V)).astype(np.float32)
    cpos, pos, vis = scattered(rng, T, n_kv, n_kv)
    vis[7:8] = False
    hurt = vis[:, 5] & (cpos[5] >= (pos // chunk * chunk))
    q, gate, hb = rng.standard_normal((T, H, D)).astype(np.float32), rng.standard_normal((T, H)).astype(np.float32), rng.standard_normal(H).astype(np.float32)
    for loud in (False, True):
        if loud:
            vc[5, 0, 3] = np.inf
        for weights in (0, 1, 2):
            d = [U.Dev(a) for a in (q, kc, vc, cpos, pack_mask(vis, n_kv), pos, hb, gate, np.array([0, n_kv, T, 0], np.int32))]
            od = U.Dev(nbytes=4 * T * H * V)
            n_scr = lib.pi_op_window_attention_scratch_floats(H, V, T)
            scr = U.Dev(np.full(n_scr, np.nan, np.float32))
            L.check(lib.pi_op_window_attention(d[0].ptr, H * D, d[1].ptr, d[2].ptr, d[3].ptr, d[4].ptr, d[5].ptr, d[6].ptr, None, d[7].ptr, H, SIGMOID, 0.21, -1.5, weights, softcap, CHUNK, chunk, 0, 0, 0, H, G, D, V, T, n_kv,
                                               scr.ptr, n_scr, od.ptr, H * V, d[8].ptr, None))
            got, want = od.get(np.float32, (T, H, V)), np.zeros((T, H, V))
            for t in range(T):
                js = np.nonzero(vis[t] & (cpos >= pos[t] // chunk * chunk))[0]
                for h in range(H):
                    s = kc[js, h // (H // G)].astype(np.float64) @ q[t, h].astype(np.float64) * np.float32(0.21) + hb[h]
                    s = softcap * np.tanh(s / softcap) if softcap and weights else s
                    w = O.sigmoid(s) if weights == 0 else np.exp(s) / (np.exp(s).sum() + (weights == 2)) if len(js) else s
                    want[t, h] = vc[js, h // (H // G)].T.astype(np.float64) @ w * O.sigmoid(gate[t, h]) * -1.5
            fine = np.isfinite(want)
            assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(got[~fine], want[~fine].astype(np.float32)) and (fine.all() or (loud and hurt.any()))
            assert rel_rms(np.where(fine, got, 0), np.where(fine, want, 0)) < 1e-5, (weights, loud)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 3, 40])
def test_launches_of_a_cancelled_run(T):
    """kernels that ask for the abort word and go on loading: a run that is cancelled ahead of them writes neither results nor partial sums, and every launch is counted once (a single token, a few, a prompt)"""
    U, lib = gpu()
    rng = np.random.default_rng(T)
    H, G, D, V, rank, E, top, n_kv = 4, 2, 64, 64, 256, 5, 2, 300
    word = U.Dev(np.zeros(16, np.int32))
    f = lambda *shape: U.Dev(rng.standard_normal(shape).astype(np.float32))
    w = lambda n, k: fasovik.upload_bf16(lib, fasovik.bf(rng, n, k, s=0.1))
    q, kc, vc, cache, x = f(T, H * 2 * D), f(n_kv, G, 2 * D), f(n_kv, G, V), f(n_kv, rank), f(T, rank)
    pos, cpos, mask = U.Dev(np.arange(n_kv - T, n_kv, dtype=np.int32)), U.Dev(np.arange(n_kv, dtype=np.int32)), U.Dev(pack_mask(np.ones((T, n_kv), bool), n_kv))
    dyn, hb, uk, uv, router, corr = U.Dev(np.array([0, n_kv, T, 0], np.int32)), f(H), w(H * D, rank), w(H * V, rank), w(E, rank), f(E)
    n_scr = max(lib.pi_op_window_attention_scratch_floats(2 * H, V, T), lib.pi_op_latent_attention_rot_scratch_floats(H, rank, 0, max(T, 8), n_kv))
    out, scr, sel = U.Dev(np.full((T, H * V), 555.0, np.float32)), U.Dev(np.full(n_scr, 777.0, np.float32)), U.Dev(np.full(T * top, 333, np.int32))
    calls = {
        "differential heads": lambda: lib.pi_op_diff_attention(q.ptr, 2 * H * D, kc.ptr, vc.ptr, cpos.ptr, mask.ptr, pos.ptr, 0.1, 0, 0, 2, 0.4, 1.0, 1e-5, H, G, D, V, T, n_kv, scr.ptr, n_scr, out.ptr, H * V, dyn.ptr, None),
        "window": lambda: lib.pi_op_window_attention(q.ptr, H * D, kc.ptr, vc.ptr, cpos.ptr, mask.ptr, pos.ptr, hb.ptr, None, None, 0, 0, 0.1, 1.0, 1, 0.0, CHUNK, 0, 0, 0, 0, H, G, D, V, T, n_kv, scr.ptr, n_scr, out.ptr, H * V,
                                                     dyn.ptr, None),
        "latent": lambda: lib.pi_op_latent_attention(q.ptr, H * D, cache.ptr, mask.ptr, uk, uv, hb.ptr, 0.1, H, D, V, rank, T, n_kv, scr.ptr, n_scr, out.ptr, H * V, dyn.ptr, None),
        "router": lambda: lib.pi_op_moe_route(router, corr.ptr, x.ptr, rank, T, top, 0, sel.ptr, out.ptr, None),
    }
    L.check(lib.pi_op_abort_begin(word.ptr, 3, None, None))
    L.check(lib.pi_op_abort_cancel(word.ptr, 3, None))
    for name, call in calls.items():
        before = word.get(np.int32)[8:15].sum()
        lib.pi_set_abort_word(word.ptr)
        try:
            L.check(call())
        finally:
            lib.pi_set_abort_word(None)
        assert np.all(out.get(np.float32) == 555.0) and np.all(scr.get(np.float32) == 777.0) and np.all(sel.get(np.int32) == 333), name
        launches = {"differential heads": 1 if T >= 32 else 2, "window": 1 if T >= 32 else 2, "latent": 2 if T > 8 else 3, "router": 1}[name]
        assert word.get(np.int32)[8:15].sum() - before == launches, name


@pytest.mark.gpu
@pytest.mark.parametrize("T,n_kv", [(40, 300), (33, 64), (2, 1100), (8, 200)])
@pytest.mark.parametrize("maps", [1, 2])
def test_scores_of_minus_infinity(T, n_kv, maps):
    """cells whose scores overflow to minus infinity have no weight, wherever they lie: at the start of every wave's and every split's range, or in all of it; a token that sees nothing else gets zeros"""
    U, lib = gpu()
    H, G, D, V = 4, 2, 64, 64
    rng = np.random.default_rng(n_kv + T)
    q = np.abs(rng.standard_normal((T, H, maps, D))).astype(np.float32) + 0.1
    kc, vc = rng.standard_normal((n_kv, G, maps, D)).astype(np.float32), rng.standard_normal((n_kv, G, V)).astype(np.float32)
    far = (np.arange(n_kv) % 64 < 32) & (np.arange(n_kv) < n_kv - T)
    kc[far] = -3e38
    cpos, pos, vis = np.arange(n_kv, dtype=np.int32), np.arange(n_kv - T, n_kv, dtype=np.int32), np.arange(n_kv)[None, :] <= np.arange(n_kv - T, n_kv)[:, None]
    vis[T - 1] = far
    args = [vis, pos, 3.0, 0, 0, maps, 0.45, 0.7, 1e-3, H, G]
    got = run_diff(U, lib, q, kc, vc, cpos, *args, True)
    near = ~far
    args[0] = vis[:T - 1][:, near]
    args[1] = pos[:T - 1]
    want = diff_attention_ref(q[:T - 1], kc[near], vc[near], cpos[near], *args)
    assert rel_rms(got[:T - 1], want) < 1e-5 and np.all(got[T - 1] == 0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("step", [0.4, 3.0, -3.0, 30.0])
@pytest.mark.parametrize("D,V,maps", [(64, 64, 1), (64, 128, 2), (36, 68, 1)])
def test_scores_that_climb_and_fall(step, D, V, maps):
    """scores that rise or fall from cell to cell, by less and by more than the maximum may lag, in tiles that all tokens see and tiles that some see; a value that is no number where nobody sees it and where two tokens do"""
    U, lib = gpu()
    H, G, T, n_kv = 4, 2, 70, 400
    rng = np.random.default_rng(D + V)
    q = np.zeros((T, H, maps, D), np.float32)
    q[..., 0], q[..., 1:] = 1.0, rng.standard_normal((T, H, maps, D - 1)) * 0.1
    kc, vc = rng.standard_normal((n_kv, G, maps, D)).astype(np.float32), rng.standard_normal((n_kv, G, V)).astype(np.float32)
    kc[..., 0] = (step * np.arange(n_kv) / 16)[:, None, None]
    vis = np.arange(n_kv)[None, :] <= np.arange(n_kv - T, n_kv)[:, None]
    vis[:, 100] = False
    vis[40:, 200] = False
    args = [np.arange(n_kv, dtype=np.int32), vis, np.arange(n_kv - T, n_kv, dtype=np.int32), 1.0, 0, 0, maps, 0.45, 0.7, 1e-3, H, G]
    want = diff_attention_ref(q, kc, vc, *args)
    # a score of size s is a sum of D fp32 terms, each rounded to s 2^-24 at worst: the exponent of its weight is off by some s 2^-24 sqrt(D)
    bound = max(1e-5, abs(step) * n_kv / 16 * 2.0 ** -24 * D ** 0.5)
    assert rel_rms(run_diff(U, lib, q, kc, vc, *args, True), want) < bound
    vc[100], vc[200, 0, 5] = np.nan, np.inf                               # (seen by none; seen by the first forty, in one value of the first key head)
    got = run_diff(U, lib, q, kc, vc, *args, True)
    assert rel_rms(got[40:], want[40:]) < bound and np.isfinite(got[:, H // G:]).all() and not np.isfinite(got[:40, :H // G]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [33, 70])
@pytest.mark.parametrize("D,V", [(64, 64), (128, 128), (36, 68)])
def test_large_values_under_a_climbing_score(D, V, T):
    """scores that climb by less than the maximum may lag, values near the top of fp32's range: weights of at most 1 keep their sums finite, as do the waves' sums together"""
    U, lib = gpu()
    H, G, n_kv = 4, 2, 400
    rng = np.random.default_rng(D + T)
    q = np.zeros((T, H, 1, D), np.float32)
    q[..., 0] = 1.0
    kc, vc = np.zeros((n_kv, G, 1, D), np.float32), (1.0 + rng.random((n_kv, G, V))).astype(np.float32)
    kc[..., 0] = (7.5 * np.arange(n_kv) / n_kv)[:, None, None]
    vis = np.arange(n_kv)[None, :] <= np.arange(n_kv - T, n_kv)[:, None]
    args = [np.arange(n_kv, dtype=np.int32), vis, np.arange(n_kv - T, n_kv, dtype=np.int32), 1.0, 0, 0, 1, 0.0, 1.0, 1e-3, H, G]
    want = diff_attention_ref(q, kc, vc, *args)
    big = np.float32(2.0 ** 119)                                          # (a token's sum at weights of at most 1: 54 effective cells of up to 2 big; at weights of up to e^7.5: past the range)
    got = run_diff(U, lib, q, kc, vc * big, *args, True)
    assert np.isfinite(got).all() and rel_rms(got.astype(np.float64) / float(big), want) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(64, 64), (128, 128), (36, 68)])
def test_large_values_beside_a_lagging_maximum(D, V):
    """three waves that each see one value near the top of fp32's range, the fourth scores that climb within its run of cells by less than its maximum may lag: what the three weigh beside them keeps their sum finite"""
    U, lib = gpu()
    H, G, T, n_kv = 2, 1, 40, 128
    q = np.zeros((T, H, 1, D), np.float32)
    q[..., 0] = 1.0
    kc, vc = np.zeros((n_kv, G, 1, D), np.float32), np.ones((n_kv, G, V), np.float32)
    kc[112:, ..., 0] = 7.5
    vc[[0, 32, 64]] = 2.5e38
    vis = np.zeros((T, n_kv), bool)
    vis[:, [0, 32, 64]] = vis[:, 96:] = True
    args = [np.arange(n_kv, dtype=np.int32), vis, np.full(T, n_kv, np.int32), 1.0, 0, 0, 1, 0.0, 1.0, 1e-3, H, G]
    want = diff_attention_ref(q, kc, vc, *args)
    got = run_diff(U, lib, q, kc, vc, *args, True)
    assert np.isfinite(got).all() and rel_rms(got / 1e38, want / 1e38) < 1e-5
