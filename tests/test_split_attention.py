"""Attention of prompts over a latent, keys, values, queries and weights in three bfloat16 parts (split_attention.hip): against the explicit fp64 sums.  Every call is given the scratch memory that the parts need, and shows by what it
left there that they were made"""
import numpy as np
import pytest

from pipeinfer_amd import lib as L
from tests.test_letevik import HALVES, NEIGHBOURS, SIGMOID, O, gpu, rel_rms, upload_bf16

BOUND = 2e-6        # fp32 sums of up to 512 + 192 + 1000 terms in tiles; rounding the products' inputs to bfloat16 would be 2e-3


def floats_of(cells, H, D, R, V):
    return (cells + 63) // 64 * 64 * 3 * (H * (D + V) + R) // 2


def state_of(T, H, V):
    """sums, maximum and denominator between two launches over the cells"""
    return T * H * (V + 2) + 3


class Call:
    """one call of the operator: tokens at `pos`, each of which sees the cells up to its own (or what `vis` says); `live` cells of n_kv are in use (the rest hold NaN), `floats` of scratch memory (none given: the parts of all cells in one launch).
    out: its output; parts(cell0): whether the scratch holds the keys of the first head's cells from cell0 on as the first operand of three parts"""
    def __init__(self, U, lib, rng, H, D, R, V, rank, n_kv, pos, pairing=HALVES, gate_width=0, sink=None, scale=None, cache=None, live=None, floats=None, vis=None):
        T, live, self.base, self.pairing, self.H, self.V = len(pos), n_kv if live is None else live, 500.0, pairing, H, V
        self.D, self.R, self.rank, self.live, self.pos, self.gate_width, self.sink, self.scale = D, R, rank, live, np.asarray(pos), gate_width, sink, (D + R) ** -0.5 if scale is None else scale
        self.Wk, self.Wv = (O.bf16_round((rng.standard_normal((H * s, rank)) / np.sqrt(rank)).astype(np.float32)) for s in (D, V))
        self.q = rng.standard_normal((T, H, D + R)).astype(np.float32)
        self.cache = np.full((n_kv, rank + R), np.nan, np.float32)
        self.cache[:live] = rng.standard_normal((live, rank + R)) if cache is None else cache
        self.g = rng.standard_normal((T, H * max(gate_width, 1) + 1)).astype(np.float32)
        words = (n_kv + 31) // 32
        self.vis = np.arange(words * 32)[None, :] <= self.pos[:, None]
        if vis is not None:
            self.vis = np.pad(vis, ((0, 0), (0, words * 32 - n_kv)))
        mask = np.packbits(self.vis, axis=1, bitorder="little").view(np.uint32)
        t = lib.pi_rotary_table_create(int(max(pos)) + 2, R, self.base) if R else None
        uk, uv = upload_bf16(lib, self.Wk), upload_bf16(lib, self.Wv)
        s = np.zeros(H, np.float32) if sink is None else np.asarray(sink, np.float32)
        q_row, out_row = H * (D + R) + 4, H * V + 3
        qd, cd, md, gd, sd, pd, dd = (U.Dev(a) for a in (np.pad(self.q.reshape(T, -1), ((0, 0), (0, 4)), constant_values=np.nan), self.cache, mask, self.g, s, self.pos.astype(np.int32), np.array([0, live, T, 0], np.int32)))
        n = max(floats_of(n_kv, H, D, R, V) if floats is None else floats, lib.pi_op_latent_attention_rot_scratch_floats(H, rank, R, T, n_kv))
        if floats is not None:
            assert n == floats, "the per-token kernels' memory is more: not what the test is about"
        scr, od = U.Dev(np.full(n, np.nan, np.float32)), U.Dev(np.full((T, out_row), 7.0, np.float32))
        L.check(lib.pi_op_latent_attention_gated(qd.ptr, q_row, cd.ptr, md.ptr, uk, uv, sd.ptr if sink is not None else None, gd.ptr if gate_width else None, self.g.shape[1], SIGMOID, max(gate_width, 1), self.scale, H, D, R, V,
                                                 rank, t, pairing, pd.ptr, T, n_kv, scr.ptr, n, od.ptr, out_row, dd.ptr, None))
        out = od.get(np.float32, (T, out_row))
        assert (out[:, H * V:] == 7.0).all()
        self.out, self.first = out[:, :H * V].reshape(T, H, V), scr.get(np.uint32, count=512 * 4)
        lib.pi_weight_free(uk)
        lib.pi_weight_free(uv)
        if t:
            lib.pi_rotary_table_free(t)

    def keys(self, h, cell0=0, cells=None):
        return self.cache[cell0:self.live if cells is None else min(cell0 + cells, self.live), :self.rank].astype(np.float64) @ self.Wk[h * self.D:(h + 1) * self.D].T.astype(np.float64)

    def parts(self, cell0=0):
        k = self.keys(0, cell0, 32)[:, :16]
        got = (self.first.view(np.uint16)[:512].astype(np.uint32) << 16).view(np.float32).reshape(2, 32, 8).transpose(1, 0, 2).reshape(32, 16)[:len(k)]      # lane l: cell l % 32, values 8 (l / 32) .. + 7
        return bool((np.abs(got - k) <= np.abs(k) * 2.0 ** -8 + np.abs(k).max() * 1e-5).all())

    def want(self, h):
        """head h of all tokens; a token's sums hold the cells that it sees and no others"""
        rot, T = {"dims": self.R, "base": self.base}, len(self.pos)
        k, v = self.keys(h), self.cache[:self.live, :self.rank].astype(np.float64) @ self.Wv[h * self.V:(h + 1) * self.V].T.astype(np.float64)
        q = self.q[:, h].astype(np.float64)
        if self.R:
            k = np.concatenate([k, self.cache[:self.live, self.rank:].astype(np.float64)], 1)
            q = np.concatenate([q[:, :self.D], np.stack([O.turn(q[t, self.D:], int(self.pos[t]), rot, self.pairing == NEIGHBOURS) for t in range(T)])], 1)
        s, vis = (q @ k.T) * self.scale, self.vis[:, :self.live]
        out = np.zeros((T, self.V))
        if np.isfinite(v).all() and np.isfinite(s).all():
            some = vis.any(1)                                          # (a token that sees nothing: zeros)
            s = np.where(vis, s, -np.inf)[some]
            m = np.maximum(s.max(1), -np.inf if self.sink is None else self.sink[h])
            e = np.exp(s - m[:, None])
            out[some] = e @ v / (e.sum(1) + (0.0 if self.sink is None else np.exp(self.sink[h] - m)))[:, None]
        else:
            for t in range(T):
                out[t] = O.softmax(s[t][vis[t]], None if self.sink is None else self.sink[h]) @ v[vis[t]]
        if self.gate_width:
            out = out * O.sigmoid(self.g[:, h * self.gate_width:(h + 1) * self.gate_width])
        return out

    def error(self, heads=None):
        heads = list(range(self.H) if heads is None else heads)
        return rel_rms(self.out[:, heads], np.stack([self.want(h) for h in heads], 1))


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,R,V,rank", [(3, 64, 0, 64, 128), (5, 64, 32, 128, 256), (2, 128, 64, 128, 512), (7, 128, 0, 64, 384), (33, 64, 32, 64, 128), (3, 128, 0, 128, 512), (4, 128, 64, 64, 256), (2, 64, 0, 128, 384)])
@pytest.mark.parametrize("T,n_kv", [(33, 33), (40, 97), (64, 320), (130, 700)])
def test_split_attention(H, D, R, V, rank, T, n_kv):
    """every shape of a head, ranks of one and of several stages, tiles of rows, queries and cells that are not full, runs that a wave does not have; gates of both widths and none, with and without a sink, both pairings"""
    U, lib = gpu()
    rng = np.random.default_rng(H * 100 + T)
    for pairing, width, sink in ((HALVES, V, True), (NEIGHBOURS, 1, False), (HALVES, 0, True)):
        c = Call(U, lib, rng, H, D, R, V, rank, n_kv, np.arange(n_kv - T, n_kv), pairing, width, rng.standard_normal(H) * 2 if sink else None)
        assert c.parts() and c.error() < BOUND, (pairing, width, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("D,R,rank", [(64, 32, 128), (128, 0, 512), (64, 0, 256), (128, 64, 512)])
@pytest.mark.parametrize("V", [64, 128])
def test_split_attention_of_many_heads(D, R, V, rank):
    """a wave for every 32 queries instead of four (many heads and tokens): every shape of a head, a last workgroup of which one wave has eight queries and one has none"""
    U, lib = gpu()
    rng = np.random.default_rng(D + R + V)
    c = Call(U, lib, rng, 128, D, R, V, rank, 390, np.arange(390 - 200, 390), NEIGHBOURS if R == 64 else HALVES, 1, rng.standard_normal(128))
    assert c.parts() and c.error(list(range(0, 128, 9)) + [127]) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("H,T", [(2, 50), (96, 384)])
def test_split_attention_in_several_launches(H, T):
    """scratch memory for the parts of 1024 cells of 2000: sums, maximum and denominator stand between the launches, by four waves and by one wave a tile"""
    U, lib = gpu()
    D, R, V, rank, n_kv = 64, 32, 64, 128, 2000
    c = Call(U, lib, np.random.default_rng(3), H, D, R, V, rank, n_kv, np.arange(n_kv - T, n_kv), HALVES, 1, np.zeros(H), floats=floats_of(1024, H, D, R, V) + state_of(T, H, V))
    assert c.parts(1024) and c.error(range(0, H, 15)) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("H,T", [(3, 70), (96, 384)])
@pytest.mark.parametrize("seen", ["any", "window", "far apart"])
def test_split_attention_of_any_mask(H, T, seen):
    """any set of cells, tokens that see none, single cells with thousands between them that nobody sees (a wave looks at 64 of its runs at a time), windows"""
    U, lib = gpu()
    rng = np.random.default_rng(H)
    D, R, V, rank, n_kv = 64, 32, 64, 128, {"any": 500, "window": 700, "far apart": 9000 if H == 3 else 2300}[seen]
    pos = np.sort(rng.integers(n_kv // 2, n_kv, T))
    cells = np.arange(n_kv)[None, :]
    vis = rng.random((T, n_kv)) < 0.3 if seen == "any" else (cells <= pos[:, None]) & (cells > pos[:, None] - 40) if seen == "window" else (cells % 2237 == pos[:, None] % 3)
    vis[5], vis[T - 33:T - 1] = False, False                          # a token, and a whole tile of queries at least in part
    for sink in (None, rng.standard_normal(H)):
        c = Call(U, lib, rng, H, D, R, V, rank, n_kv, pos, HALVES, 1, sink, vis=vis)
        heads = list(range(0, H, 31))
        assert c.parts() and c.error(heads) < BOUND
        assert not c.out[5].any() and not c.out[T - 33:T - 1].any()


@pytest.mark.gpu
@pytest.mark.parametrize("live", [600, 3072])
def test_parts_that_would_take_more_launches(live):
    """scratch memory for the keys and values of all 3072 cells as they are, or for the parts of 1920: they are written as they are, in one launch"""
    U, lib = gpu()
    H, D, V, rank, n_kv, T = 32, 128, 128, 128, 3072, 256
    c = Call(U, lib, np.random.default_rng(4), H, D, 0, V, rank, n_kv, np.arange(live - T, live), live=live, floats=n_kv * H * (D + V))
    assert not c.parts(0) and not (live > 1920 and c.parts(1920)) and c.error(range(0, H, 7)) < BOUND
    assert rel_rms(c.first.view(np.float32)[:16], c.keys(0, 0, 1)[0, :16]) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,R,V", [(5, 64, 32, 64), (6, 128, 0, 128), (96, 64, 0, 64)])
@pytest.mark.parametrize("live", [63, 64, 65, 700, 1023, 1024, 1025, 1056, 2000])
@pytest.mark.parametrize("at_once", [True, False])
def test_split_attention_over_the_cells_in_use(H, D, R, V, live, at_once):
    """fewer cells in use than there could be, which the operator learns on the device: a last run of 32 cells that is not full, whole or missing, a second launch whose cells are all, some or none of them in use; what lies behind them is
    no number"""
    U, lib = gpu()
    T, n_kv, rank = min(live, 63 if H < 96 else 384), 2000, 128        # (96 heads of 384 tokens: a wave for every 32 queries; fewer tokens of them are not taken in parts)
    floats = None if at_once else floats_of(1024, H, D, R, V) + state_of(T, H, V)
    rng = np.random.default_rng(live + H)
    c = Call(U, lib, rng, H, D, R, V, rank, n_kv, np.arange(live - T, live), HALVES, 0, rng.standard_normal(H), live=live, floats=floats)
    assert c.error(range(0, H, 17) if H > 9 else None) < BOUND
    assert c.parts(0 if at_once or live <= 1024 else 1024) or (H == 96 and T < 384)


@pytest.mark.gpu
@pytest.mark.parametrize("live", [45, 5000, 5969, 5970, 5971, 5972, 9000, 16384])
def test_split_attention_up_to_the_line_of_the_kernels_per_token(live):
    """two heads over up to 16384 cells: the parts up to some live cells, the kernels per token beyond; the ones that do not take a pass leave nothing behind"""
    U, lib = gpu()
    H, D, V, rank, n_kv, T = 2, 64, 64, 128, 16384, 40
    c = Call(U, lib, np.random.default_rng(live), H, D, 0, V, rank, n_kv, np.arange(live - T, live), HALVES, V, None, live=live)
    assert c.error() < (BOUND if c.parts() else 1e-5)
    if live < 5001 or live > 8999:
        assert c.parts() == (live < 5001)


@pytest.mark.gpu
@pytest.mark.parametrize("H,T", [(4, 140), (128, 200)])
@pytest.mark.parametrize("D,R,V", [(64, 0, 64), (128, 64, 128)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3.4e38])
def test_split_attention_of_values_out_of_range(H, T, D, R, V, bad):
    """a latent that is no number, or so large that sums with it leave fp32's range, reaches the tokens that see it and no others; where the sums stay in range they are right"""
    U, lib = gpu()
    rng = np.random.default_rng(11)
    rank, n_kv = 128, T + 30
    cache = rng.standard_normal((n_kv, rank + R)).astype(np.float32)
    cache[n_kv - 3, 5] = bad
    with np.errstate(invalid="ignore", over="ignore"):
        c = Call(U, lib, rng, H, D, R, V, rank, n_kv, np.arange(n_kv - T, n_kv), cache=cache)
        heads = range(H) if H < 9 else range(0, H, 37)
        want = np.stack([c.want(h) for h in heads], 1)
    got = c.out[:, list(heads)]
    assert c.parts() and rel_rms(got[:-3], want[:-3]) < BOUND
    if not np.isfinite(bad):
        assert not np.isfinite(c.out[-3:]).any()
        return
    for t in range(T - 3, T):                                          # (the loud cell has a token's whole mass or none of it, head by head)
        for i in range(len(got[t])):
            assert rel_rms(got[t, i], want[t, i]) < BOUND, (t, i)


@pytest.mark.gpu
@pytest.mark.parametrize("H,T", [(3, 40), (128, 200)])
@pytest.mark.parametrize("scale", [1e-30, 1e-4, 1e6, 1e17])
def test_split_attention_of_small_and_large_values(scale, H, T):
    """parts cover fp32's range: latents of any size, the queries' scale the other way"""
    U, lib = gpu()
    rng = np.random.default_rng(12)
    D, V, rank, n_kv = 128, 128, 256, 230
    cache = (rng.standard_normal((n_kv, rank)) * scale).astype(np.float32)
    c = Call(U, lib, rng, H, D, 0, V, rank, n_kv, np.arange(n_kv - T, n_kv), scale=float(D ** -0.5 / scale), cache=cache)
    assert c.parts() and c.error(range(0, H, 37) if H > 9 else None) < BOUND


def test_scratch_memory_of_the_parts():
    """six bytes for every key and value of all cells, in whole blocks of 64; nothing where a pass does not take them"""
    of = L.load().pi_op_latent_attention_prompt_scratch_floats
    assert of(32, 128, 0, 128, 512, 512, 3000) == 3008 * 12288 and of(3, 64, 32, 128, 128, 9, 64) == 64 * 912
    assert [of(3, 64, 0, 64, 128, 8, 64), of(3, 64, 16, 64, 128, 9, 64), of(3, 96, 0, 64, 128, 9, 64), of(3, 64, 0, 96, 128, 9, 64), of(3, 64, 0, 64, 64, 9, 64), of(3, 64, 0, 64, 640, 9, 64), of(3, 64, 0, 64, 0, 9, 64)] == [0] * 7


@pytest.mark.gpu
@pytest.mark.parametrize("H,T,n_kv,parts", [(96, 128, 400, False), (64, 200, 400, False), (64, 128, 400, True), (128, 256, 300, True), (16, 512, 1000, True)])
def test_which_prompts_are_taken_in_parts(H, T, n_kv, parts):
    """heads beyond a round of workgroups over few cells are quicker with keys and values as they are"""
    U, lib = gpu()
    c = Call(U, lib, np.random.default_rng(H), H, 128, 0, 128, 128, n_kv, np.arange(n_kv - T, n_kv))
    assert c.parts() == parts and c.error(range(0, H, 23)) < BOUND
