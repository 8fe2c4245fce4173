"""Attention of prompts over a latent, keys, values, queries and weights in three bfloat16 parts (split_attention.hip): against the explicit fp64 sums"""
import numpy as np
import pytest

from tests.test_letevik import HALVES, NEIGHBOURS, O, gpu, latent_case, rel_rms

BOUND = 2e-6        # fp32 sums of up to 512 + 192 + 1000 terms in tiles; rounding the products' inputs to bfloat16 would be 2e-3


class LessScratch:
    """the library, as if a pass needed no more scratch memory than `floats`"""
    def __init__(self, lib, floats):
        self.lib, self.floats = lib, floats

    def __getattr__(self, name):
        return (lambda *a: self.floats) if name == "pi_op_latent_attention_rot_scratch_floats" else getattr(self.lib, name)


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,R,V,rank", [(3, 64, 0, 64, 128), (5, 64, 32, 128, 256), (2, 128, 64, 128, 512), (7, 128, 0, 64, 384), (33, 64, 32, 64, 128)])
@pytest.mark.parametrize("T,n_kv", [(33, 33), (40, 97), (64, 320), (130, 700)])
def test_split_attention(H, D, R, V, rank, T, n_kv):
    """every shape of a head, ranks of one and several stages, tiles of rows, queries and cells that are not full, runs that a wave does not have"""
    U, lib = gpu()
    rng = np.random.default_rng(H * 100 + T)
    pos = np.arange(n_kv - T, n_kv)
    for pairing, width, sink in ((HALVES, V, True), (NEIGHBOURS, 1, False), (HALVES, 0, True)):
        got, want = latent_case(U, lib, rng, H, D, R, V, rank, n_kv, pos, 500.0, pairing, width, rng.standard_normal(H) * 2 if sink else None, (D + R) ** -0.5)
        assert rel_rms(got, want) < BOUND, (pairing, width, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("D,R", [(64, 32), (128, 0)])
def test_split_attention_of_many_heads(D, R):
    """a wave for every 32 queries instead of four (512 workgroups and more that way)"""
    U, lib = gpu()
    got, want = latent_case(U, lib, np.random.default_rng(D), 128, D, R, 64, 128, 390, np.arange(5, 390), 500.0, HALVES, 0, None, (D + R) ** -0.5)
    assert rel_rms(got, want) < BOUND


@pytest.mark.gpu
def test_split_attention_in_several_launches():
    """scratch memory for the parts of 1024 cells: sums, maximum and denominator stand between the launches"""
    U, lib = gpu()
    H, D, R, V, rank, T, n_kv = 2, 64, 32, 64, 128, 50, 2500
    floats = 1024 * 3 * (H * (D + V) + R) // 2 + T * H * (V + 2) + 3
    got, want = latent_case(U, LessScratch(lib, max(floats, 0)), np.random.default_rng(3), H, D, R, V, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, HALVES, 1, np.zeros(H), (D + R) ** -0.5)
    assert rel_rms(got, want) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3.4e38])
def test_split_attention_of_values_out_of_range(bad):
    """a latent that is no number, or so large that its sums are none, reaches the tokens that see it and no others"""
    U, lib = gpu()
    rng = np.random.default_rng(11)
    H, D, V, rank, T, n_kv = 4, 64, 64, 128, 70, 140
    cache = rng.standard_normal((n_kv, rank)).astype(np.float32)
    cache[n_kv - 3, 5] = bad
    with np.errstate(invalid="ignore", over="ignore"):
        got, want = latent_case(U, lib, rng, H, D, 0, V, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, HALVES, 0, None, D ** -0.5, cache=cache)
    assert rel_rms(got[:-3], want[:-3]) < BOUND and (not np.isfinite(got[-3:]).any() if bad != 3.4e38 else True)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-30, 1e-4, 1e6, 1e17])
def test_split_attention_of_small_and_large_values(scale):
    """parts cover fp32's range: latents of any size, the queries' scale the other way"""
    U, lib = gpu()
    rng = np.random.default_rng(12)
    H, D, V, rank, T, n_kv = 3, 128, 128, 256, 40, 200
    cache = (rng.standard_normal((n_kv, rank)) * scale).astype(np.float32)
    got, want = latent_case(U, lib, rng, H, D, 0, V, rank, n_kv, np.arange(n_kv - T, n_kv), 500.0, HALVES, 0, None, float(D ** -0.5 / scale), cache=cache)
    assert rel_rms(got, want) < BOUND
