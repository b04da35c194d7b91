"""Products of more than 128 prompt rows with hi + lo activations (crane_amd/csrc/kernels_gemm_tile.hip): the rule on the host, and on the GPU the same prompt with
cm_debug_set("gemm256") 1 (these tiles) and 0 (the 128-column kernel).

The tolerance is that of tests/test_gpu_gemm_prompts.py: where K is not split both add the same products in the same order and have the same SiLU, so that their rows are equal; where it
is split, a sum of K <= 6144 terms moves by about sqrt(K) 2^-24 of its size, and a K or V element lands on the other side of a
16-bit boundary once in a thousand.  2e-3 of the largest logit is ten times what two layers make of that; a tile, a row or a column that is lost or misplaced moves the logits
by their own size."""
import numpy as np
import pytest

from crane_amd import _lib

WS = 1 << 24
TOL = 2e-3
SHAPES = {(256, 256), (128, 384), (128, 256), (128, 192)}


def plan(m, n, k, norm=0, ws=WS):
    got = _lib.load().cm_debug_gemm_tile(m, n, k, norm, ws)
    return (got // 10000, got // 10 % 1000, got % 10) if got else None


# the figures beside the rule: each shape where it is the fastest, K in slices, widths without a tile, chips too empty
@pytest.mark.parametrize("m,n,k,norm,want", [(2048, 24576, 4096, 0, (256, 256, 1)), (2048, 6144, 4096, 0, (128, 384, 1)), (2048, 4096, 12288, 1, (128, 256, 1)), (400, 6144, 1024, 0, (128, 192, 1)),
                                             (800, 2048, 6144, 1, (128, 256, 4)), (128, 24576, 4096, 0, None), (2048, 8320, 2048, 0, None), (300, 1024, 2048, 1, None), (160, 4096, 1024, 0, None)])
def test_the_shape(m, n, k, norm, want):
    assert plan(m, n, k, norm) == want


# a tile divides the width, the slices divide the k-tiles and leave eight or more, the workspace holds them, and there are blocks enough
def test_every_plan_is_one():
    for n in (128, 1024, 2048, 3072, 4096, 6144, 6528, 6720, 8192, 12288, 24576):
        for k in (64, 512, 1024, 2048, 3264, 4096, 12288, 1056):
            for m in list(range(120, 140)) + list(range(141, 4097, 61)):
                for ws in (0, 1 << 20, WS):
                    got = plan(m, n, k, m & 1, ws)
                    if got is None:
                        continue
                    bm, bn, ks = got
                    assert m > 128 and (bm, bn) in SHAPES and n % bn == 0 and k % 64 == 0 and k // 64 % ks == 0 and k // 64 // ks >= 8
                    assert (ks == 1 or ks * m * n <= ws) and -(-m // bm) * (n // bn) * ks >= (128 if m <= 256 else 64)


# first and last rows of a tile, a row tile of one row, more k-tiles than one and an odd number of them (3264 = 51); all shapes, whole and in slices
CASES = [(1024, 3072, 16, 8, (129, 257, 385, 1025, 1409, 1536)), (2048, 6144, 32, 16, (129, 256, 385, 511, 1025, 1279)), (1024, 3264, 24, 12, (383, 1100))]


def test_the_cases_reach_every_shape():
    seen = set()
    for h, i, heads, kv, tokens in CASES:
        for m in tokens:
            for n, k, norm in (((heads + 2 * kv) * 128, h, 0), (h, heads * 128, 1), (2 * i, h, 0), (h, i, 1)):
                got = plan(m, n, k, norm)
                if got:
                    seen.add((got[0], got[1], got[2] > 1))
    assert seen >= {s + (False,) for s in SHAPES} | {(128, 256, True), (128, 192, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("h,i,heads,kv,tokens", CASES)
def test_against_the_128_column_kernel(h, i, heads, kv, tokens):
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=h, intermediate_size=i, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
               vocab_size=512, num_hidden_layers=2)
    m = Model.synthetic(cfg, seed=3, max_seq_len=1600, max_seqs=2)
    rng = np.random.default_rng(4)
    try:
        for n in tokens:
            ids = rng.integers(0, 512, n).tolist()
            rows = []
            for mode in (1, 0):
                m.debug_set("gemm256", mode)
                s = m.seq_alloc()
                rows.append(np.asarray(m.seq_forward(s, ids, 0)[0], np.float64))
                m.seq_free(s)
            assert np.isfinite(rows[0]).all() and np.abs(rows[0] - rows[1]).max() < TOL * np.abs(rows[1]).max(), n
    finally:
        m.close()


# whole products in both kernels (no slices of K, no norm in a reduction): the sums have one order and SiLU one rounding, so every bit is the same
WHOLE = [(2048, 6144, 4096, 0), (2048, 4096, 4096, 1), (2048, 24576, 4096, 0), (2048, 4096, 12288, 1)]


def test_the_products_are_whole():
    assert all(plan(*p)[2] == 1 for p in WHOLE)


@pytest.mark.gpu
def test_the_bits_of_the_128_column_kernel():
    from crane_amd import configs
    from crane_amd.backend import Model
    m = Model.synthetic(dict(configs.get_config("qwen3-8b"), vocab_size=512, num_hidden_layers=2), seed=3, max_seq_len=2048, max_seqs=1)
    try:
        for seed in (1, 2):
            ids = np.random.default_rng(seed).integers(0, 512, 2048).tolist()
            rows = []
            for mode in (1, 0):
                m.debug_set("gemm256", mode)
                s = m.seq_alloc()
                rows.append(np.asarray(m.seq_forward(s, ids, 0)[0]).copy())
                m.seq_free(s)
            assert np.array_equal(rows[0], rows[1])
    finally:
        m.close()
