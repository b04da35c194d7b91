"""GPU: the tiled matrix-core attention of prompt passes (kernels_layered_attn.hip) against the f32 FMA kernel on the same cache, at the
edges of its tiles and masks.

One attention layer without a feed-forward, bfloat16 format, the same portions with the matrix-core kernels on and off.  Both read the same
pages; the matrix cores read the query rounded to bfloat16 where the FMA kernel keeps 32 bits.  With keys and queries of unit variance
that moves a score by 2^-9 / sqrt(3) = 1.1e-3 in the mean square (d independent roundings of d products of size d^-1/2), the weights by the
same share and the largest logit by no more; everything else (weights as a 16-bit hi + lo pair, exp and log of the hardware units, the
bfloat16 rounding of the attention rows on their way into the output projection, which tips 0.3 % of the elements over) is below 3e-4.
8e-3 of the largest logit is seven times that."""
import types

import numpy as np
import pytest

from tests import gibipel_util as GI
from tests import gizezen_util as GZ
from tests import korupel_util as KO
from tests import mononex_util as MO

pytestmark = pytest.mark.gpu

TOL = 8e-3


def _run(tmp_path, U, cfg, portions, seed, **kw):
    """Logits of every fourth position and of the last 70, with the matrix-core kernels on, then off."""
    from crane_amd.backend import Model
    P = U.random_weights(cfg, seed)
    n = sum(portions)
    toks = U.tokens(n, cfg["vocab"], seed + 1)
    m = Model.from_pretrained(U.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=4, max_seq_len=2048, **kw)
    try:
        got = []
        for on in (1, 0):
            m.debug_set("lay_attn_mfma", on)
            s, at, rows = m.seq_alloc(), 0, []
            for k in portions:
                want = [i for i in range(k) if i % 4 == 0 or i >= k - 70]
                rows.append(m.step_batch([(s, toks[at:at + k], want)])[0])
                at += k
            got.append(np.concatenate(rows).astype(np.float64))
            m.seq_free(s)
        return got
    finally:
        m.close()


def _check(got):
    assert np.isfinite(got[0]).all() and np.abs(got[0] - got[1]).max() < TOL * np.abs(got[1]).max()


# key / value sizes on both sides of the padded sizes (64, 128); query rows per position 1, 3, 4; portions that start inside a tile and
# end on, before and behind a tile's edge; windows shorter than a tile, around it and over the whole context
@pytest.mark.parametrize("d,e,heads,kv,size,portions", [
    (16, 16, 4, 4, 7, (65, 16, 130)), (64, 80, 6, 2, 64, (100, 200)), (80, 64, 4, 1, 65, (63, 64, 65)), (128, 128, 8, 2, 1000, (300, 17)),
    (112, 128, 4, 1, 128, (190, 150)), (96, 48, 3, 3, 200, (64, 128, 100))])
@pytest.mark.parametrize("page", [64, 128])
def test_window_and_one_in_the_denominator(tmp_path, d, e, heads, kv, size, portions, page):
    mx = GZ.attn(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size, rot_dims=16)
    _check(_run(tmp_path, GZ, GZ.config([GZ.layer(mx, None)], vocab=96, width=64), portions, 3, kv_block_size=page))


# first tokens kept in front of the window (fewer than a tile, more than a tile, reaching into the window), a logarithmic distance term,
# values that are the keys
@pytest.mark.parametrize("d,heads,kv,size,keep,portions", [(32, 4, 2, 20, 3, (70, 150)), (128, 4, 1, 90, 70, (100, 260)), (48, 5, 5, 300, 128, (330,)),
                                                           (64, 2, 1, 5, 64, (130, 67))])
def test_kept_first_tokens_and_distance_term(tmp_path, d, heads, kv, size, keep, portions):
    mx = KO.attn(heads=heads, kv_heads=kv, dim=d, size=size, keep_first=keep)
    _check(_run(tmp_path, KO, KO.config([KO.layer("attention", None, **mx)], vocab=96, width=64), portions, 5))


# position blocks (a query sees its own block only), a linear distance term, a sink, a gate per element; block edges on and off tile edges
@pytest.mark.parametrize("d,e,heads,kv,size,portions", [(32, 16, 6, 2, 50, (200, 30)), (128, 112, 4, 2, 64, (129, 70)), (64, 64, 2, 2, 200, (150, 150))])
def test_position_blocks_and_sink(tmp_path, d, e, heads, kv, size, portions):
    mx = MO.attn(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size)
    _check(_run(tmp_path, MO, MO.config([MO.layer("attention", None, **mx)], vocab=96, width=64), portions, 7))


# mean rows of the blocks in front of the window: fewer than a tile of them, more than a tile, blocks that end in another page
@pytest.mark.parametrize("d,e,heads,kv,size,pool,portions", [(32, 16, 4, 2, 20, 6, (120, 100)), (128, 128, 4, 1, 30, 4, (300, 40)), (64, 96, 2, 2, 70, 64, (250, 65))])
def test_block_rows(tmp_path, d, e, heads, kv, size, pool, portions):
    lf = GI.left(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size, pool=pool)
    cfg = GI.config([GI.layer(lf, GI.right(), None)], vocab=96, width=64)
    _check(_run(tmp_path, GI, cfg, portions, 9))


# many key heads and query blocks, window shorter than the portion
@pytest.mark.parametrize("d,e,size,portions", [(16, 16, 300, (1025,)), (128, 128, 2000, (40, 1100)), (64, 80, 33, (1090,))])
def test_many_heads(tmp_path, d, e, size, portions):
    mx = GZ.attn(heads=64, kv_heads=64, dim=d, vdim=e, size=size, rot_dims=16)
    _check(_run(tmp_path, GZ, GZ.config([GZ.layer(mx, None)], vocab=96, width=64), portions, 11))


# ---- decode steps: the kernel for few query rows keeps 24 bits of queries and weights (three bfloat16 parts each), as the FMA kernel does, so the
# attention rows agree to a few 1e-6 and what is left is the output projection's rounding of 0.1 % of them: 1e-3 of the largest logit
TOL_FEW = 1e-3


def _few(tmp_path, U, cfg, contexts, steps, seed, **kw):
    """Three sequences with contexts of their own step together, `steps` tokens each per step; matrix-core kernels on, then off."""
    from crane_amd.backend import Model
    P = U.random_weights(cfg, seed)
    n = max(contexts) + sum(steps)
    toks = [U.tokens(n, cfg["vocab"], seed + 1 + i) for i in range(len(contexts))]
    m = Model.from_pretrained(U.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=8, max_seq_len=4096, **kw)
    got = []
    try:
        for on in (1, 0):
            m.debug_set("lay_attn_mfma", on)
            seqs, rows, at = [m.seq_alloc() for _ in contexts], [], list(contexts)
            for s, t, c in zip(seqs, toks, contexts):
                if c:
                    m.step_batch([(s, t[:c], [])], want_logits=False)      # one layer: the cached rows do not depend on the attention
            for k in steps:
                rows.append(m.step_batch([(s, t[a:a + k], list(range(k))) for s, t, a in zip(seqs, toks, at)])[0])
                at = [a + k for a in at]
            got.append(np.concatenate(rows).astype(np.float64))
            for s in seqs:
                m.seq_free(s)
    finally:
        m.close()
    assert np.isfinite(got[0]).all() and np.abs(got[0] - got[1]).max() < TOL_FEW * np.abs(got[1]).max()


# no context, one short of a tile, a tile, one more; more tiles than waves; one and several 16-row tiles per sequence; every key in one wave's
# first tile or spread over blocks (more than 24 tiles: partial sums and a merge)
@pytest.mark.parametrize("d,e,heads,kv,size,contexts,steps", [
    (16, 16, 4, 4, 7, (0, 63, 64), (1, 1, 15)), (64, 80, 6, 2, 64, (65, 127, 600), (1, 3, 1)), (128, 128, 8, 2, 1000, (1, 700, 1300), (1, 1)),
    (112, 48, 4, 1, 4000, (1600, 2500, 3100), (1, 6)), (80, 128, 16, 1, 3000, (1535, 1536, 2200), (1, 1))])
@pytest.mark.parametrize("page", [64, 128])
def test_decode_window_and_one_in_the_denominator(tmp_path, d, e, heads, kv, size, contexts, steps, page):
    mx = GZ.attn(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size, rot_dims=16)
    _few(tmp_path, GZ, GZ.config([GZ.layer(mx, None)], vocab=96, width=64), contexts, steps, 13, kv_block_size=page)


@pytest.mark.parametrize("d,heads,kv,size,keep,contexts", [(32, 4, 2, 20, 3, (0, 150, 400)), (128, 4, 1, 90, 70, (60, 161, 700)), (48, 5, 5, 300, 128, (330, 5, 1000))])
def test_decode_kept_first_tokens_and_distance_term(tmp_path, d, heads, kv, size, keep, contexts):
    mx = KO.attn(heads=heads, kv_heads=kv, dim=d, size=size, keep_first=keep)
    _few(tmp_path, KO, KO.config([KO.layer("attention", None, **mx)], vocab=96, width=64), contexts, (1, 1, 4), 15)


# a steep distance term of small arguments, r1 log(1 + r2 dist) with r2 dist down to 1e-7: 1 + x in f32 is 6e-8 off, times r1 = 1e6 a score by 0.06 and
# its weight by 6 %; log1p keeps both sides at 1e-7 of the term
def test_decode_distance_term_of_small_arguments(tmp_path):
    def weights(cfg, seed):
        P = KO.random_weights(cfg, seed)
        P["l0.mix.r1"][:] = KO.bf16_round(np.full_like(P["l0.mix.r1"], 1e6))
        P["l0.mix.r2"][:] = KO.bf16_round(np.full_like(P["l0.mix.r2"], 1e-7))
        return P
    U = types.SimpleNamespace(random_weights=weights, tokens=KO.tokens, write_checkpoint=KO.write_checkpoint)
    mx = KO.attn(heads=4, kv_heads=2, dim=32, size=1000, keep_first=3)
    _few(tmp_path, U, KO.config([KO.layer("attention", None, **mx)], vocab=96, width=64), (5, 150, 400), (1, 1, 4), 21)


@pytest.mark.parametrize("d,e,heads,kv,size,contexts", [(32, 16, 6, 2, 50, (49, 99, 100)), (128, 112, 4, 2, 64, (63, 64, 500)), (64, 64, 2, 2, 3000, (2999, 1, 2000))])
def test_decode_position_blocks_and_sink(tmp_path, d, e, heads, kv, size, contexts):
    mx = MO.attn(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size)
    _few(tmp_path, MO, MO.config([MO.layer("attention", None, **mx)], vocab=96, width=64), contexts, (1, 2, 1), 17)


@pytest.mark.parametrize("d,e,heads,kv,size,pool,contexts", [(32, 16, 4, 2, 20, 6, (19, 26, 300)), (128, 128, 4, 1, 30, 4, (33, 700, 1900)), (64, 96, 2, 2, 70, 64, (133, 134, 64))])
def test_decode_block_rows(tmp_path, d, e, heads, kv, size, pool, contexts):
    lf = GI.left(heads=heads, kv_heads=kv, dim=d, vdim=e, size=size, pool=pool)
    _few(tmp_path, GI, GI.config([GI.layer(lf, GI.right(), None)], vocab=96, width=64), contexts, (1, 1, 3), 19)
