"""Prompt attention of layer-list decoders whose long walks are shared among blocks (kernels_layered_attn.hip: lay_attn_tile_kernel): which walks (host logic, through
cm_debug_lay_attn_shares), and on the GPU against the form without a matrix core, in passes of few query tiles.

Layers without a feed-forward: no choice of experts can tip, so every row is held to the bound of tests/test_gpu_layered_attention.py, which compares the two forms on one layer
(8e-3 of the largest logit, seven times what the queries' rounding gives; up to 3.4e-3 seen where layers follow each other, 4.8e-3 with the logarithmic distance term).  Scores
and residual are scaled so that the attention decides the logits: half of a walk left out moves every row of these portions by 0.02 and more (windows; Gizezen), the median row by 0.05
(Korupel) and 0.1 (Mononex).
"""
import random

import numpy as np
import pytest

from crane_amd import _lib
from tests import gizezen_util as GZ
from tests import korupel_util as KO
from tests import mononex_util as MO

BLOCKS = 256
TOL = 8e-3


def _shares(portions, heads, kv_heads, window):
    """(start, rows) of every portion -> [(portion, first query row, share, shares)]"""
    import ctypes as C
    n, out = len(portions), (C.c_int32 * (4 * BLOCKS))()
    starts, rows = (C.c_int32 * n)(*[p[0] for p in portions]), (C.c_int32 * n)(*[p[1] for p in portions])
    total = _lib.load().cm_debug_lay_attn_shares(starts, rows, n, heads, kv_heads, window, out)
    return [tuple(out[4 * i:4 * i + 4]) for i in range(total)]


# seven key tiles of 64 are the first walk that is shared; walks are looked at while the tiles leave blocks of one round free
@pytest.mark.parametrize("start,shares", [(300, 1), (383 - 29, 1), (383 - 28, 2), (1000, 3)])
def test_walks_of_more_than_six_tiles(start, shares):
    got = _shares([(start, 30), (5, 1)], 4, 2, 1 << 40)
    assert max([s[3] for s in got], default=1) == shares
    # long walks among short ones on two key heads: more than half a round of blocks, as many as a round has, more
    assert [bool(_shares([(start, 30)] * n + [(5, 1)] * 70, 4, 2, 1 << 40)) for n in (10, 58, 59)] == [shares > 1, False, False]


def test_lists_are_whole_and_fit_one_round_of_blocks():
    rng = random.Random(5)
    seen = 0
    for _ in range(3000):
        nrep, kv = rng.choice([1, 2, 3, 4, 8]), rng.choice([1, 2, 3, 8, 16])
        portions = [(rng.randrange(6000), 1 if rng.random() < 0.7 else rng.randrange(2, 700)) for _ in range(rng.randrange(1, 60))]
        window = rng.choice([1 << 40, 4096, 300, 64])
        got = _shares(portions, nrep * kv, kv, window)
        assert len(got) * kv <= BLOCKS
        if not got:
            continue
        seen += 1
        want = [(i, q0) for i, (_, n) in enumerate(portions) for q0 in range(0, n * nrep, 64)]
        at = 0
        for seg, q0 in want:                    # a tile's shares side by side, each once
            shares = got[at][3]
            assert got[at:at + shares] == [(seg, q0, k, shares) for k in range(shares)]
            at += shares
        assert at == len(got) and at > len(want)
    assert seen > 300


def _run(tmp_path, U, cfg, start):
    """A portion of 30 rows beside one token of another sequence, three times, behind `start` tokens: all rows, with the matrix-core kernels and without."""
    from crane_amd.backend import Model
    m = Model.from_pretrained(U.write_checkpoint(str(tmp_path / "ckpt"), cfg, U.random_weights(cfg, 8)), compute_dtype="bfloat16", max_seqs=4, max_seq_len=1280)
    long, short = U.tokens(start + 90, cfg["vocab"], 40), U.tokens(60, cfg["vocab"], 41)
    got = []
    try:
        for on in (1, 0):
            m.debug_set("lay_attn_mfma", on)
            a, b = m.seq_alloc(), m.seq_alloc()
            m.step_batch([(a, long[:start], []), (b, short[:50], [])], want_logits=False)
            rows = []
            for k in range(3):
                rows.append(m.step_batch([(a, long[start + 30 * k:start + 30 * k + 30], list(range(30))), (b, short[50 + k:51 + k], None)])[0])
            got.append(np.concatenate(rows).astype(np.float64))
            m.seq_free(a)
            m.seq_free(b)
    finally:
        m.close()
    assert got[0].shape[0] == 93 and np.isfinite(got[0]).all()
    off = np.abs(got[0] - got[1]).max(-1) / np.abs(got[1]).max()
    assert off.max() < TOL, (float(off.max()), int(off.argmax()))


# walks just below and above the line, portions that end inside a tile, windows that leave some of a walk's shares empty (a layer of a shorter window beside one of a
# longer: the lists follow the longer), a single token beside them, the counters' next use
@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (48, 112), (112, 48)])
@pytest.mark.parametrize("start", [300, 383, 384, 1000])
def test_windows(tmp_path, dim, vdim, start):
    assert bool(_shares([(start, 30), (50, 1)], 4, 2, 1024)) == (start + 29 >= 384)
    layers = [GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=dim, vdim=vdim, size=size, rot_dims=16, scale=2 * dim ** -0.5), None) for size in (1024, 70, 400)]
    cfg = GZ.config(layers, vocab=96, width=256, mult=2.0, embed_scale=1.0)
    _run(tmp_path, GZ, cfg, start)


# keys kept in front of the window (in the first share, in several), the logarithmic distance term, values that are the keys
@pytest.mark.gpu
@pytest.mark.parametrize("dim,heads,kv_heads,size,keep", [(64, 4, 2, 500, 3), (128, 4, 1, 300, 200), (48, 5, 5, 1000, 70), (128, 8, 2, 400, 0)])
@pytest.mark.parametrize("start", [420, 1000])
def test_kept_first_tokens_and_distance_term(tmp_path, dim, heads, kv_heads, size, keep, start):
    assert _shares([(start, 30), (50, 1)], heads, kv_heads, size + keep)
    mixer = KO.attn(heads=heads, kv_heads=kv_heads, dim=dim, size=size, keep_first=keep)
    _run(tmp_path, KO, KO.config([KO.layer("attention", None, **mixer)], vocab=96, width=256), start)


# position blocks that are shorter than the walk the shares are made for, the linear distance term, a sink (the first share's), a gate per element
@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim,heads,kv_heads,size", [(64, 64, 4, 2, None), (128, 112, 4, 1, 700), (32, 16, 6, 2, 100)])
@pytest.mark.parametrize("start", [420, 1000])
def test_position_blocks_and_sink(tmp_path, dim, vdim, heads, kv_heads, size, start):
    assert _shares([(start, 30), (50, 1)], heads, kv_heads, 1 << 40)
    layers = [MO.layer("attention", None, **MO.attn(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=s)) for s in (size, None)]
    _run(tmp_path, MO, MO.config(layers, vocab=96, width=256), start)


# a long walk of rows that are NaN beside a sound one, both shared: the sound rows keep the bits that they have beside other sound ones, and so does the next pass on the same counters
@pytest.mark.gpu
def test_rows_that_are_no_numbers(tmp_path):
    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=64, vdim=64, size=1024), None) for _ in range(2)], vocab=96, width=256)
    assert len(_shares([(600, 30), (500, 30)], 4, 2, 1024)) == 4
    P = GZ.random_weights(cfg, 8)
    P["embed"][5] = np.nan
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=4, max_seq_len=768)
    toks, got = 7 + np.array(GZ.tokens(660, 80, 9)), []
    try:
        for t in (5, 6):
            a, b = m.seq_alloc(), m.seq_alloc()
            m.step_batch([(a, toks[:600], []), (b, np.full(500, t), [])], want_logits=False)
            rows = [m.step_batch([(a, toks[600 + 30 * k:630 + 30 * k], list(range(30))), (b, np.full(30, t), list(range(30)))])[0] for k in range(2)]
            got.append(np.stack(rows))
            m.seq_free(a)
            m.seq_free(b)
    finally:
        m.close()
    assert np.isnan(got[0][:, 30:]).all() and np.isfinite(got[1]).all() and (got[0][:, :30] == got[1][:, :30]).all()
