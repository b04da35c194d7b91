"""GPU: the tile kernel of the experts' products (kernels_layered_gemm.hip) against the plain kernels on the same rounded operands, at the
edges of its tiles.

One layer, bfloat16 format, the same step with the tile kernels on and off.  Both round the experts' inputs and inner rows to bfloat16 and
add up the exact products in f32, in another order: a sum of K = 128 .. 320 terms moves by about 1e-6 of itself, an inner row's element lands
on the other side of a rounding boundary with probability 1e-6 / 2^-8 and is then 2^-8 off -- 3e-5 in the mean square, and the same once more
in the head's input.  1e-3 of the largest logit is over ten times that; the router reads the same rows on both sides, so the choices agree."""
import numpy as np
import pytest

from oracle import gizezen_oracle as O
from tests import gibipel_util as GI
from tests import gizezen_util as GZ
from tests import korupel_util as KO
from tests import nevotar_util as NE

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _check(tmp_path, U, cfg, n, seed):
    from crane_amd.backend import Model
    m = Model.from_pretrained(U.write_checkpoint(str(tmp_path / "ckpt"), cfg, U.random_weights(cfg, seed)), compute_dtype="bfloat16", max_seqs=4,
                              max_seq_len=2560, prefill_chunk=2560)
    toks = U.tokens(n, cfg["vocab"], seed + 1)
    want = [i for i in range(n) if i % 8 == 0 or i >= n - 66]
    got = []
    try:
        for on in (1, 0):
            m.debug_set("lay_shared_gemm", on)
            s = m.seq_alloc()
            got.append(m.step_batch([(s, toks, want)])[0].astype(np.float64))
            m.seq_free(s)
    finally:
        m.close()
    assert np.isfinite(got[0]).all() and np.abs(got[0] - got[1]).max() < TOL * np.abs(got[1]).max()


# one row more than the row kernel takes, groups of no or one row, ragged last tiles, output columns that end inside a tile, inner sizes of
# the smallest and of odd numbers of k-tiles, the most groups the kernel numbers and one more (which the plain kernel keeps)
@pytest.mark.parametrize("n", [9, 65, 200])
@pytest.mark.parametrize("width,ff,shared,experts,top", [(128, 128, 128, 6, 2), (192, 320, 192, 4, 4), (320, 192, 0, 64, 3), (128, 192, 320, 65, 2)])
def test_softmax_routed_experts_and_a_shared_one(tmp_path, n, width, ff, shared, experts, top):
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=experts, top=top, ff=ff, shared=shared))], vocab=96, width=width)
    _check(tmp_path, GZ, cfg, n, 3)


# the expert of every token in the routed ones' launches: deeper, wider and narrower than they are
@pytest.mark.parametrize("ff,shared", [(128, 320), (320, 128)])
def test_a_shared_expert_of_another_size(tmp_path, ff, shared):
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=5, top=2, ff=ff, shared=shared))], vocab=96, width=192)
    _check(tmp_path, GZ, cfg, 137, 9)


# 128 x 128 tiles: enough rows and columns for 320 of them
def test_wide_tiles(tmp_path):
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=8, top=4, ff=576, shared=192))], vocab=96, width=1216)
    _check(tmp_path, GZ, cfg, 2500, 5)


def test_weights_on_the_experts_inputs_and_the_capped_product(tmp_path):
    cfg = NE.config([NE.layer("attention", NE.attn(), NE.moe(experts=6, top=3, ff=192, shared=128))], vocab=96, width=192)
    for n in (9, 150):
        _check(tmp_path, NE, cfg, n, 7)


def test_identity_experts(tmp_path):
    cfg = GI.config([GI.layer(GI.left(), GI.right(), GI.moe(experts=5, top=2, ff=128, identity=3, groups=2, keep=1, shared=192))], vocab=96, width=128)
    for n in (9, 150):
        _check(tmp_path, GI, cfg, n, 9)


def test_sigmoid_routed_experts_without_a_shared_one(tmp_path):
    cfg = KO.config([KO.layer("attention", KO.moe(experts=5, top=2, ff=192), **KO.attn())], vocab=96, width=192)
    for n in (33, 150):
        _check(tmp_path, KO, cfg, n, 11)


# the router's row kernel against the oracle in the float32 format: logits below, at and above its register sizes (16, 20, 32; more stay on the
# block-per-token form), one and two tokens per wave, a last wave with one of two
# (up to 8 rows: logits, choice and plan in one block, the expert of every token beside the groups)
@pytest.mark.parametrize("experts,shared", [(3, 28), (16, 0), (16, 28), (20, 28), (32, 0), (32, 28), (70, 12)])
@pytest.mark.parametrize("n", [1, 3, 8, 9, 1025])
def test_router_rows(tmp_path, experts, shared, n):
    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=experts, top=3, ff=24, shared=shared))], vocab=61, width=72)
    P = GZ.random_weights(cfg, 13)
    toks = GZ.tokens(n, cfg["vocab"], 14)
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="float32", max_seqs=2, max_seq_len=1088)
    try:
        got = m.step_batch([(m.seq_alloc(), toks, list(range(n)))])[0].astype(np.float64)
    finally:
        m.close()
    want = O.forward(cfg, P, toks)
    # float32 sums against float64: 1e-4 of the largest logit, as in the family's own tests; a choice within 1e-6 of a tie may fall the other way
    # for one position in a thousand
    off = np.abs(got - want).max(-1) / np.abs(want).max()
    assert np.quantile(off, 0.998) < 1e-4, (float(off.max()), int(off.argmax()))


# 8 rows, 71 logits of width 256: more products than one CU is given (tests/test_lay_router_plan.py), logits by the streaming row kernel
def test_router_of_eight_rows_on_the_whole_chip(tmp_path):
    from crane_amd import _lib
    from crane_amd.backend import Model
    assert _lib.load().cm_debug_lay_router_plan(8, 256, 70, 3, 1, 0) == 0
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=70, top=3, ff=24, shared=12))], vocab=61, width=256)
    P = GZ.random_weights(cfg, 13)
    toks = GZ.tokens(8, cfg["vocab"], 14)
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="float32", max_seqs=2, max_seq_len=64)
    try:
        got = m.step_batch([(m.seq_alloc(), toks, list(range(8)))])[0].astype(np.float64)
    finally:
        m.close()
    want = O.forward(cfg, P, toks)
    assert np.abs(got - want).max() < 1e-4 * np.abs(want).max()      # float32 sums against float64, as above


# a sequence whose rows are NaN or infinite keeps them to itself: the others of the step have the same bits as beside a sound one (3 rows: the decode
# kernels; 40: tiles, whose padding repeats the last row; portions of 30 rows: prompt attention)
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("seqs,portion", [(3, 1), (40, 1), (3, 30)])
def test_rows_that_are_no_numbers(tmp_path, bad, seqs, portion):
    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=64, vdim=64), GZ.moe(experts=6, top=2, ff=128, shared=128)) for _ in range(2)], vocab=96,
                    width=128)
    P = GZ.random_weights(cfg, 17)
    P["embed"][5] = bad
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=42, max_seq_len=128)
    try:
        got = []
        for t in (5, 6):
            ss = [m.seq_alloc() for _ in range(seqs)]
            for i, s in enumerate(ss):
                m.step_batch([(s, 7 + (np.arange(9 + i % 3) + i) % 80, [])], want_logits=False)
            step = [np.full(portion, t) if i == seqs - 1 else 7 + (np.arange(portion) + 3 * i) % 80 for i in range(seqs)]
            got.append(m.step_batch([(s, x, list(range(portion))) for s, x in zip(ss, step)])[0].reshape(seqs, portion, -1))
            for s in ss:
                m.seq_free(s)
    finally:
        m.close()
    # (the norm's tanh takes infinities to one: their logits are finite)
    assert np.isnan(got[0][-1]).all() == np.isnan(bad) and np.isfinite(got[1]).all() and (got[0][:-1] == got[1][:-1]).all()


# outputs of a number of columns that four does not divide (a gate per head, three heads): rows that are not 16-byte aligned
@pytest.mark.parametrize("n", [33, 130])
def test_columns_that_four_does_not_divide(tmp_path, n):
    cfg = GZ.config([GZ.layer(GZ.attn(heads=3, kv_heads=3), GZ.moe(experts=4, top=2, ff=128, shared=128))], vocab=97, width=128)
    _check(tmp_path, GZ, cfg, n, 11)
