"""GPU: steps of one row (kernels_layered_step.hip: norms, router and the merging of attention shares inside the products behind them) against the launches
they stand for.  Every sum is made in the same order, so the logits are the same bits."""
import numpy as np
import pytest

from tests import gizezen_util as GZ

pytestmark = pytest.mark.gpu


# every width; router logits of less and more than one batch of a wave's requests, up to a wave's lanes; inner sizes below and above one piece of 512 and no
# multiple of it, the expert of every token narrower, wider and absent; attention rows of 512, 1024 and 2048 from no, few and more shares than one batch, and of a
# width, of a number of shares or with queries in two tiles that the merging launch keeps (1950 tokens: eight shares of 2048, the most)
@pytest.mark.parametrize("width,heads,kv_heads,dim,window,experts,top,ff,shared", [
    (512, 8, 2, 64, 4096, 5, 2, 136, 72), (1024, 8, 2, 128, 1024, 14, 4, 776, 512), (2048, 8, 8, 64, 700, 64, 6, 64, 0), (4096, 16, 4, 64, 300, 63, 1, 72, 1032),
    (512, 4, 2, 48, 900, 20, 3, 520, 520), (512, 32, 1, 64, 4096, 5, 2, 136, 72), (1024, 16, 4, 64, 4096, 8, 2, 136, 72), (1024, 16, 4, 128, 4096, 8, 2, 136, 72),
    (512, 32, 8, 128, 4096, 5, 2, 136, 72)])
@pytest.mark.parametrize("context", [3, 300, 1950, 2900])
def test_against_single_launches(tmp_path, width, heads, kv_heads, dim, window, experts, top, ff, shared, context):
    from crane_amd.backend import Model
    mixer = dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, conv=4, size=window, rot_dims=dim)
    cfg = GZ.config([GZ.layer(GZ.attn(**mixer), GZ.moe(experts=experts, top=top, ff=ff, shared=shared)),
                     GZ.layer(GZ.attn(**mixer, kv_from=0), None),
                     GZ.layer(GZ.attn(**mixer), GZ.moe(experts=experts, top=top, ff=ff, shared=shared))], vocab=96, width=width)
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, GZ.random_weights(cfg, 3)), compute_dtype="bfloat16", max_seqs=4, max_seq_len=3072)
    toks = GZ.tokens(context + 3, cfg["vocab"], 4)
    out = []
    try:
        s = m.seq_alloc()
        m.step_batch([(s, toks[:context], [])], want_logits=False)
        for on in (1, 0):
            m.debug_set("lay_fused_prep", on)
            f = m.seq_fork(s)
            out.append(np.stack([m.step_batch([(f, toks[context + i:context + i + 1], None)])[0] for i in range(3)]))
            m.seq_free(f)
    finally:
        m.close()
    assert np.isfinite(out[0]).all() and (out[0] == out[1]).all()


def _bits(tmp_path, cfg, P, context, steps=4, **kw):
    """Logits of `steps` single rows behind `context` tokens: in the launches of this file's subject, then in single ones."""
    from crane_amd.backend import Model
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=4, max_seq_len=768, **kw)
    toks = GZ.tokens(context + steps, cfg["vocab"], 4)
    out = []
    try:
        s = m.seq_alloc()
        m.step_batch([(s, toks[:context], [])], want_logits=False)
        for on in (1, 0):
            m.debug_set("lay_fused_prep", on)
            f = m.seq_fork(s)
            out.append(np.stack([m.step_batch([(f, toks[context + i:context + i + 1], None)])[0] for i in range(steps)]))
            m.seq_free(f)
    finally:
        m.close()
    return out


# the row's own convolution, rotation and append: layers on borrowed keys (queries alone are convolved, nothing is appended), one to four taps on either side of a loan, five that the
# single launches keep, rotated parts of no, some and all elements, keys narrower and wider than values with padding behind either, one to four query heads on a key head; steps across a
# tile of 64 keys and a page, in one block and in shares; a page that is no power of two (divisions instead of shifts: the single launches)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps,rot", [
    (4, 2, 64, 96, (1, 4, 2), (0, 32, 64)), (8, 2, 112, 64, (3, 2, 4), (56, 0, 112)), (3, 1, 48, 128, (2, 1, 3), (48, 48, 16)), (6, 6, 128, 16, (4, 3, 1), (128, 64, 0)),
    (8, 2, 80, 80, (4, 5, 4), (80, 8, 80))])
@pytest.mark.parametrize("context,page", [(1, 64), (62, 64), (317, 64), (317, 128), (190, 192)])
def test_rows_on_their_way_into_the_attention(tmp_path, heads, kv_heads, dim, vdim, taps, rot, context, page):
    mk = lambda i, **kw: GZ.layer(GZ.attn(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, conv=taps[i], size=4096 if i < 2 else 200, rot_dims=rot[i], **kw),
                                  GZ.moe(experts=5, top=2, ff=136, shared=72))
    cfg = GZ.config([mk(0), mk(1, kv_from=0), mk(2), mk(1, kv_from=2)], vocab=96, width=512)
    a, b = _bits(tmp_path, cfg, GZ.random_weights(cfg, 5), context, kv_block_size=page)
    assert np.isfinite(a).all() and (a == b).all()


# the choice that every block makes for itself against the one whose weights are written: equal logits (the lower output first), and scores that are no numbers
@pytest.mark.parametrize("kind", ["equal", "pairs", "nan"])
@pytest.mark.parametrize("experts,top,shared", [(6, 2, 72), (14, 4, 0), (63, 5, 72)])
def test_choices_of_equal_scores_and_of_none(tmp_path, kind, experts, top, shared):
    cfg = GZ.config([GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=64, vdim=64, conv=4, rot_dims=64), GZ.moe(experts=experts, top=top, ff=136, shared=shared)) for _ in range(2)],
                    vocab=96, width=512)
    P = GZ.random_weights(cfg, 6)
    router = P["l0.mlp.router"]
    if kind == "equal":
        router[:] = router[0]
    elif kind == "pairs":
        router[1::2] = router[0:experts - experts % 2:2]
    else:
        router[experts // 2] = np.nan
    a, b = _bits(tmp_path, cfg, P, 40)
    assert np.isfinite(a).all() != (kind == "nan")
    np.testing.assert_array_equal(a, b)
