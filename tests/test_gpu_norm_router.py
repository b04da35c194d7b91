"""GPU: norm, router, choice and the experts' row lists of a pass in one launch (kernels_layered_mix.hip: lay_norm_router_kernel, and its form for prompts from 1024 rows on)
against the single launches, with the convolution tails that ride along: both sides of the line between the two forms, last blocks of one row, numbers of logits at the
edges of their registers (with the shared expert's gate 6, 16, 17 and 32; 33 stay with the single launches), one and several pieces of a row per wave.

The logits of the choice are sums of the same f32 products in another order, 1e-6 of themselves: choices agree but for ties of that size, weights move by as much; the rest is
what tests/test_gpu_layered_experts.py compares, with its tolerance."""
import pytest

from tests import gizezen_util as GZ
from tests.test_gpu_layered_experts import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 130, 1023, 1024, 1033])
@pytest.mark.parametrize("width,experts,top", [(128, 5, 2), (192, 15, 15), (1088, 16, 4), (64, 31, 1), (128, 32, 3)])
def test_one_launch_against_four(tmp_path, n, width, experts, top):
    moe = GZ.moe(experts=experts, top=top, ff=128, shared=128)
    cfg = GZ.config([GZ.layer(GZ.attn(conv=4), moe), GZ.layer(GZ.attn(conv=4, kv_from=0), moe)], vocab=96, width=width)
    _check(tmp_path, GZ, cfg, n, 21)


# portions of a prompt and single tokens of others: the tails of every segment, shorter and longer than the convolution
def test_tails_of_mixed_steps(tmp_path):
    import numpy as np

    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(conv=5), GZ.moe(experts=5, top=2, ff=128, shared=128)) for _ in range(2)], vocab=96, width=128)
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, GZ.random_weights(cfg, 4)), compute_dtype="bfloat16", max_seqs=4, max_seq_len=128)
    toks = [GZ.tokens(40, cfg["vocab"], 30 + k) for k in range(3)]
    got = []
    try:
        for on in (1, 0):
            m.debug_set("lay_shared_gemm", on)
            ss = [m.seq_alloc() for _ in toks]
            at, rows = [0, 0, 0], []
            for cut in ((9, 1, 2), (1, 20, 3), (3, 1, 5), (12, 2, 1)):
                rows.append(m.step_batch([(s, t[a:a + c], None) for s, t, a, c in zip(ss, toks, at, cut)])[0])
                at = [a + c for a, c in zip(at, cut)]
            got.append(np.concatenate(rows).astype(np.float64))
            for s in ss:
                m.seq_free(s)
    finally:
        m.close()
    assert np.isfinite(got[0]).all() and np.abs(got[0] - got[1]).max() < 1e-3 * np.abs(got[1]).max()


# rows that are NaN beside sound ones, in blocks of eight rows as in blocks of one: the sound rows keep the bits that they have beside other sound ones
@pytest.mark.parametrize("n", [130, 1027])
def test_rows_that_are_no_numbers(tmp_path, n):
    import numpy as np

    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=64, vdim=64), GZ.moe(experts=15, top=4, ff=128, shared=128)) for _ in range(2)], vocab=96, width=192)
    P = GZ.random_weights(cfg, 17)
    P["embed"][5] = np.nan
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, P), compute_dtype="bfloat16", max_seqs=4, max_seq_len=1280, prefill_chunk=2560)
    toks, got = 7 + np.array(GZ.tokens(n, 80, 18)), []
    try:
        for t in (5, 6):
            ss = [m.seq_alloc() for _ in range(3)]
            step = [toks[:n - 16], np.full(3, t), toks[:13]]
            got.append(m.step_batch([(s, x, list(range(len(x)))) for s, x in zip(ss, step)])[0])
            for s in ss:
                m.seq_free(s)
    finally:
        m.close()
    bad = slice(n - 16, n - 13)
    assert np.isnan(got[0][bad]).all() and np.isfinite(got[1]).all()
    assert (np.delete(got[0], np.r_[bad], 0) == np.delete(got[1], np.r_[bad], 0)).all()
