"""GPU: prompt attention of layer-list decoders whose long walks are shared among blocks (kernels_layered_attn.hip: lay_attn_tile_kernel) against the form without a matrix core, in
passes of few query tiles: walks just below and above the line, portions that end inside a tile, windows that leave some of a walk's shares empty (a layer of a shorter
window beside one of a longer: the lists follow the longer), single tokens beside them, the counters' next use.

Both read the same bfloat16 pages; queries are rounded to bfloat16 here and weights kept in two such parts, tests/test_gpu_gizezen.py's comparison of the two forms and its bound."""
import numpy as np
import pytest

from tests import gizezen_util as GZ

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("start", [300, 383, 384, 1000])
def test_shares_of_a_walk(tmp_path, dim, start):
    from crane_amd.backend import Model
    cfg = GZ.config([GZ.layer(GZ.attn(heads=4, kv_heads=2, dim=dim, vdim=dim, size=size), GZ.moe(experts=4, top=2, ff=128, shared=128)) for size in (1024, 70, 400)],
                    vocab=96, width=256)
    m = Model.from_pretrained(GZ.write_checkpoint(str(tmp_path / "ckpt"), cfg, GZ.random_weights(cfg, 8)), compute_dtype="bfloat16", max_seqs=4, max_seq_len=1280)
    long, short = GZ.tokens(start + 90, cfg["vocab"], 40), GZ.tokens(60, cfg["vocab"], 41)
    got = []
    try:
        for on in (1, 0):
            m.debug_set("lay_attn_mfma", on)
            a, b = m.seq_alloc(), m.seq_alloc()
            m.step_batch([(a, long[:start], []), (b, short[:50], [])], want_logits=False)
            rows = []
            for k in range(3):                  # a portion beside one token, three times
                rows.append(m.step_batch([(a, long[start + 30 * k:start + 30 * k + 30], list(range(30))), (b, short[50 + k:51 + k], None)])[0])
            got.append(np.concatenate(rows).astype(np.float64))
            m.seq_free(a)
            m.seq_free(b)
    finally:
        m.close()
    assert np.isfinite(got[0]).all()
    off = np.abs(got[0] - got[1]).max(-1) / np.abs(got[1]).max()
    # a choice of experts that the queries' rounding tips over moves its row: at most one row in thirty
    assert np.quantile(off, 0.96) < 1e-2, (float(off.max()), int(off.argmax()))
