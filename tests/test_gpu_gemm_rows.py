"""GPU: the products of 9 .. 128 rows (kernels_gemm_rows.hip) against the kernels they replace, at the edges of its tiles and of its rule.

The same step with cm_debug_set("gemm256") 1 (automatic) and 3 (the old kernels).  Both multiply bf16 hi + lo activations by bf16 weights and add
the products up in f32, in another order: a sum of K = 128 .. 2048 terms moves by about sqrt(K) 2^-24 of its size, 3e-6, and a K or V element lands
on the other side of a bf16 boundary with probability 3e-6 / 2^-8, one in a thousand -- each is then 2^-8 off, 1e-4 in the mean square over a
row.  Two layers of four products and the head: 2e-3 of the largest logit is ten times that, and a tile, a row or a slice that is lost or doubled
moves the logits by their own size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-3


def _model(H, I, heads, kv, vocab, **kw):
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=H, intermediate_size=I, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
               vocab_size=vocab, num_hidden_layers=2)
    return Model.synthetic(cfg, seed=3, max_seq_len=256, **kw)


def _close(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    assert np.isfinite(got).all() and np.abs(got - want).max() < TOL * np.abs(want).max()


# prompts: rows below, at and above each tile height; K of an odd number of k-tiles (320 = 5), widths that split K 2, 4 and 8 ways, widths of more
# than 256 column tiles that fill their last round (I 62208: 972 of 1024) and that do not (I 17408: 272 of 512)
# rows of 1280 and 5120 columns: reductions with their norm in a part of a 1024-thread workgroup and in a loop of one;
# (1024, 3072): qkv and gate_up of 6144 columns, 96 per workgroup; (128, 49152): 1024 workgroups of 96
@pytest.mark.parametrize("H,I,heads,kv", [(640, 320, 4, 2), (1024, 2048, 8, 8), (384, 17408, 6, 2), (128, 62208, 2, 1), (1024, 3072, 24, 12), (128, 49152, 2, 1), (1280, 2048, 8, 2), (5120, 1024, 8, 2)])
def test_prompts(H, I, heads, kv):
    m = _model(H, I, heads, kv, 512, max_seqs=2)
    rng = np.random.default_rng(1)
    try:
        for n in (8, 9, 15, 17, 32, 33, 63, 64, 65, 127, 128, 129):
            ids = rng.integers(0, 512, n).tolist()
            rows = []
            for mode in (1, 3):
                m.debug_set("gemm256", mode)
                s = m.seq_alloc()
                rows.append(m.seq_forward(s, ids, 0)[0])
                m.seq_free(s)
            _close(rows[0], rows[1])
    finally:
        m.close()


# decode groups, with the head: 500 column tiles (its last round 98 % full) and 300 (59 %: stays with the old kernel)
@pytest.mark.parametrize("vocab", [64000, 38400])
def test_decode_groups_and_their_head(vocab):
    m = _model(640, 1600, 8, 2, vocab, max_seqs=130)
    rng = np.random.default_rng(2)
    try:
        seqs = [m.seq_alloc() for _ in range(128)]
        for s in seqs:
            m.seq_forward(s, rng.integers(0, vocab, 5).tolist(), 0)
        for n in (9, 32, 33, 64, 65, 128):
            toks = rng.integers(0, vocab, n).tolist()
            got = []
            for mode in (1, 3):
                m.debug_set("gemm256", mode)
                rows, ids = m.step_batch_decode(seqs[:n], toks)
                assert [int(np.argmax(r)) for r in rows] == list(ids)
                got.append(rows)
                for s in seqs[:n]:
                    m.seq_truncate(s, 5)
            _close(got[0], got[1])
    finally:
        m.close()
