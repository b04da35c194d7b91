"""GPU: the decode attention on the matrix cores (attn_decode_mfma_kernel) against the vector kernel, at the edges of its tiles, shares and pages."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 15, 16, 17, 63, 64, 65, 127, 129, 700, 1100]


# One layer.  Queries and weights are two bfloat16 terms here (2^-17) and f32 there: a score of size ten moves by 8e-5, every weight by as much of itself, and the
# two terms of a weight and of the rows that go on add 2^-17 each: 1e-4 of a row, twice that here.  A tile, a row or a page that is lost or taken twice
# moves a row by a hundredth of itself and more at these lengths.  Pages smaller than a tile, as large, and larger.
@pytest.mark.parametrize("kv", ["f16", "bf16"])
@pytest.mark.parametrize("dim,heads,kv_heads,page", [(256, 8, 2, 64), (256, 8, 2, 8), (256, 8, 1, 16), (256, 6, 2, 64), (256, 2, 2, 128), (128, 8, 2, 64), (128, 8, 4, 8), (128, 8, 1, 16)])
def test_against_the_vector_kernel(kv, dim, heads, kv_heads, page):
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=512, intermediate_size=1024, num_attention_heads=heads, num_key_value_heads=kv_heads,
               head_dim=dim, vocab_size=512, num_hidden_layers=1)
    m = Model.synthetic(cfg, seed=5, max_seq_len=1280, max_seqs=16, kv_block_size=page, kv_dtype=kv)
    rng = np.random.default_rng(heads + page)
    out = []
    try:
        m.debug_set("attn_group", 0)
        seqs = [m.seq_alloc() for _ in LENGTHS]
        for s, n in zip(seqs, LENGTHS):
            m.seq_forward(s, rng.integers(0, 512, n).tolist(), 0, want_logits=False)
        toks = [rng.integers(0, 512, len(LENGTHS)).tolist() for _ in range(2)]
        for least in (1, 1 << 40):
            m.debug_set("attn_mfma_min", least)
            out.append([np.asarray(m.step_batch_decode(seqs, t)[0], np.float64).reshape(len(LENGTHS), -1) for t in toks])
            for s, n in zip(seqs, LENGTHS):
                m.seq_truncate(s, n)
    finally:
        m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and (a != b).any()                     # (another kernel)
        assert (np.abs(a - b).max(axis=1) < 2e-4 * np.abs(b).max(axis=1)).all()
