"""GPU: the attention of decode groups over 16-bit pages (kernels_attn_group.hip) against the vector kernel, which holds everything in f32, at the edges of
its tiles, shares and pages."""
import numpy as np
import pytest

from crane_amd import configs

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 62, 63, 64, 65, 127, 128, 129, 191, 254, 255, 256, 257, 319, 448, 511, 512, 513, 640, 700, 767, 768, 769, 1023, 1100]


# One layer: both sides append the same rows and read them with queries and weights of 24 bits or more, in another order (2e-7 of a row).  The rows go on
# as bfloat16 hi + lo planes, 2^-17 of an element where the two land on both sides of a rounding boundary; so do the products' inputs behind
# them: 1e-5 of a row at most, twice that here.
@pytest.mark.parametrize("kv", ["f16", "bf16"])
@pytest.mark.parametrize("heads,kv_heads,page,count", [(8, 2, 64, 26), (8, 2, 128, 26), (8, 4, 64, 13), (16, 16, 64, 13), (8, 8, 256, 7), (32, 8, 64, 26)])
def test_against_the_vector_kernel(kv, heads, kv_heads, page, count):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=512, intermediate_size=1024, num_attention_heads=heads, num_key_value_heads=kv_heads,
               head_dim=128, vocab_size=512, num_hidden_layers=1)
    m = Model.synthetic(cfg, seed=5, max_seq_len=1280, max_seqs=32, kv_block_size=page, kv_dtype=kv)
    rng = np.random.default_rng(heads + page)
    lengths = [LENGTHS[i * len(LENGTHS) // count] for i in range(count - 1)] + [LENGTHS[-1]]
    out = []
    try:
        m.debug_set("attn_mfma_min", 1 << 40)
        seqs = [m.seq_alloc() for _ in lengths]
        for s, n in zip(seqs, lengths):
            m.seq_forward(s, rng.integers(0, 512, n).tolist(), 0, want_logits=False)
        toks = [rng.integers(0, 512, count).tolist() for _ in range(2)]
        for on in (1, 0):
            m.debug_set("attn_group", on)
            out.append([np.asarray(m.step_batch_decode(seqs, t)[0], np.float64).reshape(count, -1) for t in toks])
            for s, n in zip(seqs, lengths):
                m.seq_truncate(s, n)
    finally:
        m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert (np.abs(a - b).max(axis=1) < 2e-5 * np.abs(b).max(axis=1)).all()
