"""GPU: prompt attention of few queries behind many keys, whose key tiles several blocks share (attn_prefill_fast_kernel, attn_prefill_merge_kernel), against the
same prompt in one pass, whose query tiles are enough for whole ones."""
import numpy as np
import pytest

from crane_amd import configs

pytestmark = pytest.mark.gpu


# Dense, one layer: the same cached rows, weights and sums in another order (1e-7 of a row), attention rows as bfloat16 hi + lo planes: 2^-17 of an element where
# the two land on both sides of a boundary.  Hybrid: three Gated-Delta-Net layers in front of the attention, whose chunked sums differ in order by 1e-5.
# Rows of the last pass: one, a part of a query tile, whole ones, one more; prefixes that give two shares and sixteen, a last share that ends in the
# diagonal tile, shares without a tile
@pytest.mark.parametrize("model,layers,page,tol", [("qwen3-0.6b", 1, 64, 2e-5), ("qwen3-0.6b", 1, 128, 2e-5), ("qwen3.5-0.8b", 4, 64, 1e-4)])
@pytest.mark.parametrize("prefix", [1024, 2048])
@pytest.mark.parametrize("kv", ["f16", "bf16"])
def test_against_one_pass(model, layers, page, tol, prefix, kv):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config(model), vocab_size=512)
    cfg.update(num_hidden_layers=layers)
    rng = np.random.default_rng(prefix)
    ids = rng.integers(0, 512, prefix + 200).tolist()
    rows = [2, 17, 64, 65, 130, 200]
    out = []
    for chunk in (prefix, prefix + 256):
        m = Model.synthetic(cfg, seed=3, max_seq_len=2560, max_seqs=2, prefill_chunk=chunk, kv_block_size=page, kv_dtype=kv)
        try:
            got = []
            for n in rows:
                s = m.seq_alloc()
                got.append(np.asarray(m.seq_forward(s, ids[:prefix + n], 0)[0], np.float64).ravel())
                m.seq_free(s)
            out.append(got)
        finally:
            m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.abs(a - b).max() < tol * np.abs(b).max()
