"""GPU: the chunk-parallel Gated-Delta-Net pass (the outputs inside the scan over the states for up to five chunks and 32 heads, else of all chunks
at once) against the sequential scan, at the edges of its chunks of 64 tokens, from an empty state and from one that an earlier portion left, with
one, two and three value heads per key head.

Both are f32 throughout and differ in the order of their sums (and in decays as a sum of logarithms): 1e-4 of the largest logit, the bar of the prompt
passes against the oracle."""
import numpy as np
import pytest

from crane_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [16, 32, 48])
def test_against_the_sequential_scan(values):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3.5-0.8b"), vocab_size=512, num_hidden_layers=4)
    assert cfg["linear_num_key_heads"] == 16
    cfg["linear_num_value_heads"] = values
    m = Model.synthetic(cfg, seed=5, max_seq_len=1024, max_seqs=2, kv_dtype="f32")
    rng = np.random.default_rng(values)
    try:
        for n in (64, 65, 127, 128, 129, 200, 320, 321, 512):
            ids, more = rng.integers(0, 512, n).tolist(), rng.integers(0, 512, 64 + n % 63).tolist()
            out = []
            for on in (1, 0):
                m.debug_set("gdn_chunked", on)
                s = m.seq_alloc()
                rows = [m.seq_forward(s, ids, 0)[0], m.seq_forward(s, more, n)[0], m.seq_forward(s, [7], n + len(more))[0]]
                out.append(np.concatenate([np.asarray(r, np.float64).reshape(-1) for r in rows]))
                m.seq_free(s)
            assert np.isfinite(out[0]).all() and np.abs(out[0] - out[1]).max() < 1e-4 * np.abs(out[1]).max(), n
    finally:
        m.close()
