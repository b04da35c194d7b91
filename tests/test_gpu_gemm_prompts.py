"""GPU: the products of long prompts on the LDS-DMA tiles (kernels_gemm_tile.hip) against the 128-column kernel.

The same prompt with cm_debug_set("gemm256") 1 (automatic) and 0.  Where K is not split both add the same products in the same order; where it is, a sum of
K <= 6144 terms moves by about sqrt(K) 2^-24 of its size, 5e-6, and a K or V element lands on the other side of a bf16 boundary with probability 5e-6 / 2^-8, one in
a thousand -- each is then 2^-8 off, 1e-4 in the mean square over a row.  Two layers of four products and the head: 2e-3 of the largest logit is ten
times that, and a tile, a row or a column that is lost or misplaced moves the logits by their own size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-3


# rows of a ragged last tile and of whole ones; columns of 256- and of 192-column tiles only (6528 = 34 x 192); plain, interleaved, split and added outputs; K of an
# odd number of k-tiles (3264 = 51)
@pytest.mark.parametrize("H,I,heads,kv", [(1024, 3072, 24, 12), (1024, 3264, 24, 12), (6144, 1024, 8, 8)])
def test_against_the_128_column_kernel(H, I, heads, kv):
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=H, intermediate_size=I, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
               vocab_size=512, num_hidden_layers=2)
    m = Model.synthetic(cfg, seed=3, max_seq_len=1280, max_seqs=2)
    rng = np.random.default_rng(4)
    try:
        for n in (897, 1030, 1152):
            ids = rng.integers(0, 512, n).tolist()
            rows = []
            for mode in (1, 0):
                m.debug_set("gemm256", mode)
                s = m.seq_alloc()
                rows.append(np.asarray(m.seq_forward(s, ids, 0)[0], np.float64))
                m.seq_free(s)
            assert np.isfinite(rows[0]).all() and np.abs(rows[0] - rows[1]).max() < TOL * np.abs(rows[1]).max()
    finally:
        m.close()
