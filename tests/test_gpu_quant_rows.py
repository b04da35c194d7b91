"""GPU: the int8 products of decode groups of up to 64 rows (kernels_quant_rows.hip) at the edges of their tiles and slices."""
import numpy as np
import pytest

from crane_amd import configs

pytestmark = pytest.mark.gpu


def _model(H, I, layers=1, **kw):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=H, intermediate_size=I, num_attention_heads=8, num_key_value_heads=2, head_dim=128,
               vocab_size=512, num_hidden_layers=layers)
    return Model.synthetic(cfg, seed=3, max_seq_len=128, isq="q8_0", **kw)


# K of 10 / 22 / 136 groups of four blocks in slices of one to many groups, widths of 10 .. 272 tiles, rows at the edges of one and two row tiles,
# against the same rows in a group of 128 (gemm_q8_i8_kernel).  Same codes and exact dots; <= 544 f32 additions in another order, each within
# 2^-24 of a partial sum: 544 * 6e-8 = 3.2e-5 of the row's range if nothing averages out
@pytest.mark.parametrize("H,I", [(1280, 2816), (512, 17408)])
def test_rows_of_a_group_against_a_larger_one(H, I):
    m = _model(H, I, max_seqs=2)
    rng = np.random.default_rng(5)
    try:
        for which, K, N in (("qkv0", H, 12 * 128), ("o", 1024, H), ("gate_up", H, 2 * I), ("down", I, H)):
            x = (rng.standard_normal((128, K)) * np.exp(rng.standard_normal((128, 1)))).astype(np.float32)
            want = m.debug_qgemm(0, which, x, N)
            for rows in (1, 8, 31, 32, 33, 63, 64):
                got = m.debug_qgemm(0, which, x[:rows], N)
                e = np.abs(got - want[:rows]).max(axis=1) / np.abs(want[:rows]).max(axis=1)
                assert np.isfinite(got).all() and e.max() < 3.2e-5, (which, rows, e.max())
    finally:
        m.close()


# whole rounds: the unsplit gate|up launch (272 tiles: SiLU and the next projection's codes in its epilogue) and the split ones, against the integer
# GEMVs of single sequences.  One layer; codes that land on the other side of a boundary move an output by 1 / 127 of a block's largest value
@pytest.mark.parametrize("H,I", [(1024, 17408), (1280, 2816)])
@pytest.mark.parametrize("rows", [9, 33, 64])
def test_rounds_against_the_row_kernels(H, I, rows):
    m = _model(H, I, max_seqs=66)
    rng = np.random.default_rng(6)
    try:
        seqs = [m.seq_alloc() for _ in range(rows)]
        for s in seqs:
            m.seq_forward(s, rng.integers(0, 512, 5).tolist(), 0)
        toks = rng.integers(0, 512, rows).tolist()
        out = []
        for least in (8, 0):
            m.debug_set("q_gemm_min", least)
            out.append(np.asarray(m.step_batch_decode(seqs, toks)[0], np.float64))
            for s in seqs:
                m.seq_truncate(s, 5)
        assert np.isfinite(out[0]).all() and np.abs(out[0] - out[1]).max() < 2e-2 * np.abs(out[1]).max()
    finally:
        m.close()
