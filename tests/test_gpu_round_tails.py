"""GPU: what a decode group's attention and reductions leave for the next projection (planes or codes of the rows, written by the launches that make
the rows), over numbers of sequences, splits of the tokens and row widths at which another launch writes them."""
import numpy as np
import pytest

from crane_amd import configs

pytestmark = pytest.mark.gpu


def _logits(m, rows, ctx, switch):
    rng = np.random.default_rng(rows + ctx)
    seqs = [m.seq_alloc() for _ in range(rows)]
    for s in seqs:
        m.seq_forward(s, rng.integers(0, 512, ctx + s % 3).tolist(), 0)
    toks, out = rng.integers(0, 512, rows).tolist(), []
    for key, value in switch:
        m.debug_set(key, value)
        out.append(np.asarray(m.step_batch_decode(seqs, toks)[0], np.float64))
        for s in seqs:
            m.seq_truncate(s, ctx + s % 3)
    for s in seqs:
        m.seq_free(s)
    return out


# codes: against the batched integer GEMVs, which quantise the same f32 rows themselves.  One layer of random weights: codes that land on the other side
# of a boundary (the two sides' f32 sums differ in order) move an output by 1 / 127 of a block's largest value; 2e-2 as the rounds of the row kernels.
# H 4096: the widest row of one chunk per thread, 4352: the loop above it; 1280: a part of the workgroup
@pytest.mark.parametrize("H", [1280, 4096, 4352])
@pytest.mark.parametrize("rows,ctx", [(8, 9), (20, 70), (65, 20)])
def test_codes(H, rows, ctx):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), hidden_size=H, intermediate_size=2816, num_attention_heads=8, num_key_value_heads=2, head_dim=128,
               vocab_size=512, num_hidden_layers=2)
    m = Model.synthetic(cfg, seed=3, max_seq_len=128, isq="q8_0", max_seqs=66)
    try:
        a, b = _logits(m, rows, ctx, [("q_gemm_min", 8), ("q_gemm_min", 0)])
        assert np.isfinite(a).all() and np.abs(a - b).max() < 2e-2 * np.abs(b).max()
    finally:
        m.close()


# planes: against single sequences (f32 rows throughout).  bf16 weights, hi + lo planes: 2^-17 of a row per product, two layers, f32 sums in another
# order; a K or V element on the other side of its 16-bit boundary is 2^-9 off, one in a thousand: 2e-3 as the products of such groups
@pytest.mark.parametrize("model", ["qwen3-0.6b", "qwen3.5-0.8b"])
@pytest.mark.parametrize("rows,ctx", [(9, 9), (33, 70)])
def test_planes(model, rows, ctx):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config(model), vocab_size=512, num_hidden_layers=4)
    m = Model.synthetic(cfg, seed=3, max_seq_len=128, max_seqs=rows + 2)
    rng = np.random.default_rng(rows)
    try:
        seqs = [m.seq_alloc() for _ in range(rows)]
        for s in seqs:
            m.seq_forward(s, rng.integers(0, 512, ctx + s % 3).tolist(), 0)
        toks = rng.integers(0, 512, rows).tolist()
        want = []
        for s, t in zip(seqs, toks):
            f = m.seq_fork(s)
            want.append(np.asarray(m.seq_forward(f, [t], m.seq_len(f))[0], np.float64).reshape(-1))
            m.seq_free(f)
        got = np.asarray(m.step_batch_decode(seqs, toks)[0], np.float64).reshape(rows, -1)
        want = np.stack(want)
        assert np.isfinite(got).all() and np.abs(got - want).max() < 2e-3 * np.abs(want).max()
    finally:
        m.close()


# groups that do not fill the chip, contexts below the matrix-core kernel's 768 tokens: queries, weights and their products in f32 like a single
# sequence's (the matrix cores take f16 hi + lo pairs, 22 bits at most) -- the logits are those with that kernel switched off, bit for bit
@pytest.mark.parametrize("rows,ctx", [(3, 700), (9, 300), (33, 70)])
def test_short_contexts_keep_32_bit_queries_and_weights(rows, ctx):
    from crane_amd.backend import Model
    m = Model.synthetic(dict(configs.get_config("qwen3-0.6b"), vocab_size=512, num_hidden_layers=2), seed=3, max_seq_len=768, max_seqs=rows + 1)
    try:
        a, b = _logits(m, rows, ctx, [("attn_mfma_min", 768), ("attn_mfma_min", 0)])
        assert np.isfinite(a).all() and (a == b).all()
    finally:
        m.close()


# a sequence whose rows are NaN or infinite keeps them to itself: the others of the group have the same bits as beside a sound one (products, the
# reductions, norms and quantisers behind them, attention and its combine; rows that fill 32- and 64-row tiles in part)
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("isq", [None, "q8_0"])
@pytest.mark.parametrize("rows,ctx", [(9, 9), (20, 70), (40, 70), (66, 20)])
def test_rows_that_are_no_numbers(tmp_path, bad, isq, rows, ctx):
    import json
    import os

    from crane_amd import synth
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), vocab_size=512, num_hidden_layers=2, tie_word_embeddings=False)
    w = synth.synth_weights_f32(cfg, seed=3)
    w["model.embed_tokens.weight"][5] = bad
    path = str(tmp_path / "ckpt")
    os.makedirs(path)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    synth.write_safetensors_bf16(os.path.join(path, "model.safetensors"), [(k, v.shape, synth.f32_to_bf16_bits(v)) for k, v in w.items()])
    m = Model.from_pretrained(path, max_seq_len=128, max_seqs=rows + 1, **({"isq": isq} if isq else {}))
    try:
        seqs = [m.seq_alloc() for _ in range(rows)]
        for i, s in enumerate(seqs):
            m.seq_forward(s, (6 + (np.arange(ctx + i % 3) + i) % 500).tolist(), 0)
        toks, got = (6 + np.arange(rows) % 500).tolist(), []
        for t in (5, 6):
            got.append(np.asarray(m.step_batch_decode(seqs, toks[:-1] + [t])[0], np.float32).reshape(rows, -1))
            for i, s in enumerate(seqs):
                m.seq_truncate(s, ctx + i % 3)
    finally:
        m.close()
    assert not np.isfinite(got[0][-1]).any() and np.isfinite(got[1]).all() and (got[0][:-1] == got[1][:-1]).all()
