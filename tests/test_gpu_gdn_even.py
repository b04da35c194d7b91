"""GPU: prompts and portions of an even number of tokens through the Gated-Delta-Net passes -- the convolution's window is then written where it is read --
against the same tokens with the last of each alone.

All f32, the last token's sums in another order (the fused kernel instead of the chunk-parallel or the sequential scan): 1e-4 of the largest logit, the bar of the
prompt passes against the oracle.  A window that is stale or mixed up moves the next token's channels by their own size."""
import numpy as np
import pytest

from crane_amd import configs


# around the smallest number of rows that the passes take, the chunk of 64 and the wider tiles of 512; two even portions, then an odd one, then steps of one token
@pytest.mark.gpu
@pytest.mark.parametrize("values", [16, 32])
def test_even_portions(values):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3.5-0.8b"), vocab_size=512, num_hidden_layers=4, linear_num_value_heads=values)
    m = Model.synthetic(cfg, seed=6, max_seq_len=1300, max_seqs=2, kv_dtype="f32")
    rng = np.random.default_rng(values)
    try:
        for n, more in ((14, 16), (16, 18), (18, 64), (62, 2), (64, 66), (66, 128), (510, 512), (512, 514)):
            ids = rng.integers(0, 512, n + more + 17 + 2).tolist()
            ends = [n, n + more, n + more + 17, n + more + 18, n + more + 19]
            out = []
            for alone in (False, True):
                s, at, rows = m.seq_alloc(), 0, []
                for end in ends:
                    if alone and end - at > 1:
                        m.seq_forward(s, ids[at:end - 1], at)
                        at = end - 1
                    rows.append(np.asarray(m.seq_forward(s, ids[at:end], at)[0], np.float64))
                    at = end
                m.seq_free(s)
                out.append(np.stack(rows))
            assert np.isfinite(out[0]).all() and np.abs(out[0] - out[1]).max() < 1e-4 * np.abs(out[1]).max(), (n, more)
    finally:
        m.close()


# one plane (prefill_split 1: activations in bfloat16, 2^-9 of each) against two, for the kernels that end a pass: fused under 16 rows, the rows behind a scan up to five
# chunks, the outputs of all chunks.  Four layers of two or three rounded rows in front of products and norms: 1e-2 of the largest logit as measured over models of this
# depth elsewhere, three times that here; planes that are swapped, shifted or stale move the logits by their own size.
@pytest.mark.gpu
def test_one_plane_against_two():
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3.5-0.8b"), vocab_size=512, num_hidden_layers=4)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, 512, n).tolist() for n in (9, 20, 66, 129, 400)]
    out = []
    for split in (0, 1):
        m = Model.synthetic(cfg, seed=6, max_seq_len=512, max_seqs=2, kv_dtype="f32", prefill_split=split)
        try:
            rows = []
            for p in prompts:
                s = m.seq_alloc()
                rows.append(np.asarray(m.seq_forward(s, p, 0)[0], np.float64).reshape(-1))
                m.seq_free(s)
            out.append(np.stack(rows))
        finally:
            m.close()
    assert np.isfinite(out[1]).all() and np.abs(out[0] - out[1]).max() < 3e-2 * np.abs(out[0]).max()


# the rows of a prompt's passes: whole chunks alone in front of fewer than nine rows, 128 rows more than 4096 where those are the last; a chunk that the caller gave; a short sequence
@pytest.mark.parametrize("chunk,most,tokens,passes", [
    (2048, 4224, 2048, [2048]), (2048, 4224, 2049, [2048, 1]), (2048, 4224, 2056, [2048, 8]), (2048, 4224, 2057, [2057]), (2048, 4224, 4096, [4096]), (2048, 4224, 4097, [4096, 1]),
    (2048, 4224, 4104, [4096, 8]), (2048, 4224, 4105, [4105]), (2048, 4224, 4224, [4224]), (2048, 4224, 4225, [4096, 129]), (2048, 4224, 6145, [4096, 2048, 1]), (2048, 4224, 8321, [4096, 4096, 129]),
    (2048, 2048, 4225, [2048, 2048, 129]), (2048, 2048, 2049, [2048, 1]), (512, 512, 1030, [512, 512, 6]), (5000, 5000, 5000, [5000]), (5000, 5000, 5001, [5000, 1]), (2048, 3000, 2056, [2048, 8]),
    (2048, 3000, 3000, [3000]), (1, 1, 3, [1, 1, 1])])
def test_the_passes_of_a_prompt(chunk, most, tokens, passes):
    from crane_amd import _lib
    got, rest = [], tokens
    while rest:
        got.append(_lib.load().cm_debug_prefill_pass(rest, chunk, most))
        assert 1 <= got[-1] <= min(rest, most)
        rest -= got[-1]
    assert got == passes


# a prompt in passes of up to 4096 rows, and 128 more at its end (the chunk left open), against passes of 2048 (the chunk given): one row more than a chunk (alone in either), nine, as many as a pass takes, one
# more; a second prompt behind them and a token behind that; a hybrid decoder and a dense one.  The chunked sums of three Gated-Delta-Net layers and a layer of attention in other orders: the bar of tests/test_gpu_prefill_shares.py
# 8-bit pages: codes of a row that lands on the other side of a boundary move an element by 2^-8 of its row's largest, one in a thousand of them, and so a sum of thousands of keys by far less than 1e-3
@pytest.mark.gpu
@pytest.mark.parametrize("model,layers,dtype,tol", [("qwen3.5-0.8b", 4, "f16", 1e-4), ("qwen3-0.6b", 1, "f16", 1e-4), ("qwen3-0.6b", 1, "int8", 1e-3)])
def test_long_passes(model, layers, dtype, tol):
    from crane_amd import _lib
    from crane_amd.backend import Model
    cfg = dict(configs.get_config(model), vocab_size=512, num_hidden_layers=layers)
    ids = np.random.default_rng(5).integers(0, 512, 4400).tolist()
    out = []
    for chunk in (0, 2048):
        m = Model.synthetic(cfg, seed=3, max_seq_len=4608, max_seqs=3, prefill_chunk=chunk, kv_dtype=dtype)
        try:
            got = []
            for n in (2049, 2057, 4096, 4224, 4225):
                s = m.seq_alloc()
                got.append(np.asarray(m.seq_forward(s, ids[:n], 0)[0], np.float64).ravel())
                got.append(np.asarray(m.seq_forward(s, ids[n:n + 130], n)[0], np.float64).ravel())
                got.append(np.asarray(m.seq_forward(s, [7], n + 130)[0], np.float64).ravel())
                m.seq_free(s)
            assert m.debug_read("prefill_rows", 2).tolist() == [2048, 2048 if chunk else 4224]
            with pytest.raises(_lib.CraneError):                       # several prompts in a pass: still the chunk
                m.prefill_batch([m.seq_alloc(), m.seq_alloc()], [ids[:2048], ids[:1]])
            out.append(got)
        finally:
            m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.abs(a - b).max() < tol * np.abs(b).max()
