"""GPU: prompt attention (kernels_attn_prompt.hip): many query tiles against the same prompt in portions, whose launches are small enough for attn_prefill_fast_kernel, and several
prompts in one pass against each by itself.

One layer: the cached rows and the weights are the same, and so is the order of every sum of the attention; the products around it add up in other tiles (1e-7 of a row), attention rows
travel as bfloat16 hi + lo planes, 2^-17 of an element where the two land on both sides of a boundary: 2e-5 of the largest logit, as in tests/test_gpu_prefill_shares.py."""
import numpy as np
import pytest

from crane_amd import _lib, configs

TOL = 2e-5


def _model(heads, kv, chunk, page=64, dtype="f16", seqs=2):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3-0.6b"), vocab_size=512, num_hidden_layers=1, hidden_size=512, intermediate_size=1024, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128)
    return Model.synthetic(cfg, seed=3, max_seq_len=2304, max_seqs=seqs, prefill_chunk=chunk, kv_block_size=page, kv_dtype=dtype)


def _last(m, ids):
    s = m.seq_alloc()
    row = np.asarray(m.seq_forward(s, ids, 0)[0], np.float64).ravel()
    m.seq_free(s)
    return row


# whole query tiles, one of one row behind them, a ragged one; two, four and eight query heads per key head; pages of one tile and of two; both page types; a second pass behind 1152 rows
CASES = [(32, 8, 64, "f16", (1345, 1408, 2048, 2300)), (32, 16, 128, "bf16", (1407, 1500)), (32, 4, 128, "f16", (1409,)), (40, 20, 64, "bf16", (1025, 1088))]


def test_the_cases_reach_the_kernel():
    pairs = _lib.load().cm_debug_attn_prompt_pairs
    assert all(pairs(min(n, 2048), 0, heads, kv) for heads, kv, _, _, tokens in CASES for n in tokens) and pairs(1148, 1152, 32, 8)
    assert not any(pairs(n, 0, heads, kv) for heads, kv, chunk in ((32, 8, 512), (32, 16, 512), (32, 4, 512), (40, 20, 384)) for n in range(1, chunk + 1))


# both sides of the line (figures beside the rule): prompts from their start, behind cached tokens, an odd number of query heads per key head
@pytest.mark.parametrize("rows,start,heads,kv,want", [(2048, 0, 16, 8, 0), (2688, 0, 16, 8, 0), (2816, 0, 16, 8, 1), (1344, 0, 32, 8, 0), (1408, 0, 32, 8, 1), (1792, 0, 24, 4, 0), (1920, 0, 24, 4, 1),
                                                      (4224, 0, 8, 4, 0), (2048, 2048, 16, 8, 0), (2240, 2048, 16, 8, 1), (1088, 2048, 32, 8, 1), (2048, 0, 32, 32, 0), (2048, 2048, 24, 8, 0)])
def test_the_faster_kernel(rows, start, heads, kv, want):
    assert _lib.load().cm_debug_attn_prompt_pairs(rows, start, heads, kv) == want


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,page,dtype,tokens", CASES)
def test_against_portions(heads, kv, page, dtype, tokens):
    ids = np.random.default_rng(heads + kv).integers(0, 512, 2300).tolist()
    rows = []
    for chunk in (2048, 1152, 512) if 2300 in tokens else (2048, 512 if heads == 32 else 384):
        m = _model(heads, kv, chunk, page, dtype)
        try:
            rows.append([_last(m, ids[:n]) for n in tokens])
        finally:
            m.close()
    for got in rows[:-1]:
        for a, b in zip(got, rows[-1]):
            assert np.isfinite(a).all() and np.abs(a - b).max() < TOL * np.abs(b).max()


# several sequences in one launch: tiles of every length, sequences of one row and of a tile and one; few rows, whose projection is split and added up by the rotation
@pytest.mark.gpu
@pytest.mark.parametrize("lengths", [(1, 65, 700, 64, 310, 900), (3, 40, 17, 60), (9, 1), (150, 120, 30)])
def test_several_prompts(lengths):
    rng = np.random.default_rng(1)
    prompts = [rng.integers(0, 512, n).tolist() for n in lengths]
    m = _model(32, 8, 2048, seqs=8)
    try:
        alone = [_last(m, p) for p in prompts]
        seqs = [m.seq_alloc() for _ in prompts]
        together = np.asarray(m.prefill_batch(seqs, prompts)[0], np.float64)
    finally:
        m.close()
    for a, b in zip(together, alone):
        assert np.isfinite(a).all() and np.abs(a.ravel() - b).max() < TOL * np.abs(b).max()


# head_dim 256 with an output gate (attn_prompt_wide_kernel) against the general kernel, which pages of 32 tokens take: last rows at both ends of a tile's halves and of the query groups, several
# sequences in a launch; a second pass whose keys are shared (37 and 200 rows behind 320 and 1024: shares of one tile, and of none, to eight).  The same rows and cache as above: 2e-5.
@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dtype", [(8, 2, "f16"), (4, 4, "bf16"), (16, 4, "f16")])
def test_wide_heads(heads, kv, dtype):
    from crane_amd.backend import Model
    cfg = dict(configs.get_config("qwen3.5-0.8b"), vocab_size=512, num_hidden_layers=1, full_attention_interval=1, num_attention_heads=heads, num_key_value_heads=kv)
    cfg.pop("layer_types", None)
    rng = np.random.default_rng(heads)
    prompts = [rng.integers(0, 512, n).tolist() for n in (1, 16, 31, 32, 33, 63, 64, 65, 97, 128, 193)]
    long = rng.integers(0, 512, 1224).tolist()
    rows = []
    for page in (64, 128, 32):
        got = []
        for chunk in (1024, 320):
            m = Model.synthetic(cfg, seed=3, max_seq_len=1280, max_seqs=16, prefill_chunk=chunk, kv_block_size=page, kv_dtype=dtype)
            try:
                got += [_last(m, long[:n]) for n in (357, 640, 1224)]
                if chunk == 1024:
                    got += [r.ravel() for r in np.asarray(m.prefill_batch([m.seq_alloc() for _ in prompts], prompts)[0], np.float64)]
            finally:
                m.close()
        rows.append(got)
    for a, b, c in zip(*rows):
        assert np.isfinite(a).all() and np.abs(a - c).max() < TOL * np.abs(c).max() and np.abs(b - c).max() < TOL * np.abs(c).max()
