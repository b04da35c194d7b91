"""Prompt rows in two launches where their last round of tiles would be nearly empty (crane_amd/csrc/kernels_prefill.hip: gemm_band): the rule on the host, and
on the GPU the same prompt with cm_debug_set("gemm256") 1 (bands where the rule has them) and 3 (one launch).

The tolerance is that of tests/test_gpu_gemm_prompts.py with K <= 12288: a sum whose slices of K are added in another order moves by about sqrt(K) 2^-24 of
its size, 7e-6, and a bf16 K or V element rounds to the other side with probability 7e-6 / 2^-8; 2e-3 of the largest logit is ten times what two layers make of
that, and rows that are lost or misplaced move the logits by their own size."""
import numpy as np
import pytest

from crane_amd import _lib

WS = 1 << 24
TOL = 2e-3
STORE, ADD, SILU, ACT = 0, 1, 2, 3


def band(m, n, k, epi, ws=WS):
    return _lib.load().cm_debug_gemm_band(m, n, k, epi, ws)


# the figures beside the rule; at most 256 rows, an activation behind the product, products too small to gain
@pytest.mark.parametrize("m,n,k,epi,rows", [(645, 24576, 4096, SILU, 512), (768, 24576, 4096, SILU, 512), (300, 24576, 4096, SILU, 0), (1040, 4096, 12288, ADD, 1024), (1400, 4096, 12288, ADD, 384),
                                            (1400, 6144, 4096, STORE, 0), (1290, 12288, 2048, SILU, 1280), (650, 12288, 2048, SILU, 0), (2060, 8320, 2048, STORE, 2048),
                                            (2048, 24576, 4096, SILU, 0), (2048, 4096, 12288, ADD, 0), (256, 24576, 4096, SILU, 0), (1400, 4096, 4096, ACT, 0), (300, 6144, 1024, SILU, 0)])
def test_the_first_band(m, n, k, epi, rows):
    assert band(m, n, k, epi) == rows


# whole tiles in front, at least the nine rows behind that the smallest kernel takes; nothing without a workspace that a band could not have
@pytest.mark.parametrize("n,k,epi", [(24576, 4096, SILU), (4096, 12288, ADD), (6144, 4096, STORE), (8320, 2048, STORE), (2048, 2048, ADD)])
def test_every_band_is_a_band(n, k, epi):
    for m in range(1, 4097, 7):
        for ws in (0, WS):
            rows = band(m, n, k, epi, ws)
            assert rows == 0 or (rows % 128 == 0 and 128 <= rows <= m - 9)


# prompts that are one pass each; every one of them has a product in two launches, and together they reach bands of all three epilogues from 128 to 2048 rows, of 9 rows behind and of hundreds,
# the norm behind o and down, columns behind the last 256 (8320, 16512)
CASES = [("qwen3-8b", 2, (521, 574, 645, 768, 1030, 1033, 1100, 1152, 1289, 1350, 1407, 1545)), ("qwen3.5-2b", 4, (1033, 1101, 1281, 1289, 1664, 2053, 2060, 2176, 2200, 2304)),
         ("qwen3.8-27b", 2, (280, 700, 1420))]


def products(name, layers):
    from crane_amd import configs
    c = configs.get_config(name)
    h, i, d, hq, kv = (c[x] for x in ("hidden_size", "intermediate_size", "head_dim", "num_attention_heads", "num_key_value_heads"))
    out = [("gate_up", 2 * i, h, SILU), ("down", h, i, ADD)]
    every = c.get("full_attention_interval", 1)
    if layers >= every:
        out += [("qkv", ((2 if every > 1 else 1) * hq + 2 * kv) * d, h, STORE), ("o", h, hq * d, ADD)]
    if every > 1:
        keys, values = c["linear_num_key_heads"] * 128, c["linear_num_value_heads"] * 128
        out += [("in", -(-(2 * keys + 2 * values + 2 * c["linear_num_value_heads"]) // 128) * 128, h, STORE), ("out", h, values, ADD)]
    return out


def test_the_cases_reach_bands():
    seen = set()
    for name, layers, tokens in CASES:
        for m in tokens:
            bands = {(epi, rows) for _, n, k, epi in products(name, layers) if (rows := band(m, n, k, epi))}
            assert bands, (name, m)
            seen |= bands | {(epi, m - rows < 32) for epi, rows in bands} | {"tail" for p, n, k, epi in products(name, layers) if n % 256 == 128 and band(m, n, k, epi)}
    assert {rows for x in seen if x != "tail" for rows in x[1:]} >= {128, 256, 384, 512, 640, 896, 1024, 1280, 1536, 1792, 2048}
    assert seen >= {(epi, few) for epi in (STORE, ADD, SILU) for few in (False, True)} | {"tail"}


@pytest.mark.gpu
@pytest.mark.parametrize("name,layers,tokens", CASES)
def test_bands_against_one_launch(name, layers, tokens):
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = dict(configs.get_config(name), vocab_size=512, num_hidden_layers=layers)
    if "layer_types" in cfg:
        cfg["layer_types"] = cfg["layer_types"][:layers]
    m = Model.synthetic(cfg, seed=3, max_seq_len=2304, max_seqs=2)
    rng = np.random.default_rng(5)
    try:
        for n in tokens:
            ids = rng.integers(0, 512, n).tolist()
            rows = []
            for mode in (1, 3):
                m.debug_set("gemm256", mode)
                s = m.seq_alloc()
                rows.append(np.asarray(m.seq_forward(s, ids, 0)[0], np.float64))
                m.seq_free(s)
            assert np.isfinite(rows[0]).all() and np.abs(rows[0] - rows[1]).max() < TOL * np.abs(rows[1]).max(), n
    finally:
        m.close()
