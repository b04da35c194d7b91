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


# the figures beside the rule; at most 256 rows, an activation behind the product, products too small to gain
@pytest.mark.parametrize("m,n,k,epi,rows", [(300, 24576, 4096, SILU, 256), (1400, 4096, 12288, ADD, 1024), (1400, 6144, 4096, STORE, 1280), (650, 12288, 2048, SILU, 640),
                                            (2048, 24576, 4096, SILU, 0), (2048, 4096, 12288, ADD, 0), (256, 24576, 4096, SILU, 0), (1400, 4096, 4096, ACT, 0), (300, 6144, 1024, SILU, 0)])
def test_the_first_band(m, n, k, epi, rows):
    assert _lib.load().cm_debug_gemm_band(m, n, k, epi, WS) == rows


# whole tiles in front, at least the nine rows behind that the smallest kernel takes; nothing without a workspace that a band could not have
@pytest.mark.parametrize("n,k,epi", [(24576, 4096, SILU), (4096, 12288, ADD), (6144, 4096, STORE), (8320, 2048, STORE), (2048, 2048, ADD)])
def test_every_band_is_a_band(n, k, epi):
    band = _lib.load().cm_debug_gemm_band
    for m in range(1, 4097, 7):
        for ws in (0, WS):
            rows = band(m, n, k, epi, ws)
            assert rows == 0 or (rows % 128 == 0 and 128 <= rows <= m - 9)


# bands of 128, 256, 512, 1024 and 1280 rows with 9 rows and with nearly as many as fit behind them; the norm behind o and down; columns behind the last 256 (8320)
@pytest.mark.gpu
@pytest.mark.parametrize("name,layers,tokens", [("qwen3-8b", 2, (257, 265, 384, 520, 553, 1033, 1152, 1289, 1400, 2057)), ("qwen3.5-2b", 4, (512, 649, 1033, 1152, 1545))])
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
