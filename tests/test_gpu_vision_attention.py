"""GPU: the frame attention of the vision tower (kernels_vision_attn.hip) at the edges of its tiles."""
import numpy as np
import pytest

from tests.test_qwen3_5_vl import _setup, rel

pytestmark = pytest.mark.gpu


# frames of 4, 60, 64, 68 and 132 patches (below, at and above a key tile and two query tiles), a last key tile of one merge block, frames that
# start off a 64-row boundary, several frames of one video; against the f32 oracle with the bar its other tests use
@pytest.mark.parametrize("grid", [[[1, 2, 2]], [[1, 6, 10]], [[1, 8, 8]], [[1, 2, 34]], [[1, 12, 11 * 2]], [[1, 2, 2], [1, 8, 8], [1, 2, 66], [1, 6, 10]],
                                  [[3, 6, 6], [1, 4, 4]]])
def test_against_the_oracle(grid):
    from crane_amd.backend import Model
    from oracle.qwen3_5_vision_oracle import VisionOracle
    g, cfg, w, text_w = _setup()
    n = sum(t * h * v for t, h, v in grid)
    pix = np.random.default_rng(n).standard_normal((n, g["pixel_values"].shape[1])).astype(np.float32)
    m = Model.synthetic(cfg, seed=0, max_seq_len=256, max_seqs=2)
    try:
        assert rel(m.encode_images(pix, grid), VisionOracle(cfg["vision_config"], w).forward(pix, grid)) < 1e-4
    finally:
        m.close()


# the full-width tower: images alone (64 query rows per workgroup; the first in one run of keys, the others in two with a merge) and together (128
# rows, two runs, of which the first image leaves one empty) -- the same sums of three bf16 products in another order: 24 blocks of f32 sums of <= 4096 terms, each within sqrt(4096) 2^-24 = 4e-6 of
# its size, and their re-rounding into hi + lo planes (2^-17 = 8e-6): 24 * 1.2e-5 if nothing averages out
def test_widths_and_runs_agree():
    from crane_amd import configs
    from crane_amd.backend import Model
    cfg = configs.get_config("qwen3-vl-2b")
    m = Model.synthetic(dict(cfg, text_config=dict(cfg["text_config"], num_hidden_layers=1)), seed=0, max_seq_len=256, max_seqs=1)
    grids = [[1, 6, 6], [1, 30, 36], [1, 38, 40]]
    rng = np.random.default_rng(0)
    pix = [rng.standard_normal((h * w, 1536)).astype(np.float32) for _, h, w in grids]
    try:
        alone = [m.encode_images(p, [g]) for p, g in zip(pix, grids)]
        together = m.encode_images(np.concatenate(pix), grids)
        assert rel(together, np.concatenate(alone)) < 3e-4
    finally:
        m.close()


# entries of a grid without rows (no frames, or a side of 0) cost and change nothing, whatever their other numbers; numbers whose product wraps to 0 are
# refused like any other that the patches do not match
def test_images_without_rows():
    from crane_amd import _lib
    from crane_amd.backend import Model
    g, cfg, w, text_w = _setup()
    pix = np.random.default_rng(0).standard_normal((64, g["pixel_values"].shape[1])).astype(np.float32)
    m = Model.synthetic(cfg, seed=0, max_seq_len=256, max_seqs=2)
    try:
        want = m.encode_images(pix, [[1, 8, 8]])
        for empty in ([0, 2000000000, 2], [0, 8, 4000000000], [4000000000, 0, 4000000000]):
            assert (m.encode_images(pix, [empty, [1, 8, 8]]) == want).all() and (m.encode_images(pix, [[1, 8, 8], empty]) == want).all()
        for wrong in ([2 ** 22, 2 ** 21, 2 ** 21], [2 ** 31, 2 ** 31, 4], [1, 2, 2]):
            for grid in ([wrong, [1, 8, 8]], [[1, 8, 8], wrong]):
                with pytest.raises(_lib.CraneError):
                    m.encode_images(pix, grid)
        assert (m.encode_images(pix, [[1, 8, 8]]) == want).all()
    finally:
        m.close()
