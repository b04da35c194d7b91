"""The tiles of a layer-list decoder's matrix-core products (crane_amd/csrc/kernels_layered_gemm.hip): which shape a product takes (host logic, through
cm_debug_lay_tile_shape), and on the GPU every shape against the plain kernels at ragged sizes."""
import pytest

from crane_amd import _lib
from tests import gizezen_util as GZ
from tests.test_gpu_layered_experts import _check


# (tokens, columns, inner, experts, per token, pair, columns beside, function behind it, rows * 1000 + columns; negative: the last columns in a launch of their own)
@pytest.mark.parametrize("tokens,columns,inner,experts,top,pair,beside,function,shape", [
    # 16 experts of 2048 x 4096, 4 per token, and one of every token: the figures beside the rule
    (100, 2048, 4096, 16, 4, 1, 2048, 0, 64064), (200, 2048, 4096, 16, 4, 1, 2048, 0, 128192), (450, 4096, 2048, 16, 4, 0, 4096, 0, 128192),
    (700, 2048, 4096, 16, 4, 1, 2048, 0, 192128), (1200, 4096, 2048, 16, 4, 0, 4096, 0, 192128), (2048, 2048, 4096, 16, 4, 1, 2048, 0, 256256),
    (2048, 4096, 2048, 16, 4, 0, 4096, 0, 256256),
    # 14 experts of 768 x 1024
    (326, 768, 1024, 14, 4, 1, 512, 0, 64064), (326, 1024, 768, 14, 4, 0, 1024, 0, 64064), (2048, 768, 1024, 14, 4, 1, 512, 0, 128128),
    (2048, 1024, 768, 14, 4, 0, 1024, 0, 192128),
    # one matrix: columns behind the last whole tile, a function that only the two smaller shapes know
    (2048, 4128, 4096, 0, 0, 0, 0, 0, -128128), (2048, 4096, 4096, 0, 0, 0, 0, 0, 128128), (326, 1032, 1024, 0, 0, 0, 0, 0, 64064),
    (2048, 6144, 4096, 0, 0, 0, 0, 0, 128192), (2048, 6144, 4096, 0, 0, 0, 0, 1, 128128)])
def test_the_shape_whose_rounds_take_the_least(tokens, columns, inner, experts, top, pair, beside, function, shape):
    assert _lib.load().cm_debug_lay_tile_shape(tokens, columns, inner, experts, top, pair, beside, function) == shape


# every shape of either product, odd numbers of k-tiles, ragged rows and columns (the products' tolerance: tests/test_gpu_layered_experts.py)
@pytest.mark.gpu
@pytest.mark.parametrize("n,width,ff,shared,experts,first,second", [
    (1300, 1600, 1088, 704, 8, 256256, 192128), (1000, 1088, 1088, 320, 16, 128192, 128128), (700, 1088, 1088, 320, 16, 192128, 128128),
    (1700, 1088, 1088, 320, 16, 192128, 128192), (2100, 1216, 576, 192, 8, 192128, 256256)])
def test_experts_on_every_shape(tmp_path, n, width, ff, shared, experts, first, second):
    plan = _lib.load().cm_debug_lay_tile_shape
    assert plan(n, ff, width, experts, 4, 1, shared, 0) == first and plan(n, width, ff, experts, 4, 0, width, 0) == second
    cfg = GZ.config([GZ.layer(GZ.attn(), GZ.moe(experts=experts, top=4, ff=ff, shared=shared))], vocab=96, width=width)
    _check(tmp_path, GZ, cfg, n, 3)


# 32 gates behind 4096 columns (their sigmoid in the small launch), and 3 behind 640 whose function stays inside the tile kernel
@pytest.mark.gpu
@pytest.mark.parametrize("n,width,heads,kv_heads,tail", [(2000, 4096, 32, 16, True), (130, 192, 3, 3, False)])
def test_last_columns(tmp_path, n, width, heads, kv_heads, tail):
    mixer = GZ.attn(heads=heads, kv_heads=kv_heads, dim=64, vdim=64)
    cols = (heads + 2 * kv_heads) * 64 + heads
    assert (_lib.load().cm_debug_lay_tile_shape(n, cols, width, 0, 0, 0, 0, 0) < 0) == tail
    _check(tmp_path, GZ, GZ.config([GZ.layer(mixer, None)], vocab=96, width=width), n, 5)


# one matrix on tiles in pairs (an even number of 128- or 192-wide ones): a projection of 5 k-tiles, ragged rows, a last row tile of 4 rows and none
@pytest.mark.gpu
@pytest.mark.parametrize("n,width,shape", [(1300, 3072, 128128), (1028, 4096, 128128), (2000, 6144, 128192), (2048, 6144, 128192)])
def test_tiles_in_pairs(tmp_path, n, width, shape):
    assert _lib.load().cm_debug_lay_tile_shape(n, width, 320, 0, 0, 0, 0, 0) == shape
    _check(tmp_path, GZ, GZ.config([GZ.layer(GZ.attn(heads=5, kv_heads=5, dim=64, vdim=64), None)], vocab=96, width=width), n, 7)
