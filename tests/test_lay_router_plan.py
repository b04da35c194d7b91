"""Host logic of a layer-list decoder's router in decode steps (crane_amd/csrc/kernels_layered.hip: lay_router_decode_fits through
cm_debug_lay_router_plan): one launch on one CU while there is little to multiply, the streaming row kernel on the whole chip otherwise -- no GPU.
(What the routes compute is held to the oracle in tests/test_gpu_layered_experts.py.)"""
import pytest

from crane_amd import _lib


def one_launch(rows, width, outputs, top=4, shared=1, offset=0):
    return _lib.load().cm_debug_lay_router_plan(rows, width, outputs, top, shared, offset)


# measured on both sides of the lines (up to 17 logits 8 rows of 4096, up to 33 logits 2^18 products, more 2^17): the faster one is taken
@pytest.mark.parametrize("rows,width,outputs,one", [
    (1, 1024, 14, 1), (8, 1024, 14, 1), (1, 4096, 16, 1), (8, 2048, 16, 1), (8, 4096, 16, 1), (8, 4104, 16, 0), (8, 1024, 24, 1), (4, 2048, 24, 1),
    (8, 512, 32, 1), (1, 4096, 32, 1), (8, 1024, 32, 0), (8, 2048, 32, 0), (2, 1024, 48, 1), (8, 512, 48, 0), (1, 1024, 64, 1), (4, 1024, 64, 0),
    (8, 4096, 64, 0), (1, 512, 128, 1), (1, 1024, 128, 0), (1, 4096, 256, 0)])
def test_the_faster_route(rows, width, outputs, one):
    assert one_launch(rows, width, outputs) == one


def test_refusals():
    assert one_launch(8, 64, 4) == 1 and one_launch(9, 64, 4) == 0                  # rows of the streaming kernel
    assert one_launch(1, 72, 70) == 1 and one_launch(1, 76, 70) == 0                # whole 16-byte pieces of a row of the matrix ...
    assert all(one_launch(1, 72, 70, offset=o) == 0 for o in (2, 4, 8)) and one_launch(1, 72, 70, offset=16) == 1      # ... from a 16-byte boundary
    assert one_launch(1, 72, 70, top=64) == 1 and one_launch(1, 72, 70, top=65) == 0
