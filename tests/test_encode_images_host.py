"""What Model.encode_images hands to its caller, with the library's call replaced by one that writes a known pattern -- no GPU."""
import ctypes as C
import gc

import numpy as np
import pytest

from crane_amd.backend import Model


class Lib:
    """cm_vision_encode: a quarter as many rows as patches, element i of the features = i."""
    cm_vocab_size = staticmethod(lambda h: 16)
    cm_hidden_size = staticmethod(lambda h: 96)
    cm_destroy = staticmethod(lambda h: None)
    cm_vision_features = staticmethod(lambda h, n: n // 4 * 96)

    @staticmethod
    def cm_vision_encode(h, pix, n, grid, images, out, rows):
        C.cast(rows, C.POINTER(C.c_size_t))[0] = n // 4
        np.ctypeslib.as_array(out, (n // 4 * 96,))[:] = np.arange(n // 4 * 96)
        return 0


# the features own exactly their rows: no view that keeps the upper bound on them (four times as many) alive
@pytest.mark.parametrize("patches", [4, 16, 4096])
def test_features_own_their_rows(patches):
    got = Model(1, Lib).encode_images(np.zeros((patches, 8), np.float32), [[1, 2, patches // 2]])
    gc.collect()
    assert got.base is None and got.flags.owndata and got.flags.c_contiguous and got.flags.writeable
    assert got.shape == (patches // 4, 96) and got.dtype == np.float32
    assert (got.reshape(-1) == np.arange(got.size)).all()
