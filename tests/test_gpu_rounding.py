"""GPU: sums whose rounding is written out in the kernels, so that 16-bit pages and 8-bit codes stay what they are under another compiler or another way of exchanging lanes,
against the same roundings in numpy: equal, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from crane_amd import _lib

pytestmark = pytest.mark.gpu

F = np.float32


def _ptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def _fma(a, b, c):
    """a b + c with one rounding: the product is exact in 64 bits of significand, and a sum that these round onto a boundary of 24 has a chance of 2^-40."""
    return (a.astype(np.longdouble) * b.astype(np.longdouble) + c.astype(np.longdouble)).astype(F)


# one row, an odd number of heads, a block of heads that is not full, K slices
@pytest.mark.parametrize("n,heads,slices", [(1, 1, 1), (75, 3, 1), (117, 8, 4), (33, 5, 2)])
def test_rotation_of_prompt_rows(n, heads, slices):
    rng = np.random.default_rng(n)
    parts = rng.standard_normal((slices, n, 2 * heads, 128)).astype(F)
    angle = rng.uniform(0, 6.28, (n, 64))
    cos, sin = np.cos(angle).astype(F), np.sin(angle).astype(F)
    out = np.empty((2, heads, n, 128), F)
    assert _lib.load().cm_debug_rope_rows(_ptr(parts), n, heads, slices, _ptr(cos), _ptr(sin), _ptr(out)) == 0
    x = parts[0]
    for p in parts[1:]:
        x = x + p
    k, c, s = x[:, :heads], np.tile(cos, 2)[:, None], np.tile(sin, 2)[:, None]
    other = np.roll(k, 64, axis=-1)
    y = other * s * np.where(np.arange(128) < 64, F(-1), F(1))
    want = np.where(np.arange(128) % 4 < 2, _fma(k, np.broadcast_to(c, k.shape), y), k * c + y)
    assert np.array_equal(out[0], want.transpose(1, 0, 2)) and np.array_equal(out[1], x[:, heads:].transpose(1, 0, 2))


# a key of zeros, one query channel and no decay: y is the state's first row times the query's scale, and what is left is the norm's sum of squares
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_norm_of_a_gated_delta_step(seed):
    heads, kd = 32, 32 * 128
    rng = np.random.default_rng(seed)
    proj = np.zeros(4 * kd + 2 * heads, F)
    proj[0:kd:128] = 32                                    # silu(32) = 32 in 32 bits, and so is 32 / sqrt(32^2 + 1e-6) = 1
    proj[3 * kd:4 * kd] = 32
    proj[4 * kd:] = -200                                   # no update, no decay
    conv = np.zeros((3 * kd, 4), F)
    conv[:, 3] = 1
    state = np.zeros((heads, 128, 128), F)
    state[:, 0] = rng.standard_normal((heads, 128))
    out = np.empty((heads, 128), F)
    assert _lib.load().cm_debug_gdn_step(_ptr(proj), _ptr(conv), _ptr(state), heads, _ptr(out)) == 0
    y = state[:, 0] * F(0.08838834764831845)
    q = y.reshape(heads, 4, 32)
    t = _fma(q, q, np.roll(q, 16, axis=-1) * np.roll(q, 16, axis=-1))[..., :16]
    for half in (8, 4, 2, 1):
        t = t[..., :half] + t[..., half:2 * half]
    t = t[..., 0]
    tot = ((t[:, 0] + t[:, 1]) + t[:, 2]) + t[:, 3]
    rms = F(1) / np.sqrt(_fma(tot, np.full_like(tot, 2.0 ** -7), np.full_like(tot, 1e-6)))
    assert np.array_equal(out, y * rms[:, None] * F(32))
