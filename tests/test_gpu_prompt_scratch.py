"""GPU: the buffers of prompts and of decode groups where the card has no room for them.  Allocations fail by a limit that the test sets (cm_debug_set "alloc_most"), before the runtime is asked."""
import numpy as np
import pytest

from crane_amd import _lib, configs

pytestmark = pytest.mark.gpu

CFG = dict(configs.get_config("qwen3.5-0.8b"), vocab_size=512, num_hidden_layers=4)
IDS = np.random.default_rng(2).integers(0, 512, 2300).tolist()


def _model(**kw):
    from crane_amd.backend import Model
    return Model.synthetic(CFG, seed=3, max_seq_len=4608, max_seqs=4, **kw)


def _row(m):
    s = m.seq_alloc()
    row = np.asarray(m.seq_forward(s, IDS, 0)[0]).copy()
    m.seq_free(s)
    return row


def _rows(m):
    return m.debug_read("prefill_rows", 2).tolist()


@pytest.fixture(scope="module")
def by_chunks():
    m = _model(prefill_chunk=2048)
    try:
        return _row(m)
    finally:
        m.close()


# 4224 rows: 140 MB of projection rows; 2048: 68 MB of those, 92 of chunked sums; the products' workspace 67 MB
def test_no_room_for_long_passes(by_chunks):
    m = _model()
    try:
        m.debug_set("alloc_most", 120_000_000)
        assert np.array_equal(_row(m), by_chunks) and _rows(m) == [2048, 2048]
        m.debug_set("alloc_most", -1)
        assert np.array_equal(_row(m), by_chunks) and _rows(m) == [2048, 2048]        # fixed with the first prompt
    finally:
        m.close()


def test_no_room_at_all_and_then_some(by_chunks):
    m = _model()
    try:
        m.debug_set("alloc_most", 70_000_000)
        for _ in range(2):
            with pytest.raises(_lib.CraneError):
                _row(m)
        m.debug_set("alloc_most", 120_000_000)
        assert np.array_equal(_row(m), by_chunks)
    finally:
        m.close()


# (635 MB for 4224 rows, asked for where twice that is free)
@pytest.mark.parametrize("free,rows", [(0, 2048), (1_250_000_000, 2048), (1_300_000_000, 4224), (-1, 4224)])
def test_the_free_memory_decides(by_chunks, free, rows):
    m = _model()
    try:
        m.debug_set("free_memory", free)
        row = _row(m)
        assert _rows(m) == [2048, rows] and np.array_equal(row, by_chunks) == (rows == 2048)
        assert np.abs(row - by_chunks).max() < 1e-4 * np.abs(by_chunks).max()
    finally:
        m.close()


def test_no_room_for_a_group():
    m = _model()
    try:
        seqs = [m.seq_alloc() for _ in range(2)]
        for s in seqs:
            m.seq_forward(s, IDS[:40], 0)
        m.debug_set("alloc_most", 1_000_000)                     # (128 projection rows: 4 MB)
        for _ in range(2):
            with pytest.raises(_lib.CraneError):
                m.step_batch_decode(seqs, [1, 2])
        m.debug_set("alloc_most", -1)
        a = np.asarray(m.step_batch_decode(seqs, [1, 2], want_logits=True)[0]).copy()
    finally:
        m.close()
    m = _model()
    try:
        seqs = [m.seq_alloc() for _ in range(2)]
        for s in seqs:
            m.seq_forward(s, IDS[:40], 0)
        assert np.array_equal(a, np.asarray(m.step_batch_decode(seqs, [1, 2], want_logits=True)[0]))
    finally:
        m.close()
