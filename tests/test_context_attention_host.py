"""Host side of the prefill context attention: the extend entry's
validation messages (no kernel launch), and the tests' metadata helper."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from akv_amd import _lib, context_attention as ca

from harness import attention_metadata, plain_segments, window_segments


def test_validation_messages():
    q = torch.zeros((4, 8, 64), dtype=torch.bfloat16)
    k = torch.zeros((4, 1, 64), dtype=torch.bfloat16)
    ind = torch.zeros(2, dtype=torch.int64)
    with pytest.raises(ValueError, match="both query and KV positions"):
        ca.extend_attention_fwd(q, k, k, q, k, k, ind, ind, ind, None, True, None, 4,
                                context_q_positions=torch.zeros(4, dtype=torch.int64))
    with pytest.raises(ValueError, match="must align with Q/KV"):
        ca.extend_attention_fwd(q, k, k, q, k, k, ind, ind, ind, None, True, None, 4,
                                context_q_positions=torch.zeros(3, dtype=torch.int64),
                                context_kv_positions=torch.zeros(2, dtype=torch.int64))
    with pytest.raises(ValueError, match="requires page_size=1"):
        ca.extend_attention_fwd(q, k, k, q, k, k, ind, ind, ind, None, True, None, 4, page_size=16,
                                context_q_positions=torch.zeros(4, dtype=torch.int64),
                                context_kv_positions=torch.zeros(2, dtype=torch.int64))
    with pytest.raises(ValueError, match="custom mask"):
        ca.extend_attention_fwd(q, k, k, q, k, k, ind, ind, ind, torch.ones(1), True, None, 4)


def test_split_bytes_names_the_batches_it_takes():
    need = _lib.load().akv_context_attention_split_bytes
    assert need(1, 64, 8, 64, -1, 200, 200, 20000) > 0
    assert need(1, 64, 8, 64, 0, 200, 200, 20000) > 0  # no window either
    assert need(1, 64, 8, 64, 128, 200, 200, 20000) == 0  # a window
    assert need(65, 64, 8, 64, -1, 6500, 100, 20000) == 0  # too many segments
    assert need(1, 64, 8, 64, -1, 4096, 4096, 20000) == 0  # the plain launch fills the chip
    # short segments that fill a round of the plain launch
    assert need(64, 28, 4, 128, -1, 64 * 18, 28, 64 * 1900) == 0
    assert need(32, 40, 8, 128, -1, 32 * 18, 29, 32 * 2268) == 0
    # a workspace that goes with the batch
    assert need(1, 64, 8, 64, -1, 16, 16, 1000) < 10 << 20
    assert need(1, 64, 8, 64, -1, 200, 200, 20000) > 60 << 20


@pytest.mark.parametrize("why,changes", [("window", {27: 128}), ("segments", {15: 65}), ("no workspace", {36: None}),
                                         ("short workspace", {37: 64}), ("workspace alignment", {36: (1 << 20) + 8})])
def test_split_refuses(why, changes):
    """Each is refused before any device pointer is looked at: all of them
    are null here, so a call that passed this check would stop at the next."""
    lib = _lib.load()
    fn = lib.akv_context_attention_split
    args = [None if t is _lib.c_void_p else 0 for t in fn.argtypes]
    good = {15: 1, 16: 8, 17: 1, 18: 64, 21: _lib.AKV_I32, 23: _lib.AKV_I32, 26: _lib.AKV_I32, 27: -1, 29: 0.125,
            32: _lib.AKV_BF16, 35: 4, 36: 1 << 20, 37: 1 << 30}
    for at, value in {**good, **changes}.items():
        args[at] = value
    assert fn(*args) == _lib.AKV_EINVAL
    assert "akv_context_attention_split: needs no window" in _lib.last_error(), why
    for at, value in good.items():
        args[at] = value
    assert fn(*args) == _lib.AKV_EINVAL
    assert "null device pointer" in _lib.last_error()


def test_metadata_helper_splits_segments():
    """Two query segments; the second reads one key (occurrence 5) before
    its own births; a plain request follows with occurrence ids offset."""
    window = SimpleNamespace(
        segment_query_starts=np.array([0, 3]), segment_query_ends=np.array([3, 5]),
        occurrence_raw_tokens=np.array([0, 1, 2, 3, 4, 1]), occurrence_positions=np.array([0, 1, 2, 3, 4, 0]),
        birth_occurrences=np.arange(5), segment_key_occurrences=np.array([0, 1, 2, 5, 3, 4]),
        segment_key_offsets=np.array([0, 3, 6]))
    seg = window_segments(window)
    np.testing.assert_array_equal(seg.query_lengths, [3, 2])
    np.testing.assert_array_equal(seg.prefix_lengths, [0, 1])
    np.testing.assert_array_equal(seg.prefix, [5])
    np.testing.assert_array_equal(seg.prefix_positions, [0])
    np.testing.assert_array_equal(seg.query_positions, [0, 1, 2, 3, 4])
    meta = attention_metadata([seg, plain_segments(3, 2)], torch.arange(100, 111))
    c = meta.cpu
    np.testing.assert_array_equal(c.qo_indptr, [0, 3, 5, 7])
    np.testing.assert_array_equal(c.kv_indptr, [0, 0, 1, 4])
    np.testing.assert_array_equal(c.occurrences, [5, 6, 7, 8])
    np.testing.assert_array_equal(meta.kv_indices.numpy(), [105, 106, 107, 108])
    np.testing.assert_array_equal(c.query_positions, [0, 1, 2, 3, 4, 3, 4])
    np.testing.assert_array_equal(c.kv_positions, [0, 0, 1, 2])
