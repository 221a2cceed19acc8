"""Many chunk pairs packed a column at a time give the bytes of the table packed pair by pair, and
refuse what that refuses."""
import ctypes as C

import numpy as np
import pytest

from satsuma2_amd import api


def rows(n):
    rng = np.random.default_rng(n)
    seqs = [bytes(rng.choice(list(b"ACGTN"), int(k)).astype(np.uint8)) for k in rng.integers(0, 90, 2 * n)]
    return [api.ChunkPair(seqs[k], seqs[n + k], *(int(v) for v in rng.integers(0, 1 << 30, 4)),
                          q_record_len=int(rng.integers(-1, 1 << 30)) if k % 3 else -1, fast=k % 2) for k in range(n)]


@pytest.mark.parametrize("n", [31, 32, 33, 200])
def test_same_table(n):
    pairs = rows(n)
    arr, keep = api._pairs_array(pairs)
    for k, p in enumerate(pairs):
        one, keep1 = api._pairs_array([p])
        for f, _ in api.Pair._fields_:
            assert getattr(arr[k], f) == getattr(one[0], f), f


@pytest.mark.parametrize("field,value", [("t_record", 1.5), ("tseq", "ACGT"), ("fast", "x")])
def test_refused(field, value):
    for n in (1, 40):
        pairs = rows(n)
        setattr(pairs[n // 2], field, value)
        with pytest.raises((TypeError, C.ArgumentError, ValueError)):
            api._pairs_array(pairs)


@pytest.mark.parametrize("value", [np.uint64(7), np.int64(5), True, 1 << 31, (1 << 31) + 5, (1 << 32) + 3, 1 << 63, 1 << 64,
                                   -(1 << 63) - 1, -5, np.array(4)])
@pytest.mark.parametrize("field", ["t_record", "q_record_len", "fast"])
def test_integers_of_any_type(field, value):
    """Record arrays hold uint64; what one pair is packed to, many are."""
    pairs = rows(40)
    setattr(pairs[11], field, value)
    arr, _ = api._pairs_array(pairs)
    for k in (0, 11, 39):
        one, _ = api._pairs_array(pairs[k:k + 1])
        for f, _ in api.Pair._fields_:
            assert getattr(arr[k], f) == getattr(one[0], f), (k, f)
