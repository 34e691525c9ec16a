"""How the kernel of whole layers deals a decode step's attention to its blocks, on the CPU: every cached key of every head is walked once, every piece has a place of
its own, and what brings a head's pieces together waits for places that are written, all of them."""
import ctypes
import random

import numpy as np
import pytest

from infinicore_infer_amd.kernels.lib import get_lib


def _pieces(positions, kv_heads, units):
    lib = get_lib()
    pos = np.array(positions, dtype=np.int32)
    heads = len(positions) * kv_heads
    cap = heads + units
    out, spans = np.zeros((cap, 6), dtype=np.int32), np.zeros((heads, 2), dtype=np.int32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    n = lib.ic_decode_chain_pieces(ptr(pos), len(positions), kv_heads, units, ptr(out), cap, ptr(spans))
    assert 0 < n <= cap
    return out[:n], spans


def _check(positions, kv_heads, units):
    pieces, spans = _pieces(positions, kv_heads, units)
    seen, places = {}, {}
    for w, row, kvh, lo, hi, place in pieces.tolist():
        assert 0 <= w < units and lo < hi <= positions[row] + 1
        seen.setdefault((row, kvh), []).append((lo, hi, w))
        assert place not in places and 0 <= place < len(positions) * kv_heads + units
        places[place] = (row, kvh)
    whole = spans[0][0] > spans[0][1]
    for row, pos in enumerate(positions):
        for kvh in range(kv_heads):
            mine = sorted(seen[(row, kvh)])
            assert mine[0][0] == 0 and mine[-1][1] == pos + 1 and all(a[1] == b[0] for a, b in zip(mine, mine[1:]))
            s = row * kv_heads + kvh
            first, last = spans[s].tolist()
            if whole:
                assert first > last and len(mine) == 1
            else:
                assert [w for _, _, w in mine] == list(range(first, last + 1))
                assert all(places[s + w] == (row, kvh) for w in range(first, last + 1))
    # what a block's plan must have room for, as the rule that admits a step counts it
    heads, total = len(positions) * kv_heads, sum((p + 64) // 64 for p in positions) * kv_heads
    assert np.bincount(pieces[:, 0]).max() <= max(-(-heads // units), min(heads, -(-total // units) + 1))


@pytest.mark.parametrize("positions,kv_heads,units", [
    ([0], 1, 256), ([63], 8, 256), ([64], 8, 256), ([600], 8, 256), ([2063], 36, 256), ([2063], 8, 256), ([16300], 2, 256), ([0] * 8, 36, 256),
    ([2100, 2000, 1950, 1900, 2050, 2001, 1999, 2002], 36, 256), ([4000, 0, 1, 62, 63, 64, 65, 2], 8, 64), ([5, 700], 36, 304)])
def test_every_key_once_and_every_piece_a_place(positions, kv_heads, units):
    _check(positions, kv_heads, units)


def test_random_steps():
    rng = random.Random(5)
    for _ in range(1500):
        longest = int(2 ** rng.uniform(0, 14))
        _check([rng.randrange(longest) for _ in range(rng.randint(1, 8))], rng.choice([1, 2, 3, 8, 36, 64]), rng.choice([64, 128, 228, 256, 304]))
