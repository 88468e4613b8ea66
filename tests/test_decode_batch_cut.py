"""The cut of a decode batch into split-K chunks, on the host: a batch whose
sequences are about as long as each other keeps the cut its size gives, a
ragged one is cut finer, neither needs more than the workspace query's bound,
and the array-backed step refuses what its array cannot hold before any work
(256 compute units, as without a device).
"""
import ctypes
import random

import pytest

from tinymetalagent_amd import runtime as R

TILE, CUS = 32, 256


def _chunking(positions, layers, kv):
    chunk, chunks = ctypes.c_size_t(), ctypes.c_size_t()
    arr = (ctypes.c_size_t * len(positions))(*positions)
    R.check(R.load_library().te_hip_attention_decode_chunking(arr, 0, len(positions), layers, kv, 0,
                                                              ctypes.byref(chunk), ctypes.byref(chunks)))
    return chunk.value, chunks.value


def _cut_of_the_size(positions, layers, kv):
    """Chunks of the longest sequence for 3.5 workgroups per CU of equal work."""
    tiles = [(p + TILE) // TILE for p in positions]
    per = max(2, -(-sum(tiles) * layers * kv // (CUS * 7 // 2)))
    return -(-max(tiles) // per)


@pytest.mark.parametrize("layers,kv,positions", [
    (28, 4, [2048] * 16), (28, 4, [4096] * 16), (36, 2, [1024] * 64), (24, 2, [8192] * 8), (36, 2, [8192] * 2),
    (28, 4, [2048 - 20 * i for i in range(16)]), (28, 4, [600] * 10), (28, 2, [511, 512, 480, 500, 470])])
def test_even_batch_keeps_the_cut_of_its_size(layers, kv, positions):
    assert _chunking(positions, layers, kv)[1] == _cut_of_the_size(positions, layers, kv)


@pytest.mark.parametrize("layers,kv,positions,chunks", [
    (28, 4, [1531, 15877, 9040, 4211, 12798, 2345, 7007, 10662], 8), (28, 4, [2000, 10, 20, 300, 50, 40, 60, 100], 8),
    (28, 4, [512] + [40] * 40, 3)])
def test_ragged_batch_is_cut_finer(layers, kv, positions, chunks):
    assert _cut_of_the_size(positions, layers, kv) < chunks == _chunking(positions, layers, kv)[1]


def test_no_batch_needs_more_than_its_workspace():
    lib, rng, heads, d = R.load_library(), random.Random(3), 8, 128
    for _ in range(3000):
        seqs, layers, kv = rng.randint(1, 64), rng.choice([1, 2, 5, 28, 36, 80]), rng.choice([1, 2, 4, 8])
        top = rng.choice([1, 31, 300, 2100, 9000, 131072])
        positions = [rng.randrange(top) for _ in range(seqs)] if rng.random() < 0.7 else [top] * seqs
        arr = (ctypes.c_size_t * seqs)(*positions)
        held = lib.te_hip_attention_decode_workspace_bytes(arr, 0, seqs, layers, heads, kv, d)
        assert held >= seqs * layers * heads * _chunking(positions, layers, kv)[1] * (d + 2) * 4, positions


def test_array_backed_step_refuses_a_cut_beyond_its_array():
    """One long sequence among short ones: the chunks its size needs (342 of 3
    tiles, 21.7 MiB of partials) exceed the 16 MiB array, though longer ones
    would fit it.  Refused on the host: no pointer is used."""
    layers, heads, kv, d, positions = 1, 16, 2, 128, [32767] + [1] * 7
    chunks = _chunking(positions, layers, kv)[1]
    assert chunks == 342 and len(positions) * layers * heads * chunks * (d + 2) * 4 > 16 << 20
    arr = (ctypes.c_size_t * len(positions))(*positions)
    p = ctypes.c_void_p(4096)
    st = R.load_library().te_hip_attention_decode_step_noalloc_f16(
        p, p, p, None, None, None, p, p, p, p, arr, 0, len(positions), layers, 32768, heads, kv, d, p, None)
    assert st == R.TE_STATUS_UNSUPPORTED
