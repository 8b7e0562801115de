"""The host arithmetic by which a chunk chooses its slices: what it adds up, and that a call does not wait for it."""
import time

import numpy as np

from hipml_amd import attn


def slices_of_all(pos0, tok, n_head, n_kv, splits):
    """The definition: block by block of 8 tasks (32 tokens of a head), as many slices as its last token's key tiles take."""
    group, tiles = n_head // n_kv, -(-(pos0 + tok) // 64)
    ntask, per_slice = -(-tok // 32) * group, -(-tiles // splits)
    total = 0
    for tb in range(-(-ntask // 8)):
        seq = pos0 + min((min(tb * 8 + 7, ntask - 1) // group + 1) * 32, tok)
        total += max(1, min(splits, -(-(-(-seq // 64)) // per_slice)))
    return total


def test_slices_of_all_blocks():
    rng = np.random.default_rng(3)
    lib = attn.lib()
    for _ in range(4000):
        n_kv = int(rng.integers(1, 9))
        n_head = n_kv * int(rng.integers(1, 13))
        tok, pos0 = int(np.exp(rng.uniform(0.0, np.log(5000)))), int(np.exp(rng.uniform(0.0, np.log(20_000)))) - 1
        splits = int(rng.integers(2, 65))
        assert lib.hipml_dbg_chunk_slices_of_all(pos0, tok, n_head, n_kv, splits) == slices_of_all(pos0, tok, n_head, n_kv, splits)


def test_choosing_slices_takes_no_time():
    # one KV head's 500 blocks near position 0, 62 counts: block by block 165 us on the CPU that this was found on, and 4 so
    lib, args = attn.lib(), (0, 16_000, 8, 1, 64)
    best = 1.0
    for _ in range(50):
        start = time.perf_counter()
        for _ in range(20):
            lib.hipml_dbg_chunk_q8_slices(*args)
        best = min(best, (time.perf_counter() - start) / 20)
    assert best < 40e-6, best
