"""Chunks over the cache, and over its registered f16 copy, for which fewer key slices run than the caller's scratch holds: the result is the oracle's (the gate of
the chunk kernels) and that of a call which asks for those slices, and the rest of the scratch is left alone."""
import ctypes

import numpy as np
import pytest
import torch

from hipml_amd import attn

N_HEAD, N_KV, HD = 24, 4, 256


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("tok,pos0,splits,n_head,n_kv", [
    (450, 1800, 12, 24, 4),   # every block of tokens with all slices, a ragged last tile
    (353, 5003, 14, 24, 4),   # twelve blocks, two rounds of workgroups in one
    (900, 100, 8, 24, 4),     # blocks near position 0 with fewer slices than the last
    (700, 0, 8, 24, 4), (600, 40, 8, 32, 8), (1501, 90, 12, 14, 2)])
def test_fewer_slices_than_the_scratch_holds(tok, pos0, splits, n_head, n_kv, dtype):
    from oracle import binding as orc
    from gpu_util import SCALE, dev, host, report
    from test_gpu_prefill import GATE
    attn.init(0)
    lib = attn.lib()
    used = lib.hipml_dbg_chunk_q8_slices(pos0, tok, n_head, n_kv, splits)
    assert 2 <= used < splits and lib.hipml_dbg_chunk_wg_splits(pos0, tok, n_head, n_kv, splits) == 0
    assert lib.hipml_dbg_chunk_q8_slices(pos0, tok, n_head, n_kv, used) == used
    r = orc.Rng(0x511C_0000 + tok * 131 + pos0)
    stride = pos0 + tok + 3
    kb = orc.quantize(dtype, r.normal_array((n_kv, stride, HD))).reshape(n_kv, stride, -1)
    vb = orc.quantize(dtype, r.normal_array((n_kv, stride, HD))).reshape(n_kv, stride, -1)
    q, gate = r.normal_array((tok, n_head, HD)), dev(r.normal_array((tok, n_head, HD)))
    qd, kd, vd = dev(q), dev(kb), dev(vb)
    acc, ml = attn.chunk_scratch(tok, n_head, splits)
    acc.fill_(7.0), ml.fill_(7.0)
    out, asked, gated_rows, work = (torch.full((tok + 1, n_head, HD), float("nan"), device="cuda") for _ in range(4))
    out16 = torch.full((tok + 1, n_head, HD), float("nan"), dtype=torch.float16, device="cuda")
    args = (n_head, n_kv, HD, pos0, tok, dtype + 1, stride, acc, ml)
    attn.chunk_attention_q8_split(qd, kd, vd, out, *args, splits)
    attn.chunk_attention_q8_split_gate(qd, kd, vd, gate, gated_rows, *args, splits)
    attn.chunk_attention_q8_split_gate_f16(qd, kd, vd, gate, work, out16, *args, splits)
    torch.cuda.synchronize()
    assert bool((acc[used:] == 7.0).all()) and bool((ml[used:] == 7.0).all())
    attn.chunk_attention_q8_split(qd, kd, vd, asked, *args, used)
    two = torch.empty((tok, n_head, HD), device="cuda")
    attn.q_gate(out[:tok].contiguous(), gate, two)
    torch.cuda.synchronize()
    want = orc.attn_chunk_kv(q, kb, vb, n_head, n_kv, HD, pos0, tok, stride, SCALE, n_threads=8, dtype=dtype)
    assert report(f"chunk {tok}@{pos0}, {used} of {splits} slices", want, host(out[:tok]), *GATE)[0]
    assert torch.equal(asked[:tok], out[:tok])
    assert torch.equal(two, gated_rows[:tok]) and torch.equal(out16[:tok], two.to(torch.float16))
    for x in (out, asked, gated_rows, out16):
        assert bool(x[tok].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("tok,pos0,splits,t64", [
    (96, 1700, 10, 0),    # a count that leaves the first block a slice short: the kernel of 32 tokens per wave
    (420, 5003, 12, 1), (1079, 492, 8, 0),
    (64, 1819, 10, 0), (33, 1400, 8, 0)])  # few tokens behind less than 2,048 rows, which read the copy
def test_fewer_slices_over_a_registered_copy(tok, pos0, splits, t64, dtype):
    from test_gpu_kv_f16 import run_chunk_f16
    from test_gpu_kv_shadow import Attached, attend
    from oracle import binding as orc
    attn.init(0)
    took = ctypes.c_int()
    used = attn.lib().hipml_dbg_chunk_f16_slices(pos0, tok, N_HEAD, N_KV, splits, ctypes.byref(took))
    assert splits == attn.chunk_slices(pos0, tok, N_KV) and 2 <= used < splits and took.value == t64
    r = orc.Rng(0x511C_1000 + tok)
    stride = pos0 + tok + 5
    kb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    vb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    q = r.normal_array((tok, N_HEAD, HD))
    with Attached(kb, vb, stride, pos0 + tok, dtype=dtype) as c:
        got = attend(q, c.k, c.v, pos0, tok, stride, splits, dtype=dtype + 1)
    by_hand = run_chunk_f16(q, kb, vb, pos0, tok, stride, used, dtype=dtype)
    assert np.array_equal(got.view(np.uint32), by_hand.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("tok,pos0,splits,cache", [
    (64, 2048, 12, True), (1, 2048, 12, True), (33, 5000, 16, True), (64, 2047, 12, False), (65, 2048, 12, False)])
def test_few_tokens_read_the_cache_beside_a_registered_copy(tok, pos0, splits, cache, dtype):
    # both sides of the rule's two lines; the registered copy is made NaN after its conversion, so a call that reads it shows
    from test_gpu_kv_f16 import run_chunk_f16
    from test_gpu_kv_shadow import Attached, attend
    from gpu_util import dev
    from oracle import binding as orc
    attn.init(0)
    r = orc.Rng(0x511C_2000 + tok)
    stride = pos0 + tok + 5
    kb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    vb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    q = r.normal_array((tok, N_HEAD, HD))
    plain = attend(q, dev(kb), dev(vb), pos0, tok, stride, splits, dtype=dtype + 1)
    with Attached(kb, vb, stride, pos0 + tok, dtype=dtype) as c:
        if cache:
            c.copy.fill_(0xFF)
        got = attend(q, c.k, c.v, pos0, tok, stride, splits, dtype=dtype + 1)
    if cache:
        assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))
    else:
        took = ctypes.c_int()
        most = min(splits, attn.chunk_slices(pos0, tok, N_KV))
        used = attn.lib().hipml_dbg_chunk_f16_slices(pos0, tok, N_HEAD, N_KV, most, ctypes.byref(took))
        assert np.array_equal(got.view(np.uint32), run_chunk_f16(q, kb, vb, pos0, tok, stride, used, dtype=dtype).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("tok,pos0", [(768, 1300), (900, 900), (1400, 1700)])
def test_a_scratch_with_room_for_tiles_that_would_not_pay(tok, pos0, dtype):
    from oracle import binding as orc
    from gpu_util import SCALE, dev, report
    from test_gpu_prefill import GATE
    from test_gpu_kv_shadow import attend
    attn.init(0)
    splits = attn.chunk_splits(pos0, tok, N_KV)
    assert splits > attn.chunk_slices(pos0, tok, N_KV) >= 2
    assert attn.lib().hipml_dbg_chunk_makes_tiles(pos0, tok, N_HEAD, N_KV, splits) == 0
    r = orc.Rng(0x511C_3000 + tok)
    stride = pos0 + tok + 5
    kb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    vb = orc.quantize(dtype, r.normal_array((N_KV, stride, HD))).reshape(N_KV, stride, -1)
    q = r.normal_array((tok, N_HEAD, HD))
    got = attend(q, dev(kb), dev(vb), pos0, tok, stride, splits, dtype=dtype + 1)
    rows = np.array([0, 31, 32, 400, tok - 33, tok - 1], dtype=np.int32)
    want = orc.attn_chunk_kv(q, kb, vb, N_HEAD, N_KV, HD, pos0, tok, stride, SCALE, rows=rows, n_threads=8, dtype=dtype)
    assert report(f"chunk {tok}@{pos0} without tiles", want, got[rows], *GATE)[0]
    assert np.isfinite(got).all()


@pytest.mark.parametrize("tok,pos0,use", [(1024, 8192, 2), (672, 8192, 4), (2048, 100_000, 4), (800, 6500, 3), (800, 1000, 0)])
def test_where_a_chunk_makes_tiles(tok, pos0, use):
    # and never in a scratch of a slice less than hipml_attn_chunk_splits says
    lib, splits = attn.lib(), attn.chunk_splits(pos0, tok, N_KV)
    assert lib.hipml_dbg_chunk_makes_tiles(pos0, tok, N_HEAD, N_KV, splits) == use
    assert lib.hipml_dbg_chunk_makes_tiles(pos0, tok, N_HEAD, N_KV, splits - 1) == 0


def test_the_slices_that_run_fit_the_scratch():
    # never more than asked for, never one alone (that is another kernel's sums), and no other count where the blocks fill the
    # chip by themselves
    lib = attn.lib()
    rng = np.random.default_rng(7)
    took = ctypes.c_int()
    for _ in range(3000):
        n_kv = int(rng.integers(1, 9))
        n_head = n_kv * int(rng.integers(1, 9))
        tok, pos0 = (int(np.exp(rng.uniform(0.0, np.log(top)))) for top in (6000, 200_000))
        splits = int(rng.integers(2, 65))
        used = lib.hipml_dbg_chunk_q8_slices(pos0, tok, n_head, n_kv, splits)
        assert 2 <= used <= splits
        over_tiles = lib.hipml_dbg_chunk_f16_slices(pos0, tok, n_head, n_kv, splits, ctypes.byref(took))
        assert 2 <= over_tiles <= splits
        blocks = ((tok + 31) // 32 * (n_head // n_kv) + 7) // 8
        if n_kv * blocks >= 512:
            assert used == over_tiles == splits
        assert lib.hipml_dbg_chunk_wg_splits(pos0, tok, n_head, n_kv, splits) <= splits
