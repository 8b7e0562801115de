"""How the front end's launches are laid out (by rows, or flat with the V rows behind) and where long calls are cut into several
launches: the same bits as calls of few rows, and nothing beside the rows."""
import numpy as np
import pytest
import torch

from hipml_amd import attn

HD, N_ROT, THETA, EPS = 256, 64, 1e7, 1e-6


def flat(n_heads, n_kv, rows, append):
    return attn.lib().hipml_dbg_front_flat(n_heads, n_kv, rows, int(append)) != 0


def test_which_launches_are_flat():
    # where a quarter of the waves would have no row
    assert [flat(5, 1, rows, False) for rows in (249, 250, 2048)] == [False, True, True]
    assert [flat(3, 1, rows, True) for rows in (249, 250, 2048)] == [False, True, True]
    assert not any(flat(h, kv, 2048, True) for h, kv in ((24, 4), (48, 8), (28, 2), (32, 8), (16, 2), (14, 2), (5, 1), (2, 1)))
    assert not any(flat(h, kv, 2048, False) for h, kv in ((24, 4), (3, 1), (6, 1)))


@pytest.mark.parametrize("n_heads,n_kv,append", [(4, 1, False), (5, 1, False), (8, 1, False),
                                                 (1, 1, True), (3, 3, True), (6, 1, True), (7, 1, True), (1, 1, False)])
def test_rows_found_by_a_product(n_heads, n_kv, append):
    # every wave of the largest flat launch of these heads: its row is the quotient
    rows = max((r for r in range(1, 32_769) if flat(n_heads, n_kv, r, append)), default=0)
    for d, n in ((n_heads + n_kv, rows), (n_kv, rows)):
        if rows and d > 1:
            waves = np.arange(d * n, dtype=np.uint64)
            inverse = np.uint64((0xFFFFFFFF + d) // d)
            assert int(inverse) < 1 << 32
            assert np.array_equal(waves * inverse >> np.uint64(32), waves // np.uint64(d))


def run(dtype, qg, k, v, qw, kw, n_heads, n_kv, pos0, stride, cuts, caches):
    """The chunk's front end (with append where dtype is not None) as one call per piece between two cuts."""
    rows = qg.shape[0]
    q, gate = (torch.full((rows + 1, n_heads, HD), 7.0, device="cuda") for _ in range(2))
    kd = torch.cat((k, torch.full_like(k[:1], 7.0)))
    kc, vc = (c.clone() for c in caches)
    shape = (n_heads, n_kv, HD, N_ROT, THETA, EPS)
    for a, b in zip(cuts, cuts[1:]):
        if dtype is None:
            attn.chunk_front(qg[a:], kd[a:], q[a:], gate[a:], qw, kw, *shape, pos0 + a, b - a)
        else:
            attn.chunk_front_encode(dtype, qg[a:], kd[a:], v[a:], q[a:], gate[a:], qw, kw, kc, vc, *shape, pos0 + a, b - a, stride)
    torch.cuda.synchronize()
    assert all(bool((t[rows] == 7.0).all()) for t in (q, gate, kd))
    return q, gate, kd, kc, vc


def same(one, many):
    for name, a, b in zip(("q", "gate", "k", "k cache", "v cache"), one, many):
        assert torch.equal(a, b), name


def inputs(n_heads, n_kv, rows, seed):
    attn.init(0)
    attn.rope_table(THETA, N_ROT, 131_072)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    made = [torch.randn(s, device="cuda", generator=gen) for s in ((rows, n_heads, 2 * HD), (rows, n_kv, HD), (rows, n_kv, HD))]
    return made + [1.0 + 0.1 * torch.randn(HD, device="cuda", generator=gen) for _ in range(2)]


# both sides of the rule's line, ragged last workgroups, one and several KV heads
@pytest.mark.gpu
@pytest.mark.parametrize("n_heads,n_kv,rows,dtype,is_flat", [
    (24, 4, 257, 1, False), (5, 1, 249, None, False), (5, 1, 250, None, True), (5, 1, 251, 0, False), (3, 1, 337, 0, True),
    (3, 1, 337, 1, True), (1, 1, 513, 0, True), (2, 2, 513, 1, True), (8, 1, 171, None, True)])
def test_one_launch_has_the_bits_of_small_ones(n_heads, n_kv, rows, dtype, is_flat):
    assert flat(n_heads, n_kv, rows, dtype is not None) == is_flat and not flat(n_heads, n_kv, 47, dtype is not None)
    made = inputs(n_heads, n_kv, rows, rows * 100 + n_heads)
    pos0, stride = 1000, 1000 + rows + 5
    caches = [torch.full((n_kv, stride, 144 if dtype == 1 else 272), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(2)]
    args = (n_heads, n_kv, pos0, stride)
    one = run(dtype, *made, *args, [0, rows], caches)
    same(one, run(dtype, *made, *args, [*range(0, rows, 47), rows], caches))
    if dtype is not None:
        for c in one[3:]:
            assert bool((c[:, :pos0] == 0x5A).all()) and bool((c[:, pos0 + rows:] == 0x5A).all())
            assert not bool((c[:, pos0:pos0 + rows] == 0x5A).all(dim=2).any())


@pytest.mark.gpu
@pytest.mark.parametrize("append", [False, True])
def test_a_chunk_that_leaves_the_table(append):
    # angles of positions past the table are computed on the device, where that is allowed: by rows, whatever the shape
    rows, n_heads, n_kv = (600, 3, 1) if append else (600, 5, 1)
    made = inputs(n_heads, n_kv, rows, 11)
    assert flat(n_heads, n_kv, rows, append)
    pos0, stride = 131_072 - rows + 1, 131_080
    caches = [torch.full((n_kv, stride, 272), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(2)]
    args = (n_heads, n_kv, pos0, stride)
    dtype = 0 if append else None
    with pytest.raises(attn.HipmlError):
        run(dtype, *made, *args, [0, rows], caches)
    attn.rope_allow_device_angles(1)
    try:
        one, many = (run(dtype, *made, *args, cuts, caches) for cuts in ([0, rows], [*range(0, rows, 47), rows]))
    finally:
        attn.rope_allow_device_angles(0)
    same(one, many)
    assert bool(one[0][:rows].isfinite().all())


@pytest.mark.gpu
@pytest.mark.parametrize("n_heads,n_kv,dtype", [(2, 1, 0), (2, 1, None), (1, 1, 1)])
def test_a_chunk_longer_than_a_launch(n_heads, n_kv, dtype):
    rows = 32_770  # a launch holds 32,768: by rows, and flat (one head)
    made = inputs(n_heads, n_kv, rows, 5)
    pos0, stride = 9, 9 + rows + 2
    caches = [torch.full((n_kv, stride, 144 if dtype == 1 else 272), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(2)]
    args = (n_heads, n_kv, pos0, stride)
    same(run(dtype, *made, *args, [0, rows], caches), run(dtype, *made, *args, [0, 20_000, 32_767, rows], caches))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [0, 1])
def test_a_bulk_append_longer_than_a_launch(dtype):
    attn.init(0)
    n_kv, rows, start, src0 = 2, 32_771, 11, 3
    stride, row_bytes = start + rows + 2, 144 if dtype else 272
    k, v = (torch.randn((src0 + rows, n_kv, HD), device="cuda") for _ in range(2))
    whole, pieces = ([torch.full((n_kv, stride, row_bytes), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(2)] for _ in range(2))
    attn.kv_encode_bulk(dtype, k, v, *whole, n_kv, HD, stride, start, src0, rows)
    for a, b in ((0, 16_000), (16_000, 32_767), (32_767, rows)):
        attn.kv_encode_bulk(dtype, k[src0 + a:], v[src0 + a:], *pieces, n_kv, HD, stride, start + a, 0, b - a)
    torch.cuda.synchronize()
    for a, b in zip(whole, pieces):
        assert torch.equal(a, b) and bool((a[:, :start] == 0x5A).all()) and bool((a[:, start + rows:] == 0x5A).all())
        assert not bool((a[:, start:start + rows] == 0x5A).all(dim=2).any())
