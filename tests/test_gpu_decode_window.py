"""Batched decode, a window of workers: a worker takes whole turns of its four waves (128 rows) where the batch has an item of at
most eight columns, any number of tiles of 32 rows where every item is wider.  Depths around both, against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import binding as orc  # noqa: E402
from hipml_amd import attn  # noqa: E402
from gpu_util import N_HEADS, HD, SCALE, dev, host, decode_scratch, report  # noqa: E402
from test_gpu_decode import KERNEL_CLASS  # noqa: E402


@pytest.mark.parametrize("depths,cols", [
    ((1, 32, 33, 127, 128, 129), (1,) * 6),       # at most one turn each
    ((4100, 2048, 1), (1, 1, 1)),                 # several workers a slot, and a slot of one key
    ((3969, 640, 2100, 97), (3, 1, 3, 1)),        # wide and narrow items
    ((3969, 4095), (3, 3))])                      # wide items alone
def test_whole_turns(depths, cols):
    attn.init(0)
    n_kv, slots = 4, len(depths)
    stride = max(depths) + 5
    r = orc.Rng(0x7D2A + sum(depths))
    kb = orc.quantize(0, r.normal_array((slots, n_kv, stride, HD))).reshape(slots, n_kv, stride, -1)
    vb = orc.quantize(0, r.normal_array((slots, n_kv, stride, HD))).reshape(slots, n_kv, stride, -1)
    pos = [(d + c - 1, d + c) for d, n in zip(depths, cols) for c in range(n)]
    slot_of = [s for s, n in enumerate(cols) for _ in range(n)]
    rows = len(pos)
    splits = attn.batch_splits(stride, n_kv, slots)
    q = r.normal_array((rows, N_HEADS, HD))
    kd, vd, qd = dev(kb), dev(vb), dev(q)
    acc, ml = decode_scratch(N_HEADS, splits, rows)
    acc.fill_(float("nan")), ml.fill_(float("nan"))
    out = torch.full((rows, N_HEADS, HD), float("nan"), device="cuda")
    attn.attn_decode_batch_cols(0, torch.tensor(pos, dtype=torch.int32, device="cuda"), qd, kd, vd, acc, ml, out, N_HEADS, n_kv,
                                HD, stride, SCALE, splits, kd[0].numel(), N_HEADS * splits * HD, N_HEADS * splits * 2,
                                N_HEADS * HD, list(cols))
    torch.cuda.synchronize()
    got = host(out)
    for i in range(rows):
        want = orc.attn_decode_kv(q[i], kb[slot_of[i]], vb[slot_of[i]], N_HEADS, n_kv, HD, pos[i][1], SCALE, stride=stride)
        assert report(f"row {i}, {pos[i][1]} keys", want.ravel(), got[i].ravel(), *KERNEL_CLASS)[0]
    assert np.isfinite(got).all()
