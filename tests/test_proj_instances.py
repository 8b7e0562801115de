"""That tests/proj_instances.py names a shape for every variant of the projection kernels that any call can take."""
import pytest

import proj_instances as inst

M = sorted({*range(1, 400, 13), *range(400, 20_000, 197), *range(20_000, 130_000, 7_777), 1024, 1345, 2048, 5120, 6144, 12_288})


@pytest.mark.parametrize("k", [64, 256, 1088, 1280, 5120, 32_768, 34_560, 36_096])
def test_every_row_kernel_has_a_shape(k):
    named = {inst.row_variant(*shape) for shape in inst.ROWS}
    assert len(named) == len(inst.ROWS)
    named |= {inst.row_variant(*shape) for shape in inst.WIDE}
    taken = {inst.row_variant(m, k, rows): (m, rows) for m in M for rows in range(1, 129)}
    assert not {c: s for c, s in taken.items() if c not in named}


@pytest.mark.parametrize("x16", [0, 1])
@pytest.mark.parametrize("k", [64, 128, 1024])
def test_every_tile_has_a_shape(k, x16):
    named = {(inst.gemm_tile(m, k_, t, h), h) for m, k_, t, h in inst.TILES}
    assert len(named) == len(inst.TILES)
    tokens = [*range(1, 700, 17), *range(700, 4200, 83)]
    taken = {(inst.gemm_tile(m, k, t, x16), x16): (m, t) for m in M for t in tokens}
    assert not {c: s for c, s in taken.items() if c not in named}


def test_every_packed_tile_has_a_shape():
    named = {inst.gemm_choice(*shape) for shape in inst.PACKED}
    assert len(named) == len(inst.PACKED) and min(named) >= 300
    tokens = [*range(1, 700, 17), *range(700, 4200, 83)]
    taken = {inst.gemm_choice(m, k, t, g): (m, k, t, g) for m in M for t in tokens for k in (1024, 5120) for g in (0, 1, 2)}
    assert not {c: s for c, s in taken.items() if c >= 300 and c not in named}


@pytest.mark.parametrize("m,k", [(12_288, 5120), (1024, 5120), (5120, 6144)])
def test_the_models_projections_are_among_them(m, k):
    named = {inst.row_variant(*shape) for shape in inst.ROWS + inst.WIDE}
    assert all(inst.row_variant(m, k, rows) in named for rows in range(1, 129))


@pytest.mark.parametrize("k", [256, 4864, 5120, 6144, 8192])
@pytest.mark.parametrize("rows", [5, 6, 7, 8])
def test_weights_that_fill_the_chip_are_read_once_for_five_to_eight_rows(k, rows):
    # two passes of four rows over these take the chip twice: 1.3 to 1.6 times one pass of eight
    for m in (6145, 7168, 8192, 10_240, 11_264, 12_288 if k <= 6144 else 11_200):
        assert inst.row_kernel(m, k, rows) // 10_000 == 108, m
