"""Shapes that between them run every variant of the projection kernels, as the library itself names the variant a call
takes (test_proj_instances.py holds that none is missing, test_gpu_proj_instances.py runs them)."""
from hipml_amd import attn


def row_kernel(m, k, rows):
    """kernel * 10^6 + a * 10^4 + b * 100 + c: 0 the row kernel, 1 digits (activation rows a pass, weight rows of a group), 2
    blocks and 3 units (activation tiles, weight rows, last tile half dead); W at a 16-byte boundary."""
    return attn.lib().hipml_dbg_rows_kernel(m, k, rows, 1)


def row_variant(m, k, rows):
    """The same with what the code leaves out: the kernel that streams units takes its weights by 16-byte requests where k is of
    whole 256-value chunks, by dwords elsewhere."""
    kernel = row_kernel(m, k, rows)
    return kernel, kernel // 1_000_000 == 3 and k % 256 == 0


def gemm_tile(m, k, tokens, x16):
    """(place in the table of tiles, whole sectors of weights), W at a 64-byte boundary."""
    sectors = int(k % 1024 == 0)
    return attn.lib().hipml_dbg_gemm_tile(m, k, tokens, sectors, x16), sectors


def gemm_choice(m, k, tokens, rows):
    """100 * route (1 the rows as they lie, 2 f16 row by row, 3 packed) + place in the route's table of tiles, for a call with
    scratch over f32 rows (0), f32 rows with a gate (1) or f16 rows (2), W at a 64-byte boundary."""
    return attn.lib().hipml_dbg_gemm_choice(m, k, tokens, int(k % 1024 == 0), rows)


# (weight rows, k, activation rows): ragged in the rows of a workgroup, k of 19 chunks or 37 units (uneven shares of the
# waves, several turns of every ring, a last run of one chunk), more runs than waves, one chunk in all
ROWS = [
    (3, 2368, 1), (3, 34560, 1), (1032, 32768, 1), (5117, 4864, 1), (1003, 2560, 2), (5180, 4864, 2), (2069, 4864, 2),
    (3, 4864, 3), (1032, 4864, 3), (2069, 4864, 3), (12281, 4864, 3), (1003, 34560, 4), (597, 4864, 5), (5117, 6144, 4),
    (12281, 4864, 4), (12281, 4864, 5), (8190, 8448, 7), (9973, 5120, 8), (6156, 4864, 9), (8230, 4864, 9),
    (6156, 4864, 25), (6156, 4864, 17), (8230, 4864, 25), (8230, 4864, 17), (6156, 4864, 41), (6156, 4864, 33),
    (8230, 4864, 41), (8230, 4864, 33), (6156, 4864, 57), (6156, 4864, 49), (8230, 4864, 57), (8230, 4864, 49),
    (3, 2368, 9), (3, 2368, 3), (2069, 2368, 17), (4143, 2368, 3), (2618, 2368, 17), (5180, 2368, 3),
    (3106, 2368, 17), (6156, 2368, 3), (8230, 2368, 9), (8230, 2368, 3), (2069, 2368, 49), (1345, 2368, 81), (773, 1280, 115), (4143, 2368, 17),
    (2740, 2368, 33), (5180, 2368, 17), (4082, 2368, 33), (6156, 2368, 17), (4143, 2368, 33), (8230, 2368, 17),
]
# And of every tile of the kernel that streams units by 16-byte requests (k of whole 256-value chunks, one among them): ragged in
# both directions, several workgroups of 8 and of 24 rows, waves with no unit or uneven shares
WIDE = [
    (3, 256, 9), (1003, 1280, 30), (2069, 1280, 31), (517, 1280, 125), (5180, 4864, 16), (645, 1280, 115), (771, 1280, 127),
    (517, 1280, 115), (1029, 1280, 125), (1349, 1280, 81), (773, 1280, 115), (1637, 1280, 65), (1029, 1280, 115),
    (1541, 1280, 125), (1541, 1280, 115), (261, 1280, 125), (2053, 256, 125), (2053, 1280, 97), (5117, 4864, 24), (5117, 4864, 70),
]
# (weight rows, k, tokens, f16 activations)
TILES = [
    (12380, 704, 580, 0), (10996, 704, 258, 0), (10996, 704, 143, 0), (239, 1408, 51, 0), (239, 704, 51, 0),
    (12380, 704, 649, 1), (10996, 704, 258, 1), (7190, 704, 212, 1), (239, 1408, 51, 1), (239, 704, 51, 1),
    (239, 5120, 51, 0), (2173, 3072, 97, 0), (5460, 3072, 74, 0), (12380, 3072, 74, 0), (10996, 3072, 143, 0),
    (6671, 3072, 534, 0), (10996, 3072, 258, 0), (12380, 3072, 396, 0), (12380, 3072, 649, 0), (8228, 3072, 74, 0),
    (1069, 3072, 210, 0),
    (239, 1024, 51, 1), (2173, 3072, 97, 1), (7363, 3072, 97, 1), (10996, 3072, 258, 1), (10996, 3072, 396, 1),
    (12380, 3072, 396, 1), (7363, 3072, 985, 1), (10996, 3072, 143, 1), (1069, 3072, 210, 1), (7363, 3072, 210, 1),
]
# (weight rows, k, tokens, rows as above): calls with scratch whose rows are packed, every tile of that kernel once
PACKED = [
    (5522, 1024, 69, 1), (8280, 3072, 69, 0), (12380, 2048, 69, 1), (16554, 1024, 69, 1), (8280, 1024, 137, 1),
    (16554, 1024, 137, 1), (12380, 2048, 273, 0), (12380, 3072, 137, 1), (8280, 2048, 392, 1), (12380, 2048, 392, 2),
    (16554, 2048, 273, 0), (10996, 2048, 789, 0),
]
