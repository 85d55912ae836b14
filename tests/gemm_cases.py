"""Shapes of the prefill GEMM by the launch that the planner gives them on 256 CUs, for the tests of its kernels: a test cannot
choose a tile, so each shape here is kept with its tile and K splits, and a planner that moves it fails the check of this table."""

import collections
import ctypes

from heteromega_amd import _lib

CUS = 256

Plan = collections.namedtuple("Plan", "tile row_blocks waves k_groups buffers tiles_per_barrier splits partial_bytes")


def gemm_plan(m, cols, k, large_scales=False, cus=CUS):
    """The launch of m rows, cols columns (gate and up of a fused call together) and K = k."""
    out = (ctypes.c_int64 * 8)()
    fn = ctypes.CDLL(_lib.LIB_PATH).hm_gemm_plan_of
    fn.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_int32, ctypes.c_void_p]
    fn.restype = None
    fn(m, cols, k // 128, cus, int(large_scales), out)
    return Plan(*out)


def runs(plan, k):
    """K tiles of each K group of each split."""
    count = plan.splits * plan.k_groups
    base, longer = divmod(k // 128, count)
    sizes = [base + (i < longer) for i in range(count)]
    return [sizes[s * plan.k_groups:(s + 1) * plan.k_groups] for s in range(plan.splits)]


# {tile: [(rows, columns, K tiles, K splits)]}. Per tile: unsplit calls with every remainder of the longest run behind the
# pipeline's loop of as many K tiles as there are LDS buffers (and at least one trip of that loop), K groups of equal and of
# unequal runs for each where there are K groups, and calls with K splits.
TILES = {
    0: [(18, 3968, 24, 1), (17, 1024, 22, 1), (17, 128, 21, 1), (17, 128, 16, 1), (17, 128, 13, 1), (17, 128, 20, 1),
        (17, 128, 17, 1), (31, 5120, 37, 3), (19, 4096, 64, 4)],
    1: [(33, 9216, 24, 1), (33, 9216, 21, 1), (33, 9216, 16, 1), (33, 9216, 13, 1), (33, 9216, 20, 1), (33, 9216, 17, 1),
        (33, 4864, 48, 3)],
    2: [(49, 9216, 32, 1), (49, 9216, 29, 1), (49, 9216, 20, 1), (49, 9216, 19, 1), (49, 9216, 24, 1), (49, 9216, 21, 1),
        (49, 9216, 28, 1), (49, 9216, 25, 1), (51, 5120, 56, 3)],
    3: [(17, 18432, 16, 1), (17, 18432, 15, 1), (17, 18432, 10, 1), (17, 18432, 9, 1), (17, 18432, 12, 1), (17, 18432, 11, 1),
        (17, 18432, 14, 1), (17, 18432, 13, 1), (17, 6656, 37, 4), (17, 6656, 38, 4)],
    4: [(33, 18432, 16, 1), (33, 18432, 15, 1), (33, 18432, 10, 1), (33, 18432, 9, 1), (33, 18432, 12, 1), (33, 18432, 11, 1),
        (33, 18432, 14, 1), (33, 18432, 13, 1), (65, 2816, 48, 5)],
    5: [(49, 18432, 16, 1), (49, 18432, 15, 1), (49, 18432, 10, 1), (49, 18432, 9, 1), (49, 18432, 12, 1), (49, 18432, 11, 1),
        (49, 18432, 14, 1), (49, 18432, 13, 1), (49, 9216, 33, 3), (97, 2432, 56, 6)],
    6: [(65, 18432, 12, 1), (65, 18432, 11, 1), (65, 18432, 8, 1), (65, 18432, 7, 1), (65, 18432, 10, 1), (65, 18432, 9, 1),
        (67, 9216, 39, 3), (65, 3072, 64, 8)],
    7: [(81, 18432, 12, 1), (81, 18432, 11, 1), (81, 18432, 8, 1), (81, 18432, 13, 1), (81, 18432, 10, 1), (81, 18432, 9, 1),
        (81, 9216, 64, 3), (256, 9216, 30, 1)],
    8: [(97, 18432, 16, 1), (97, 18432, 15, 1), (97, 18432, 10, 1), (97, 18432, 17, 1), (97, 18432, 12, 1), (97, 18432, 19, 1),
        (97, 18432, 14, 1), (97, 18432, 13, 1), (97, 5632, 48, 5), (200, 11264, 17, 1)],
    9: [(113, 18432, 16, 1), (113, 18432, 23, 1), (113, 18432, 18, 1), (113, 18432, 25, 1), (113, 18432, 20, 1),
        (113, 18432, 19, 1), (113, 18432, 14, 1), (113, 18432, 21, 1), (113, 9216, 48, 3)],
    10: [(129, 18432, 8, 1), (129, 18432, 5, 1), (129, 18432, 6, 1), (129, 18432, 7, 1), (65, 9216, 39, 7), (65, 11264, 33, 5)],
    11: [(161, 24576, 8, 1), (161, 24576, 5, 1), (161, 24576, 6, 1), (161, 24576, 7, 1), (161, 2816, 64, 11),
        (81, 18432, 27, 3)],
    12: [(200, 24576, 8, 1), (200, 24576, 5, 1), (200, 24576, 6, 1), (200, 24576, 7, 1), (97, 11264, 39, 5), (97, 11264, 40, 5)],
    13: [(240, 24576, 8, 1), (240, 24576, 5, 1), (240, 24576, 6, 1), (240, 24576, 7, 1), (113, 11264, 56, 5),
        (113, 9216, 56, 7)],
    14: [(97, 18432, 8, 1), (65, 18432, 5, 1), (97, 18432, 6, 1), (81, 18432, 7, 1), (97, 2816, 64, 11), (97, 4352, 56, 7)],
}
