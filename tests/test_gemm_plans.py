"""CPU checks that the shapes of the GEMM's GPU tests get the launches that those tests are for (the planner is host code)."""

import pytest

from gemm_cases import CUS, TILES, gemm_plan, runs


def test_every_tile_is_covered():
    # every tile that the planner ever takes, over rows, columns and K up to those of a prompt chunk
    taken = {gemm_plan(m, 128 * c, 128 * kt).tile for m in (17, 33, 49, 65, 81, 97, 113, 129, 161, 200, 240, 300, 512, 2048)
             for c in (1, 3, 8, 16, 24, 32, 40, 72, 80, 108, 144, 192, 224) for kt in (1, 4, 9, 16, 24, 32, 40, 64, 108, 112)}
    assert taken == set(TILES) == set(range(len(TILES)))


@pytest.mark.parametrize("tile", sorted(TILES))
def test_tile_cases(tile):
    remainders, uneven, split = set(), set(), False
    for m, cols, kt, splits in TILES[tile]:
        p = gemm_plan(m, cols, 128 * kt)
        assert (p.tile, p.splits) == (tile, splits), (m, cols, kt, p)
        r = runs(p, 128 * kt)
        if splits > 1:
            split = True
            assert 0 < p.partial_bytes == splits * m * cols * 4 <= 32 << 20
        elif max(r[0]) > p.buffers:
            (remainders if len(set(r[0])) == 1 else uneven).add(max(r[0]) % p.buffers)
    p = gemm_plan(*TILES[tile][0][:2], 128 * TILES[tile][0][2])
    assert split and remainders == set(range(p.buffers))
    assert uneven == (set(range(p.buffers)) if p.k_groups > 1 else set())


def test_other_files_cases():
    """What the comments of other GPU tests say about a launch."""
    import test_gpu_bounds
    import test_gpu_ffn
    import test_gpu_linear

    for module in (test_gpu_bounds, test_gpu_ffn, test_gpu_linear):
        for m, cols, k, splits in module.GEMM_SPLITS:
            assert gemm_plan(m, cols, k).splits == splits, (module.__name__, m, cols, k)
    assert CUS == 256
