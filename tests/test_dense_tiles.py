"""Dense GEMM on tiles of many sizes: where they are chosen (CPU), and the
kernel at the edges of its tiles, stages and slices (GPU; whole numbers whose sums
are exact in fp16 and in any order, so the result is torch's fp32 product, bit for
bit)."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))

CUT = [(32, 32), (32, 64), (64, 64), (64, 128)]  # whole or in slices
TILES = CUT + [(96, 128), (64, 192), (96, 192), (128, 192), (96, 256), (128, 256)]


@pytest.mark.parametrize("cus", [256, 304, 64])
def test_tiles_stand_in_for_one_launch(cus):
    import numpy as np
    import streamk
    rng = np.random.default_rng(cus)
    seen = set()
    for _ in range(6000):
        m, n = int(2 ** rng.uniform(0, 13)), 256 * int(2 ** rng.uniform(0, 5.3))
        k = 64 * int(2 ** rng.uniform(0, 7.5))
        t, (_, p) = streamk.tile(m, n, k, cus), streamk.plan(m, n, k, cus)
        if t is None:
            continue
        seen.add(t[:2])
        rows, cols, slices = t
        tiles = -(-m // rows) * -(-n // cols)
        assert (rows, cols) in TILES and tiles <= 4 * cus
        assert len(streamk.launches(m, n, k, cus)) == 1 and streamk.launches(m, n, k, cus)[0]["slices"] == p["k_slices"]
        assert slices in (1, 2, 4) and slices <= p["k_slices"]
        if slices > 1:  # the plan's scratch holds their sums and counters
            assert (rows, cols) in CUT and p["tile_cols"] == 128
            assert tiles * slices <= cus and tiles <= 1024
            assert tiles * rows * cols * slices <= p["sk_tiles"] * 128 * 128 * p["k_slices"]
    assert len(seen) >= 9
    assert streamk.tile(4096, 4352, 4096) is None and streamk.tile(777, 4352, 10240) is None


@pytest.mark.parametrize("m,n,k,slower", [
    (576, 1536, 4544, (64, 64, 1)), (240, 3328, 4096, (64, 64, 1)),
    (130, 7424, 3328, (64, 64, 1)), (265, 3840, 3072, (64, 64, 1)), (172, 5376, 9920, (64, 64, 1)),
    (1486, 5376, 3008, (128, 256, 1)), (4798, 2048, 128, (96, 256, 1)), (1703, 10752, 128, (128, 256, 1)),
    (586, 768, 16256, (64, 128, 4)), (449, 1024, 6208, (64, 128, 4))])
def test_tiles_that_were_slower_are_not_taken(m, n, k, slower):
    """Sizes at which a tile took 1.05 to 1.3 times the best one or the plan's launch, most of them by
    a choice that knew only operands in the last-level cache."""
    import streamk
    assert streamk.tile(m, n, k) != slower


def _check(m, n, k, top):
    import torch
    import streamk
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(m + n + k)
    A, B = (torch.randint(-top, top + 1, (r, k), device="cuda:0", generator=gen).half() for r in (m, n))
    C = torch.full((m + 1, n), 7.0, dtype=torch.half, device="cuda:0")
    streamk.gemm(A, B, C[:m])
    want = A.float() @ B.float().t()
    torch.cuda.synchronize()
    assert want.abs().max().item() < 2048
    assert torch.equal(C[:m].float(), want)
    assert (C[m] == 7.0).all()  # nothing past the last row


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m", [1, 31, 65, 200])
def test_stages(tile, m):
    """One stage to past the end of the longest ring, even and odd, and columns that 192 does
    not divide."""
    import streamk
    streamk.force_tile(*tile)
    try:
        for stages in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11):
            _check(m, 512, 64 * stages, 1)
        _check(m, 256, 320, 1)
        _check(m, 1536, 320, 1)
    finally:
        streamk.force_tile(0)


@pytest.mark.gpu
@pytest.mark.parametrize("polls", [-1, 0, 1])  # 0 and 1: shares left to the last arrival
@pytest.mark.parametrize("tile", CUT + [(-1, 0)])
@pytest.mark.parametrize("m,n,k,slices", [(33, 256, 1024, 4), (100, 512, 1344, 4), (129, 512, 832, 3), (300, 1280, 576, 2)])
def test_slices(tile, m, n, k, slices, polls):
    """Slices of equal and unequal length; (-1, 0): the 128 x 128 tiles they stand in for."""
    import streamk
    streamk.force_tile(*tile, slices)
    streamk.force_finish_polls(polls)
    try:
        if tile[0] > 0:
            assert streamk.tile(m, n, k) == tile + (slices,)
        for _ in range(2):
            _check(m, n, k, 1)
    finally:
        streamk.force_finish_polls(-1)
        streamk.force_tile(0)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(64, 512, 512), (291, 1280, 896), (100, 512, 10240), (777, 2048, 1024), (1514, 3072, 1600),
                                   (885, 6912, 704), (701, 5632, 832)])
def test_chosen_tiles(m, n, k):
    import streamk
    assert streamk.tile(m, n, k) is not None
    _check(m, n, k, 1)
