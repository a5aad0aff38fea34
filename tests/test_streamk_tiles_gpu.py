"""GPU tests of the dense GEMM's kernels at the edges of their tiles, stages and
slices.  Operands are whole numbers in [-2, 2] and at most 448 deep, so every sum
stays below 2048 in magnitude and is exact in fp16 and in any order of addition:
the result is torch's fp32 product, bit for bit.  (Deeper sums, for slices, use
{-1, 0, 1}.)"""
import os
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))


@pytest.fixture(scope="module")
def env():
    import torch
    import streamk
    assert torch.cuda.is_available()
    return torch, streamk


@pytest.fixture(autouse=True)
def planned(env):
    """The plan's own launches, also where tiles of other sizes would be taken."""
    env[1].force_tile(-1)
    yield
    env[1].force_tile(0)


def _check(env, m, n, k, top, tile):
    torch, streamk = env
    assert streamk.tile(m, n, k) is None
    _, plan = streamk.plan(m, n, k)
    assert (plan["tile_rows"], plan["tile_cols"]) == tile
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
    return plan


# one stage to seven: every place where the loops of two and of six slabs are left
@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("m,n,tile", [(1281, 8192, (256, 256)), (1535, 6400, (256, 256)), (601, 8192, (128, 256)),
                                      (767, 5632, (128, 256)), (1, 256, (128, 128)), (300, 1024, (128, 128))])
def test_stages(env, m, n, stages, tile):
    assert env[1].launches(m, n, 64 * stages)[0] == {
        "rows": tile[0], "cols": tile[1], "waves": 8, "slices": 1,
        "tiles": -(-m // tile[0]) * (n // tile[1])}
    _check(env, m, n, 64 * stages, 2, tile)


# ... and over a deeper k, in the loops of four waves (all but the last)
@pytest.mark.parametrize("stages", [0, 1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("m,n,k,tile", [(1999, 8192, 768, (256, 256)), (1535, 6400, 2048, (256, 256)),
                                        (1001, 8192, 3072, (128, 256)), (767, 5632, 4096, (128, 256)),
                                        (1300, 3328, 6144, (128, 256)),  # 143 tiles, dealt out one by one
                                        (1076, 7424, 5120, (256, 256))])
def test_deep_stages(env, m, n, k, stages, tile):
    assert env[1].launches(m, n, k + 64 * stages)[0]["waves"] == (8 if m == 1076 else 4)
    _check(env, m, n, k + 64 * stages, 1, tile)


@pytest.mark.parametrize("polls", [-1, 0, 1])  # 0 and 1: shares left to the last arrival
@pytest.mark.parametrize("m,n,k,tile", [
    (2049, 8192, 1024, (256, 256)),   # 32 stream-K tiles in quarters, most of them with one row or none
    (2100, 8192, 1088, (256, 256)),   # ... 52 rows; slices of unequal length
    (4000, 4352, 832, (256, 256)),    # 16 tiles, 64 quarters, up to three slices
    (129, 256, 512, (128, 128)), (300, 1280, 768, (128, 128)), (128, 512, 1216, (128, 128)),
    (5000, 512, 576, (128, 128)),     # whole tiles only
    (777, 4352, 7232, (128, 128)),    # 119 tiles of 128 x 256 in two slices of unequal length, 9 rows in the last
    (2048, 2048, 7168, (128, 128)), (129, 16384, 7232, (128, 128)),
])
def test_slices(env, m, n, k, tile, polls):
    import marlin
    torch, streamk = env
    first = streamk.launches(m, n, k)[0]
    sliced = first["slices"] > 1
    assert sliced == (m != 5000) and (first["rows"], first["cols"]) == ((128, 256) if k >= 7168 else (128, 128))
    marlin.release()
    streamk.force_finish_polls(polls)
    try:
        for _ in range(2):
            _check(env, m, n, k, 1, tile)
    finally:
        streamk.force_finish_polls(-1)
    # the slices' sums had their room: nothing ran in the place of the launch above
    sums = first["tiles"] * first["slices"] * first["rows"] * first["cols"] * 4
    assert (marlin.scratch_bytes()[0] >= sums) if sliced else marlin.scratch_bytes() == (0, 0)


def test_deep_tiles_under_capture(env):
    """Sizes that run in slices outside a capture are captured on a stream without scratch."""
    torch, streamk = env
    m, n, k = 777, 4352, 7168
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(5)
    A, B = (torch.randint(-1, 2, (r, k), device="cuda:0", generator=gen).half() for r in (m, n))
    C = streamk.gemm(A, B)
    want = A.float() @ B.float().t()
    assert torch.equal(C.float(), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        streamk.gemm(A, B, C)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C.float(), want)
        assert torch.equal(streamk.gemm(A, B).float(), want)


@pytest.mark.parametrize("m,n,k", [(777, 4352, 7232), (2048, 2048, 7168), (129, 16384, 7232), (1000, 4096, 10304)])
def test_deep_tiles_have_the_same_bits_under_capture(env, m, n, k):
    """In two slices outside a capture and whole within one: the sums are added up in the same order."""
    torch, streamk = env
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(k)
    A, B = (torch.randn((r, k), device="cuda:0", generator=gen).half() for r in (m, n))
    want = streamk.gemm(A, B)
    C = torch.zeros_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        streamk.gemm(A, B, C)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)
        assert torch.equal(streamk.gemm(A, B), want)
