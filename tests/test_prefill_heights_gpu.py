"""GPU tests of the four-wave prefill kernel's tile heights and of how the k
slices of a tile finish it together, against the CPU oracle (fp32 sums in
another order: the bounds of test_gemm_gpu.py)."""
import os
import sys

import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))


@pytest.fixture(scope="module")
def env():
    import torch
    import marlin
    assert torch.cuda.is_available()
    return torch, marlin


@pytest.fixture(scope="module")
def problem():
    n, k = 512, 2304  # 36 stages: halves and slices of odd lengths
    out = {}
    for g in (128, -1):
        A, _, _, B, sp = O.make_problem(257, n, k, g, seed=n + g)
        out[g] = (A, B, sp, O.gemm(A, B, sp, n, g))
    return n, k, out


@pytest.mark.parametrize("polls", [-1, 0, 1])  # 0 and 1: shares left to the last arrival
@pytest.mark.parametrize("slices", [1, 2, 3, 5, 6, 8])
@pytest.mark.parametrize("rows", [80, 96, 112, 128])
def test_heights_and_slices(env, problem, rows, slices, polls):
    torch, marlin = env
    n, k, cases = problem
    marlin.force_kernel(2)
    marlin.force_tile_rows(rows)
    marlin.force_k_slices(slices)
    marlin.force_finish_polls(polls)
    dev = torch.device("cuda:0")
    try:
        for g, (A, B, sp, want) in cases.items():
            dA, dB, ds = (torch.from_numpy(x).to(dev) for x in (A, B, sp))
            ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
            for m in (1, rows - 16, rows - 1, rows, rows + 1, 2 * rows + 1):
                _, plan = marlin.plan(m, n, k, g)
                assert (plan["kernel"], plan["tile_rows"], plan["k_slices"]) == (2, rows, slices)
                C = torch.full((m + 1, n), 7.0, dtype=torch.half, device=dev)
                marlin.mul(dA[:m], dB, C[:m], ds, ws)
                again = torch.empty_like(C[:m])
                marlin.mul(dA[:m], dB, again, ds, ws)
                torch.cuda.synchronize()
                assert torch.equal(C[:m], again)
                assert (C[m] == 7.0).all()  # nothing past the last row
                r = O.compare(C[:m].cpu().numpy(), want[:m])
                assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.rel_mean_abs_err <= 1e-3, (g, m)
    finally:
        marlin.force_kernel(0)
        marlin.force_tile_rows(0)
        marlin.force_k_slices(0)
        marlin.force_finish_polls(-1)


@pytest.mark.parametrize("rows", [80, 96, 112])
@pytest.mark.parametrize("groupsize", [128, -1])
def test_dequantised_weights_bit_exact(env, rows, groupsize):
    """One-hot rows return rows of the dequantised weight, every k of both k halves of three
    slices."""
    torch, marlin = env
    n, k = 256, 768
    _, _, _, B, sp = O.make_problem(1, n, k, groupsize, seed=rows)
    W = O.dequant(B, sp, k, n, groupsize)
    if groupsize == -1:
        W = W * O.unpack_scales(sp, False)
    dev = torch.device("cuda:0")
    A = np.eye(k, dtype=np.float16)
    C = torch.empty((k, n), dtype=torch.half, device=dev)
    ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
    marlin.force_kernel(2)
    marlin.force_tile_rows(rows)
    try:
        for slices in (1, 3):
            marlin.force_k_slices(slices)
            marlin.mul(torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev), C,
                       torch.from_numpy(sp).to(dev), ws)
            torch.cuda.synchronize()
            assert np.array_equal(C.cpu().numpy().view(np.uint16), W.view(np.uint16))
    finally:
        marlin.force_kernel(0)
        marlin.force_tile_rows(0)
        marlin.force_k_slices(0)


@pytest.mark.parametrize("m,n,k", [(690, 4608, 4096), (140, 11008, 4864), (565, 1792, 2816), (529, 768, 4992),
                                   (236, 3072, 4352)])
@pytest.mark.parametrize("rows", [0, -1])  # by cost (some of them in whole row blocks, without slices), and in slices
def test_slices_captured_without_scratch(env, rows, m, n, k):
    """Problems that run in slices are captured on a stream that has no scratch, without any:
    nothing is allocated, and the replays are right whatever runs in between.  On a stream
    that has scratch the graph repeats the bits of the eager call."""
    torch, marlin = env
    marlin.force_rows(rows)
    try:
        assert rows == 0 or marlin.rows_plan(m, n, k, 128) is None
        _captured_without_scratch(torch, marlin, m, n, k)
    finally:
        marlin.force_rows(0)


def _captured_without_scratch(torch, marlin, m, n, k):
    dev = torch.device("cuda:0")
    assert marlin.plan(m, n, k, 128)[1]["k_slices"] > 1
    A, _, _, B, sp = O.make_problem(m, n, k, 128, seed=m)
    dA, dB, ds = (torch.from_numpy(x).to(dev) for x in (A, B, sp))
    ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
    eager = torch.empty((m, n), dtype=torch.half, device=dev)
    marlin.mul(dA, dB, eager, ds, ws)
    torch.cuda.synchronize()
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int))
    want = O.gemm(A[rows], B, sp, n, 128)
    marlin.release()  # (a new stream may have the handle of one that had scratch)
    cold, warm = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(warm):
        marlin.mul(dA, dB, eager, ds, ws)
    torch.cuda.synchronize()
    held = marlin.scratch_bytes()
    for side in (cold, warm):
        C = torch.zeros_like(eager)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            marlin.mul(dA, dB, C, ds, ws)
        assert marlin.scratch_bytes() == held
        for _ in range(3):
            C.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert side is cold or torch.equal(C, eager)
            r = O.compare(C[rows].cpu().numpy(), want)
            assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.rel_mean_abs_err <= 1e-3
            marlin.mul(dA[:17], dB, torch.empty((17, n), dtype=torch.half, device=dev), ds, ws)
        held = marlin.scratch_bytes()
        del graph
