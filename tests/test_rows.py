"""Column strips with up to 64 rows per workgroup: where they are chosen (CPU), and the
kernel at the edges of its strip sets, row blocks and k range (GPU) -- the oracle at the
tolerance of the other kernels (one fp16 rounding of weights and result, fp32 sums:
max|C - C_ref| <= 1e-2 max|C_ref|, mean 1e-3, as in test_gemm_gpu.py) and, with one-hot
rows, the dequantised weights bit for bit."""
import os
import sys

import numpy as np
import pytest

import _oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))

PAIRS = [(1, 1), (2, 1), (3, 1), (2, 2), (3, 2), (4, 2), (6, 2), (2, 3), (3, 3), (4, 3), (5, 3), (6, 3),
         (4, 4), (5, 4), (6, 4), (8, 2), (8, 3), (8, 4)]
CASES = [(pair, g) for pair in PAIRS for g in (128, -1) if (pair, g) != ((4, 4), -1)]


@pytest.mark.parametrize("groupsize", [128, -1])
def test_where_the_rows_stay_together(groupsize):
    import marlin
    rng = np.random.default_rng(1)
    seen = set()
    for _ in range(60000):
        m, n, k = int(2 ** rng.uniform(0, 11)), 256 * int(2 ** rng.uniform(0, 6.8)), 128 * int(2 ** rng.uniform(0, 7))
        t = marlin.rows_plan(m, n, k, groupsize)
        if t is None:
            continue
        strips, rows = t
        seen.add((strips, rows // 16))
        assert m > 16 and k >= (640 if rows > 16 else 2048) and ((strips, rows // 16), groupsize) in CASES
        assert rows == 16 or m > rows - 16
        assert -(-(n // 16) // strips) * -(-m // rows) <= 2.7 * 256
    if groupsize == 128:
        assert marlin.rows_plan(491, 2048, 5760, 128) == (4, 64)  # (one problem in a thousand)
        seen.add((4, 4))
    assert sorted(seen) == sorted(pair for pair, g in CASES if g == groupsize)  # none that nothing reaches
    for pair in ((7, 4), (4, 4)):  # what does not exist cannot be forced
        marlin.force_rows(*pair)
        try:
            forced = marlin.rows_plan(64, 4096, 4096, groupsize) == (pair[0], 16 * pair[1])
            assert forced == ((pair, groupsize) in CASES)
        finally:
            marlin.force_rows(0)
    for m, n, k in [(16, 4096, 4096), (2048, 4096, 4096), (64, 4096, 512)]:
        assert marlin.rows_plan(m, n, k, groupsize) is None
    # an override of the plan is an override of this choice, too
    assert marlin.rows_plan(46, 18432, 4480, groupsize) is not None
    for force, off in [(marlin.force_kernel, 0), (marlin.force_strips, 0), (marlin.force_k_slices, 0),
                       (marlin.force_tile_rows, 0), (marlin.force_row_halves, 0), (marlin.force_finish_polls, -1)]:
        force(64 if force is marlin.force_tile_rows else 1)
        try:
            assert marlin.rows_plan(46, 18432, 4480, groupsize) is None
        finally:
            force(off)


@pytest.mark.parametrize("m,n,k,groupsize", [(1015, 256, 7296, -1), (1531, 512, 8448, 128), (2008, 512, 5888, 128), (1229, 256, 10496, 128),
                                              (1316, 512, 5504, -1), (1654, 1024, 5504, 128), (123, 6912, 1280, 128),
                                              (161, 5376, 1280, 128), (64, 25600, 1280, 128)])
def test_not_where_it_was_slower(m, n, k, groupsize):
    """Sizes at which the kernel took 1.09 to 1.47 times the plan's launch."""
    import marlin
    assert marlin.rows_plan(m, n, k, groupsize) is None


@pytest.mark.parametrize("m,n,k,groupsize,kernel", [
    (15, 18176, 4608, -1, 1), (14, 21504, 6656, -1, 1), (16, 16640, 4224, -1, 1), (10, 512, 13184, -1, 1),
    (13, 5888, 4992, 128, 3), (14, 2048, 5504, -1, 3), (9, 3072, 6912, -1, 3), (10, 768, 7296, 128, 3), (9, 512, 8192, -1, 3)])
def test_few_rows_take_the_faster_kernel(m, n, k, groupsize, kernel):
    """Sizes at which streaming (1) or column strips (3) took 1.08 to 1.19 times the other's time."""
    import marlin
    assert marlin.plan(m, n, k, groupsize)[1]["kernel"] == kernel


@pytest.mark.parametrize("m,n,k,groupsize", [(47, 7168, 9472, 128), (48, 7168, 9984, 128), (46, 7424, 11776, -1),
                                              (46, 7936, 11008, 128), (44, 7168, 11648, 128), (1342, 512, 6400, 128)])
def test_a_deep_k_streams(m, n, k, groupsize):
    """Sizes at which the kernel took 1.10 to 1.21 times the plan's launch: 33 to 48 rows over a
    deep k, where the streaming kernel's fit reads high, and rows far beyond an XCD's L2."""
    import marlin
    assert marlin.rows_plan(m, n, k, groupsize) is None


@pytest.mark.parametrize("m,n,k,groupsize", [(96, 4096, 4096, 128), (128, 4096, 4096, 128), (64, 8192, 4096, 128),
                                              (141, 3840, 1536, 128), (179, 3072, 1536, 128), (36, 12288, 1280, 128)])
def test_where_the_plan_was_slower(m, n, k, groupsize):
    """Sizes at which the plan's launch took 1.2 times the kernel's time and more, three of them
    of ten and twelve groups."""
    import marlin
    assert marlin.rows_plan(m, n, k, groupsize) is not None


@pytest.mark.parametrize("m,n,k,groupsize", [(64, 28672, 8192, 128), (45, 12288, 4096, -1), (144, 2048, 1792, 128),
                                             (491, 2048, 5760, 128)])
def test_the_probes_follow_this_kernel(m, n, k, groupsize):
    """The floor beside a problem is that of the launch that computes it."""
    import marlin
    strips, rows = marlin.rows_plan(m, n, k, groupsize)
    parts = -(-m // rows)
    assert marlin.probe_split(m, n, k, groupsize) == {
        "kernel": 4, "grid": -(-(n // 16) // strips) * parts, "strips": strips, "row_parts": parts,
        "granules_per_wg": 0, "wgs_per_tile": 0}
    marlin.force_rows(-1)
    try:
        assert marlin.probe_split(m, n, k, groupsize)["kernel"] in (1, 3)
    finally:
        marlin.force_rows(0)


def _gemm(A, B, s, n):
    import torch
    import marlin
    dev = torch.device("cuda:0")
    m = A.shape[0]
    C = torch.full((m + 1, n), 7.0, dtype=torch.half, device=dev)
    ws = torch.zeros(max(n // 128, 1) * 16, dtype=torch.int, device=dev)
    marlin.mul(torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev), C[:m], torch.from_numpy(s).to(dev), ws)
    torch.cuda.synchronize()
    assert (C[m] == 7.0).all() and not ws.any().item()  # nothing past the last row
    return C[:m].cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("pair,groupsize", CASES)
def test_rows_against_the_oracle(pair, groupsize):
    """Row counts around a workgroup's, strip sets that do and do not divide the columns, and k
    ranges of one chunk per wave, fewer, and an uneven number."""
    import marlin
    strips, blocks = pair
    marlin.force_rows(strips, blocks)
    try:
        assert marlin.rows_plan(17, 256, 512, groupsize) == (strips, 16 * blocks)
        for m in (17, 16 * blocks + 1, 32 * blocks, 70):
            for n, k in ((256, 512), (768, 1152), (1024, 2688 if groupsize == 128 else 2624)):
                A, q, s, B, sp = O.make_problem(m, n, k, groupsize, seed=m + n + k)
                r = O.compare(_gemm(A, B, sp, n), O.gemm(A, B, sp, n, groupsize))
                assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.cosine >= 0.9999, (m, n, k, r)
    finally:
        marlin.force_rows(0)


@pytest.mark.gpu
@pytest.mark.parametrize("pair,groupsize", CASES)
def test_rows_return_dequantised_weights(pair, groupsize):
    import marlin
    strips, blocks = pair
    n, k, m = 512, 640, 64
    _, q, s, B, sp = O.make_problem(1, n, k, groupsize, seed=strips + blocks)
    W = O.dequant(B, sp, k, n, groupsize)
    if groupsize == -1:
        W = W * O.unpack_scales(sp, False)  # fp16(q-8) * s, one rounding
    marlin.force_rows(strips, blocks)
    try:
        for base in range(0, k, m):
            A = np.zeros((m, k), np.float16)
            A[np.arange(m), base + np.arange(m)] = 1.0
            assert np.array_equal(_gemm(A, B, sp, n).view(np.uint16), W[base:base + m].view(np.uint16)), base
    finally:
        marlin.force_rows(0)


@pytest.mark.gpu
@pytest.mark.parametrize("pair,groupsize", CASES)
def test_rows_of_few_chunks(pair, groupsize):
    """From no chunk of 64 k-values in most waves to two, three and four in each: the last two
    are steps of their own.  One row part and several."""
    import marlin
    marlin.force_rows(*pair)
    try:
        for k in (256, 384, 512, 1024, 1408, 1536, 2048) + (() if groupsize == 128 else (128, 192, 576, 1088, 1600)):
            for m in (17, 16 * pair[1] + 3):
                A, q, s, B, sp = O.make_problem(m, 256, k, groupsize, seed=m + k)
                r = O.compare(_gemm(A, B, sp, 256), O.gemm(A, B, sp, 256, groupsize))
                assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.cosine >= 0.9999, (m, k, r)
    finally:
        marlin.force_rows(0)


@pytest.mark.gpu
@pytest.mark.parametrize("pair,k", [((8, 3), 5120), ((8, 3), 5888), ((8, 4), 3072), ((8, 4), 3200), ((8, 4), 4096), ((8, 4), 4736), ((8, 4), 8192)])
@pytest.mark.parametrize("groupsize", [128, -1])
def test_rows_over_a_deep_k(pair, k, groupsize):
    """From where weights are requested three chunks ahead: chunks per wave that the ring of
    three does and does not divide and that differ between waves, ragged rows, one-hot rows."""
    import marlin
    n = 512
    if groupsize == -1 and k % 1024:
        k -= 64  # an odd number of chunks
    marlin.force_rows(*pair)
    try:
        for m in (33, 16 * pair[1], 100):
            A, q, s, B, sp = O.make_problem(m, n, k, groupsize, seed=m + k)
            r = O.compare(_gemm(A, B, sp, n), O.gemm(A, B, sp, n, groupsize))
            assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.rel_mean_abs_err <= 1e-3, (m, r)
        W = O.dequant(B, sp, k, n, groupsize)
        if groupsize == -1:
            W = W * O.unpack_scales(sp, False)  # fp16(q-8) * s, one rounding
        rows = np.random.default_rng(k).permutation(k)[:200]
        one = np.zeros((len(rows), k), np.float16)
        one[np.arange(len(rows)), rows] = 1.0
        assert np.array_equal(_gemm(one, B, sp, n).view(np.uint16), W[rows].view(np.uint16))
    finally:
        marlin.force_rows(0)


@pytest.mark.gpu
def test_probes_of_every_pair_run():
    import torch
    import marlin
    n, k = 1280, 1152
    B = torch.randint(-2**31, 2**31 - 1, (k // 16, 2 * n), dtype=torch.int32, device="cuda:0")
    for (strips, blocks), g in CASES:
        marlin.force_rows(strips, blocks)
        try:
            assert marlin.probe_split(70, n, k, g)["kernel"] == 4
            for kind in (0, 1):
                marlin.probe(kind, B, n, k, 70, g)
        finally:
            marlin.force_rows(0)
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,g", [(46, 18432, 4480, 128), (45, 12288, 4096, -1), (144, 2048, 1792, 128), (111, 512, 4992, 128)])
def test_chosen_and_captured(m, n, k, g):
    """By cost, against fp32 of the same weights; twice the same bits, in a replayed graph too."""
    import torch
    import marlin
    assert marlin.rows_plan(m, n, k, g) is not None
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(m)
    q = torch.randint(0, 16, (k, n), dtype=torch.int32, device=dev, generator=gen)
    s = (torch.rand((1 if g == -1 else k // g, n), device=dev, generator=gen) * 0.019 + 0.001).half()
    A = torch.randn((m, k), device=dev, generator=gen).half()
    B, sp = marlin.pack_weights(q), marlin.pack_scales(s, g != -1)
    ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
    C = torch.zeros((m, n), dtype=torch.half, device=dev)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        marlin.mul(A, B, C, sp, ws)
        side.synchronize()
        want = C.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            marlin.mul(A, B, C, sp, ws)
    ref = A.float() @ ((q - 8).float() * s.float().repeat_interleave(k // s.shape[0], 0))
    assert (want.float() - ref).norm() <= 1.2e-3 * ref.norm()
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)
        marlin.mul(A, B, C, sp, ws)
        torch.cuda.synchronize()
        assert torch.equal(C, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,g", [(10, 768, 11392, 128), (16, 4096, 11008, 128), (9, 512, 12288, -1), (17, 16128, 2176, 128)])
def test_few_rows_captured_without_scratch(m, n, k, g):
    """Problems that the streaming kernel shares out are captured on a stream that has no
    scratch, as column strips, to the bits of an eager call on that kernel, and replayed between
    eager calls; the capture allocates nothing."""
    import torch
    import marlin
    assert marlin.plan(m, n, k, g)[1]["partial_kib"] > 0
    dev = torch.device("cuda:0")
    A, q, s, B, sp = O.make_problem(m, n, k, g, seed=m + n)
    want = O.gemm(A, B, sp, n, g)
    dA, dB, dS = (torch.from_numpy(x).to(dev) for x in (A, B, sp))
    C = torch.empty((m, n), dtype=torch.half, device=dev)
    ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
    marlin.mul(dA, dB, C, dS, ws)
    torch.cuda.synchronize()
    marlin.force_kernel(3)
    strips = _gemm(A, B, sp, n)
    marlin.force_kernel(0)
    marlin.release()  # (a new stream may have the handle of one that had scratch)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        marlin.mul(dA, dB, C, dS, ws)
    assert marlin.scratch_bytes() == (0, 0)
    for _ in range(3):
        C.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(C.cpu().numpy().view(np.uint16), strips.view(np.uint16)) and not ws.any().item()
        r = O.compare(C.cpu().numpy(), want)
        assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.rel_mean_abs_err <= 1e-3, r
        r = O.compare(_gemm(A, B, sp, n), want)
        assert r.max_abs_err <= 1e-2 * r.max_abs_ref, r


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,g", [(9, 512, 1024, 128), (16, 256, 512, -1), (13, 768, 1152, 128), (40, 256, 512, 128),
                                     (300, 512, 1152, -1), (41, 2304, 2048, 128), (64, 1024, 4096, -1)])
def test_operands_that_start_anywhere(m, n, k, g):
    """Views into larger storage: A off by one half, B by one word, or both.  Loads straight into
    LDS are for operands that start on 16 bytes; these take kernels that load to registers."""
    import torch
    import marlin
    assert m > 8 and (marlin.plan(m, n, k, g)[1]["kernel"] == 3 or marlin.rows_plan(m, n, k, g) is not None)
    dev = torch.device("cuda:0")
    A, q, s, B, sp = O.make_problem(m, n, k, g, seed=m + k)
    want = O.gemm(A, B, sp, n, g)
    store_a = torch.zeros(m * k + 8, dtype=torch.half, device=dev)
    store_b = torch.zeros(B.size + 4, dtype=torch.int32, device=dev)
    dS = torch.from_numpy(sp).to(dev)
    ws = torch.zeros(n // 128 * 16, dtype=torch.int, device=dev)
    for off_a, off_b in ((1, 0), (0, 1), (3, 2), (4, 0)):
        dA, dB = store_a[off_a:off_a + m * k].view(m, k), store_b[off_b:off_b + B.size].view(B.shape)
        dA.copy_(torch.from_numpy(A))
        dB.copy_(torch.from_numpy(B))
        C = torch.full((m + 1, n), 7.0, dtype=torch.half, device=dev)
        marlin.mul(dA, dB, C[:m], dS, ws)
        torch.cuda.synchronize()
        assert (C[m] == 7.0).all() and not ws.any().item()
        r = O.compare(C[:m].cpu().numpy(), want)
        assert r.max_abs_err <= 1e-2 * r.max_abs_ref and r.rel_mean_abs_err <= 1e-3, (off_a, off_b, r)
