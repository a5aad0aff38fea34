"""CPU tests of the weight conversion's host side: what the C entries refuse before
anything is launched.  No GPU work."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))

PROB_SHAPE = 1


@pytest.mark.parametrize("B,s_packed,scales", [
    (1 << 30, 1 << 29, 1 << 29),             # scales packed onto themselves
    (1 << 30, 1 << 29, (1 << 29) + 2046),    # the last byte of the packed ones
    (1 << 30, (1 << 20) + 1024, 1 << 29),    # inside the weight
    ((1 << 20) + 1024, 1 << 29, 1 << 28),
    (1 << 29, (1 << 29) + 1024, 1 << 28),    # the two outputs
    (1 << 30, 1 << 29, (1 << 30) - 2046),    # scales that run into the words
])
def test_pack_refuses_operands_that_overlap(B, s_packed, scales):
    import marlin
    k, n, gs = 256, 512, 128
    assert marlin._lib.marlin_amd_pack(1 << 20, k, n, gs, 0, scales, n, 1, B, s_packed, 0, None) == PROB_SHAPE


def test_problems_no_grid_holds_are_refused():
    """... with the code that sends the Python calls to the tensor operations."""
    import marlin
    lib, P = marlin._lib, 1 << 20
    deep = 16 * 65536  # a row of workgroups per 16 rows: one too many
    assert lib.marlin_amd_pack_words(P, deep, 64, 1 << 40, 0, None) == PROB_SHAPE
    assert lib.marlin_amd_pack(P, deep, 64, 128, 0, 1 << 50, 64, 1, 1 << 40, 1 << 52, 0, None) == PROB_SHAPE
    assert lib.marlin_amd_quantize(P, 4 * 65536, 64, 4, 0, P, P, P, 0, None) == PROB_SHAPE
    # 32 threads, or 256, per group of a column: 2^32 threads
    assert lib.marlin_amd_quantize(P, 8192, 65536, 4, 1, P, P, P, 0, None) == PROB_SHAPE
    assert lib.marlin_amd_quantize(P, 132 * 256, 65536, 132, 1, P, P, P, 0, None) == PROB_SHAPE


def test_what_counts_as_looking_on():
    """Function modes see the tensor operations; a default device does not ask to."""
    import torch
    import marlin
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert marlin._can_tell and not marlin._looked_on()
    with torch.device("cpu"):
        assert not marlin._looked_on()
        with Mode():
            assert marlin._looked_on()
    with Mode():
        assert marlin._looked_on()
    assert not marlin._looked_on()


def test_without_torchs_own_names_the_tensor_operations_run(monkeypatch):
    import marlin
    monkeypatch.setattr(marlin, "_can_tell", False)
    assert marlin._looked_on()


def test_what_the_kernels_do_not_take_is_left_to_the_tensor_operations():
    """... with its own results and its own refusals, group sizes of every kind among them."""
    import torch
    import marlin
    binding = marlin._torch_binding
    w, B = torch.ones(256, 256).half(), torch.empty(16, 512, dtype=torch.int32)
    for tensor in (w, w.t(), w.float(), w[0], [1.0], None):
        for group in (-1, 128, 0, 2 ** 40, 128.0, None):
            assert binding.quantize(tensor, group) is None
            assert binding.pack(tensor, w, B, w, 256, 256, group) is False
    _, q, s = marlin.quantize(w, 128)
    assert q.shape == w.shape and s.shape == (2, 256)
    with pytest.raises(ZeroDivisionError):
        marlin.quantize(w, 0)
    with pytest.raises(RuntimeError):
        marlin.quantize(w, 2 ** 40)
    with pytest.raises(TypeError):
        marlin.quantize(w, 128.0)


def test_the_devices_own_compute_units_decide_how_long_groups_are_quantised():
    """A workgroup per 64 columns fills a small device sooner, and then takes rounds of them."""
    import marlin
    launches = marlin._lib.marlin_amd_quantize_launches
    assert launches(4096, 4096, 128, 0, 256) == launches(4096, 4096, -1, 1, 256) == 1
    assert launches(1024, 4096, -1, 0, 256) == 1 and launches(4096, 4096, -1, 0, 256) == 3
    # 256 workgroups: one round of 256 compute units, four of 64
    assert launches(2048, 16384, -1, 0, 256) == 1 and launches(2048, 16384, -1, 0, 64) == 3
    assert launches(2048, 16384, -1, 0, 0) == 0
