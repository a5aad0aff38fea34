"""Dense fp16 GEMM with a stream-K tail (the reference's gemm/streamk_gemm) over
the C ABI of libmarlin_amd.so: C = A @ B.T with A (m, k) and B (n, k) in fp16,
fp32 accumulation.  The GEMM always runs in the HIP library; a missing library
is an import-time error."""
import ctypes

from native import lib as _lib, torch_binding as _torch_binding

_P, _I = ctypes.c_void_p, ctypes.c_int
_lib.streamk_amd_check.restype = _I
_lib.streamk_amd_check.argtypes = [_I, _I, _I]
_lib.streamk_amd_plan.restype = _I
_lib.streamk_amd_plan.argtypes = [_I, _I, _I, _I, _P]
_lib.streamk_amd_launches.restype = _I
_lib.streamk_amd_launches.argtypes = [_I, _I, _I, _I, _I, _P]
_lib.streamk_amd_tile.restype = _I
_lib.streamk_amd_tile.argtypes = [_I, _I, _I, _I, _P]
_lib.streamk_amd_force_tile.restype = None
_lib.streamk_amd_force_tile.argtypes = [_I, _I, _I]
_lib.streamk_amd_tile_coord.restype = None
_lib.streamk_amd_tile_coord.argtypes = [_I, _I, _I, _P]
_lib.streamk_amd_slice_coord.restype = None
_lib.streamk_amd_slice_coord.argtypes = [_I, _I, _I, _P]
_lib.streamk_amd_force_finish_polls.restype = None
_lib.streamk_amd_force_finish_polls.argtypes = [_I]
_lib.streamk_amd_last_error.restype = ctypes.c_char_p


def check(m, n, k):
    """Return code streamk_gemm_tn would give for these sizes (no GPU touched)."""
    return _lib.streamk_amd_check(m, n, k)


def plan(m, n, k, cus=256):
    """The split of the output tiles (tile_rows x tile_cols) into data-parallel and stream-K tiles."""
    out = (ctypes.c_int * 8)()
    rc = _lib.streamk_amd_plan(m, n, k, cus, out)
    keys = ("tiles_m", "tiles_n", "dp_tiles", "sk_tiles", "k_slices", "grid", "tile_rows", "tile_cols")
    return rc, dict(zip(keys, out))


def tile(m, n, k, cus=256):
    """(rows, cols, slices) of the tiles that compute the problem in one launch, in place of the
    plan's, or None."""
    out = (ctypes.c_int * 3)()
    _lib.streamk_amd_tile(m, n, k, cus, out)
    return tuple(out) if out[0] > 0 else None


def force_tile(rows, cols=0, slices=1):
    """Tiles that compute every problem, in place of the plan's (0 = by cost, -1 = never; calling
    thread only)."""
    _lib.streamk_amd_force_tile(int(rows), int(cols), int(slices))


def launches(m, n, k, cus=256, scratch=True):
    """The launches that compute the plan's tiles, unless tile() names others;
    `scratch`: whether there is room for partial sums."""
    out = (ctypes.c_int * 10)()
    count = _lib.streamk_amd_launches(m, n, k, cus, int(scratch), out)
    keys = ("rows", "cols", "waves", "tiles", "slices")
    return [dict(zip(keys, out[5 * i:5 * i + 5])) for i in range(count)]


def tile_coord(tile, tiles_m, tiles_n):
    """(row tile, column tile) of a tile number."""
    out = (ctypes.c_int * 2)()
    _lib.streamk_amd_tile_coord(tile, tiles_m, tiles_n, out)
    return out[0], out[1]


def slice_coord(block, tiles, slices):
    """(tile, slice) of a workgroup of a launch of slices."""
    out = (ctypes.c_int * 2)()
    _lib.streamk_amd_slice_coord(block, tiles, slices, out)
    return out[0], out[1]


def force_finish_polls(polls):
    """How often a workgroup looks for the other slices of its tile before it leaves them its
    share of the sums; -1 = the default (calling thread only)."""
    _lib.streamk_amd_force_finish_polls(int(polls))


def gemm(A, B, C=None):
    """C (m, n) = A (m, k) @ B (n, k).T on the current stream; returns C."""
    return _torch_binding.dense(A, B, C)
