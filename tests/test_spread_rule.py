"""The rule that chooses a tiling (no GPU: the device counts as one of 256 compute units): the alternatives that spread a head are
used only while all groups of the call fit one launch, the dense ones only where the default would need taller tiles, and batch tiles
that are asked for are kept."""
import ctypes

import pytest

from flashrnn_amd._lib import DTYPE_IDS, FUNCTION_IDS, load_library

DIMS = (32, 64, 96, 128, 160, 192, 256, 320, 384, 448, 512, 640, 768, 1024)


def _plan(function, dtype, B, N, D, backward):
    v = [ctypes.c_int() for _ in range(4)]
    rc = load_library().frnn_fused_plan(FUNCTION_IDS[function], DTYPE_IDS[dtype], B, N, D, backward, *map(ctypes.byref, v))
    return tuple(x.value for x in v) if rc == 0 else None


@pytest.mark.parametrize("function", list(FUNCTION_IDS))
@pytest.mark.parametrize("dtype", list(DTYPE_IDS))
def test_a_spread_tiling_always_fits_one_launch(monkeypatch, function, dtype):
    differ = 0
    for D in DIMS:
        for backward in (0, 1):
            for B, N in ((1, 1), (5, 2), (16, 4), (33, 3), (64, 1), (256, 3)):
                monkeypatch.delenv("FRNN_FUSED_VARIANT", raising=False)
                monkeypatch.delenv("FRNN_TILE_ROWS", raising=False)
                p = _plan(function, dtype, B, N, D, backward)
                if p is None:
                    continue
                monkeypatch.setenv("FRNN_FUSED_VARIANT", "1")  # (no such entry: the default)
                q = _plan(function, dtype, B, N, D, backward)
                assert 16 * p[0] * p[1] * p[2] % D == 0
                if p[2] < q[2]:  # dense: half the workgroups per head, tiles of half the height or no more launches
                    assert p[0] == 8 and 2 * p[2] == q[2] and p[3] <= max(q[3], 8 * (32 // p[2]) * p[2])
                    continue
                if p[:3] != q[:3]:
                    differ += 1
                    assert p[2] >= q[2] and 1 < p[2] <= 32 and N * -(-B // 4) <= 8 * (32 // p[2])
                    assert p[3] == N * -(-B // 4) * p[2]  # 4-row tiles, all in one launch
                    monkeypatch.delenv("FRNN_FUSED_VARIANT")
                    monkeypatch.setenv("FRNN_TILE_ROWS", "16")
                    t = _plan(function, dtype, B, N, D, backward)
                    assert t[:3] == q[:3] or t[3] == N * -(-B // 16) * t[2]
    assert differ > 0 or function == "elman"


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("function,D,backward,lim,default,dense", [("lstm", 256, 0, 8, 4, 2), ("slstm", 256, 0, 8, 4, 2), ("gru", 256, 0, 4, 4, 2),
                                                                   ("gru", 384, 0, 4, 6, 3), ("gru", 256, 1, 8, 4, 2)])
def test_the_dense_tiling_begins_where_the_default_needs_taller_tiles(monkeypatch, function, dtype, D, backward, lim, default, dense):
    room = 8 * (32 // default)
    for N in (1, 2, 3, 40, 200):
        last = room // N * lim  # rows of the largest batch that the default still takes with tiles of `lim` rows
        for B in {1, max(1, last), last + 1, 2 * last + 2, 5 * last + 7}:
            p = _plan(function, dtype, B, N, D, backward)
            launches, packed = -(-N * -(-B // 16) // room), -(-N * -(-B // 16) // (8 * (32 // dense)))
            assert p[2] == (dense if N * -(-B // lim) > room and (launches <= 1 or 8 * packed < 5 * launches) else default), (B, N, p)
    B = room * lim + 1  # (never where a height is asked for)
    monkeypatch.setenv("FRNN_TILE_ROWS", "16")
    assert _plan(function, dtype, B, 1, D, backward)[2] == default


def test_calls_that_fit_the_static_scratch_keep_fitting():
    """The dense tiling's exchange words can exceed the library's static scratch where the default's do not: such a call keeps the
    default there (null tensors: the size is checked first, then the pointers)."""
    lib = load_library()
    for function, B, N in (("lstm", 256, 3), ("slstm", 180, 3), ("gru", 100, 3)):
        args = [FUNCTION_IDS[function], DTYPE_IDS["bfloat16"], 0, B, 4, N, 256] + [None] * 8
        rc = lib.frnn_fused_forward_static(*args)
        assert "static scratch" not in lib.frnn_last_error().decode(), (rc, lib.frnn_last_error())


@pytest.mark.parametrize("function", list(FUNCTION_IDS))
@pytest.mark.parametrize("dtype", list(DTYPE_IDS))
def test_a_session_takes_no_more_than_the_default_tiling(monkeypatch, function, dtype):
    """A decode session holds its workgroups for as long as it is open: those of the default tiling of its heads, also where a sequence
    call of the same size spreads them over more (in tilings that split tiles; those that do not keep the number of waves)."""
    lib, spread = load_library(), 0
    for D in DIMS:
        for B, N in ((1, 1), (4, 2), (8, 3), (33, 1)):
            waves, wgs = ctypes.c_int(), ctypes.c_int()
            if lib.frnn_fused_decode_workgroups(FUNCTION_IDS[function], DTYPE_IDS[dtype], B, N, D, ctypes.byref(waves), ctypes.byref(wgs)):
                continue  # (does not fit the device at once)
            monkeypatch.setenv("FRNN_FUSED_VARIANT", "1")  # (no such entry: the default)
            monkeypatch.setenv("FRNN_TILE_ROWS", "4")
            q = _plan(function, dtype, B, N, D, 0)
            monkeypatch.delenv("FRNN_FUSED_VARIANT")
            monkeypatch.delenv("FRNN_TILE_ROWS")
            p = _plan(function, dtype, B, N, D, 0)
            spread += p[0] * p[3] > q[0] * q[3]
            assert wgs.value * waves.value <= q[0] * q[3], (D, B, N)
    assert spread > 0 or function == "elman"


@pytest.mark.parametrize("function", list(FUNCTION_IDS))
@pytest.mark.parametrize("dtype", list(DTYPE_IDS))
def test_the_workspace_of_a_call_serves_its_tiling_beside_a_session(monkeypatch, function, dtype):
    """Workspace is asked for before a call, which may meet a session that was opened since: the default tiling at 4-row tiles needs no
    more of it than the spread tiling that it replaces."""
    lib = load_library()
    for D in DIMS:
        for backward in (0, 1):
            for B, N in ((1, 1), (5, 2), (16, 4), (33, 3), (64, 1)):
                p = _plan(function, dtype, B, N, D, backward)
                if p is None or 16 * p[0] * p[1] * p[2] == D:  # (no wave shares a tile: kept beside a session)
                    continue
                args = (FUNCTION_IDS[function], DTYPE_IDS[dtype], B, 7, N, D, backward)
                asked = lib.frnn_fused_workspace_bytes(*args)
                monkeypatch.setenv("FRNN_FUSED_VARIANT", "1")
                default = _plan(function, dtype, B, N, D, backward)
                monkeypatch.setenv("FRNN_TILE_ROWS", "4")
                assert p[:3] == default[:3] or 0 < lib.frnn_fused_workspace_bytes(*args) <= asked, (D, backward, B, N)
                monkeypatch.delenv("FRNN_FUSED_VARIANT")
                monkeypatch.delenv("FRNN_TILE_ROWS")
