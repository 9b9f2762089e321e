"""The rule that chooses a tiling (no GPU: the device counts as one of 256 compute units): the alternatives that spread a head are
used only while all groups of the call fit one launch, and batch tiles that are asked for are kept."""
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
                if p[:3] != q[:3]:
                    differ += 1
                    assert p[2] >= q[2] and 1 < p[2] <= 32 and N * -(-B // 4) <= 8 * (32 // p[2])
                    assert p[3] == N * -(-B // 4) * p[2]  # 4-row tiles, all in one launch
                    monkeypatch.delenv("FRNN_FUSED_VARIANT")
                    monkeypatch.setenv("FRNN_TILE_ROWS", "16")
                    t = _plan(function, dtype, B, N, D, backward)
                    assert t[:3] == q[:3] or t[3] == N * -(-B // 16) * t[2]
    assert differ > 0 or function == "elman"
