"""Which calls get workgroups that only fetch operands (no GPU: the device counts as one of 256 compute units)."""
import pytest

from flashrnn_amd._lib import DTYPE_IDS, FUNCTION_IDS, load_library


def fetch_workgroups(function, dtype, B, T, N, D, backward):
    return load_library().frnn_fused_fetch_workgroups(FUNCTION_IDS[function], DTYPE_IDS[dtype], B, T, N, D, backward)


# forward: one for each group, or fewer with up to 32 KB a step each (8 for the 12 groups of an XCD, 4 for 7); not 2 for 6, 3 or 5 groups of more
@pytest.mark.parametrize("function,B,N,D,want", [("lstm", 8, 3, 256, 8), ("lstm", 64, 3, 256, 48), ("lstm", 256, 3, 256, 64), ("gru", 250, 3, 256, 64), ("lstm", 70, 3, 256, 32), ("slstm", 140, 3, 256, 32),
                                                 ("lstm", 128, 3, 320, 0), ("lstm", 256, 3, 640, 0), ("slstm", 256, 3, 384, 0), ("lstm", 256, 12, 64, 0), ("lstm", 16, 1, 768, 8), ("gru", 16, 2, 640, 8),
                                                 ("lstm", 64, 3, 768, 0), ("lstm", 16, 1, 512, 0)])
def test_forward(function, B, N, D, want):
    assert fetch_workgroups(function, "bfloat16", B, 512, N, D, 0) == want
    assert fetch_workgroups(function, "bfloat16", B, 24, N, D, 0) == 0 and fetch_workgroups(function, "float32", B, 512, N, D, 0) == 0
    assert fetch_workgroups(function, "bfloat16", 1, 65536, 1, D, 0) == 0


# backward: one for each group or none, 4-row tiles only beyond the last-level cache (36 bytes a unit and step: B16 N4 D192 T606 and T607)
@pytest.mark.parametrize("function,B,T,N,D,want", [("lstm", 128, 28, 3, 256, 48), ("lstm", 256, 64, 3, 256, 48), ("lstm", 8, 1024, 3, 256, 0), ("slstm", 16, 606, 4, 192, 0),
                                                   ("slstm", 16, 607, 4, 192, 16), ("slstm", 16, 2048, 2, 384, 0), ("lstm", 16, 4096, 4, 192, 0), ("gru", 128, 512, 3, 256, 48), ("gru", 200, 1024, 3, 256, 80), ("gru", 256, 1024, 3, 256, 0)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_backward(function, dtype, B, T, N, D, want):
    assert fetch_workgroups(function, dtype, B, T, N, D, 1) == want


def test_errors():
    assert fetch_workgroups("lstm", "bfloat16", 0, 8, 1, 256, 0) < 0 and fetch_workgroups("lstm", "bfloat16", 1, 8, 1, 100, 0) < 0
