"""Reverse kernels that do half of a step's adjoint in the wait of the step before: sequences of one step and a few, ragged tiles of each height, wave
pairs and single waves, both ends of the rule, against the oracle."""
import pytest

from parity import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 5])
@pytest.mark.parametrize("function,dtype,B,N,D", [("lstm", "bfloat16", 5, 2, 256), ("lstm", "float16", 6, 1, 768), ("lstm", "bfloat16", 3, 1, 1024), ("slstm", "bfloat16", 7, 3, 192),
                                                  ("slstm", "float16", 5, 1, 640), ("gru", "bfloat16", 131, 2, 256), ("gru", "float16", 6, 1, 512), ("gru", "bfloat16", 70, 3, 384),
                                                  ("lstm", "float32", 3, 1, 256), ("lstm", "float32", 5, 1, 512)])
def test_matches_the_oracle(gpu, function, dtype, B, T, N, D):
    print(f"case early adjoint {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    check_case(gpu, function, B, T, N, D, dtype, "hip_fused", seed=T, init="randn")
