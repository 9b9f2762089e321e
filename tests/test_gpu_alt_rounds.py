"""Alternating backend: head dims around the lines at which its step kernels change the order and the number of the
fragments that a wave requests at once (forward: more than 512 units of a one-gate cell, 8 k-steps of 32 units per round
and 4 waves; backward: at least 4 k-steps, one for each wave, and for the GRU no more than the 32 of a round)."""
import pytest

from parity import check_case

pytestmark = pytest.mark.gpu

CASES = [
    # forward rounds: last head dim of the 4-step rounds, first of the 8-step ones (one wave has a fifth k-step), a full round,
    # one k-step into the second
    ("elman", 3, 9, 1, 512, "bfloat16"),
    ("elman", 17, 9, 2, 544, "bfloat16"),
    ("elman", 5, 9, 1, 544, "float16"),
    ("elman", 33, 9, 1, 1024, "bfloat16"),
    ("elman", 2, 9, 1, 1056, "bfloat16"),
    # ... and the 4-step rounds again where the launch has more than 288 workgroups of 16 units x 16 rows: 272, 306 and 320 of them
    ("elman", 64, 5, 2, 544, "bfloat16"),
    ("elman", 129, 5, 1, 544, "float16"),
    ("elman", 65, 5, 1, 1024, "bfloat16"),
    # backward: k-steps (gates x units / 32) below, at and above one for each wave, and one into the second round
    ("elman", 5, 9, 2, 96, "bfloat16"),
    ("elman", 5, 9, 2, 128, "bfloat16"),
    ("gru", 17, 9, 2, 32, "bfloat16"),
    ("lstm", 17, 9, 2, 32, "float16"),
    ("slstm", 1, 9, 3, 32, "bfloat16"),
    ("gru", 3, 9, 1, 320, "bfloat16"),
    ("gru", 3, 9, 1, 352, "bfloat16"),
]


@pytest.mark.parametrize("function,B,T,N,D,dtype", CASES)
def test_alternating_backend_at_the_edges_of_its_rounds(gpu, function, B, T, N, D, dtype):
    print(f"case alt rounds {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    check_case(gpu, function, B, T, N, D, dtype, "hip", seed=3)
