"""Dense tilings (8 waves on half the workgroups of the default, taken by large batches): every tile height against the oracle, single
steps with the bits of the sequence, and their waits that run out."""
import pytest
import torch

from parity import check_case
from test_gpu_decode import _device_inputs
from test_gpu_wait_runs_out import test_waits_that_run_out_end_the_kernels_and_are_reported as check_wait

pytestmark = pytest.mark.gpu


# (4, 8 and 16 rows by the rule, the last tile ragged; the bound on an element: see test_gpu_spread_tilings.py)
@pytest.mark.parametrize("function,dtype,B,N,D", [("lstm", "bfloat16", 3, 66, 256), ("lstm", "float16", 173, 3, 256), ("lstm", "bfloat16", 517, 2, 256),
                                                  ("slstm", "bfloat16", 173, 3, 256), ("slstm", "float16", 517, 2, 256), ("gru", "bfloat16", 131, 2, 256),
                                                  ("gru", "float16", 177, 3, 256), ("gru", "bfloat16", 517, 2, 256), ("gru", "bfloat16", 81, 2, 384),
                                                  ("gru", "float16", 161, 2, 384), ("gru", "bfloat16", 641, 1, 384)])
def test_every_tile_height_matches_the_oracle(gpu, function, dtype, B, N, D):
    print(f"case dense {function} {dtype} B{B} N{N} D{D}", flush=True)
    check_case(gpu, function, B, 3, N, D, dtype, "hip_fused", seed=37, init="randn")


@pytest.mark.parametrize("function,B,N,D", [("lstm", 173, 3, 256), ("gru", 131, 2, 256), ("gru", 161, 2, 384), ("slstm", 517, 2, 256)])
def test_steps_give_the_bits_of_a_sequence(gpu, function, B, N, D):
    from flashrnn_amd import flashrnn, flashrnn_step, make_carry

    T = 6
    x = _device_inputs(gpu, function, B, T, N, D, "bfloat16", seed=41)
    with torch.no_grad():
        ref, _ = flashrnn(x["Wx"], x["R"], x["b"], x["states"], function=function, backend="hip_fused", dtype="bfloat16")
    s, carry = x["states"], make_carry(x["states"])
    for t in range(T):
        s = flashrnn_step(x["Wx"][:, t:t + 1].contiguous(), x["R"], x["b"], s, function=function, dtype="bfloat16", carry=carry)
        assert torch.equal(s[:, :, 0], ref[:, :, t]), t


@pytest.mark.parametrize("function,D", [("lstm", 256), ("slstm", 256), ("gru", 256), ("gru", 384)])
def test_waits_that_run_out(gpu, monkeypatch, function, D):
    monkeypatch.setenv("FRNN_FUSED_VARIANT", "4")
    check_wait(gpu, monkeypatch, function, "bfloat16", 8, D, 4, False, False)
