"""Forward kernels that store the outputs of a step behind the first probe of the next one: sequences of one step and a few, ragged tiles of 4
and of 8 rows, both ends of the rule, with and without a gate cache, against the oracle; and single steps, whose only step has no next."""
import pytest
import torch

from parity import check_case
from test_gpu_decode import _device_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 5])
@pytest.mark.parametrize("function,dtype,B,N,D", [("lstm", "bfloat16", 5, 2, 256), ("lstm", "float16", 77, 4, 256), ("slstm", "bfloat16", 7, 3, 192), ("slstm", "bfloat16", 131, 4, 192),
                                                  ("gru", "bfloat16", 6, 1, 512), ("gru", "float16", 70, 3, 320), ("lstm", "bfloat16", 66, 2, 384)])
def test_outputs_of_every_step_are_stored(gpu, function, dtype, B, T, N, D):
    from flashrnn_amd import flashrnn, flashrnn_step, make_carry

    print(f"case stores behind the probe {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    check_case(gpu, function, B, T, N, D, dtype, "hip_fused", seed=T, init="randn")
    x = _device_inputs(gpu, function, B, T, N, D, dtype, seed=T)
    with torch.no_grad():
        ref, last = flashrnn(x["Wx"], x["R"], x["b"], x["states"], function=function, backend="hip_fused", dtype=dtype)
    assert torch.equal(last, ref[:, :, -1:])
    s, carry = x["states"], make_carry(x["states"])
    for t in range(T):
        s = flashrnn_step(x["Wx"][:, t:t + 1].contiguous(), x["R"], x["b"], s, function=function, dtype=dtype, carry=carry)
        assert torch.equal(s[:, :, 0], ref[:, :, t]), t
