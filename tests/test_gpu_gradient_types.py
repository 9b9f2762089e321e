"""Gradients of the weights in the storage type, written by the kernels: bit for bit the fp32 sums rounded, whatever the types of R and b;
and the initial state that a call without one begins at, cleared by the call."""
import pytest
import torch

from flashrnn_amd import FlashRNNConfig, flashrnn
from flashrnn_amd.flashrnn import DTYPE_DICT, rnn_function_registry

pytestmark = pytest.mark.gpu


# (one split and several; heads of one and of several workgroups; n: not whole numbers of 256 elements)
@pytest.mark.parametrize("function,dtype,B,T,N,D,backend", [("lstm", "bfloat16", 5, 7, 3, 256, "hip_fused"), ("gru", "float16", 9, 70, 1, 96, "hip_fused"),
                                                            ("slstm", "bfloat16", 8, 140, 2, 64, "hip_fused"), ("elman", "bfloat16", 33, 40, 1, 32, "hip"),
                                                            ("lstm", "float16", 3, 5, 1, 160, "hip"), ("lstm", "float32", 4, 9, 1, 64, "hip_fused")])
def test_narrow_gradients_are_the_rounded_sums(gpu, function, dtype, B, T, N, D, backend):
    print(f"case gradient types {function} {dtype} B{B} T{T} N{N} D{D} {backend}", flush=True)
    Gr, Gw, _, Gt, S = rnn_function_registry[function]["gates_states"]
    kdt = DTYPE_DICT[dtype]
    g = torch.Generator(device=gpu).manual_seed(3)
    Wx = torch.randn(B, T, Gw, N, D, generator=g, device=gpu).to(kdt).requires_grad_(True)
    R = (torch.randn(Gr, N, D, D, generator=g, device=gpu) / D ** 0.5).to(kdt)
    b = (torch.randn(Gt, N, D, generator=g, device=gpu) * 0.1).to(kdt)
    ds = torch.randn(S, B, T, N, D, generator=g, device=gpu).to(kdt)
    cfg = FlashRNNConfig(backend=backend, function=function, dtype=dtype, head_dim=D, num_heads=N, batch_size=B)

    def run(rt, bt, states):
        leaves = (Wx, R.to(rt).requires_grad_(True), b.to(bt).requires_grad_(True))
        junk = torch.full((S * B * N * D + 4096,), float("nan"), device=gpu, dtype=kdt)  # (what the next allocation may find)
        del junk
        out, _ = flashrnn(*leaves, states, config=cfg)
        return (out.detach(),) + torch.autograd.grad(out, leaves, grad_outputs=ds)

    ref = run(torch.float32, torch.float32, torch.zeros(S, B, 1, N, D, device=gpu, dtype=kdt))
    for rt in (kdt, torch.float32):
        for bt in (kdt, torch.float32):
            got = run(rt, bt, None)
            assert got[2].dtype == rt and got[3].dtype == bt
            for x, y in zip(got, ref):
                assert torch.equal(x, y.to(x.dtype))
