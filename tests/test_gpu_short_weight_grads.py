"""Weight gradients of short calls: the GEMM that writes dR itself and sums db on the side, at the edges of its rule and of its stages of
32 rows, against the split GEMM with its reduction (same operands: only the order of the sums differs)."""
import pytest
import torch

from flashrnn_amd import FlashRNNConfig, flashrnn
from flashrnn_amd.flashrnn import DTYPE_DICT, rnn_function_registry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backend", ["hip_fused", "hip"])
@pytest.mark.parametrize("function,dtype,B,T,N,D", [("lstm", "bfloat16", 1, 1, 1, 32), ("lstm", "bfloat16", 5, 19, 3, 256), ("gru", "float16", 3, 11, 2, 96),
                                                    ("slstm", "bfloat16", 2, 16, 1, 192), ("gru", "bfloat16", 31, 33, 1, 128), ("lstm", "float16", 32, 16, 1, 64),
                                                    ("lstm", "bfloat16", 27, 19, 2, 64), ("elman", "bfloat16", 4, 256, 1, 768), ("elman", "bfloat16", 5, 205, 2, 640),
                                                    ("lstm", "bfloat16", 7, 3, 1, 160), ("lstm", "bfloat16", 2, 5, 1, 320), ("gru", "float32", 5, 51, 1, 96),
                                                    ("lstm", "float32", 3, 7, 2, 64)])
def test_one_split_gives_the_sums_of_several(gpu, monkeypatch, function, dtype, B, T, N, D, backend):
    print(f"case short weight grads {function} {dtype} B{B} T{T} N{N} D{D} {backend}", flush=True)
    Gr, Gw, _, Gt, S = rnn_function_registry[function]["gates_states"]
    g = torch.Generator(device=gpu).manual_seed(5)
    kdt = DTYPE_DICT[dtype]
    Wx = torch.randn(B, T, Gw, N, D, generator=g, device=gpu).to(kdt).requires_grad_(True)
    R = (torch.randn(Gr, N, D, D, generator=g, device=gpu) / D ** 0.5).requires_grad_(True)  # (fp32 leaves: the sums as they are)
    b = (torch.randn(Gt, N, D, generator=g, device=gpu) * 0.1).requires_grad_(True)
    cfg = FlashRNNConfig(backend=backend, function=function, dtype=dtype, head_dim=D, num_heads=N, batch_size=B)
    ds = torch.randn(S, B, T, N, D, generator=g, device=gpu).to(kdt)

    def grads():
        states, _ = flashrnn(Wx, R, b, None, config=cfg)
        return states.detach(), torch.autograd.grad(states, (Wx, R, b), grad_outputs=ds)

    states, one = grads()
    monkeypatch.setenv("FRNN_GEMM_SPLITS", "3")
    _, several = grads()
    assert torch.equal(one[0], several[0]) and torch.equal(one[2], several[2])
    rows = B * T
    h = torch.cat([torch.zeros_like(states[0][:, :1]), states[0][:, :-1]], 1).double().abs().reshape(rows, N, D)
    # a sum of `rows` products in fp32, in any order, is within rows * 2^-24 of the sum of their sizes (the GRU's g gate: its cotangent is
    # that of the candidate times r < 1)
    gate = [2, 0, 1] if function == "gru" else range(Gr)
    dg = one[0].double().abs().reshape(rows, Gw, N, D)
    size = torch.stack([torch.matmul(dg[:, k].permute(1, 2, 0).contiguous(), h.permute(1, 0, 2).contiguous()) for k in gate])
    slack = 1 + 2 ** -7  # (the GEMM's operand of the g gate is rounded to the storage type once more)
    assert ((one[1] - several[1]).abs().double() <= 2 * rows * 2.0 ** -24 * size * slack).all()
    if backend == "hip_fused" and function == "lstm":
        ref = torch.stack([torch.matmul(one[0].double().reshape(rows, Gw, N, D)[:, k].permute(1, 2, 0).contiguous(),
                                        torch.cat([torch.zeros_like(states[0][:, :1]), states[0][:, :-1]], 1).double().reshape(rows, N, D).permute(1, 0, 2).contiguous())
                           for k in range(Gr)])
        assert ((one[1].double() - ref).abs() <= rows * 2.0 ** -24 * size).all()
