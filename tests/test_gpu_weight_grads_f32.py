"""fp32 weight gradients: the GEMM at its three tile sides, with rows that end within a stage of 32, sequences shorter and longer than a
stage and several splits, against the products of the pass's own dWx and h in 64 bits."""
import pytest
import torch

from flashrnn_amd import FlashRNNConfig, flashrnn
from flashrnn_amd.flashrnn import rnn_function_registry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("function", ["lstm", "elman"])
@pytest.mark.parametrize("B,T,N,D", [(1, 1, 1, 128), (67, 1, 2, 128), (5, 51, 2, 256), (40, 31, 1, 384), (3, 700, 1, 128), (9, 64, 3, 64), (7, 37, 2, 96), (16, 33, 1, 512)])
def test_f32_weight_gradients(gpu, function, B, T, N, D):
    print(f"case f32 weight grads {function} B{B} T{T} N{N} D{D}", flush=True)
    Gr, Gw, _, Gt, S = rnn_function_registry[function]["gates_states"]
    g = torch.Generator(device=gpu).manual_seed(8)
    Wx = torch.randn(B, T, Gw, N, D, generator=g, device=gpu).requires_grad_(True)
    R = (torch.randn(Gr, N, D, D, generator=g, device=gpu) / D ** 0.5).requires_grad_(True)
    b = (torch.randn(Gt, N, D, generator=g, device=gpu) * 0.1).requires_grad_(True)
    s0 = torch.randn(S, B, 1, N, D, generator=g, device=gpu)
    cfg = FlashRNNConfig(backend="hip_fused", function=function, dtype="float32", head_dim=D, num_heads=N, batch_size=B)
    out, _ = flashrnn(Wx, R, b, s0, config=cfg)
    dWx, dR, db = torch.autograd.grad(out, (Wx, R, b), torch.randn(out.shape, generator=g, device=gpu))
    rows = B * T
    h = torch.cat([s0[0], out.detach()[0, :, :-1]], 1).double().reshape(rows, N, D).permute(1, 0, 2).contiguous()
    dg = dWx.double().reshape(rows, Gw, N, D).permute(1, 2, 3, 0).contiguous()
    for k in range(Gr):
        # (a sum of `rows` products in fp32, in any order, is within rows * 2^-24 of the sum of their sizes)
        size = torch.matmul(dg[k].abs(), h.abs())
        assert ((dR[k].double() - torch.matmul(dg[k], h)).abs() <= rows * 2.0 ** -24 * size).all()
        size_b = dg[k].abs().sum(-1)
        assert ((db[k].double() - dg[k].sum(-1)).abs() <= rows * 2.0 ** -24 * size_b).all()
