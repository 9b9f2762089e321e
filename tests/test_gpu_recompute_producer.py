"""Recompute mode, heads of one workgroup, 16-bit types: the reverse kernels whose producer wave loads the operands and stages h
(csrc/frnn_plan.h, bwd_producer_wave), at the edges of its ring of three sets and of its 4-row tiles, by both store paths, and the truncated
scan, in which that wave only takes part in the barriers."""
import pytest
import torch

from flashrnn_amd import FlashRNNConfig, flashrnn
from oracle import make_inputs
from parity import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("function", ["lstm", "slstm", "gru"])
@pytest.mark.parametrize("D,dtype", [(32, "bfloat16"), (64, "float16"), (96, "bfloat16"), (96, "float16")])
@pytest.mark.parametrize("B,T", [(1, 1), (5, 2), (3, 3), (9, 4), (6, 8)])
def test_matches_oracle_with_both_store_paths(gpu, monkeypatch, function, D, dtype, B, T):
    print(f"case recompute producer {function} B{B} T{T} N2 D{D} {dtype}", flush=True)
    for cut in (False, True):
        check_case(gpu, function, B, T, 2, D, dtype, "hip_fused", seed=91, init="randn",
                   options=dict(recompute_gates=True, gradient_recurrent_cut=cut))
    kdt = getattr(torch, dtype)
    inp = make_inputs(function, B, T, 2, D, 91, init="randn")
    cfg = FlashRNNConfig(backend="hip_fused", function=function, dtype=dtype, head_dim=D, num_heads=2, recompute_gates=True,
                         gradient_recurrent_clipval=0.5)
    res = []
    for stores in ("0", "1"):
        monkeypatch.setenv("FRNN_PRODUCER_STORES", stores)
        leaves = [inp[k].to(gpu, kdt).requires_grad_() for k in ("Wx", "R", "b", "states")]
        out, _ = flashrnn(*leaves, config=cfg)
        res.append(torch.autograd.grad(out, leaves, inp["dstates"].to(gpu, kdt)))
    assert all(torch.equal(x, y) for x, y in zip(*res))
