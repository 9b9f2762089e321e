"""Heads of one workgroup, 16-bit types: outputs stored by the compute waves and by the producer wave, which the library picks by size, give the same
bits at the edges of the producer's ring and of the 4-row tiles, and so does what it picks on either side of its lines."""
import pytest
import torch

from flashrnn_amd import FlashRNNConfig, flashrnn
from oracle import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("function", ["lstm", "slstm", "gru", "elman"])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("B,T,N", [(1, 1, 1), (5, 2, 2), (3, 3, 1), (9, 4, 2), (6, 8, 3), (261, 5, 4)])
def test_store_paths_agree(gpu, monkeypatch, function, D, B, T, N):
    print(f"case store rule {function} B{B} T{T} N{N} D{D}", flush=True)
    inp = make_inputs(function, B, T, N, D, 17, init="randn")
    dtype = torch.float16 if N == 2 else torch.bfloat16
    cfg = FlashRNNConfig(backend="hip_fused", function=function, dtype=str(dtype)[6:], head_dim=D, num_heads=N)
    res = []
    for stores in ("0", "1", None):
        if stores is None:
            monkeypatch.delenv("FRNN_PRODUCER_STORES")
        else:
            monkeypatch.setenv("FRNN_PRODUCER_STORES", stores)
        leaves = [inp[k].to(gpu, dtype).requires_grad_() for k in ("Wx", "R", "b", "states")]
        out, _ = flashrnn(*leaves, config=cfg)
        grads = torch.autograd.grad(out, leaves, inp["dstates"].to(gpu, dtype))
        with torch.no_grad():
            res.append([out.detach(), flashrnn(*leaves, config=cfg)[0], *grads])
    for other in res[1:]:
        assert all(torch.equal(x, y) for x, y in zip(res[0], other))
    assert torch.equal(res[0][0], res[0][1])
