"""The single-step kernel of the fused backend (16-bit types) at every head dimension: the bits of the sequence kernel, whose order of
summation depends on its tiling (own slice first, k split in two, chains that take turns); taller tiles keep the scan kernel."""
import pytest
import torch

from oracle import make_inputs

pytestmark = pytest.mark.gpu

DIMS = (32, 64, 96, 128, 160, 192, 256, 320, 384, 448, 512, 640, 768, 1024)
CASES = [(f, D, "bfloat16", 5, 2, 0) for f in ("lstm", "slstm", "gru", "elman") for D in DIMS]
CASES += [(f, D, "float16", 19, 1, rows) for f, D, rows in (("lstm", 192, 0), ("gru", 512, 0), ("slstm", 320, 4), ("lstm", 256, 16), ("slstm", 512, 8), ("gru", 192, 16), ("elman", 640, 16),
                                                            ("elman", 96, 8), ("lstm", 1024, 16), ("gru", 64, 8))]


@pytest.mark.parametrize("function,D,dtype,B,N,rows", CASES)
def test_steps_give_the_bits_of_the_sequence(gpu, monkeypatch, function, D, dtype, B, N, rows):
    from flashrnn_amd import FlashRNNConfig, flashrnn, flashrnn_step, make_carry

    print(f"case step kernel {function} D{D} {dtype} rows={rows}", flush=True)
    if rows:
        monkeypatch.setenv("FRNN_TILE_ROWS", str(rows))
    T, kdt = 4, {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    x = {k: v.to(gpu, kdt).contiguous() for k, v in make_inputs(function, B, T, N, D, 41, init="randn", round_to=kdt).items()}
    cfg = FlashRNNConfig(head_dim=D, num_heads=N, function=function, dtype=dtype, forward_clipval=0.6 if D in (32, 640) else None)
    with torch.no_grad():
        ref, _ = flashrnn(x["Wx"], x["R"], x["b"], x["states"], config=cfg)
    s, carry = x["states"], make_carry(x["states"])
    for t in range(T):
        s = flashrnn_step(x["Wx"][:, t:t + 1].contiguous(), x["R"], x["b"], s, config=cfg, carry=carry)
        assert torch.equal(s[:, :, 0], ref[:, :, t]), (t, float((s[:, :, 0] != ref[:, :, t]).float().mean()))
