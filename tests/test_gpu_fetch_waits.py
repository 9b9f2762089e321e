"""Waits that run out in reverse launches with workgroups that fetch operands: the host leaves a workgroup of every head out of the scan (FRNN_SPIN_LIMIT=-3)
while those workgroups stay.  (The forward kernel is the same one with and without them: test_gpu_wait_runs_out.py has its waits.)  Every workgroup has to end by its own bounds, the call has to report the wait, the outputs have to be NaN, and nothing is left behind."""
import pytest
import torch

from oracle import make_inputs
from test_fetch_rule import fetch_workgroups
from test_gpu_wait_runs_out import KDT, _reported, _workgroups_per_head

pytestmark = pytest.mark.gpu

# 16- and 8-row tiles, wave pairs beyond the last-level cache
CASES = [("slstm", "bfloat16", 20, 26, 256, 16), ("lstm", "float16", 9, 33, 320, 8),
         ("gru", "bfloat16", 16, 26, 256, 8), ("slstm", "bfloat16", 16, 2500, 192, 4)]


@pytest.mark.parametrize("handshake", [False, True])
@pytest.mark.parametrize("function,dtype,B,T,D,rows", CASES)
def test_launches_with_workgroups_that_fetch_end_and_report(gpu, monkeypatch, function, dtype, B, T, D, rows, handshake):
    from flashrnn_amd import FlashRNNConfig, flashrnn, last_status

    print(f"case fetch wait runs out {function} {dtype} B{B} T{T} D{D} rows={rows} handshake={handshake}", flush=True)
    monkeypatch.setenv("FRNN_TILE_ROWS", str(rows))
    assert fetch_workgroups(function, dtype, B, T, 1, D, 1) > 0
    inp = make_inputs(function, B, T, 1, D, 7, init="zeros", round_to=KDT[dtype])
    cfg = FlashRNNConfig(head_dim=D, num_heads=1, batch_size=B, function=function, dtype=dtype)
    Wx, R, b = (inp[k].to(gpu, KDT[dtype]).requires_grad_(True) for k in ("Wx", "R", "b"))

    def forward():
        st, _ = flashrnn(Wx, R, b, None, config=cfg)
        torch.cuda.synchronize()
        return st

    def backward(st):
        g = torch.autograd.grad(st, [Wx, b], grad_outputs=torch.ones_like(st))
        torch.cuda.synchronize()
        return g

    good = forward()
    good_g = backward(good)
    assert not _reported()
    st = forward()
    if not handshake:
        monkeypatch.setenv("FRNN_AGENT_STORES", "1")  # (the handshake at the start of the kernels would give up first)
    monkeypatch.setenv("FRNN_SPIN_LIMIT", "-3")
    g = backward(st)
    k = _workgroups_per_head(function, dtype, B, D, 1)
    assert k > 1 and last_status("backward") == 1 and _reported()
    assert torch.isnan(g[1][:, :, :D - D // k].float()).all()
    monkeypatch.delenv("FRNN_SPIN_LIMIT")
    monkeypatch.delenv("FRNN_AGENT_STORES", raising=False)
    again = forward()
    again_g = backward(again)
    assert not _reported()
    assert torch.equal(again, good) and all(torch.equal(x, y) for x, y in zip(again_g, good_g))
