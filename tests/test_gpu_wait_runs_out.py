"""A wait between the workgroups of a head that really probes and runs out (spin limit -1: the first probe that does not
find every word ends the wait).  Whether a wait of a call runs out depends on the timing of that call; either way every
kernel ends normally, a call that reports nothing has the right results, and one that reports a failed wait has NaN in
the outputs of the workgroup that gave up."""
import pytest
import torch

from oracle import make_inputs

pytestmark = pytest.mark.gpu

KDT = {"bfloat16": torch.bfloat16, "float32": torch.float32, "float16": torch.float16}
# function, dtype, B, N, D, recompute: one case per form of the wait (pairs of words in one and in several rounds, single
# words of 16 and 32 bits, destinations in groups, wave pairs that share the receive, the wait split around the rebuild)
CASES = [
    ("lstm", "bfloat16", 8, 1, 256, False),
    ("gru", "float16", 5, 1, 320, False),
    ("slstm", "bfloat16", 16, 1, 768, False),
    ("lstm", "bfloat16", 9, 1, 1024, False),
    ("elman", "bfloat16", 3, 1, 512, False),
    ("elman", "float32", 4, 1, 256, False),
    ("lstm", "float32", 4, 1, 512, False),
    ("gru", "float32", 3, 1, 640, False),
    ("slstm", "bfloat16", 8, 1, 192, True),
    ("lstm", "bfloat16", 64, 1, 192, True),
]


@pytest.mark.parametrize("function,dtype,B,N,D,recompute", CASES)
def test_waits_that_run_out_end_the_kernels_and_are_reported(gpu, monkeypatch, function, dtype, B, N, D, recompute):
    from flashrnn_amd import FlashRNNConfig, check_status, flashrnn, last_status

    print(f"case wait runs out {function} {dtype} B{B} N{N} D{D} recompute={recompute}", flush=True)
    kdt, T = KDT[dtype], 48
    inp = make_inputs(function, B, T, N, D, 7, init="zeros", round_to=kdt if kdt != torch.float32 else None)
    cfg = FlashRNNConfig(head_dim=D, num_heads=N, batch_size=B, function=function, dtype=dtype, recompute_gates=recompute)
    Wx, R, b = (inp[k].to(gpu, kdt).requires_grad_(True) for k in ("Wx", "R", "b"))

    def forward():
        st, _ = flashrnn(Wx, R, b, None, config=cfg)
        torch.cuda.synchronize()
        return st

    def backward(st):
        g = torch.autograd.grad(st, [Wx, b], grad_outputs=torch.ones_like(st))
        torch.cuda.synchronize()
        return g

    def reported():
        try:
            check_status()
        except RuntimeError:
            return True
        return False

    good = forward()
    good_g = backward(good)
    assert not reported()
    st = forward()
    monkeypatch.setenv("FRNN_AGENT_STORES", "1")  # (no handshake at the start of the kernels: it would give up first)
    monkeypatch.setenv("FRNN_SPIN_LIMIT", "-1")
    g = backward(st)
    failed_b = last_status("backward") == 1
    assert reported() == failed_b
    bad = forward()
    failed_f = last_status("forward") == 1
    assert reported() == failed_f
    monkeypatch.delenv("FRNN_SPIN_LIMIT")
    monkeypatch.delenv("FRNN_AGENT_STORES")
    if failed_f:
        assert torch.isnan(bad[0]).any()
    else:
        assert torch.equal(bad, good)
    if failed_b:
        assert torch.isnan(g[1].float()).any()
    else:
        assert all(torch.equal(x, y) for x, y in zip(g, good_g))
    again = forward()  # and nothing is left behind
    again_g = backward(again)
    assert not reported()
    assert torch.equal(again, good) and all(torch.equal(x, y) for x, y in zip(again_g, good_g))
