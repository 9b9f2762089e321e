"""A wait between the workgroups of a head that runs out inside the time loop.  The host leaves one workgroup of every head out
of the launch (FRNN_SPIN_LIMIT=-3), so that the others wait for its words in vain, in the first step that waits, whatever the
timing: every workgroup of the head has to give up, leave the loop together with all its waves and end normally, the call has
to report it, and the outputs of those workgroups have to be NaN."""
import ctypes

import pytest
import torch

from oracle import make_inputs

pytestmark = pytest.mark.gpu

KDT = {"bfloat16": torch.bfloat16, "float32": torch.float32, "float16": torch.float16}
# function, dtype, B, D, batch rows per tile, recompute: at least one case per form of the forward and of the reverse wait
CASES = [
    # 16-bit types, forward: pairs of words behind the own slice, with and without a producer wave; single words
    ("lstm", "bfloat16", 8, 256, 4, False),
    ("slstm", "bfloat16", 16, 768, 8, False),
    ("slstm", "bfloat16", 8, 192, 4, False),
    # ... 16 words per probe, in one round and in several, with and without the own slice in front (GRU at 16 rows: lane conditions)
    ("gru", "bfloat16", 5, 1024, 4, False),
    ("gru", "float16", 20, 1024, 8, False),
    ("gru", "bfloat16", 17, 1024, 16, False),
    ("lstm", "bfloat16", 16, 640, 16, False),
    ("slstm", "bfloat16", 16, 640, 16, False),
    # ... wave pairs that split k forward, the destinations and the sources in reverse, in one round and in several
    ("lstm", "bfloat16", 9, 1024, 4, False),
    ("slstm", "float16", 16, 1024, 8, False),
    ("lstm", "bfloat16", 16, 1024, 16, False),
    # ... reverse: up to 32 words per probe; lane conditions and give-up in front of the next probe
    ("gru", "float16", 16, 512, 16, False),
    ("elman", "bfloat16", 3, 1024, 4, False),
    # ... recompute mode: the wait split around the rebuild, at 16-row tiles with lane conditions
    ("slstm", "bfloat16", 8, 192, 4, True),
    ("lstm", "bfloat16", 12, 256, 8, True),
    ("lstm", "float16", 16, 192, 16, True),
    ("slstm", "bfloat16", 16, 128, 16, True),
    ("gru", "bfloat16", 16, 256, 16, True),
    # fp32: the 4x4x1 form, without a split, in wave pairs, in fours over the device (with a pause between reverse probes)
    ("gru", "float32", 4, 256, 4, False),
    ("lstm", "float32", 4, 320, 4, False),
    ("lstm", "float32", 4, 384, 4, False),
    ("slstm", "float32", 3, 512, 4, False),
    ("gru", "float32", 4, 512, 4, False),
    ("gru", "float32", 3, 640, 4, False),
    ("lstm", "float32", 4, 1024, 4, False),
    # ... the 16x16x4 form: one round and several, few words and 16 per probe
    ("lstm", "float32", 16, 256, 16, False),
    ("gru", "float32", 16, 160, 16, False),
    ("elman", "float32", 16, 512, 16, False),
    ("elman", "float32", 8, 1024, 8, False),
]


def _workgroups_per_head(function, dtype, B, D, backward):
    from flashrnn_amd._lib import DTYPE_IDS, FUNCTION_IDS, load_library

    v = [ctypes.c_int() for _ in range(4)]
    assert load_library().frnn_fused_plan(FUNCTION_IDS[function], DTYPE_IDS[dtype], B, 1, D, backward, *map(ctypes.byref, v)) == 0
    return v[2].value


def _reported():
    from flashrnn_amd import check_status

    try:
        check_status()
    except RuntimeError:
        return True
    return False


@pytest.mark.parametrize("handshake", [False, True])
@pytest.mark.parametrize("function,dtype,B,D,rows,recompute", CASES)
def test_waits_that_run_out_end_the_kernels_and_are_reported(gpu, monkeypatch, function, dtype, B, D, rows, recompute, handshake):
    from flashrnn_amd import FlashRNNConfig, flashrnn, last_status

    print(f"case wait runs out {function} {dtype} B{B} D{D} rows={rows} recompute={recompute} handshake={handshake}", flush=True)
    monkeypatch.setenv("FRNN_TILE_ROWS", str(rows))
    kdt, T = KDT[dtype], 13
    inp = make_inputs(function, B, T, 1, D, 7, init="zeros", round_to=kdt if kdt != torch.float32 else None)
    cfg = FlashRNNConfig(head_dim=D, num_heads=1, batch_size=B, function=function, dtype=dtype, recompute_gates=recompute)
    Wx, R, b = (inp[k].to(gpu, kdt).requires_grad_(True) for k in ("Wx", "R", "b"))

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
    kb = _workgroups_per_head(function, dtype, B, D, 2 if recompute else 1)
    assert kb > 1 and last_status("backward") == 1 and _reported()
    assert torch.isnan(g[1][:, :, :D - D // kb].float()).all()  # db of every workgroup that ran
    kf = _workgroups_per_head(function, dtype, B, D, 0)
    bad = forward()
    if kf > 1:
        assert last_status("forward") == 1 and _reported()
        assert torch.isnan(bad[0][..., :D - D // kf].float()).all()  # h of every workgroup that ran, all steps
    else:  # (a head of one workgroup waits for nobody)
        assert not _reported() and torch.equal(bad, good)
    monkeypatch.delenv("FRNN_SPIN_LIMIT")
    monkeypatch.delenv("FRNN_AGENT_STORES", raising=False)
    again = forward()  # and nothing is left behind
    again_g = backward(again)
    assert not _reported()
    assert torch.equal(again, good) and all(torch.equal(x, y) for x, y in zip(again_g, good_g))


@pytest.mark.parametrize("function,dtype,B,D", [("lstm", "bfloat16", 8, 256), ("gru", "float16", 8, 1024), ("lstm", "float32", 4, 512)])
def test_heads_with_all_their_workgroups_are_not_touched(gpu, monkeypatch, function, dtype, B, D):
    """Calls that wait for nobody keep their grid whole under the same setting: single steps and truncated backpropagation."""
    from flashrnn_amd import FlashRNNConfig, flashrnn, flashrnn_step, make_carry

    print(f"case nobody left out {function} {dtype} B{B} D{D}", flush=True)
    kdt, T = KDT[dtype], 5
    inp = make_inputs(function, B, T, 1, D, 3, init="zeros", round_to=kdt if kdt != torch.float32 else None)
    Wx, R, b = (inp[k].to(gpu, kdt).requires_grad_(True) for k in ("Wx", "R", "b"))
    cfg = FlashRNNConfig(head_dim=D, num_heads=1, batch_size=B, function=function, dtype=dtype, gradient_recurrent_cut=True)
    st, _ = flashrnn(Wx, R, b, None, config=cfg)
    s0 = torch.zeros_like(st[:, :, :1]).detach()

    def calls():
        g = torch.autograd.grad(st, [Wx, b], grad_outputs=torch.ones_like(st), retain_graph=True)
        step = flashrnn_step(Wx[:, :1].detach().contiguous(), R.detach(), b.detach(), s0, config=cfg, carry=make_carry(s0))
        torch.cuda.synchronize()
        return (*g, step)

    want = calls()
    monkeypatch.setenv("FRNN_SPIN_LIMIT", "-3")
    got = calls()
    assert not _reported()
    assert all(torch.equal(x, y) for x, y in zip(got, want))
