"""Decode sessions beside each other and beside sequence calls: the workgroups of all of them stay on the device together, so they
run in the default tilings, and forward calls keep their bits."""
import pytest
import torch

from test_gpu_decode import IDLE, _device_inputs

pytestmark = pytest.mark.gpu

CASES = [("lstm", 4, 1, 768, "bfloat16"), ("slstm", 3, 1, 384, "float16"), ("gru", 4, 1, 1024, "bfloat16"), ("gru", 2, 1, 640, "float16"),
         ("lstm", 4, 1, 512, "float32"), ("slstm", 4, 1, 256, "float32"), ("gru", 16, 4, 192, "float32"), ("lstm", 4, 8, 320, "float32"), ("lstm", 3, 1, 160, "float32")]


@pytest.mark.parametrize("function,B,N,D,dtype", CASES)
def test_two_sessions_and_a_sequence_call_beside_one(gpu, function, B, N, D, dtype):
    from flashrnn_amd import FlashRNNDecoder, check_status, flashrnn

    print(f"case sessions {function} B{B} N{N} D{D} {dtype}", flush=True)
    T = 6
    x = _device_inputs(gpu, function, B, T, N, D, dtype, seed=91)
    y = _device_inputs(gpu, function, B, T, N, D, dtype, seed=92)

    def sequence(v, train=False):
        if not train:
            with torch.no_grad():
                return flashrnn(v["Wx"], v["R"], v["b"], v["states"], function=function, dtype=dtype)[0]
        leaves = [v[k].clone().requires_grad_() for k in ("Wx", "R", "b", "states")]
        out = flashrnn(*leaves, function=function, dtype=dtype)[0]
        return [out.detach(), *torch.autograd.grad(out, leaves, grad_outputs=torch.ones_like(out))]

    ref_x, ref_y, trained = sequence(x), sequence(y), sequence(y, True)
    torch.cuda.current_stream().synchronize()
    kw = dict(function=function, dtype=dtype, idle_polls=IDLE)
    with FlashRNNDecoder(x["R"], x["b"], x["states"], **kw) as one, FlashRNNDecoder(y["R"], y["b"], y["states"], **kw) as two:
        out_x, out_y = [], []
        for t in range(T):  # both make progress in turn
            out_x.append(one.step(x["Wx"][:, t:t + 1].contiguous()))
            out_y.append(two.step(y["Wx"][:, t:t + 1].contiguous()))
    torch.cuda.current_stream().synchronize()
    assert torch.equal(torch.cat(out_x, 2), ref_x) and torch.equal(torch.cat(out_y, 2), ref_y)
    with FlashRNNDecoder(x["R"], x["b"], x["states"], **kw) as one:
        out_x = [one.step(x["Wx"][:, :2].contiguous())]
        beside, again = sequence(y), sequence(y, True)
        check_status()
        out_x.append(one.step(x["Wx"][:, 2:6].contiguous()))
    torch.cuda.current_stream().synchronize()
    assert torch.equal(beside, ref_y) and torch.equal(again[0], trained[0])
    assert torch.equal(torch.cat(out_x, 2), ref_x)
    # (the reverse scan's sums over workgroups come in another order: two roundings of the storage type, by the longest chain of steps)
    eps = {"float32": 2.0 ** -19, "float16": 2.0 ** -10, "bfloat16": 2.0 ** -7}[dtype]
    for a, b in zip(again[1:], trained[1:]):
        assert torch.isfinite(a.float()).all()
        assert float((a.float() - b.float()).norm() / b.float().norm()) < eps
    again = sequence(y, True)  # closed: the tilings of a device without sessions
    assert all(torch.equal(a, b) for a, b in zip(again, trained))


def test_a_session_that_idled_out_is_none(gpu):
    """Sequence calls look at the kernel, not at close(): a session that nobody closed counts while it runs."""
    from flashrnn_amd import FlashRNNDecoder, flashrnn

    print("case sessions idle", flush=True)
    x = _device_inputs(gpu, "lstm", 4, 4, 1, 768, "bfloat16", seed=93)

    def train():
        leaves = [x[k].clone().requires_grad_() for k in ("Wx", "R", "b", "states")]
        out = flashrnn(*leaves)[0]
        return [out.detach(), *torch.autograd.grad(out, leaves, grad_outputs=torch.ones_like(out))]

    alone = train()
    dec = FlashRNNDecoder(x["R"], x["b"], x["states"], idle_polls=1 << 14)
    dec.kernel_stream.synchronize()  # (nobody posts)
    assert all(torch.equal(a, b) for a, b in zip(train(), alone))  # (the spread tilings again)
    dec.close()
