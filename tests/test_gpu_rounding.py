"""What is rounded where in the 16-bit types, against values known exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("function", ["lstm", "slstm"])
@pytest.mark.parametrize("D,B", [(64, 256), (256, 64), (512, 32)])  # one workgroup, tall tiles and several workgroups per head
def test_fp16_cell_states_are_rounded_once(gpu, function, D, B):
    """c = i z + f c' with i = f = 1 exactly: the stored state is the fp16 value nearest to the exact sum, not to its fp32 value.
    tanh(2^-6) and tanh(2^-7) bring sums of 32 and more, and of 16 and more, so near to the middle between two fp16 values that
    the fp32 value is that middle.  z comes from a step with f = 0, unrounded in the carry."""
    from flashrnn_amd import flashrnn, flashrnn_step, make_carry

    print(f"case rounding {function} D{D} B{B}", flush=True)
    N, S = 2, 2 if function == "lstm" else 4
    gen = torch.Generator().manual_seed(83)
    zeros = dict(dtype=torch.float16, device=gpu)
    R, b = torch.zeros(4, N, D, D, **zeros), torch.zeros(4, N, D, **zeros)
    e = torch.randint(4, 6, (B, N, D), generator=gen)
    c0 = ((torch.randint(0, 1024, (B, N, D), generator=gen) / 1024 + 1) * 2.0 ** e).to(gpu, torch.float16)
    x_z = ((torch.randint(0, 2, (B, N, D), generator=gen) * 2 - 1) * 2.0 ** (e - 11)).to(gpu, torch.float16)

    def wx(f):
        x = torch.zeros(B, 1, 4, N, D, **zeros)
        x[:, 0, 0] = 1.0 if function == "slstm" else 60000.0  # (sLSTM: i = exp(1 - m) with m = max(1, -+60000 + 1) = 1)
        x[:, 0, 1] = f
        x[:, 0, 2] = x_z
        return x

    s0 = torch.zeros(S, B, 1, N, D, **zeros)
    s0[1, :, 0] = c0
    if function == "slstm":
        s0[2:] = 1.0  # n, m
    no_c = s0.clone()
    no_c[1] = 0
    carry = make_carry(no_c)
    flashrnn_step(wx(-60000.0), R, b, no_c, function=function, dtype="float16", carry=carry)
    z = carry[1]
    # (numpy rounds 64 bits to 16 in one step)
    want = torch.from_numpy((z.double() + c0.double()).cpu().numpy().astype("float16")).to(gpu)
    assert int(((z + c0.float()).half() != want).sum()) > 0  # (there are sums that two roundings get wrong)
    got = flashrnn_step(wx(60000.0), R, b, s0, function=function, dtype="float16", carry=make_carry(s0))
    assert torch.equal(got[1, :, 0], want)
    with torch.no_grad():
        seq, _ = flashrnn(wx(60000.0), R, b, s0, function=function, dtype="float16")
    assert torch.equal(seq[1, :, 0], want)
