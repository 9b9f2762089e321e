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


@pytest.mark.parametrize("variant", ["", "1"])  # the tiling of a small call and the default one
@pytest.mark.parametrize("function,B,N,D", [("lstm", 16, 4, 256), ("lstm", 16, 2, 512), ("slstm", 16, 3, 320), ("lstm", 16, 2, 768), ("slstm", 16, 2, 192)])
def test_partial_sums_between_workgroups_keep_their_bits(gpu, monkeypatch, function, B, N, D, variant):
    """ds0 of h is R^T dg, and dg is what dWx holds (the product takes it rounded).  fp32 sums of 4 D products are off by about sqrt(4 D)
    2^-25 of the result, 2^-20 here, so about 2^-20 / 2^-11 = 0.2 % of them round to the farther of two fp16 values; if the workgroups' shares are
    rounded to 15 mantissa bits on their way, 3 % do."""
    from flashrnn_amd import flashrnn

    print(f"case partial sums {function} B{B} N{N} D{D} variant={variant}", flush=True)
    if variant:
        monkeypatch.setenv("FRNN_FUSED_VARIANT", variant)
    S = 2 if function == "lstm" else 4
    gen = torch.Generator().manual_seed(85)
    mk = lambda *s: torch.randn(*s, generator=gen).to(gpu, torch.float16)
    Wx, b, ds = mk(B, 1, 4, N, D).requires_grad_(True), mk(4, N, D) * 0.1, mk(S, B, 1, N, D)
    R = (mk(4, N, D, D).float() / D ** 0.5).half()
    s0 = mk(S, B, 1, N, D)
    if function == "slstm":
        s0[2] = s0[2].abs() + 1
    s0.requires_grad_(True)
    out, _ = flashrnn(Wx, R, b, s0, function=function, dtype="float16")
    dwx, ds0 = torch.autograd.grad(out, [Wx, s0], grad_outputs=ds)
    dg = dwx[:, 0].double().permute(1, 2, 0, 3).contiguous()             # [4, N, B, D]
    want = torch.matmul(dg, R.double()).sum(0).transpose(0, 1)            # sum over gates and rows of R[g, n, row, col]
    want = torch.from_numpy(want.cpu().numpy().astype("float16")).to(gpu)
    wrong = float((ds0[0, :, 0] != want).float().mean())
    print(f"rounded to the other neighbour: {wrong:.5f}", flush=True)
    assert wrong < 5e-3


@pytest.mark.parametrize("function", ["lstm", "gru"])
@pytest.mark.parametrize("D", [64, 256])
def test_the_sum_of_two_products_is_fused_with_the_carried_state(gpu, function, D):
    """c = fma(f, c', i z) and h = fma(z, h', (1 - z) n), the second product rounded: the bits that calls have always had.  The gates come out
    of steps that leave one of them alone (an fp32 state is stored as it is); 64 bits of mantissa hold the exact sums."""
    import numpy as np

    from flashrnn_amd import flashrnn, flashrnn_step

    print(f"case fused sum {function} D{D}", flush=True)
    B, N, big, S = 16, 2, 1e4, 2 if function == "lstm" else 1
    G = 4 if function == "lstm" else 3
    gen = torch.Generator().manual_seed(86)
    R, b = torch.zeros(G, N, D, D, device=gpu), torch.zeros(4, N, D, device=gpu)
    pre, prev = torch.randn(G, B, N, D, generator=gen), torch.randn(B, N, D, generator=gen)

    def step(gates, carried, run=None):
        x = torch.zeros(B, 1, G, N, D)
        for g, v in enumerate(gates):
            x[:, 0, g] = v
        s0 = torch.zeros(S, B, 1, N, D)
        s0[S - 1, :, 0] = carried
        args = (x.to(gpu), R, b, s0.to(gpu))
        with torch.no_grad():
            out = flashrnn_step(*args, function=function, dtype="float32") if run is None else flashrnn(*args, function=function, dtype="float32")[0]
        return out[S - 1, :, 0].cpu().numpy()

    if function == "lstm":  # gates i, f, z, o
        i, f, z = step((pre[0], -big, big, 0), 0.0), step((-big, pre[1], 0, 0), 1.0), step((big, -big, pre[2], 0), 0.0)
        gates, plain = (pre[0], pre[1], pre[2], 0), i * z
    else:                   # gates r, z, n
        f, z = step((0, pre[1], 0), 1.0), step((0, -big, pre[2]), 0.0)
        gates, plain = (0, pre[1], pre[2]), (np.float32(1) - f) * z
    carried = prev.numpy()
    want = (f.astype(np.longdouble) * carried.astype(np.longdouble) + plain.astype(np.longdouble)).astype(np.float32)
    assert (want != f * carried + plain).any()
    assert np.array_equal(step(gates, prev), want) and np.array_equal(step(gates, prev, run="sequence"), want)
