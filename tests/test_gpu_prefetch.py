"""Workgroups of a scan's launch that only fetch its operands into L2: the same bits with and without them, at the edges of their rule and of
their work (short sequences, ragged tiles, fewer compute units left than groups, several launches), and single calls against the oracle."""
import pytest
import torch

from parity import check_case
from test_fetch_rule import fetch_workgroups
from test_gpu_decode import IDLE, _device_inputs

pytestmark = pytest.mark.gpu

# T: 24 is the longest sequence that goes without.  B250 N3 D256: 12 groups of an XCD share 8 such workgroups, B120 N4 the 15 groups of an XCD 2
CASES = [("lstm", "bfloat16", 5, 24, 3, 256), ("lstm", "bfloat16", 5, 25, 3, 256), ("slstm", "float16", 9, 26, 4, 192), ("gru", "bfloat16", 250, 31, 3, 256),
         ("lstm", "float16", 250, 33, 3, 256), ("lstm", "bfloat16", 517, 27, 2, 256), ("slstm", "bfloat16", 120, 29, 4, 192), ("lstm", "bfloat16", 9, 37, 1, 768),
         ("elman", "bfloat16", 17, 39, 1, 1024), ("gru", "float32", 6, 35, 3, 160), ("lstm", "float32", 33, 30, 2, 256), ("gru", "bfloat16", 131, 32, 2, 384),
         # reverse: pairs of waves, ragged 8- and 16-row tiles, several launches
         ("lstm", "float16", 7, 45, 1, 512), ("slstm", "bfloat16", 3, 25, 1, 448), ("gru", "bfloat16", 18, 49, 2, 512), ("lstm", "bfloat16", 99, 28, 4, 192),
         ("gru", "float16", 67, 26, 3, 256), ("slstm", "float16", 131, 27, 3, 256), ("gru", "bfloat16", 517, 25, 2, 256),
         ("gru", "bfloat16", 77, 26, 3, 320)]

# forward and backward launches that have them (in the first launch of the call): all, 8 for 12 groups of an XCD, 4 for 7, 5 for 10
FORWARD = [("lstm", "bfloat16", 5, 25, 3, 256), ("gru", "bfloat16", 250, 31, 3, 256), ("lstm", "float16", 70, 33, 3, 256), ("slstm", "float16", 130, 26, 4, 192), ("gru", "float16", 131, 32, 2, 384)]
# 16-row tiles, 8-row tiles of each cell, the GRU's dense tiling, pairs of waves beyond the last-level cache
BACKWARD = [("lstm", "float16", 250, 33, 3, 256), ("lstm", "bfloat16", 99, 28, 4, 192), ("slstm", "bfloat16", 120, 29, 4, 192), ("gru", "float16", 101, 40, 3, 256), ("gru", "bfloat16", 77, 26, 3, 320),
            ("gru", "bfloat16", 199, 27, 3, 256), ("gru", "float16", 171, 26, 3, 256), ("slstm", "float16", 9, 1100, 4, 192), ("slstm", "bfloat16", 6, 6500, 1, 192)]


@pytest.mark.parametrize("function,dtype,B,T,N,D", CASES + [c for c in FORWARD + BACKWARD if c not in CASES])
def test_same_bits_with_and_without(gpu, monkeypatch, function, dtype, B, T, N, D):
    from flashrnn_amd import check_status, flashrnn

    print(f"case prefetch {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    case = (function, dtype, B, T, N, D)
    assert case not in FORWARD or fetch_workgroups(*case, 0) > 0
    assert case not in BACKWARD or fetch_workgroups(*case, 1) > 0
    x = _device_inputs(gpu, function, B, T, N, D, dtype, seed=43)
    dstates = x.pop("dstates")
    for k in x:
        x[k].requires_grad_(True)
    out = []
    for workgroups in ("0", "1", None):  # none, one per XCD, as many as the rule takes
        monkeypatch.delenv("FRNN_PREFETCH", raising=False)
        if workgroups is not None:
            monkeypatch.setenv("FRNN_PREFETCH", workgroups)
        st, _ = flashrnn(x["Wx"], x["R"], x["b"], x["states"], function=function, backend="hip_fused", dtype=dtype)
        out.append((st, *torch.autograd.grad(st, list(x.values()), grad_outputs=dstates)))
    check_status()
    for other in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(out[0], other))


@pytest.mark.parametrize("function,dtype,B,T,N,D", [("lstm", "bfloat16", 7, 41, 3, 256), ("gru", "float16", 131, 26, 2, 256), ("slstm", "float32", 5, 28, 2, 128),
                                                  ("gru", "bfloat16", 6, 26, 1, 512), ("slstm", "bfloat16", 99, 25, 4, 192)])
def test_matches_the_oracle(gpu, function, dtype, B, T, N, D):
    print(f"case prefetch oracle {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    check_case(gpu, function, B, T, N, D, dtype, "hip_fused", seed=47)


def _leaves(x):
    dstates = x.pop("dstates")
    return [v.requires_grad_(True) for v in (x["Wx"], x["R"], x["b"], x["states"])], dstates


def _pass(leaves, dstates, function, dtype):
    from flashrnn_amd import flashrnn

    st, _ = flashrnn(*leaves, function=function, backend="hip_fused", dtype=dtype)
    return (st, *torch.autograd.grad(st, leaves, grad_outputs=dstates))


def test_beside_heads_of_one_workgroup_on_another_stream(gpu):
    """Nothing orders those behind a launch whose workgroups ask for a compute unit each."""
    from flashrnn_amd import check_status

    wide, narrow = ("lstm", "bfloat16", 128, 64, 3, 256), ("gru", "bfloat16", 256, 64, 12, 64)
    print("case prefetch beside another stream", wide, narrow, flush=True)
    assert all(fetch_workgroups(*wide, b) > 0 and fetch_workgroups(*narrow, b) == 0 for b in (0, 1))
    args, want = [], []
    for (f, dt, B, T, N, D), seed in ((wide, 5), (narrow, 6)):
        args.append((*_leaves(_device_inputs(gpu, f, B, T, N, D, dt, seed=seed)), f, dt))
        want.append(_pass(*args[-1]))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for order in ((0, 1), (1, 0), (0, 1)):
        got = [None, None]
        for i in order:
            with torch.cuda.stream(streams[i]):
                got[i] = _pass(*args[i])
        torch.cuda.synchronize()
        check_status()
        for i in (0, 1):
            assert all(torch.equal(a, b) for a, b in zip(got[i], want[i])), (order, i)


def test_captured_and_replayed_beside_a_session(gpu):
    """Whether a call is made beside a session is decided at its capture; replayed beside one, it keeps the workgroups that it was captured with."""
    from flashrnn_amd import FlashRNNDecoder, check_status, flashrnn

    function, dtype, B, T, N, D = "lstm", "bfloat16", 64, 40, 3, 256
    print(f"case prefetch captured {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
    assert fetch_workgroups(function, dtype, B, T, N, D, 0) > 0
    x = _device_inputs(gpu, function, B, T, N, D, dtype, seed=7)
    y = _device_inputs(gpu, function, 4, 6, 1, D, dtype, seed=8)

    def call(v):
        with torch.no_grad():
            return flashrnn(v["Wx"], v["R"], v["b"], v["states"], function=function, dtype=dtype)[0]

    first, tokens = call(x), call(y)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(x)
    fresh = torch.randn_like(x["Wx"]).mul_(0.5)
    for Wx in (x["Wx"].clone(), fresh):
        x["Wx"].copy_(Wx)
        want = call(x)
        torch.cuda.current_stream().synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.current_stream().synchronize()
        assert torch.equal(out, want)
        out.zero_()
        got = []
        with FlashRNNDecoder(y["R"], y["b"], y["states"], function=function, dtype=dtype, idle_polls=IDLE) as session:
            for t in range(6):
                got.append(session.step(y["Wx"][:, t:t + 1].contiguous()))
                if t in (1, 3):
                    graph.replay()
                    torch.cuda.current_stream().synchronize()
                    check_status()
        torch.cuda.current_stream().synchronize()
        assert torch.equal(out, want) and torch.equal(torch.cat(got, 2), tokens)
    assert not torch.equal(first, want)
