"""Workgroups of a scan's launch that only fetch its operands into L2: the same bits with and without them, at the edges of their rule and of
their work (short sequences, ragged tiles, fewer compute units left than groups, several launches), and single calls against the oracle."""
import pytest
import torch

from parity import check_case
from test_gpu_decode import _device_inputs

pytestmark = pytest.mark.gpu

# T: 24 is the longest sequence that goes without.  B250 N3 D256: 12 groups of an XCD share 8 such workgroups, B120 N4 the 15 groups of an XCD 2
CASES = [("lstm", "bfloat16", 5, 24, 3, 256), ("lstm", "bfloat16", 5, 25, 3, 256), ("slstm", "float16", 9, 26, 4, 192), ("gru", "bfloat16", 250, 31, 3, 256),
         ("lstm", "float16", 250, 33, 3, 256), ("lstm", "bfloat16", 517, 27, 2, 256), ("slstm", "bfloat16", 120, 29, 4, 192), ("lstm", "bfloat16", 9, 37, 1, 768),
         ("elman", "bfloat16", 17, 39, 1, 1024), ("gru", "float32", 6, 35, 3, 160), ("lstm", "float32", 33, 30, 2, 256), ("gru", "bfloat16", 131, 32, 2, 384),
         # reverse: pairs of waves, ragged 8- and 16-row tiles, several launches
         ("lstm", "float16", 7, 45, 1, 512), ("slstm", "bfloat16", 3, 25, 1, 448), ("gru", "bfloat16", 18, 49, 2, 512), ("lstm", "bfloat16", 99, 28, 4, 192),
         ("gru", "float16", 67, 26, 3, 256), ("slstm", "float16", 131, 27, 3, 256), ("gru", "bfloat16", 517, 25, 2, 256),
         ("gru", "bfloat16", 77, 26, 3, 320)]


@pytest.mark.parametrize("function,dtype,B,T,N,D", CASES)
def test_same_bits_with_and_without(gpu, monkeypatch, function, dtype, B, T, N, D):
    from flashrnn_amd import check_status, flashrnn

    print(f"case prefetch {function} {dtype} B{B} T{T} N{N} D{D}", flush=True)
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
