"""The work that users of this package give it, as a list of cases that can be timed.

A case is one call (or one short chain of calls) of the public functions: ``flashrnn`` with gradients (a training step's
recurrence), ``flashrnn`` without (inference over a sequence) and ``flashrnn_step`` (token-by-token decoding).  The listed
cases are the package's benchmark configurations, the points of its batch and head-dimension sweeps at both ends, and the
short, ragged and less common calls (fp16, recompute mode, clipping, fp32 master weights) that its tests exercise.

Fields of a case: ``call`` (train, infer, step), ``function``, ``dtype`` (kernel type), ``backend``, B, T, N, D, ``weights``
(type in which the caller keeps R and b: the kernel type, or fp32 master weights that are cast on every call), ``init`` (zeros:
no states passed; randn: a given initial state), ``grad_on`` (cotangent on all states, or on h only as in a language model),
``recompute`` (no gate cache) and ``clip`` (gradient_recurrent_clipval, 0: off).
"""
import math

import torch

from flashrnn_amd import FlashRNNConfig, flashrnn, flashrnn_step, make_carry
from flashrnn_amd.flashrnn import DTYPE_DICT, rnn_function_registry

_BYTES = {"bfloat16": 2, "float16": 2, "float32": 4}


def _case(name, call, function, dtype, B, T, N, D, backend="hip_fused", weights=None, init="zeros", grad_on="all", recompute=False,
          clip=0.0):
    return dict(name=name, call=call, function=function, dtype=dtype, backend=backend, B=B, T=T, N=N, D=D,
                weights=weights or dtype, init=init, grad_on=grad_on, recompute=recompute, clip=clip)


def listed():
    return [
        # token-by-token decoding of a small batch: 16 dependent tokens, state and fp32 carry handed from call to call
        _case("step_lstm_b8_n3_d256", "step", "lstm", "bfloat16", 8, 16, 3, 256, init="randn"),
        # inference in fp32 over a short sequence: the smallest whole-sequence call
        _case("infer_lstm_f32_b4_t256_n1_d64", "infer", "lstm", "float32", 4, 256, 1, 64),
        # a short, ragged training step (odd batch, odd length), where launches and host time count
        _case("train_lstm_b5_t19_n3_d256", "train", "lstm", "bfloat16", 5, 19, 3, 256),
        # the configuration that the package's metric is quoted on
        _case("train_lstm_b8_t1024_n3_d256", "train", "lstm", "bfloat16", 8, 1024, 3, 256, init="randn"),
        # long sequences, one workgroup per head
        _case("train_gru_b16_t2048_n4_d128", "train", "gru", "bfloat16", 16, 2048, 4, 128),
        # a language-model block: sLSTM, cotangent on h only, fp32 master weights, the longest sequence
        _case("train_slstm_b16_t4096_n4_d192", "train", "slstm", "bfloat16", 16, 4096, 4, 192, weights="float32", grad_on="h"),
        # the alternating backend on a wide Elman cell
        _case("train_elman_hip_b32_t1024_n1_d1024", "train", "elman", "bfloat16", 32, 1024, 1, 1024, backend="hip"),
        # large-batch training, small heads: the end of the batch sweep, where the device is full
        _case("train_lstm_b256_t1024_n12_d64", "train", "lstm", "bfloat16", 256, 1024, 12, 64),
        # large-batch training, heads that span several workgroups
        _case("train_lstm_b256_t1024_n3_d256", "train", "lstm", "bfloat16", 256, 1024, 3, 256, weights="float32"),
        # one wide head: the end of the head-dimension sweep
        _case("train_lstm_b16_t1024_n1_d768", "train", "lstm", "bfloat16", 16, 1024, 1, 768),
        # fp32 training
        _case("train_lstm_f32_b16_t1024_n1_d512", "train", "lstm", "float32", 16, 1024, 1, 512),
        # fp16 with a ragged batch and length, activation memory saved by recompute mode, recurrent gradients clipped
        _case("train_lstm_f16_b33_t515_n8_d96_recompute", "train", "lstm", "float16", 33, 515, 8, 96, init="randn", recompute=True, clip=1.0),
    ]


# head dimensions of the fused kernels (the decode and alternating paths take them too) and of recompute mode
_DIMS = (32, 64, 96, 128, 160, 192, 256, 320, 384, 448, 512, 640, 768, 1024)
_RECOMPUTE_DIMS = (32, 64, 96, 128, 192, 256)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges above: sizes spread over their logarithm, odd ones included."""
    kind = rng.choices(("train", "infer", "train_f32", "train_hip", "step"), (5, 2, 1, 1, 1))[0]
    function = rng.choices(("lstm", "slstm", "gru", "elman"), (4, 2, 2, 1))[0]
    dtype = rng.choices(("bfloat16", "float16"), (3, 1))[0]
    backend, recompute, clip = "hip_fused", False, 0.0
    if kind == "train_f32":
        call, dtype = "train", "float32"
        D = rng.choice([d for d in _DIMS if d <= 512])
        B, T = _log_int(rng, 1, 64), _log_int(rng, 16, 1024)
    elif kind == "train_hip":
        call, backend = "train", "hip"
        D = rng.choice(_DIMS)
        B, T = _log_int(rng, 1, 64), _log_int(rng, 16, 512 if function != "elman" else 1024)
    elif kind == "step":
        call, backend = "step", rng.choice(("hip_fused", "hip"))
        D = rng.choice(_DIMS)
        B, T = _log_int(rng, 1, 64), _log_int(rng, 4, 64)
    else:
        call = kind
        D = rng.choice(_DIMS)
        if call == "infer" and rng.random() < 0.25:
            dtype, D = "float32", rng.choice([d for d in _DIMS if d <= 512])
        recompute = call == "train" and function != "elman" and D in _RECOMPUTE_DIMS and rng.random() < 0.15
        clip = 1.0 if call == "train" and rng.random() < 0.2 else 0.0
        B, T = _log_int(rng, 1, 256), _log_int(rng, 16, 4096)
    N = rng.randint(1, max(1, 768 // D))
    # no more tokens than the largest listed case has, and (wide heads need several launches at large batches) no more than
    # about 2048 x 16 rows at D >= 512
    most = (256 * 1024 * 768) // (N * D)
    if D >= 512:
        most = min(most, 2048 * 16)
    if dtype == "float32":
        most = min(most, 1024 * 16)
    T = max(4, min(T, most // B))
    weights = "float32" if call == "train" and rng.random() < 0.3 else dtype
    return dict(call=call, function=function, dtype=dtype, backend=backend, B=B, T=T, N=N, D=D, weights=weights,
                init="randn" if call == "step" else rng.choice(("zeros", "randn")), grad_on=rng.choice(("all", "h")), recompute=recompute,
                clip=clip)


def prepare(case, seed):
    """Inputs with the distributions of the package's tests: Wx ~ N(0, 1), R ~ N(0, 1/D), small biases."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kdt, wdt = DTYPE_DICT[case["dtype"]], DTYPE_DICT[case["weights"]]
    Gr, Gw, _, Gt, S = rnn_function_registry[case["function"]]["gates_states"]
    B, T, N, D = case["B"], case["T"], case["N"], case["D"]

    def randn(*shape, dtype=kdt):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32 if dtype == torch.float32 else dtype)

    st = {"case": case}
    st["R"] = (randn(Gr, N, D, D, dtype=torch.float32) / D ** 0.5).to(wdt)
    st["b"] = (randn(Gt, N, D, dtype=torch.float32) * 0.1).to(wdt)
    st["states"] = None
    if case["init"] == "randn":
        s0 = randn(S, B, 1, N, D)
        if case["function"] == "slstm":
            s0[2] = s0[2].abs() + 1.0  # (a state that the cell can reach: n >= 1)
        st["states"] = s0
    st["config"] = FlashRNNConfig(backend=case["backend"], function=case["function"], dtype=case["dtype"], head_dim=D, num_heads=N,
                                  batch_size=B, recompute_gates=case["recompute"], gradient_recurrent_clipval=case["clip"] or None)
    if case["call"] == "step":
        st["Wx"] = [randn(B, 1, Gw, N, D) for _ in range(T)]
        return st
    st["Wx"] = randn(B, T, Gw, N, D)
    if case["call"] == "train":
        ds = randn(S, B, T, N, D)
        if case["grad_on"] == "h":
            ds[1:] = 0
        st["dstates"] = ds
        for k in ("Wx", "R", "b", "states"):
            if st[k] is not None:
                st[k].requires_grad_(True)
    return st


def run(st):
    case = st["case"]
    if case["call"] == "step":
        s, carry, out = st["states"], make_carry(st["states"]), []
        for wx in st["Wx"]:
            s = flashrnn_step(wx, st["R"], st["b"], s, config=st["config"], carry=carry)
            out.append(s)
        return {"states": out, "carry": carry}
    if case["call"] == "infer":
        with torch.no_grad():
            states, last = flashrnn(st["Wx"], st["R"], st["b"], st["states"], config=st["config"])
        return {"states": states, "last": last}
    leaves = {k: st[k] for k in ("Wx", "R", "b", "states") if st[k] is not None}
    states, _ = flashrnn(st["Wx"], st["R"], st["b"], st["states"], config=st["config"])
    grads = torch.autograd.grad(states, list(leaves.values()), grad_outputs=st["dstates"])
    return {"states": states.detach(), **{"d" + k: v for k, v in zip(leaves, grads)}}


def work(case):
    """Inputs read once, outputs written once; the recurrent product forward, its transpose and dR backward."""
    Gr, Gw, _, Gt, S = rnn_function_registry[case["function"]]["gates_states"]
    B, T, N, D = case["B"], case["T"], case["N"], case["D"]
    es, ws = _BYTES[case["dtype"]], _BYTES[case["weights"]]
    tokens, unit = B * T, N * D
    seq = tokens * unit * es
    params = (Gr * unit * D + Gt * unit) * ws
    s0 = S * B * unit * es
    flops = 2.0 * tokens * Gr * unit * D
    if case["call"] == "train":
        given = s0 if case["init"] == "randn" else 0
        # read Wx, the cotangent, R, b (and s0); write the states and the gradients of what was given
        return {"bytes": float(seq * (2 * Gw + 2 * S) + 2 * params + 2 * given), "flops": 3 * flops}
    if case["call"] == "step":
        return {"bytes": float(seq * (Gw + S) + params + s0 + 2 * S * B * unit * 4), "flops": flops}
    return {"bytes": float(seq * (Gw + S) + params + (s0 if case["init"] == "randn" else 0)), "flops": flops}


def tolerance(case):
    """About four times the largest relative difference seen (per output) against the other backend, whose sums run in
    another order, and against an fp32 run on the same inputs: bf16 training 2-4.7e-3, sequences without gradients 1.7e-3;
    fp16 5e-4 and 2.2e-4; fp32 against the other order 7e-7 (up to 2e-6 element-wise over 1024 steps)."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    train = case["call"] == "train"
    return {"rel": (1.6e-2 if train else 7e-3) if case["dtype"] == "bfloat16" else (2e-3 if train else 1e-3)}


class _ClampGrad(torch.autograd.Function):
    """Identity whose cotangent is clamped to [-v, v]."""

    @staticmethod
    def forward(ctx, x, v):
        ctx.v = v
        return x.view_as(x)

    @staticmethod
    def backward(ctx, g):
        return g.clamp(-ctx.v, ctx.v), None


def _cell(function, x, y, b, s):
    """One step of a cell.  The stabiliser of the sLSTM is held constant in its adjoint, and the guard max(n, 1) is
    transparent there, as in the kernels."""
    sig, tanh = torch.sigmoid, torch.tanh
    if function == "elman":
        return (tanh(x[0] + y[0] + b[0]),)
    if function == "gru":
        r, z = sig(x[0] + y[1] + b[1]), sig(x[1] + y[2] + b[2])
        return (z * s[0] + (1 - z) * tanh(x[2] + b[3] + r * (y[0] + b[0])),)
    i, f, z, o = (x[k] + y[k] + b[k] for k in range(4))
    if function == "lstm":
        c = sig(f) * s[1] + sig(i) * tanh(z)
        return (sig(o) * tanh(c), c)
    lf = torch.nn.functional.logsigmoid(f) + s[3].detach()
    m = torch.where(s[2] == 0, i, torch.maximum(i, lf)).detach()
    i, f = torch.exp(i - m), torch.exp(lf - m)
    c, n = f * s[1] + i * tanh(z), f * s[2] + i
    n = n + (n.clamp(min=1.0) - n).detach()
    return (sig(o) * c / n, c, n, m)


def exact(case, seed):
    """What ``run`` returns, in 64 bits: the parameters and inputs as the kernels take them (rounded to the kernel type)."""
    st = prepare(case, seed)
    Gr, _, _, _, S = rnn_function_registry[case["function"]]["gates_states"]
    kdt, (B, N, D) = DTYPE_DICT[case["dtype"]], (case["B"], case["N"], case["D"])
    step, train = case["call"] == "step", case["call"] == "train"
    leaf = {"Wx": torch.cat(st["Wx"], 1) if step else st["Wx"], "R": st["R"], "b": st["b"], "states": st["states"]}
    leaf = {k: v.detach().to(kdt).double().requires_grad_(train) for k, v in leaf.items() if v is not None}
    s = tuple(leaf["states"][:, :, 0].unbind(0)) if "states" in leaf else tuple(leaf["Wx"].new_zeros(B, N, D) for _ in range(S))
    with torch.set_grad_enabled(train):
        R = leaf["R"].permute(1, 3, 0, 2).reshape(N, D, Gr * D).contiguous()
        b, out = leaf["b"].unbind(0), []
        for t, wx in enumerate(leaf["Wx"].unbind(1)):
            if case["clip"] and t:
                s = (_ClampGrad.apply(s[0], case["clip"]),) + s[1:]
            y = torch.bmm(s[0].transpose(0, 1), R).reshape(N, B, Gr, D).permute(2, 1, 0, 3)
            s = _cell(case["function"], wx.unbind(1), y.unbind(0), b, s)
            out.append(torch.stack(s))
        states = torch.stack(out, 2)
    if step:
        return {"states": [x[:, :, None] for x in out], "carry": out[-1]}
    if not train:
        return {"states": states, "last": states[:, :, -1:]}
    grads = torch.autograd.grad(states, list(leaf.values()), grad_outputs=st["dstates"].double())
    return {"states": states.detach(), **{"d" + k: v for k, v in zip(leaf, grads)}}
