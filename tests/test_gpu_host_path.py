"""flashrnn() through the host module (csrc/host_torch.cpp) against the autograd function in Python, which every call takes that the
module does not: the same bits, and the same behaviour towards autograd."""
import pytest
import torch
import torch.utils.checkpoint

from oracle import make_inputs


class _Mode(torch.overrides.TorchFunctionMode):
    """Any active mode sends a call down the general path."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _leaves(gpu, function="lstm", B=5, T=7, N=2, D=64, dtype=torch.bfloat16, weights=None):
    inp = make_inputs(function, B, T, N, D, 3, init="randn", round_to=torch.bfloat16)
    return [inp["Wx"].to(gpu, dtype).requires_grad_(), inp["R"].to(gpu, weights or dtype).requires_grad_(),
            inp["b"].to(gpu, weights or dtype).requires_grad_(), inp["states"].to(gpu, dtype).requires_grad_()]


def test_only_plain_calls_take_the_host_module():
    import importlib

    fr = importlib.import_module("flashrnn_amd.flashrnn")
    cfg = fr.FlashRNNConfig(head_dim=32, num_heads=1)
    x = [torch.zeros(2, 3, 4, 1, 32), torch.nn.Parameter(torch.zeros(4, 1, 32, 32)), torch.zeros(4, 1, 32)]
    assert fr._plain(cfg, *x, None) and fr._plain(cfg, *x, torch.zeros(2, 2, 1, 1, 32))
    assert not fr._plain(fr.FlashRNNConfig(head_dim=32, num_heads=1, input_shape="TBGHD"), *x, None)
    assert not fr._plain(fr.FlashRNNConfig(head_dim=32, num_heads=1, initial_val=0.5), *x, None)
    assert not fr._plain(cfg, x[0].as_subclass(type("Sub", (torch.Tensor,), {})), x[1], x[2], None)
    with _Mode():
        assert not fr._plain(cfg, *x, None)
    with torch.autograd.forward_ad.dual_level():
        assert not fr._plain(cfg, *x, None)
    seen = []
    torch.func.vmap(lambda w: (seen.append(fr._plain(cfg, w, x[1], x[2], None)), w)[1])(x[0][None])
    torch.jit.trace(lambda w: (seen.append(fr._plain(cfg, w, x[1], x[2], None)), w + 1)[1], x[0], check_trace=False)
    assert seen == [False, False]


@pytest.mark.gpu
@pytest.mark.parametrize("function,D,backend,options,dtype,weights", [
    ("lstm", 256, "hip_fused", {}, torch.bfloat16, None), ("gru", 64, "hip", {}, torch.bfloat16, None),
    ("slstm", 64, "hip_fused", {"recompute_gates": True}, torch.float16, torch.float32),
    ("lstm", 64, "hip_fused", {"gradient_recurrent_clipval": 0.5, "forward_clipval": 0.7}, torch.float32, None),
    ("elman", 32, "hip", {"gradient_recurrent_cut": True}, torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("given", [True, False])
def test_both_paths_give_the_same_bits(gpu, function, D, backend, options, dtype, weights, given):
    from flashrnn_amd import FlashRNNConfig, flashrnn

    name = {torch.bfloat16: "bfloat16", torch.float16: "float16", torch.float32: "float32"}[dtype]
    print(f"case host path {function} D{D} {backend} {options} {name}", flush=True)
    cfg = FlashRNNConfig(backend=backend, function=function, dtype=name, head_dim=D, num_heads=2, **options)
    leaves = _leaves(gpu, function, D=D, dtype=dtype, weights=weights)
    leaves[0] = torch.cat([leaves[0].detach()] * 2, dim=1)[:, ::2].requires_grad_()  # (not contiguous)
    if not given:
        leaves = leaves[:3]

    def run():
        out, last = flashrnn(*leaves, config=cfg)
        g = torch.autograd.grad([out, last], leaves, [out.detach(), last.detach()])
        return [out.detach(), last.detach(), *g]

    got = run()
    with _Mode():
        ref = run()
    with torch.no_grad():
        plain = flashrnn(*leaves, config=cfg)
    for x, y in zip(got + list(plain), ref + ref[:2]):
        assert x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.gpu
def test_autograd_meets_the_function_it_knows(gpu):
    from flashrnn_amd import flashrnn

    print("case host path autograd", flush=True)
    leaves = _leaves(gpu)
    out, _ = flashrnn(*leaves)
    one = torch.autograd.grad(out.float().sum(), leaves, retain_graph=True)
    two = torch.autograd.grad(out.float().sum(), leaves[1:2])  # (a part of the inputs, and the graph a second time)
    assert torch.equal(one[1], two[0])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.float().sum(), leaves)
    out, _ = flashrnn(*leaves)  # no second derivative: an error where it is asked for
    g = torch.autograd.grad((out.float() ** 2).sum(), leaves[0], create_graph=True)[0]
    with pytest.raises(RuntimeError, match="once_differentiable"):
        g.float().sum().backward()
    packed = []  # saved-tensor hooks see what the function saves, and the reverse pass what they give back
    with torch.autograd.graph.saved_tensors_hooks(lambda x: (packed.append(x.shape), x.cpu())[1], lambda x: x.to(gpu)):
        out, _ = flashrnn(*leaves)
    hooked = torch.autograd.grad(out.float().sum(), leaves)
    assert len(packed) >= 5 and all(torch.equal(x, y) for x, y in zip(one, hooked))
    out = torch.utils.checkpoint.checkpoint(lambda *x: flashrnn(*x)[0], *leaves, use_reentrant=False)  # (its hooks end the second call early)
    again = torch.autograd.grad(out.float().sum(), leaves)
    assert all(torch.equal(x, y) for x, y in zip(one, again))
    R = leaves[1].detach().clone().requires_grad_()
    out, _ = flashrnn(leaves[0], R, *leaves[2:])
    with torch.no_grad():
        R.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out.float().sum(), leaves[0])
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda w: flashrnn(w, *[x.detach() for x in leaves[1:]])[0])(leaves[0].detach()[None])
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
        flashrnn(torch.autograd.forward_ad.make_dual(leaves[0].detach(), torch.ones_like(leaves[0])), *leaves[1:])
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_compiled_caller(gpu):
    """torch.compile of a caller: its graph breaks at the call, which takes the Python path."""
    from flashrnn_amd import flashrnn

    print("case host path compiled caller", flush=True)
    leaves = _leaves(gpu)

    def loss(*x):
        return flashrnn(*x)[0].float().square().sum()

    ref = torch.autograd.grad(loss(*leaves), leaves)
    got = torch.autograd.grad(torch.compile(loss, backend="eager")(*leaves), leaves)
    assert all(torch.equal(x, y) for x, y in zip(ref, got))


@pytest.mark.gpu
def test_compiled_autograd(gpu):
    from flashrnn_amd import FlashRNNConfig, flashrnn

    print("case host path compiled autograd", flush=True)
    for options in ({}, {"gradient_recurrent_clipval": 0.25, "recompute_gates": True}):
        cfg = FlashRNNConfig(head_dim=64, num_heads=2, **options)
        leaves = _leaves(gpu)
        ref = torch.autograd.grad(flashrnn(*leaves, config=cfg)[0].float().square().sum(), leaves)
        value = flashrnn(*leaves, config=cfg)[0].float().square().sum()
        with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
            value.backward()
        assert all(torch.equal(x, y.grad) for x, y in zip(ref, leaves))


@pytest.mark.gpu
def test_threads_share_the_record_of_failed_waits(gpu):
    import threading

    from flashrnn_amd import check_status, flashrnn

    print("case host path threads", flush=True)
    x = [v.detach() for v in _leaves(gpu, D=256)]
    ref, results = flashrnn(*x)[0], [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            results[i] = [flashrnn(*x)[0] for _ in range(50)]
            torch.cuda.current_stream().synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    check_status()
    assert all(torch.equal(y, ref) for r in results for y in r)


@pytest.mark.gpu
def test_a_failed_wait_is_named_behind_more_calls_than_the_ring_holds(gpu, monkeypatch):
    from flashrnn_amd import check_status, flashrnn, last_status

    print("case host path status ring", flush=True)
    x = [v.detach() for v in _leaves(gpu, T=2, D=256)]
    with torch.no_grad():
        for _ in range(4100):
            flashrnn(*x)
        check_status()
        monkeypatch.setenv("FRNN_SPIN_LIMIT", "-2")
        flashrnn(*x)
        monkeypatch.delenv("FRNN_SPIN_LIMIT")
        assert last_status("forward") == 1
        with pytest.raises(RuntimeError, match="forward of lstm B5 T2 N2 D256"):
            flashrnn(*x)
        flashrnn(*x)
    check_status()
    assert last_status("forward") == 0


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["R", "b", "states"])
def test_tensors_of_another_device_are_refused_on_the_host(gpu, monkeypatch, name):
    """Weights or a state left on the CPU: an error before anything is launched, on every path."""
    from flashrnn_amd import FlashRNNConfig, FlashRNNDecoder, flashrnn, flashrnn_step

    print(f"case host path device {name}", flush=True)

    def inputs(D, T=4):
        x = dict(zip(("Wx", "R", "b", "states"), (v.detach() for v in _leaves(gpu, D=D, T=T))))
        x[name] = x[name].cpu()
        return x

    refused = pytest.raises(RuntimeError, match="is on cpu|got a CPU tensor")
    for D in (64, 16):  # (two heads of 16 units run as one)
        with refused:
            flashrnn(**inputs(D))
    x = inputs(64)
    with _Mode(), refused:
        flashrnn(**x)
    x["Wx"].requires_grad_()
    with refused:
        flashrnn(**x)
    with refused:
        flashrnn(**inputs(64), config=FlashRNNConfig(head_dim=64, num_heads=2, backend="hip"))
    with refused:
        flashrnn_step(**inputs(64, T=1))
    with refused:
        FlashRNNDecoder(*[inputs(64)[k] for k in ("R", "b", "states")])
    monkeypatch.setenv("FRNN_TEST_MAX_BATCH", "2")  # (ranges of the batch)
    with refused:
        flashrnn(**inputs(64))


@pytest.mark.gpu
def test_the_last_result_of_a_kind_outlives_its_word(gpu, monkeypatch):
    """A backward call that failed stays the last backward call, however many forward calls use the words behind it."""
    from flashrnn_amd import check_status, flashrnn, last_status

    print("case host path last status", flush=True)
    leaves = _leaves(gpu, T=2, D=256)
    out, _ = flashrnn(*leaves)
    monkeypatch.setenv("FRNN_SPIN_LIMIT", "-2")
    torch.autograd.grad(out.float().sum(), leaves)
    monkeypatch.delenv("FRNN_SPIN_LIMIT")
    with pytest.raises(RuntimeError, match="backward of lstm B5 T2 N2 D256"):
        check_status()
    with torch.no_grad():
        for _ in range(4200):
            flashrnn(*leaves)
    assert last_status("backward") == 1 and last_status("forward") == 0
    check_status()


@pytest.mark.gpu
def test_a_word_stays_with_its_call_until_that_is_launched(gpu):
    """Another thread's call that took its words and is not launched yet, while this one makes more calls than there are words."""
    import ctypes

    from flashrnn_amd import _lib, check_status, flashrnn

    print("case host path late launch", flush=True)
    x = [v.detach() for v in _leaves(gpu, T=2, D=256)]
    host, stream = _lib.load_host(), torch.cuda.current_stream().cuda_stream
    one, shared, *late = host.status_take(1, 2, 7, 9, 3, 512, stream)
    with torch.no_grad():
        for _ in range(4200):
            flashrnn(*x)
    torch.cuda.synchronize()
    for word in (one, shared):  # what its kernel does where a wait runs out
        ctypes.c_int.from_address(word).value = 1
    for slot in late:
        host.status_launched(slot)
    with pytest.raises(RuntimeError, match=r"earlier fused call \(backward of gru B7 T9 N3 D512\)"):
        check_status()
    check_status()


@pytest.mark.gpu
def test_other_threads_run_while_a_call_waits_for_a_word(gpu):
    """Where every word is taken, a call of the general path waits for the device, and not with the interpreter lock."""
    import threading
    import time

    from flashrnn_amd import _lib, flashrnn

    print("case host path lock", flush=True)
    x = [v.detach() for v in _leaves(gpu, T=4000, D=256)]
    host, stream = _lib.load_host(), torch.cuda.current_stream().cuda_stream
    gaps, done = [], threading.Event()

    def tick():
        last = time.perf_counter()
        while not done.is_set():
            time.sleep(0.001)
            gaps.append(time.perf_counter() - last)
            last += gaps[-1]

    with torch.no_grad():
        flashrnn(*x)
        torch.cuda.synchronize()
        for _ in range(100):  # (about 3 ms each)
            flashrnn(*x)
    thread, longest = threading.Thread(target=tick), 0.0
    thread.start()
    for _ in range(4200):
        t = time.perf_counter()
        host.status_launched(host.status_take(0, 0, 5, 4000, 2, 256, stream)[2])
        longest = max(longest, time.perf_counter() - t)
    done.set()
    thread.join()
    torch.cuda.synchronize()
    print(f"longest wait for a word {longest * 1e3:.1f} ms, longest pause of the other thread {max(gaps) * 1e3:.1f} ms", flush=True)
    assert longest > 0.05 and max(gaps) < longest / 2
