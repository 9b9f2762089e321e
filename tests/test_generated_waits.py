"""Waits in the generated code of kernels whose loads have to stay in flight over a step.  What a source line asks for can be
lost in the compiler's counting of outstanding loads (it takes the lower count where two paths meet), which shows in no
result, only in the time; so the built device code is read back."""
import os
import re

import pytest

from test_kernel_resources import LLVM, ROOT, _disassemble

BUILD = os.path.join(ROOT, "flashrnn_amd", "csrc", "build")


def _functions(obj, tmp):
    path = os.path.join(BUILD, obj)
    if not os.path.exists(path):
        pytest.fail(f"{path} is missing: build the library first (make -C flashrnn_amd/csrc)")
    if not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("no llvm-objdump in this image")
    out, name = {}, None
    for line in _disassemble(path, str(tmp)).splitlines():
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            name = m.group(1)
            out[name] = []
        elif name and line.strip():
            out[name].append(line.split("//")[0].strip())
    return out


def _vmcnt(lines):
    return [int(m.group(1)) for t in lines for m in [re.search(r"s_waitcnt .*vmcnt\((\d+)\)", t)] if m]


@pytest.mark.parametrize("obj", ["fused_bwd_1_0.o", "fused_bwd_1_2.o"])
def test_producer_wave_of_the_slstm_waits_for_no_load_of_the_last_iteration(obj, tmp_path):
    """Between two barriers the producer wave hands over operands that it requested two iterations before and requests new
    ones: with n loads per iteration at least n are in flight, whatever path led there, and no wait may ask for fewer."""
    kernels = {k: v for k, v in _functions(obj, tmp_path).items()
               if re.search(r"fused_bwd_kernelILi1E\w+?Li(64ELi4|96ELi6)ELi1ELi1ELi4ELb0ELb[01]E", k)}
    assert len(kernels) == 4, sorted(kernels)
    for name, code in kernels.items():
        bars = [i for i, t in enumerate(code) if t.startswith("s_barrier")]
        steps = [code[a:b] for a, b in zip(bars, bars[1:])]
        steps = [s for s in steps if any("ds_write_b128" in t for t in s) and any("buffer_load_dwordx4" in t for t in s)]
        loads = [sum("buffer_load_dwordx4" in t for t in s) for s in steps]
        n = min(loads)
        assert n >= 6 and loads.count(n) >= 3 and set(loads) <= {n, 3 * n}, (name, loads)  # (3n: the first requests)
        short = [w for s, m in zip(steps, loads) for w in _vmcnt(s) if m == n and w < n]
        assert not short, f"{name}: waits of vmcnt {short} with {n} loads per iteration"


@pytest.mark.parametrize("obj,kernel", [
    ("fused_fwd_3_1.o", r"ILi3EfLi(448|512|640)ELi4E\w+?Li16E"), ("fused_fwd_2_0.o", r"ILi2E\w+?Li768ELi4E\w+?Li16E"),
    ("fused_fwd_2_2.o", r"ILi2E\w+?Li768ELi4E\w+?Li16E")])
def test_masks_of_a_probe_of_16_words_stay_in_scalar_registers(obj, kernel, tmp_path):
    """Forward, tallest tiles: from the last request of a probe to the barrier behind the copy of its words to LDS no mask is
    fetched back from a vector register, to which the compiler moves scalar values that it has no room for."""
    kernels = {k: v for k, v in _functions(obj, tmp_path).items() if re.search("fused_fwd_kernel" + kernel, k)}
    assert kernels
    for name, code in kernels.items():
        probes = [i for i, (a, b) in enumerate(zip(code, code[1:])) if "load_dwordx" in a and "sc1" in a and not ("load_dwordx" in b and "sc1" in b)]
        assert len(probes) >= 4, name  # (two rounds of a step, two steps per turn of the loop)
        for i in probes:
            end = next(j for j in range(i, len(code)) if code[j].startswith("s_barrier") or (j > i and "sc1" in code[j] and "dwordx" in code[j]))
            back = sum("v_readlane" in t for t in code[i:end])
            assert back <= 4, f"{name}: {back} masks fetched back behind the probe at {i}"


def test_alternating_lstm_step_in_fp32_requests_its_product_before_it_waits(tmp_path):
    """The operands of the adjoint are requested in front of the product and waited for behind it: on the way to the block of
    its first MFMA, which waits for the fragments, there is no wait for a load."""
    (code,) = [v for k, v in _functions("frnn_alt.o", tmp_path).items() if "alt_step_bwd_kernelILi0EfE" in k]
    first = next(i for i, t in enumerate(code) if "mfma" in t)
    waits = [i for i, t in enumerate(code[:first]) if re.search(r"vmcnt\(", t)]
    early = [i for i in waits if first - i > 20]
    assert not early, code[early[0] - 5:early[0] + 3]


def test_operands_of_an_elman_step_stay_where_they_arrive(tmp_path):
    """Reverse kernels of 10 and 12 waves: of the operands that a step requests, few are moved to another register, each behind a
    wait for its load (with a closure beside the step that nobody calls there was one more in each of the two loops)."""
    kernels = {k: v for k, v in _functions("fused_bwd_3_0.o", tmp_path).items() if re.search(r"fused_bwd_kernelILi3E\w+?Li(160ELi10|192ELi12)ELi1ELi1ELi4E", k)}
    assert len(kernels) == 2, sorted(kernels)
    for name, code in kernels.items():
        arrive = {m.group(1) for t in code for m in [re.match(r"buffer_load_ushort (v\d+),", t)] if m}
        moved = [t for t in code for m in [re.match(r"v_mov_b32_e32 v\d+, (v\d+)$", t)] if m and m.group(1) in arrive]
        assert arrive and len(moved) <= 8, (name, moved)
