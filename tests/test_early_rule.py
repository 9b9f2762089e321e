"""Which reverse kernels do half of a step's adjoint ahead of time: the tilings where it was measured to gain, and none of those where it loses
(csrc/frnn_plan.h, read by the host's compiler)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "flashrnn_amd", "csrc")
NC = {"lstm": 4, "slstm": 5, "gru": 4}
# cell, type, D, waves, workgroups, rows
GAINS = [("lstm", "bf16", 192, 4, 6, 4), ("lstm", "bf16", 256, 4, 8, 4), ("lstm", "f16", 768, 4, 24, 4), ("lstm", "f16", 1024, 4, 32, 4), ("lstm", "bf16", 384, 4, 6, 8),
         ("slstm", "bf16", 192, 4, 6, 4), ("slstm", "f16", 384, 4, 12, 4), ("slstm", "bf16", 640, 4, 20, 4), ("slstm", "f16", 256, 4, 16, 4), ("slstm", "bf16", 512, 4, 8, 4),
         ("gru", "bf16", 192, 4, 3, 4), ("gru", "f16", 320, 4, 10, 4), ("gru", "bf16", 512, 4, 16, 4), ("gru", "bf16", 256, 8, 2, 8), ("lstm", "f32", 512, 4, 32, 4), ("lstm", "f32", 768, 4, 48, 4)]
LOSES = [("slstm", "bf16", 128, 4, 4, 4), ("slstm", "bf16", 448, 4, 14, 4), ("slstm", "bf16", 512, 4, 16, 4), ("slstm", "f16", 512, 4, 16, 4), ("slstm", "f16", 640, 4, 20, 4),
         ("slstm", "f16", 768, 4, 24, 4), ("slstm", "bf16", 1024, 4, 32, 4), ("gru", "bf16", 640, 4, 10, 4), ("gru", "f16", 768, 4, 12, 4), ("lstm", "bf16", 192, 4, 3, 4),
         ("slstm", "bf16", 192, 4, 3, 4), ("lstm", "f32", 1024, 4, 64, 4), ("slstm", "f32", 256, 4, 16, 4), ("lstm", "f32", 256, 4, 8, 4), ("lstm", "bf16", 256, 4, 4, 16)]


@pytest.fixture(scope="module")
def early(tmp_path_factory):
    src = tmp_path_factory.mktemp("rule") / "rule.cpp"
    cases = [c for g in (GAINS, LOSES) for c in g]
    calls = "\n".join(f"  putchar('0' + frnn::bwd_adjoint_early({3 if f == 'gru' else 4}, {NC[f]}, {D}, {w}, 1, {k}, {r}, {4 if t == 'f32' else 2}, {str(t == 'f16').lower()}, false));"
                      for f, t, D, w, k, r in cases)
    src.write_text(f'#include "{CSRC}/frnn_plan.h"\n#include <cstdio>\nint main() {{\n{calls}\n}}\n')
    exe = str(src.with_suffix(""))
    subprocess.run(["g++", "-std=c++17", "-o", exe, str(src)], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return dict(zip(cases, out))


@pytest.mark.parametrize("case,want", [(c, "1") for c in GAINS] + [(c, "0") for c in LOSES])
def test_the_first_half_is_done_early_where_it_pays(early, case, want):
    assert early[case] == want
