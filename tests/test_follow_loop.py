"""The loop of the workgroups that fetch operands ahead of a scan (csrc/frnn_follow.h), run by the host against scans that are played to it: what it
fetches, and that it ends, whatever the scan does."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "flashrnn_amd", "csrc")
PLAY = r"""
#include <algorithm>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <vector>
using std::max; using std::min;
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_s_sleep(x) ++now
#define __hip_atomic_load(p, order, scope) (*(p))  // (the status word)
static int now = 0;  // pauses of the loop: the clock of the scan that is played
#include "frnn_follow.h"

// groups, T, pauses per step, start (pause at which the scan begins), stop (step at which it stops, -1: none), fails (pause at which the status word is set, -1: never),
// at (where the groups run: 1 here, -1 elsewhere, 0 never known), spin_limit, wave, waves
int main(int, char** v) {
  const int groups = atoi(v[1]), T = atoi(v[2]), per = atoi(v[3]), start = atoi(v[4]), stop = atoi(v[5]), fails = atoi(v[6]), at = atoi(v[7]), limit = atoi(v[8]),
            wave = atoi(v[9]), waves = atoi(v[10]);
  int status = 0;
  std::vector<std::vector<int>> got(groups);
  int ahead = 0;
  auto steps = [&]() {
    if (fails >= 0 && now >= fails) status = 1;
    const int b = now < start ? 0 : min(T, (now - start) / per);
    return stop >= 0 ? min(b, stop) : b;
  };
  steps();
  frnn::prefetch_follow(0, 1, groups, T, wave, waves, &status, limit, [&](int) { return now >= start ? at : 0; }, [&](int) { return steps(); },
                        [&](int g, int t, int, int) { got[g].push_back(t); ahead = max(ahead, t + 1 - steps()); });
  bool rising = true;
  long n = 0;
  for (auto& s : got) { n += s.size(); for (size_t i = 1; i < s.size(); ++i) rising = rising && s[i] > s[i - 1]; }
  printf("%d %ld %d %d %d\n", now, n, ahead, (int)rising, got[0].empty() ? -1 : got[0].back());
}
"""


@pytest.fixture(scope="module")
def play(tmp_path_factory):
    src = tmp_path_factory.mktemp("follow") / "play.cpp"
    src.write_text(PLAY)
    exe = str(src.with_suffix(""))
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", exe, str(src)], check=True)

    def run(groups=1, T=100, per=3, start=0, stop=-1, fails=-1, at=1, limit=1 << 22, wave=0, waves=4):
        args = [str(a) for a in (groups, T, per, start, stop, fails, at, limit, wave, waves)]
        out = subprocess.run([exe, *args], check=True, capture_output=True, text=True, timeout=60).stdout.split()
        return dict(zip(("pauses", "fetched", "ahead", "rising", "last"), map(int, out)))

    return run


@pytest.mark.parametrize("at", [0, 1])
@pytest.mark.parametrize("T", [25, 100, 65535])
def test_every_step_is_fetched_once_and_some_steps_ahead(play, T, at):
    r = play(T=T, at=at)
    assert r == dict(pauses=r["pauses"], fetched=T, ahead=6, rising=1, last=T - 1)


def test_two_groups_of_one_wave(play):
    assert play(groups=8)["fetched"] == 200  # (waves 4: this wave has groups 0 and 4)


def test_steps_that_are_over_are_left_out(play):
    r = play(T=4000, per=3, start=-3000)  # begins 1000 steps late
    assert r["rising"] == 1 and r["last"] == 3999 and r["fetched"] <= 3006


def test_a_group_that_has_ended_is_not_waited_for(play):
    assert play(T=100, start=-1000)["pauses"] <= 1


def test_a_group_of_another_xcd_is_let_go(play):
    """Its words need never become visible here: a loop that waited for them would hold its launch for as long as its bound of probes lasts."""
    assert play(at=-1, stop=0)["pauses"] <= 1
    r = play(at=-1, start=20, stop=0)  # not known at first
    assert r["fetched"] == 6 and r["pauses"] <= 22


@pytest.mark.parametrize("at", [0, 1])
def test_the_loop_ends_with_a_scan_that_stops(play, at):
    assert play(at=at, stop=4, fails=500)["pauses"] <= 500 + 64 + 3  # the status word says so
    assert play(at=at, stop=4)["pauses"] <= (1 << 15) + 32           # nobody says so
    assert play(at=at, stop=4, limit=256)["pauses"] <= 256 + 32
    assert play(at=at, limit=-2)["fetched"] == 0
