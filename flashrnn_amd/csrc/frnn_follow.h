// The loop of a workgroup that fetches operands ahead of a scan (frnn_prefetch.h).  On its own, without device types, so that the host's compiler
// reads it too.
#pragma once

namespace frnn {

// Steps ahead of the one that is being computed.  3 are too few where the device moves much (forward, B64 N3 D256 -0.3 % instead of -13 %, B256
// -9 instead of -18), 12 are as good as 6 but for B256 (-15: 12 steps of 12 groups no longer stay in an L2 beside what is stored).
constexpr int kPrefetchAhead = 6;
constexpr int kPrefetchPolls = 1 << 15;    // probes that see no step before such a workgroup ends
// Sequences up to this length go without (training pass, bf16: B256 N3 D256 T19 130.7 -> 131.9 us, T32 189.5 -> 180.1; B5 T19 93.0 -> 93.5, T64 141.8 -> 139.1)
constexpr int kPrefetchMinSteps = 24;
// Forward scans beyond this length as well: the tag of a word, t % 65535 + 1, which tells how far a group is, then says nothing
// to a workgroup that starts late.
constexpr int kPrefetchMaxSteps = 65535;

// Its groups are first, first + stride, ... below `groups`; its waves share them out, or share one.
// begun(group): the number of steps that the group has begun, as far as is known; request(group, step, part, parts): fetch this
// wave's part of the operands of a step.  here(group): 1 if the group runs on the XCD of this workgroup, -1 if not, 0 as long as that is not
// known.  What is fetched is of use on this XCD only, and a group on another one keeps its words there.
template <typename Here, typename Begun, typename Request>
__device__ __forceinline__ void prefetch_follow(int first, int stride, int groups, int Tn, int wave, int waves, const int* status, int spin_limit, Here here, Begun begun,
                                                Request request) {
  const int mine = first < groups ? (groups - first + stride - 1) / stride : 0;  // groups of this workgroup
  const int parts = mine > 0 && waves >= mine ? waves / mine : 1;                // waves per group
  const int part = wave % parts;
  int next[2], grp[2];
  bool placed[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = wave / parts + k * waves;
    grp[k] = first + i * stride;
    next[k] = i < mine ? 0 : Tn;
    placed[k] = false;
  }
  for (int polls = 0; polls <= min(spin_limit, kPrefetchPolls); ++polls) {
    if (next[0] >= Tn && next[1] >= Tn) break;
    bool did = false;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (next[k] >= Tn) continue;
      if (!placed[k]) {
        const int at = here(grp[k]);
        placed[k] = at > 0;
        if (at < 0) { next[k] = Tn; continue; }
      }
      const int b = begun(grp[k]), goal = min(b + kPrefetchAhead, Tn);
      next[k] = max(next[k], min(b, Tn));  // (late: what is behind is of no use any more)
      for (; next[k] < goal; ++next[k]) {
        request(grp[k], next[k], part, parts);
        did = true;
      }
    }
    if (did) { polls = 0; continue; }
    __builtin_amdgcn_s_sleep(4);
    if ((polls & 63) == 63 && __builtin_amdgcn_readfirstlane(__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) break;
  }
}

}  // namespace frnn
