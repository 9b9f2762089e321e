// Workgroups that fetch the operands of the coming steps into the L2 of an XCD (heads of several workgroups).
//
// A compute unit's vector memory returns in the order in which it was asked, whichever wave asked.  A scan whose workgroups exchange
// words in every step therefore waits, with its words, for every operand that some wave of the same compute unit has requested
// from HBM meanwhile, a producer wave's included: ~1900 cycles, more the more the device moves, against ~700 for the words.  (Forward, T = 1024,
// a build whose Wx is always the same two steps', i.e. in L2: LSTM B8 N3 D256 0.874 -> 0.833 ms, B256 1.783 -> 1.481.)  The scans leave
// compute units idle, and those of the same XCD share its L2.  So a launch gets a few more workgroups, each on a compute unit of its
// own, which request what the scan will need some steps later; the scan's own requests find it in L2.
// They follow the groups (forward: a group's step is read off the words that its workgroups exchange, in passing; reverse: the group writes it down, as
// the 2 bits of a step that its words carry are lost as soon as such a workgroup falls 6 steps behind), nobody waits for them, and they end with the last step requested, when their groups turn out to run on another XCD, or
// when these stop: a failed wait, or no step for kPrefetchPolls probes.
//
// Forward kernel, bf16, T = 1024, without and with: LSTM N3 D256 B8 0.883 -> 0.840 ms, B16 0.900 -> 0.842, B64 0.965 -> 0.854, B128 1.231 ->
// 1.083, B256 1.787 -> 1.527; sLSTM N4 D192 B16 0.905 -> 0.832, B256 2.805 -> 2.401; GRU N3 D256 B16 0.839 -> 0.773, B256 1.492 -> 1.243.
#pragma once
#include "frnn_exchange.h"
#include "frnn_follow.h"

namespace frnn {

__device__ __forceinline__ u32x4 make_rsrc4(const void* p, size_t bytes) {  // (make_rsrc as a register tuple, for inline asm)
  const u64 a = (u64)p;
  return u32x4{(unsigned)a, (unsigned)(a >> 32) & 0xffffu, (unsigned)(bytes > 0x7fffffffu ? 0x7fffffffu : bytes), 0x00020000u};
}
// The kernel's arguments through a pointer that the compiler knows nothing about: what one role of a kernel reads through it is loaded
// where that role needs it.  Read as the kernel's parameter, the loads are shared with the scan's, in front of the branches between the
// roles, and stay in scalar registers over the time loop; the scans at the limit then move masks and pointers to vector registers
// and back in every step.
template <typename Args> __device__ __forceinline__ const __attribute__((address_space(4))) Args* own_args() {
  typedef const __attribute__((address_space(4))) Args* args_t;
  args_t p = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}
// 16 bytes per lane to the LDS address `lds` + 16 * lane (out of range: no memory traffic)
__device__ __forceinline__ void load_to_lds(u32x4 r, unsigned voff, unsigned soff, unsigned lds) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff), "s"(lds) : "memory", "m0");
#pragma clang diagnostic pop
}

// (none may land in the LDS of a workgroup that comes later)
__device__ __forceinline__ void all_fetched() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Does a group run on this XCD?  (prefetch_follow's here(); `words`: its words of xcd_handshake, or null: as the launch has placed it)
template <int KW> __device__ __forceinline__ int group_here(const int* words, int lane) {
  if (!words) return 1;
  const int own = own_xcd(), v = lane < KW ? __hip_atomic_load(words + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : own;
  return __any(v != 0 && v != own) ? -1 : __all(v != 0) ? 1 : 0;
}

// Steps begun, off the first word of a forward group's two exchange slots (`slots`, LLW words each): h of step t carries the tag of t, which
// is t + 1 in sequences that get such workgroups.
template <int LLW> __device__ __forceinline__ int forward_steps_begun(const u64* slots) {
  const unsigned v0 = (unsigned)ll_load(slots), v1 = (unsigned)ll_load(slots + LLW);
  return __builtin_amdgcn_readfirstlane((int)(max(v0, v1) >> 16));
}

// One wave's part of `planes` planes of `rows` (of up to TR) rows of PPR 16-byte pieces; k: the instruction that is next for this wave
template <int PPR, int PLANES, int TR>
__device__ __forceinline__ void fetch_rows(u32x4 r, unsigned so, unsigned row_bytes, unsigned plane_bytes, int rows, int lane, int& k, int parts, unsigned junk) {
  constexpr int NP = PLANES * TR * PPR, NI = (NP + 63) / 64;
  for (; k < NI; k += parts) {
    const int c = lane + 64 * k, q = c % PPR, row = c / PPR % TR, plane = c / (PPR * TR);
    load_to_lds(r, c < NP && row < rows ? row * row_bytes + plane * plane_bytes + q * 16 : kInvalidOff, so, junk);
  }
  k -= NI;
}

// The forward scan's Wx (16-bit types): TR rows x GW gates x D units of a step.  `junk`: LDS address of 1 KB that nobody reads.
template <int KW, int GW, int D, int TR, int LLW>
__device__ __forceinline__ void prefetch_wx(const void* Wx, const u64* ll, const int* status, const int* xcd, int first, int stride, int groups, int grp0, int N, int B, int Tn, int wave, int waves,
                                            int lane, int spin_limit, unsigned junk) {
  constexpr int ES = 2;
  const unsigned ND = (unsigned)N * D;
  const u32x4 r = make_rsrc4(Wx, (size_t)B * Tn * GW * ND * ES);
  prefetch_follow(first, stride, groups, Tn, wave, waves, status, spin_limit,
    [&](int g) { return group_here<KW>(xcd ? xcd + (size_t)(grp0 + g) * 32 : nullptr, lane); },
    [&](int g) { return forward_steps_begun<LLW>(ll + (size_t)(grp0 + g) * 3 * LLW); },
    [&](int g, int t, int part, int parts) {
      const int n = (grp0 + g) % N, bt = (grp0 + g) / N, rows = min(TR, B - bt * TR);
      const unsigned so = (((unsigned)bt * TR * Tn + t) * GW * ND + n * D) * ES;
      int k = part;
      fetch_rows<D * ES / 16, GW, TR>(r, so, Tn * GW * ND * ES, ND * ES, rows, lane, k, parts, junk);
    });
  all_fetched();
}

// The reverse scan's operands of a step: the gate cache (NCP values per element), the planes DSM of the cotangent and SPM of the states before
// the step.  `begun`: where group 0 keeps its number of steps begun, the others `stride_words` apart.
template <typename T, int KW, int S, int NCP, int SPM, int DSM, int D, int TR>
__device__ __forceinline__ void prefetch_reverse(const void* cache, const void* states, const void* dstates, const unsigned* begun, size_t stride_words, const int* status, const int* xcd, int first,
                                                 int stride, int groups, int grp0, int N, int B, int BS, int Tn, int wave, int waves, int lane, int spin_limit, unsigned junk) {
  constexpr int ES = (int)sizeof(T), PPR = D * ES / 16;
  const unsigned ND = (unsigned)N * D;
  const u32x4 rSt = make_rsrc4(states, ((size_t)(S - 1) * BS + B) * Tn * ND * ES), rDs = make_rsrc4(dstates, ((size_t)(S - 1) * BS + B) * Tn * ND * ES);
  const u32x4 rCa = make_rsrc4(cache, (size_t)Tn * N * B * D * NCP * ES);
  prefetch_follow(first, stride, groups, Tn, wave, waves, status, spin_limit,
    [&](int g) { return group_here<KW>(xcd ? xcd + (size_t)(grp0 + g) * 32 : nullptr, lane); },
    [&](int g) { return __builtin_amdgcn_readfirstlane((int)ll_load(begun + (size_t)(grp0 + g) * stride_words)); },
    [&](int g, int i, int part, int parts) {
      const int t = Tn - 1 - i, n = (grp0 + g) % N, bt = (grp0 + g) / N, rows = min(TR, B - bt * TR);
      int k = part;
      fetch_rows<NCP * ES, D / 16, TR>(rCa, (((unsigned)t * N + n) * (D / 16) * B + bt * TR) * 16 * NCP * ES, 16 * NCP * ES, (unsigned)B * 16 * NCP * ES, rows, lane, k, parts, junk);
#pragma unroll
      for (int p = 0; p < S; ++p) {
        const unsigned so = (((unsigned)(p * BS + bt * TR) * Tn + t) * ND + n * D) * ES;
        if ((DSM >> p) & 1) fetch_rows<PPR, 1, TR>(rDs, so, Tn * ND * ES, 0, rows, lane, k, parts, junk);
        if ((SPM >> p) & 1 && t > 0) fetch_rows<PPR, 1, TR>(rSt, so - ND * ES, Tn * ND * ES, 0, rows, lane, k, parts, junk);
      }
    });
  all_fetched();
}

}  // namespace frnn
