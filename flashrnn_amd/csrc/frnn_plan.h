// The static tiling table of the fused kernels: which (D, WAVES, UTW, KW) are compiled for each
// (gate-row count, storage type), forward and backward.  Replaces the reference's constraint
// solver + JIT bisection (flashrnn/flashrnn/flashrnn.py:429-589, cuda_init_parametric.py:92-358).
//
// X(D, VARIANT, WAVES, UTW, KW, MTR):  D = 16 * UTW * WAVES * KW, or half or a quarter of that where two or four waves share
// every unit tile (fwd_k_split, bwd_dest_split);  MTR = the largest batch tile (4, 8 or 16 rows)
// this tiling is compiled for: taller tiles keep more state per lane, and where that would spill registers to
// scratch memory the tile height stops below (a large batch then runs as more groups, in several launches if
// the workgroups of a head wait for each other).  No compiled kernel uses scratch memory; a test checks the
// compiler's resource report of every instantiation.
//   R registers per lane = UTW * G_r * D / 8 (bf16) or UTW * G_r * D / 4 (f32), over the waves that share a tile; a workgroup of
//   4 waves (one per SIMD) may use up to 512 VGPRs per lane, one of 8 waves 256, of 16 waves 128.
// VARIANT 0 is the default.  VARIANTS 2 and 3, where a head dim has them, spread the head over more workgroups: 3, the
// wider one, or else 2, is used instead of the default while all groups of the call fit one launch with 4-row
// batch tiles (measured faster up to a launch that fills the device, slower where the default still takes one launch and
// they would take two; not while a decode session runs, see pick_beside).  VARIANT 4 packs the head into half the workgroups of the default, two waves per SIMD: a large batch then
// runs on tiles of half the height (see pick_plan).  To try another tiling add an X(D, 1, ...) entry and run with FRNN_FUSED_VARIANT=1.  The alternatives that were measured and lost (4 waves x 2 tiles for
// D = 128, 8 x 2 waves for D = 256, ...) are not compiled in.
// Forward and backward tile independently (the gate cache layout does not depend on the plan).
#pragma once

namespace frnn {
struct Plan {
  int D, variant, waves, utw, kw, max_tr;
  int cooperative = 0;  // host side only: launch the kernel as a cooperative one (see fused_*_tu.hip)
  int recompute = 0;    // host side only: the reverse kernel of recompute mode
  int left_out = 0;     // host side only, tests of the failure path: workgroups at the end of the grid that are not launched
  int order = 0;        // forward: > 1: sums over k in this many parts, as a tiling whose waves split k does (see pick_beside)
};

// Resident operand of the forward product: a wave holds UTW*G_r*KS fragments of R.  When they alone
// would take more than 400 of the 512 registers a wave has at one wave per SIMD (LSTM D = 1024: all
// 512), those of the last RLK k-steps live in LDS instead (as many as bring the rest down to 352, and
// as fit beside the two h buffers) and are read back one k-step ahead as the A operand of their MFMAs.
constexpr int fwd_lds_ksteps(int GR, int D, int WAVES, int UTW, int esize) {
  const int KM = esize == 4 ? 4 : 32, FR = esize == 4 ? 1 : 4, FRB = esize == 4 ? 4 : 16;
  const int KS = D / KM, per = UTW * GR * FR, regs = per * KS;
  if (!(WAVES <= 4 && regs > 336)) return 0;
  const int want = (regs - 320 + per - 1) / per;
  const int room = (160 * 1024 - 2 * 16 * D * esize - 1024) / (WAVES * UTW * GR * 64 * FRB);
  return want < room ? want : room;
}

// Waves per unit tile, forward: tilings with 16 * UTW * WAVES * KW = KSP * D, KSP = 2 or 4, have KSP waves of a workgroup share
// a tile.  Each keeps R for one part of k (D / KSP of it) and multiplies it with that part of h; all but the first hand their
// sums to the first through LDS, which alone does the gate math of the tile.  Two reasons to do so:
//   the operand of a tile is more than the 512 registers of a wave hold (16-bit D = 1024; fp32 from D = 384 on), or
//   the product of a step is long against the exchange: the head then takes KSP times the workgroups and multiplies for 1 / KSP
//   of the time.  fp32 (8 cycles per k, see fwd_form_4x4x1), LSTM B16 N1 T256, forward: D = 512 as 16 workgroups
//   of pairs 0.543 ms, as 32 of fours 0.470; D = 256 as 4 / 8 / 16 workgroups 0.441 / 0.369 / 0.312; D = 128 as 2 / 4 / 8 0.300 /
//   0.279 / 0.254.  16-bit (16 cycles per gate and 32 k) from D = 384 on: LSTM D = 384 0.282 -> 0.274, D = 512 0.317 -> 0.292,
//   D = 640 0.363 -> 0.340, D = 768 0.394 -> 0.363; sLSTM 0.298 -> 0.285 .. 0.409 -> 0.381; GRU D = 1024 0.430 -> 0.364, D = 768 0.334 ->
//   0.319, D = 640 0.315 -> 0.298 (D = 512 and less no gain); below that the pairs lose what they cannot do, multiply the own slice in
//   front of the wait (D = 256 0.217 -> 0.244).
// fp32 heads beyond 512 units take D / 16 = 40, 48 or 64 workgroups, more than the 32 compute units of an XCD: such a group
// spreads over the device (decode_block) and exchanges at agent scope.
constexpr int fwd_k_split(int D, int WAVES, int UTW, int KW) { return 16 * WAVES * UTW * KW / D; }
// the dense alternatives of the tables (host: pick_plan; not for the resident decode kernel, whose groups all have 4 rows)
constexpr int kDenseVariant = 4;
// Forward kernels whose launch may get workgroups that fetch Wx into L2 (frnn_prefetch.h): the gated cells in the 16-bit types, 2 to 8 workgroups per head, and from
// 20 on those whose waves split k (training pass, Wx from memory, bf16 T = 1024: B16 N1 LSTM D640 2773 -> 2756 us, D768 3054 -> 3046, GRU 2591 -> 2578, 2832 -> 2804).
// (Forward, T = 512, all sizes from B1 N1 to B256 N3, without and with: those -2 to -15 % where the call has more to move than the last-level cache holds, +-0.5 where
// not.  10 to 16 workgroups, whose steps last longer than a trip to HBM, -0.4 to +0.1, fp32, 3 to 28 workgroups, -0.5 to +0.8; and the role itself, a branch and its
// registers, made their scans 1 to 2 % slower: LSTM bf16 B64 N3 D768 T = 256 935 -> 948 us, GRU B256 N3 D640 1034 -> 1050, fp32 LSTM B8 N3 D448 429 -> 439, sLSTM D160
// 313 -> 318.  Elman, one load per step: -1.4 to +1.0 % at any batch.)
constexpr bool fwd_prefetched(int GR, int D, int WAVES, int UTW, int KW, int esize) {
  return esize == 2 && GR >= 3 && KW > 1 && (KW <= 8 || (KW >= 20 && KW < 32 && fwd_k_split(D, WAVES, UTW, KW) > 1));
}
// Forward kernel, fp32 at 4-row tiles, cells with 3 or 4 recurrent gates: the product runs on v_mfma_f32_4x4x1_16B_f32
// (see the kernel), when the whole operand, D / KSP registers per tile in that form, fits the registers of a wave (512 in
// workgroups of up to 4 waves, 256 with up to 8: D = 96 as 6 waves).
constexpr bool fwd_form_4x4x1(int GR, int D, int WAVES, int UTW, int KW, int TR, int esize) {
  return esize == 4 && TR == 4 && GR >= 3 && (WAVES <= 4 ? UTW * D / fwd_k_split(D, WAVES, UTW, KW) <= 384 : WAVES <= 8 && UTW * D <= 96);
}
// (16-bit kernels whose waves split k: the whole operand in registers)
constexpr bool fwd_k_split16(int D, int WAVES, int UTW, int KW, int esize) {
  return esize == 2 && fwd_k_split(D, WAVES, UTW, KW) > 1;
}
// Forward kernel: one more wave per workgroup that fetches Wx for the compute waves.  A vector memory instruction that a
// compute wave issues behind the exchange wait delays its MFMAs (~70 cycles each on the chain of dependent steps), one
// issued in front of the wait delays the probe (a wave's memory operations return in order).  The producer wave has a
// queue of its own: it loads the Wx of the whole workgroup three steps ahead and writes the Wx of the next step into an
// LDS buffer, from which the compute waves take their elements with LDS reads.  For the kernels with steps of ~2000 cycles
// (16-bit types, 4- and 8-row tiles, heads of several workgroups of 4 waves) that stay within the 256 registers a wave has when
// five share four SIMDs (heads of one workgroup of up to 8 waves, where every load is on the chain: the gated cells,
// GRU B16 T2048 N4 D128 forward 0.915 -> 0.826 ms), and for the cells with four gates: LSTM D = 256 forward 0.944 -> 0.887 ms per 1024 steps, sLSTM
// D = 192 0.961 -> 0.914; the GRU (three loads per step to save) measured +1.5 % to -0.8 %, Elman the same to 0.3 %.
constexpr bool fwd_producer_wave(int GR, int D, int WAVES, int UTW, int KW, int TR, int esize) {
  // (heads of one workgroup: every load is on the chain; the Elman cell, one load per step, measured 0 to +10 % with the wave)
  // (wave pairs that split k up to D = 512, 128 registers of R: forward, B8 N1 T256, without and with: LSTM D = 384 0.286 -> 0.273 ms,
  // D = 512 0.327 -> 0.293; D = 640, 160 registers, spills with five waves)
  if (KW == 1) return esize == 2 && GR >= 3 && TR == 4 && WAVES <= 8 && UTW == 1;
  return esize == 2 && GR == 4 && KW > 1 && TR <= 8 && WAVES == 4 && UTW * GR * (D / 32) * 4 / fwd_k_split(D, WAVES, UTW, KW) <= (TR == 4 && fwd_k_split(D, WAVES, UTW, KW) == 1 ? 160 : 128);
}
// Forward kernel: may the producer wave also store the outputs of a step (16-byte pieces, one step late) instead of the
// compute lanes (2 bytes per state and lane at 4-row tiles)?  Exists for the heads that run as one workgroup with a
// producer wave; the host picks these instantiations by cell, cache and number of groups (fwd_producer_stores_pay; measured: LSTM
// B256 N12 D64 forward -20 %, but +5-9 % at B = 16, where the stores of the compute lanes are hidden anyway).
constexpr bool fwd_producer_stores(int GR, int D, int WAVES, int UTW, int KW, int TR, int esize) {
  return KW == 1 && fwd_producer_wave(GR, D, WAVES, UTW, KW, TR, esize);
}
// Backward kernel: the same producer wave for the operands of a step (gate cache, s_(t-1), the cotangent of the
// states), for the heads that run as one workgroup: there every load of the compute waves is on the chain of dependent
// steps, and a step (~1600 cycles) is shorter than a fetch from HBM, which their one-step prefetch therefore waits for
// (a timing-only build without these loads runs GRU D = 128 backward 35 % faster).  The producer wave loads four steps
// ahead and leaves the operands of the next step in LDS.  Not for truncated backpropagation
// (no barrier per step to hand over at: that variant of the step keeps its own loads).  All four cells: GRU B16 T2048
// N4 D128 1.396 -> 1.049 ms, Elman B16 T1024 N12 D64 0.312 -> 0.261, N6 D128 0.386 -> 0.301.
// Recompute mode: Wx in the place of the gate cache, and h_(t-1) straight into the buffer that the rebuilt product reads, so the compute
// waves load nothing, keep two operand sets instead of three and have the registers for both operands without accumulation registers.
// Whole backward pass, T = 256, without and with: LSTM B33 N8 D96 (fp16, T515) 609 -> 490 us, sLSTM 392 -> 285, GRU 264 -> 201; B16 N12 D64 LSTM 223 ->
// 152, sLSTM 261 -> 165, GRU 196 -> 125; B16 N4 D32 172 -> 116, 207 -> 126, 166 -> 101; B256 N12 D64, mostly bytes, 613 -> 534, 750 -> 572, 492 ->
// 477; B256 N24 D32 709 -> 586, 818 -> 715, 583 -> 426.  Not the GRU's 8 waves at D = 128, which have 170 registers each beside a ninth.
constexpr bool bwd_producer_wave(int GR, int nc, int D, int WAVES, int UTW, int KW, int TR, int esize, bool rc) {
  // (nc = 5, the sLSTM: its 8-wave kernel spills at the 170 registers that nine waves leave each)
  if (rc) return esize == 2 && KW == 1 && TR == 4 && WAVES <= 6 && UTW == 1;
  return esize == 2 && KW == 1 && TR == 4 && (WAVES <= 6 || (WAVES <= 8 && nc <= 4)) && UTW == 1;
}
// LDS bytes of the hand-over buffers of that wave (two steps): the gate cache (nc values per element, padded to an even
// number), s_(t-1) and the cotangent (s states each) of the workgroup's UT_WG tiles of TR rows x 16 units, and 16
// spare bytes
constexpr int bwd_producer_bytes(int nc, int s, int ut_wg, int TR, int esize) {
  return 2 * ut_wg * TR * 16 * ((nc + 1) / 2 * 2 + 2 * s) * esize + 16;
}
// Backward kernel: may the producer wave also store dWx (see fwd_producer_stores)?  Not the 8-wave kernels (D = 128): one
// workgroup of nine waves per compute unit is all that their 166 registers allow, and there the variant measured slower
// (LSTM bf16 B256 T1024 N6 D128 reverse kernel 1.46 -> 1.58 ms, GRU 1.18 -> 1.21).
constexpr bool bwd_producer_stores(int GR, int nc, int D, int WAVES, int UTW, int KW, int TR, int esize, bool rc) {
  return bwd_producer_wave(GR, nc, D, WAVES, UTW, KW, TR, esize, rc) && WAVES <= 6;
}
// Waves per tile position, backward: with 16 * UTW * WAVES * KW = DSP * D, DSP = 2 or 4 waves of a workgroup share a position
// and split the destinations of the reverse product between them.  fp32 (4x4x1 form): each keeps R^T (own gate rows x
// destinations) for every DSP-th group of 4 destination workgroups, G_r * D / (4 DSP) registers; 16-bit (16x16x32 form): for one
// half of the destination workgroups.  Each sends the partial sums it computes itself; the first wave alone owns the
// position's elements (gate math, loads, stores).  There is no sum to hand over (but see RSP in the kernel), so the split pays from
// smaller heads on than forward.  Reverse kernel, B8 N1 T256: 16-bit LSTM D = 192 as 6 workgroups of pairs instead of 3 0.227 -> 0.214 ms,
// D = 256 0.257 -> 0.241, D = 320 0.279 -> 0.249, D = 384 0.305 -> 0.276, D = 448 0.333 -> 0.297, D = 512 0.359 -> 0.323, D = 640 0.411 ->
// 0.382, D = 768 0.455 -> 0.432; sLSTM the same within 2 %, but D = 256 slower with 8 workgroups (0.263 -> 0.289) and 0.247 with 16 of
// fours; GRU D = 320 0.248 -> 0.232, D = 512 0.316 -> 0.299, D = 1024 0.508 -> 0.477, the others no gain.
// fp32 LSTM B16 N1 T256: D = 128 as 2 / 4 / 8 workgroups 0.422 / 0.325 / 0.278, D = 256 as 4 / 8 / 16 0.462 / 0.368 / 0.321, D = 512
// as 16 / 32 0.623 / 0.528.
constexpr int bwd_dest_split(int D, int WAVES, int UTW, int KW) { return 16 * WAVES * UTW * KW / D; }
// Backward kernel: LDS bytes of the two dWx hand-over buffers of the producer-store instantiations
// ([gate][row][unit], and [row][unit] for the GRU's g-gate cotangent), behind the operand hand-over buffers
constexpr int bwd_producer_store_bytes(int gw, bool gru, int D, int TR, int esize) {
  return 2 * (gw * TR * (D + 8) + (gru ? TR * (D + 8) : 0)) * esize;
}
// Forward kernel: do the k-steps over the workgroup's own slice of h run in front of the exchange wait?  Heads of
// 2..16 workgroups (up to 12 where part of the operand lives in LDS) whose slice is a whole number of k-steps; not the fp32
// kernels whose operand alone takes 256 registers, at the tile heights where they keep 2 or 4 elements per lane
// (with the two-part product they spill).  The host reads this for the delay of the first probe.
constexpr bool fwd_own_slice_first(int GR, int D, int WAVES, int UTW, int KW, int TR, int esize) {
  const int KM = esize == 4 ? 4 : 32, KS = D / KM;
  return KW > 1 && KW <= 16 && !fwd_form_4x4x1(GR, D, WAVES, UTW, KW, TR, esize) && !fwd_k_split16(D, WAVES, UTW, KW, esize) &&
         (fwd_lds_ksteps(GR, D, WAVES, UTW, esize) == 0 || KW <= 12) && (D / KW) % KM == 0 &&
         !(esize == 4 && UTW * GR * KS >= 256 && TR >= (KW > 8 ? 8 : 16));
}
// Forward kernel: the outputs of a step are stored behind the first probe of the next step, while it is on its way, instead of in front
// of it.  For the gated cells in the 16-bit types whose product over the own slice comes before the probe: workgroups of 4 waves, up to 8
// per head at 4-row tiles and 5 at 8-row tiles; their first probe mostly finds the words.  (A second one has to wait for the stores.)  Forward, T =
// 384: LSTM N3 D256 B16 0.325 -> 0.302 ms, B64 0.338 -> 0.314, B128 0.422 -> 0.404, N2 D320 B16 0.341 -> 0.333, sLSTM N4 D192 B16 0.321 -> 0.297, B128
// 0.474 -> 0.441, GRU N3 D256 B16 0.314 -> 0.296, N2 D384 0.350 -> 0.337, D512 0.397 -> 0.394.  Elsewhere the words come later than the first probe:
// 8-row tiles of 6 and more workgroups +2 to +6 %, waves that split k +4 to +10, 10 workgroups and more +5 to +8, 16-row tiles and the
// dense tilings +2 to +9, fp32 +4 to +9; the Elman cell -1.5 to +0.5.
constexpr bool fwd_stores_behind_probe(int GR, int D, int WAVES, int UTW, int KW, int TR, int esize) {
  return esize == 2 && GR >= 3 && WAVES == 4 && KW <= (TR == 4 ? 8 : TR == 8 ? 5 : 0) && fwd_own_slice_first(GR, D, WAVES, UTW, KW, TR, esize);
}
// Reverse kernels with an instantiation for launches that have workgroups which fetch its operands into L2 (frnn_prefetch.h): gated cells in the 16-bit
// types, 8- and 16-row tiles of up to 5 workgroups per head (the GRU 8-row tiles), and the sLSTM's pairs of 6 workgroups (nc: values of the gate cache).
// Whole backward pass, bf16, T = 512, without and with: LSTM B128 N3 D256 784 -> 752 us, B256 1261 -> 1174, sLSTM B128 N3 D256 879 -> 813, B256 N4
// D192 1385 -> 1285, GRU B128 N2 D320 736 -> 717, N3 D256 714 -> 708, in its dense tiling of 2 (65 to 80 groups; training pass) B171 and B200 N3 D256 T = 256 742 -> 729, 760 -> 744, T = 1024
// 2783 -> 2799, 2848 -> 2866; the pairs of 6 beyond the last-level cache: bf16 and fp16 B16 N4 T2048 D192 1809 -> 1746, 1819 -> 1751.
// Elsewhere: GRU B16 N1 D512 592 -> 596, LSTM B8 T1024 N3 D256 912 -> 930, B16
// N1 D384 551 -> 562, D512 650 -> 649, sLSTM B16 N4 D128 400 -> 415, taller tiles of 6 to 10 workgroups -0.5 to +2.7 %, fp32 -0.3 to +4, recompute mode +-1.  The
// sLSTM's other pairs, beyond the last-level cache: 10 and 12 workgroups, bf16, whose steps are longer, -0.4 and -0.7 %, which is no second kernel's worth; 14 -3 % in
// bf16, -2 in fp16, 16 -2.5 and +7.5, 20 +1.8, 24 -8.5 and +2.4: one type's gain is the other's loss, and they are left without.
constexpr bool bwd_prefetched(int GR, int nc, int D, int WAVES, int UTW, int KW, int TR, int esize, bool rc) {
  return esize == 2 && (GR == 4 || (GR == 3 && TR == 8)) && KW > 1 && !rc && UTW == 1 &&
         (TR == 4 ? nc == 5 && bwd_dest_split(D, WAVES, UTW, KW) == 2 && KW == 6 : bwd_dest_split(D, WAVES, UTW, KW) == 1 && KW <= 5);
}
// Reverse kernel, heads of several workgroups: the half of a step's adjoint that does not depend on the running cotangent is done behind the
// first probe of the step before, while the words travel.  16-bit gated cells at tilings that wait in one round (backward pass, bf16, T = 512: LSTM B8 T1024 N3
// D256 959 -> 912 us, B16 N4 D192 462 -> 431, N1 D384 588 -> 551, D512 680 -> 650, D640 830 -> 751, D768 937 -> 847, D1024 1094 -> 1043,
// GRU N3 D256 502 -> 460, D512 648 -> 592, D1024 1008 -> 963).  Not where it loses (kernels of the same tree that differ in nothing else):
// - the sLSTM's pairs of 4 and of more than 12 workgroups, but in bf16 20 and 24.  It needs a step's operands one wait earlier, and has the most of them: as soon
//   as a call has more to read than the last-level cache holds they come from memory, and these steps wait for them (fp16, T = 2000, B32 D128 1540 -> 1782, D448
//   2562 -> 2716, D512 2698 -> 3248, D640 T1046 1711 -> 1813, D768 3616 -> 3826, D1024 T653 1478 -> 1559, bf16 D512 2938 -> 3261, D1024 1214 -> 1239; where the
//   cache holds them, D448 +5 %, D128 and D512 to D1024 -2 to -6).  6 to 12 gain either way (D320 -4 to -7 %, D384 T4096 -10), as do bf16 at 20 (D640 -3 to -6)
//   and 24 (D768 -7 to +0.9), its fours (D256) and its single waves.
// - the GRU's single waves at 10 and 12 workgroups, 4-row tiles (D640, D768: +2.2 and +2.3 % at B1, -1.3 to +1.0 else; at 7 -3.2 to +0.4),
// - four gates at 3 workgroups or less, 4-row tiles (LSTM B160 N2 D192 T256 328 -> 333, T1024 1175 -> 1203, sLSTM 0 to +0.9 %; the GRU -3),
// - tiles of 8 and 16 rows of up to 5 workgroups, whose probes come back sooner than 2 or 4 elements are done, unless the operands are in
//   L2 (LSTM B256 N3 D256 1250 without either, 1261 with this, 1174 with both) or the cell is the GRU (1030 -> 954),
// - fp32, but for the LSTM's 4-row tiles of 16 to 48 workgroups (T = 256, B16 D256 359 -> 351, D384 537 -> 532, D512 625 -> 603, D640 1073 -> 1054, D768
//   1280 -> 1263; D1024, 64 workgroups, B1 1097 -> 1136, B4 1052 -> 1100; N3 D128 -1 %, sLSTM D256 +3, D128 +9, taller tiles +5 to +6),
// - the Elman cell, which has no more to prepare than a product (+-1 to +8 %).
constexpr bool bwd_adjoint_early(int GR, int nc, int D, int WAVES, int UTW, int KW, int TR, int esize, bool fp16, bool fetched) {
  const int dsp = bwd_dest_split(D, WAVES, UTW, KW);
  if (UTW != 1 || GR == 1) return false;
  if (esize == 4) return GR == 4 && nc == 4 && KW >= 16 && KW <= 48 && TR == 4;
  if (TR > 4) return GR == 3 || KW > 5 || fetched;
  if (GR == 3) return dsp > 1 || KW < 10;
  if (nc == 5 && dsp == 2) return (KW >= 6 && KW <= 12) || (!fp16 && KW > 16 && KW < 32);
  return KW > 3;
}
}

// Measured on MI355X (T = 1024, bf16): when the head fits one workgroup, one tile per wave and
// 8..16 waves (2..4 per SIMD, so one wave's gate math hides behind another's MFMAs) beats 4 waves
// with several tiles each; when it does not fit, 4 waves with one tile each and more workgroups
// beat fewer, fuller workgroups (the step is a dependency chain, not a throughput problem).
// ---- 4 recurrent gate rows per unit (lstm, slstm) --------------------------------------------
// (D = 1024, forward and backward: workgroups of two wave pairs, see fwd_k_split / bwd_dest_split; the reverse kernels
// stop at 8-row tiles: at 16 rows the sLSTM's, with four states, and the fp16 LSTM's spill, and the bf16 LSTM's, which
// does not, takes twice as long per launch as at 8 rows: LSTM bf16 B256 T512 12.5 against 12.8 ms)
#define FRNN_PLANS_GR4_BF16(X) \
  X(256, 4, 8, 1, 2, 16) \
  X(384, 2, 4, 1, 12, 4) X(448, 2, 4, 1, 14, 4) X(512, 2, 4, 1, 16, 4) X(640, 2, 4, 1, 20, 4) X(768, 2, 4, 1, 24, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 8) X(192, 0, 12, 1, 1, 4) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 32, 16)
#define FRNN_BWD_PLANS_GR4_BF16(X) \
  X(192, 2, 4, 1, 6, 4) X(256, 2, 4, 1, 8, 4) X(320, 2, 4, 1, 10, 4) X(384, 2, 4, 1, 12, 4) X(448, 2, 4, 1, 14, 4) X(512, 2, 4, 1, 16, 4) X(640, 2, 4, 1, 20, 4) X(768, 2, 4, 1, 24, 4) \
  X(160, 2, 2, 1, 5, 16) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 4) X(192, 0, 4, 1, 3, 16) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 32, 8)
// slstm backward: as above, but D = 160 as 5 workgroups of 2 waves (10 waves of 168 registers each spill at every tile height)
#define FRNN_BWD_PLANS_SLSTM_BF16(X) \
  X(128, 2, 4, 1, 2, 16) X(128, 3, 4, 1, 4, 4) X(192, 2, 4, 1, 6, 4) X(256, 2, 4, 1, 16, 4) X(320, 2, 4, 1, 10, 4) X(384, 2, 4, 1, 12, 4) X(448, 2, 4, 1, 14, 4) X(512, 2, 4, 1, 16, 4) X(640, 2, 4, 1, 20, 4) X(768, 2, 4, 1, 24, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 8) X(128, 0, 8, 1, 1, 8) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 32, 8)
// slstm: its heavier gate math tips D = 192 forward to 3 workgroups of 4 waves (1.19 against 1.26 ms)
#define FRNN_PLANS_SLSTM_BF16(X) \
  X(256, 4, 8, 1, 2, 16) \
  X(384, 2, 4, 1, 12, 4) X(448, 2, 4, 1, 14, 4) X(512, 2, 4, 1, 16, 4) X(640, 2, 4, 1, 20, 4) X(768, 2, 4, 1, 24, 4) \
  X(160, 2, 2, 1, 5, 16) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 8) X(192, 0, 4, 1, 3, 16) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 32, 16)
// fp32: a 16-unit tile of a gated cell takes G_r * D / 4 registers of a wave (D in the 4x4x1 form of the 4-row tiles).
// Forward, D = 384 .. 512: workgroups of two wave pairs, 4-row tiles only (see fwd_k_split; D = 16 * (WAVES / 2) * KW);
// D = 640 .. 1024: one tile per workgroup, k split over its four waves, groups that span the device (D = 16 * KW)
#define FRNN_PLANS_GR4_F32(X) \
  X(128, 2, 4, 1, 4, 4) X(128, 3, 4, 1, 8, 4) X(160, 2, 4, 1, 5, 4) X(192, 2, 4, 1, 6, 4) X(192, 3, 4, 1, 12, 4) X(256, 2, 4, 1, 8, 4) X(256, 3, 4, 1, 16, 4) \
  X(320, 2, 4, 1, 10, 4) X(320, 3, 4, 1, 20, 4) X(384, 3, 4, 1, 24, 4) X(448, 3, 4, 1, 28, 4) X(512, 3, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) \
  X(320, 0, 4, 1, 5, 8) X(384, 0, 4, 1, 12, 4) X(448, 0, 4, 1, 14, 4) X(512, 0, 4, 1, 16, 4) \
  X(640, 0, 4, 1, 40, 4) X(768, 0, 4, 1, 48, 4) X(1024, 0, 4, 1, 64, 4)
// (backward, D = 384 .. 512: workgroups of two wave pairs, D = 640 .. 1024: one tile position per workgroup, 4-row tiles
// only; see bwd_dest_split)
#define FRNN_BWD_PLANS_GR4_F32(X) \
  X(64, 2, 2, 1, 2, 16) X(64, 3, 4, 1, 4, 4) X(96, 3, 4, 1, 6, 4) X(128, 2, 4, 1, 4, 4) X(128, 3, 4, 1, 8, 4) X(160, 2, 4, 1, 5, 4) X(160, 3, 4, 1, 10, 4) X(192, 2, 4, 1, 6, 4) X(192, 3, 4, 1, 12, 4) \
  X(256, 2, 4, 1, 8, 4) X(256, 3, 4, 1, 16, 4) X(320, 2, 4, 1, 10, 4) X(320, 3, 4, 1, 20, 4) X(384, 3, 4, 1, 24, 4) X(448, 3, 4, 1, 28, 4) X(512, 3, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 8) X(96, 0, 2, 1, 3, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 8) \
  X(320, 0, 4, 1, 5, 8) X(384, 0, 4, 1, 12, 4) X(448, 0, 4, 1, 14, 4) X(512, 0, 4, 1, 16, 4) \
  X(640, 0, 4, 1, 40, 4) X(768, 0, 4, 1, 48, 4) X(1024, 0, 4, 1, 64, 4)
// slstm fp32 backward: the same, from the same measurements
#define FRNN_BWD_PLANS_SLSTM_F32(X) \
  X(64, 2, 2, 1, 2, 16) X(64, 3, 4, 1, 4, 4) X(96, 3, 4, 1, 6, 4) X(128, 2, 4, 1, 4, 4) X(128, 3, 4, 1, 8, 4) X(160, 2, 4, 1, 5, 4) X(160, 3, 4, 1, 10, 4) X(192, 2, 4, 1, 6, 4) X(192, 3, 4, 1, 12, 4) \
  X(256, 2, 4, 1, 8, 4) X(256, 3, 4, 1, 16, 4) X(320, 2, 4, 1, 10, 4) X(320, 3, 4, 1, 20, 4) X(384, 3, 4, 1, 24, 4) X(448, 3, 4, 1, 28, 4) X(512, 3, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 8) X(96, 0, 2, 1, 3, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 8) \
  X(320, 0, 4, 1, 5, 8) X(384, 0, 4, 1, 12, 4) X(448, 0, 4, 1, 14, 4) X(512, 0, 4, 1, 16, 4) \
  X(640, 0, 4, 1, 40, 4) X(768, 0, 4, 1, 48, 4) X(1024, 0, 4, 1, 64, 4)
// ---- 3 recurrent gate rows per unit (gru) ----------------------------------------------------
#define FRNN_PLANS_GR3_BF16(X) \
  X(256, 4, 8, 1, 2, 16) X(384, 4, 8, 1, 3, 16) \
  X(640, 2, 4, 1, 20, 4) X(768, 2, 4, 1, 24, 4) X(1024, 2, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 16) X(192, 0, 12, 1, 1, 16) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 16) X(1024, 0, 4, 1, 16, 16)
#define FRNN_BWD_PLANS_GR3_BF16(X) \
  X(256, 4, 8, 1, 2, 16) \
  X(192, 2, 4, 1, 3, 16) X(320, 2, 4, 1, 10, 4) X(512, 2, 4, 1, 16, 4) X(1024, 2, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 8) X(192, 0, 12, 1, 1, 4) \
  X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 16, 16)
#define FRNN_PLANS_GR3_F32(X) \
  X(128, 2, 4, 1, 4, 4) X(128, 3, 4, 1, 8, 4) X(160, 2, 4, 1, 5, 4) X(192, 2, 4, 1, 6, 4) X(192, 3, 4, 1, 12, 4) X(256, 2, 4, 1, 8, 4) X(256, 3, 4, 1, 16, 4) \
  X(320, 2, 4, 1, 10, 4) X(320, 3, 4, 1, 20, 4) X(384, 3, 4, 1, 24, 4) X(448, 3, 4, 1, 28, 4) X(512, 3, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) \
  X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 12, 4) X(448, 0, 4, 1, 14, 4) X(512, 0, 4, 1, 16, 4) \
  X(640, 0, 4, 1, 40, 4) X(768, 0, 4, 1, 48, 4) X(1024, 0, 4, 1, 64, 4)
#define FRNN_BWD_PLANS_GR3_F32(X) \
  X(64, 2, 2, 1, 2, 16) X(64, 3, 4, 1, 4, 4) X(96, 3, 4, 1, 6, 4) X(128, 2, 4, 1, 4, 4) X(128, 3, 4, 1, 8, 4) X(160, 2, 4, 1, 5, 4) X(160, 3, 4, 1, 10, 4) X(192, 2, 4, 1, 6, 4) X(192, 3, 4, 1, 12, 4) \
  X(256, 2, 4, 1, 8, 4) X(256, 3, 4, 1, 16, 4) X(320, 2, 4, 1, 10, 4) X(320, 3, 4, 1, 20, 4) X(384, 3, 4, 1, 24, 4) X(448, 3, 4, 1, 28, 4) X(512, 3, 4, 1, 32, 4) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 2, 1, 3, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) \
  X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 12, 4) X(448, 0, 4, 1, 14, 4) X(512, 0, 4, 1, 16, 4) \
  X(640, 0, 4, 1, 40, 4) X(768, 0, 4, 1, 48, 4) X(1024, 0, 4, 1, 64, 4)
// ---- 1 recurrent gate row per unit (elman) ---------------------------------------------------
#define FRNN_PLANS_GR1_BF16(X) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 16) X(192, 0, 12, 1, 1, 16) \
  X(256, 0, 16, 1, 1, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 8, 3, 1, 4) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) \
  X(768, 0, 8, 1, 6, 16) X(1024, 0, 8, 1, 8, 8)
#define FRNN_BWD_PLANS_GR1_BF16(X) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 8, 1, 1, 16) X(160, 0, 10, 1, 1, 16) X(192, 0, 12, 1, 1, 16) \
  X(256, 0, 16, 1, 1, 16) X(320, 0, 4, 1, 5, 16) X(384, 0, 8, 1, 3, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 8, 1, 4, 16) X(640, 0, 4, 1, 10, 16) \
  X(768, 0, 8, 1, 6, 16) X(1024, 0, 8, 1, 8, 4)
// (fp32: a 16-unit tile costs D / 4 MFMAs of 32 cycles per step whatever the batch tile, so heads from D = 128 on are
// spread over D / 64 workgroups with one tile per wave: D = 256 as one workgroup of 4 waves x 4 tiles took 8.0 ms
// per 1024 steps forward + backward, as 4 workgroups it takes 2.7)
#define FRNN_PLANS_GR1_F32(X) \
  X(96, 2, 2, 1, 3, 16) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) \
  X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 8) X(1024, 0, 4, 1, 16, 8)
#define FRNN_BWD_PLANS_GR1_F32(X) \
  X(96, 2, 2, 1, 3, 16) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 16) X(128, 0, 4, 1, 2, 16) X(160, 0, 2, 1, 5, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) \
  X(320, 0, 4, 1, 5, 16) X(384, 0, 4, 1, 6, 16) X(448, 0, 4, 1, 7, 16) X(512, 0, 4, 1, 8, 16) X(640, 0, 4, 1, 10, 16) X(768, 0, 4, 1, 12, 16) X(1024, 0, 4, 1, 16, 8)

// ---- reverse scan in recompute mode (no gate cache): R and R^T are both resident, so only the head
// dims whose two operands fit the registers beside the working set; same tilings as above where those
// fit (gru D = 192 runs as 3 workgroups of 4 waves here: 12 waves have 168 registers each).  D = 320 (and 384 for the
// GRU, three gate rows) at 4-row tiles only; the 4-gate cells spill at D = 384, the GRU at D = 512.
#define FRNN_BWD_RC_PLANS_GR4_BF16(X) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 4) X(128, 0, 4, 1, 2, 16) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 8) X(320, 0, 4, 1, 5, 4)
// slstm: D = 192 stops at 8-row tiles (its 16-row kernel, with both operands resident and four states, spills)
#define FRNN_BWD_RC_PLANS_SLSTM_BF16(X) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 4) X(128, 0, 4, 1, 2, 16) X(192, 0, 4, 1, 3, 8) X(256, 0, 4, 1, 4, 8) X(320, 0, 4, 1, 5, 4)
#define FRNN_BWD_RC_PLANS_GR3_BF16(X) \
  X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16) X(96, 0, 6, 1, 1, 8) X(128, 0, 8, 1, 1, 8) X(192, 0, 4, 1, 3, 16) X(256, 0, 4, 1, 4, 16) X(320, 0, 4, 1, 5, 4) X(384, 0, 4, 1, 6, 4)
#define FRNN_BWD_RC_PLANS_GR4_F32(X) X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16)
#define FRNN_BWD_RC_PLANS_GR3_F32(X) X(32, 0, 2, 1, 1, 16) X(64, 0, 4, 1, 1, 16)
#define FRNN_BWD_RC_PLANS_NONE(X)
