// C entry points of the prefill attention kernel (fk_prefill_kernel.h):
// fk_paged_prefill (FlashAttnPrefill with a block table) and fk_varlen_prefill
// (dense keys: FlashAttnPrefill without one, and FlashAttnVarlen).  This file
// instantiates the kernel at D = DV in {64, 128, 256} with bf16 and fp8 pages
// and dense keys; fk_prefill_heads.hip instantiates the other head sizes.
#include <algorithm>

#include "fk_prefill_kernel.h"

namespace fk {
namespace {

// (query / key, value) head sizes the library is built for.
bool prefill_heads_supported(int d, int dv, bool fp8_pages) {
  if (fp8_pages) return d == dv && (d == 64 || d == 128 || d == 256);
  if (d == dv)
    return d == 32 || d == 64 || d == 72 || d == 80 || d == 96 || d == 128 || d == 256;
  return d == 192 && dv == 128;
}

template <int D>
void launch_prefill_d(bool paged, bool fp8, bool split, const PrefillParams& P, dim3 grid,
                      const int32_t* bt, const int32_t* cu_q, const int32_t* cu_k,
                      hipStream_t stream) {
  if (paged && fp8)
    launch_prefill<true, true, D, D>(split, P, grid, bt, cu_q, cu_k, stream);
  else
    launch_prefill_bf16<D, D>(paged, split, P, grid, bt, cu_q, cu_k, stream);
}

// Query tokens per work-group.
int64_t prefill_wg_tokens(int gqa, int col_blocks) {
  const int hw = gqa < kPrefillWaves ? gqa : kPrefillWaves;
  return static_cast<int64_t>(kPrefillWaves / hw) * 16 * col_blocks;
}

// Launch shape of a prefill call, from the host-side bounds alone (the plan
// entry point and the launch agree on it).
struct PrefillShape {
  int col_blocks;     // 16-query column blocks per wave
  int64_t wg_tokens;  // query tokens per work-group
  int64_t qblocks;    // query blocks per sequence (grid z before the key parts)
  bool may_pair;      // causal pairs of blocks may occur
  int hsplit;         // work-groups per kv head (head groups of up to 4)
  int ks;             // key parts within a work-group (1 or 2)
  int xs;             // key parts over work-groups (1: none), with a workspace
  int ks_plain;       // ks of the same call without a workspace (xs = 1)
  bool part_f32;      // the key parts' O in fp32 rather than bf16
};

// MLA's head sizes (one_col_block_built): two column blocks a wave, or one.  Two serve 32
// queries with each K / V byte read from LDS but make half as many work-groups; with too
// few of them CUs stay idle and each one's block takes longer.  Two where their
// work-groups (a causal pair counts as one) pass half of the CUs, or their keys are long
// enough that parts of them make up for it: 1800 and 2^17 over all work-groups, 2^19 for
// causal pairs, which see half and run in one part.  A block of 128 of at most 64 queries
// would be half empty: one.  Measured on one box, us, one / two (heads of 192 / 128):
//   causal, 16 heads: 1x256 13.2 / 20.1, 1x1024 27 / 33, 1x2048 43 / 48, 4x512 20 / 27,
//     32x33 7.3 / 8.8; 877 and 1200 47 / 40, 1x3000 111 / 75, 4x1024 42.2 / 39.5, 16x400
//     47 / 40
//   not causal, 16 heads: 1x512 over 1024 22 / 26, 1x1024 over 1024 23 / 28, 92 and 95 over
//     745 17 / 19; 598 over 2279 43 / 34, 62 .. 107 over 3340 37 / 27; 1x512 over
//     4096 44 / 39, 1x2000 over 2000 61 / 51, 8x200 over 1000 35 / 32; 128 heads: 4x256
//     over 512 83 / 67, 8x200 over 1000 300 / 210
bool two_col_blocks(int64_t batch, int64_t total_q, int64_t max_seqlen_q, int64_t max_seqlen_k,
                    int64_t grid_x, int64_t wg_tokens, int causal) {
  if (2 * max_seqlen_q <= wg_tokens) return false;
  const bool pairs = causal && max_seqlen_k < 2 * max_seqlen_q;
  int64_t blocks = batch * ((max_seqlen_q + wg_tokens - 1) / wg_tokens);
  if (total_q > 0) blocks = std::min(blocks, total_q / wg_tokens + batch);
  const int64_t wgs = grid_x * (pairs ? (blocks + 1) / 2 : blocks);
  const int64_t keys = std::max(max_seqlen_k, max_seqlen_q);
  return 2 * wgs > num_cus() ||
         (pairs ? wgs * keys >= int64_t(1) << 19 : keys >= 1800 && wgs * keys >= int64_t(1) << 17);
}

// total_q: the rows of q, or 0 if unknown.
PrefillShape prefill_shape(bool paged, bool fp8, int64_t batch, int64_t total_q,
                           int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads,
                           int num_kv_heads, int head_size, int head_size_v, int causal) {
  PrefillShape sh;
  const int gqa = num_heads / num_kv_heads;
  const int hw = gqa < kPrefillWaves ? gqa : kPrefillWaves;  // query heads per work-group
  sh.hsplit = (gqa + hw - 1) / hw;
  sh.col_blocks = col_blocks_for(head_size, head_size_v);
  if (one_col_block_built(head_size, head_size_v) &&
      !two_col_blocks(batch, total_q, max_seqlen_q, max_seqlen_k,
                      static_cast<int64_t>(num_kv_heads) * sh.hsplit,
                      prefill_wg_tokens(gqa, 2), causal))
    sh.col_blocks = 1;
  const int64_t wg_tokens = prefill_wg_tokens(gqa, sh.col_blocks);
  sh.wg_tokens = wg_tokens;
  sh.qblocks = (max_seqlen_q + wg_tokens - 1) / wg_tokens;
  // Key split when the 4-wave launch would leave SIMDs with one wave: fewer
  // work-groups than two per CU.  A causal sequence with fewer cached keys than
  // twice its queries pairs its blocks two per work-group; max_seqlen_k (a
  // bound on every sequence's keys, 0 = unknown) tells whether that can happen.
  const bool may_pair = causal && max_seqlen_k > 0 && max_seqlen_k < 2 * max_seqlen_q;
  sh.may_pair = may_pair;
  const int64_t wgs = static_cast<int64_t>(num_kv_heads) * sh.hsplit * batch *
                      (may_pair ? (sh.qblocks + 1) / 2 : sh.qblocks);
  sh.ks = ((std::max(head_size, head_size_v) <= 192 || paged) && wgs < 2LL * num_cus()) ? 2 : 1;
  sh.ks_plain = sh.ks;
  sh.xs = 1;
  sh.part_f32 = part_in_f32(head_size, head_size_v);
  const int64_t ncu = num_cus();
  // Where the key split would run (fewer 4-wave work-groups than two per CU):
  // 4-wave work-groups, two per CU, with each block's keys in xs parts over
  // work-groups, instead of one 8-wave key-split work-group per block, for
  // chunks over cached keys (blocks not paired) and, at head sizes up to 64 with
  // bf16 pages, for causal pairs.  xs = floor(2 CUs / work-groups) when that is
  // at least 2 and fills 7/8 of the two-per-CU slots; else the parts run in two
  // rounds of the slots, and xs = floor(4 CUs / work-groups), the most that two
  // rounds hold (the ceiling of one round's, taken before, ran as many rounds of
  // longer parts; same box, us, whole call: Qwen3-8B heads 1x800 over 8192 168 ->
  // 126, 1x1100 over 8192 244 -> 189, over 16000 on fp8 pages 568 -> 403, 2x600 over
  // 6000 171 -> 135, MLA 877 and 1200 over 2669 and 3300 194.5 -> 167.6; where the
  // quotients agree nothing changes).  At most kMaxKeyParts, and only while a part
  // keeps at least 20 stages of 32 keys (40
  // above head size 64: a dense 2048-token non-causal prompt at 16 / 16 / 80
  // heads, 2 parts of 32 stages, went 48.8 -> 52.9).
  // Measured on MI355X (whole call, µs, key split -> this; same box, A/B in
  // alternating processes, two rounds averaged): Qwen3-8B heads (32 / 8 / 128)
  // 1x512 over 8192 102.9 -> 91.2, 2x512 over 4096 92.8 -> 86.5, 3x512 over 4096
  // 160.2 -> 145.9, fp8 pages 1x512 over 8192 114.7 -> 109.8; Qwen3-Next heads
  // (16 / 2 / 256) 1x512 over 8192 116.0 -> 106.4, 2x512 over 4096 109.4 ->
  // 103.5; Whisper heads (20 / 20 / 64) 4x512 over 4096 112.9 -> 80.4, 2x512
  // over 4096 57.2 -> 47.8, 1x512 over 8192 54.9 -> 48.5, prompts 1x2048 45.2 ->
  // 40.8, 2x2048 80.5 -> 61.7, 1x4096 132.0 -> 93.7; dense keys, 1x512 over 8192
  // at Qwen3-8B heads 98.6 -> 90.1 and at MLA's (16 / 16 / 192 / 128, not
  // causal) 92.7 -> 81.2, 2x512 over 4096 93.7 -> 89.4.  In single probes, causal
  // pairs at head 128 and 256 were slower this way (1x2048: 58.9 -> 68.3 and
  // 65.7 -> 73.8; they keep the key split with split pairs), and so were short
  // parts (Whisper heads 2x1024 at 3 parts of 12 stages: 31.6 -> 33.2).
  if (sh.ks == 2 && wgs > 0 &&
      (!may_pair || (!fp8 && std::max(head_size, head_size_v) <= 64))) {
    const int64_t slots = 2 * ncu;
    int64_t xs = slots / wgs;
    const bool one_round = xs >= 2 && 8 * wgs * xs >= 7 * slots;
    if (!one_round) xs = 2 * slots / wgs;
    xs = std::min<int64_t>(xs, kMaxKeyParts);
    const double stages = static_cast<double>(std::max(max_seqlen_k, max_seqlen_q) +
                                              (may_pair ? wg_tokens : 0)) /
                          kStageKeys;  // the heaviest work-group's stages (a pair's)
    const double min_stages = std::max(head_size, head_size_v) <= 64 ? 20.0 : 40.0;
    // (Keys too few for the parts of two rounds: the fewest that leave no slot idle.)
    if (!one_round && stages < min_stages * xs)
      xs = std::min<int64_t>((slots + wgs - 1) / wgs, kMaxKeyParts);
    if (xs >= 2 && stages >= min_stages * xs && sh.qblocks * xs <= 65535) {
      sh.ks = 1;
      sh.xs = static_cast<int>(xs);
      return sh;
    }
  }
  // Otherwise, work-group key split when even the key split leaves CUs without
  // a work-group (one work-group per CU at this size): each block's keys in xs
  // parts over xs work-groups, merged by prefill_merge_kernel.  xs minimises an
  // estimate of the call's time (µs; constants measured on MI355X): the heaviest work-group
  // streams S stages of 32 keys (all of max_seqlen_k; a causal pair of blocks
  // about max_seqlen_k plus one block) at kStageUs per stage and key-split half,
  // plus kBlockUs per block (its queries, the first stage's latency, the rows);
  // the work-groups run ceil(wgs * xs / CUs) rounds; the parts' states are
  // written and read back at kMergeBytesPerUs, plus kMergeUs for the merge's
  // launch.  Short blocks (prompts) keep one part: their per-block costs stay.
  // (The constants were fitted with the parts' O in fp32; the estimate keeps
  // those bytes, so that its choices stay the measured ones.)
  if (wgs > 0 && wgs < ncu) {
    constexpr double kStageUs = 1.2, kBlockUs = 6.0, kMergeUs = 3.0;
    constexpr double kMergeBytesPerUs = 2.5e6;
    const int64_t keys = std::max(max_seqlen_k, max_seqlen_q);
    const int blocks = may_pair ? 2 : 1;
    const double S = static_cast<double>(keys + (may_pair ? wg_tokens : 0)) / kStageKeys;
    const double row_bytes =
        static_cast<double>(batch) * max_seqlen_q * num_heads * (head_size_v + kPartMl) * 4;
    double best = S / sh.ks * kStageUs + blocks * kBlockUs;
    for (int xs = 2; xs <= kMaxKeyParts; ++xs) {
      if (S < 4.0 * xs * sh.ks || sh.qblocks * xs > 65535) break;
      const double rounds = static_cast<double>((wgs * xs + ncu - 1) / ncu);
      const double t = rounds * (S / (sh.ks * xs) * kStageUs + blocks * kBlockUs) +
                       xs * row_bytes / kMergeBytesPerUs + kMergeUs;
      if (t < best) {
        best = t;
        sh.xs = xs;
      }
    }
  }
  return sh;
}

// The launch's item order: the number of sequences for the kernel's longest-first order
// (PrefillParams::lpt), or 0 for the grid's own (sequence by sequence, block index
// slowest).  items: an upper bound of the launch's query blocks (pairs count twice).
//
// Longest first fills the tail of a ragged launch and leaves no gaps for the absent
// blocks of its shorter sequences, but every work-group pays for finding its item, about
// 0.045 us a sequence, and it takes a sequence's blocks together: at equal lengths the
// light last blocks no longer come last, and where the grid's x is not a multiple of the
// 8 XCDs a sequence's blocks read its keys through several L2s.  Measured on one box,
// whole calls, us, own order / longest first (lengths uniform in the range given):
//   equal lengths: 9 x 200 at 32 / 8 / 128 22 / 33, 64 x 100 39 / 48, 64 x 200 at 64 / 8 /
//     64 80 / 119, 64 x 32 over 2000 at 16 / 2 / 256 113 / 170
//   ragged and short: 64 x (4 .. 40) 14 / 19, a vision batch of 64 x (15 .. 60) 12.7 / 18.7
//   ragged: 5 x (60 .. 600) 36 / 24, 16 x (150 .. 1500) 228 / 155, 16 x (75 .. 300) over
//     (1000 .. 4000) 238 / 167, 2 x (150 .. 1500) 71 / 40
//   ragged, many: 64 x (60 .. 600) 198 / 213, at 64 / 8 / 64 206 / 255
//   equal lengths whose keys pass the caches: 64 x 200 over 1000 399 / 372, at 16 / 2 / 256
//     507 / 378, 64 x 600 at 16 / 2 / 256 512 / 412
//   prompts nearly alike: 2 x 2000, rows 92 % of the longest's, 77 / 70, 96 % 76 / 74, 100 %
//     80 / 82; 4 x 1000, 91 % 46 / 42, 96 % 47 / 46, 100 % 49 / 51; 32 x 600, 91 % 157 / 162
//   chunks of one length over contexts alike / down to 3/4 / down to 1/4 of the longest:
//     16 x 256 over 4000 304 / 315, 293 / 288, 266 / 210; 4 x 512 over 4000 147 / 156, 145 /
//     144, 143 / 139; 32 x 128 over 4000 at 16 / 2 / 256 390 / 390, 406 / 330, 375 / 251; over
//     shorter ones 16 x 256 over 1000 92 / 102, 88 / 92, 87 / 75, 8 x 512 over 1000 101 /
//     110, 96 / 103, 91 / 102
//   not causal, 16 heads of 72, lengths alike: 16 x 1500 307 / 238, 32 x 700 167 / 131, 64 x
//     300 93 / 86, 8 x 1500 (61 MB) 122 / 123, 16 x 300 22 / 22, 32 x 150 21 / 25; 20 heads of
//     64 16 x 1500 238 / 244; 16 heads of 192 / 128 over other keys: 1226 and 1217 over 1454 and
//     2192 99 / 76, 4 x 1200 over 950 .. 1600 114 / 92, 3 x 1070 .. 1250 over 180 .. 275 30 / 30
// so it is taken when
//   - the launch holds more work-groups than CUs (else each has a CU to itself in any
//     order) of four stages or more, with long keys already at 3/4 of them, and
//   - the lengths differ: the rows are fewer than 90 % of batch * max_seqlen_q, 96 % where
//     an item's stages are 30 and half of sequences times rounds or more (total_q 0: unknown,
//     taken as ragged), or 48 stages and more are mostly cached keys, or, not causal, 16 and
//     more are of other lengths than the queries: the host does not know the keys' lengths
//     (taken as ragged too).  And the search stays small against an item's stages: at most
//     9 sequences times rounds of the slots for each; or
//   - over four rounds and more the batch's keys exceed what holds them: the last-level
//     cache, or, where a work-group computes 64 rows for each key read (head size 256),
//     the L2s; not causal (no light last blocks to lose) from three rounds, 8 stages and
//     48 MB on where a head's blocks stay on one XCD.
// Head 256 with one or two blocks a sequence in one round keeps its own order (the L2s)
// below 96 stages (32 x 32 over 1000 36 / 46; over 1000 .. 4000 99 / 88).
int prefill_order(const PrefillShape& sh, int xs, int64_t batch, int64_t total_q,
                  int64_t max_seqlen_q, int64_t max_seqlen_k, int num_kv_heads, int head_size,
                  int head_size_v, int causal, int window_left, int elem, int64_t items) {
  if (batch > 64 || items * xs > 65535) return 0;
  if (batch == 1) return 1;  // (its blocks in order, at no cost)
  const double ncu = num_cus();
  const double gx = static_cast<double>(num_kv_heads) * sh.hsplit * xs / (sh.may_pair ? 2 : 1);
  double keys = static_cast<double>(std::max(max_seqlen_k, max_seqlen_q));
  if (window_left >= 0)
    keys = std::min(keys, static_cast<double>(window_left) + static_cast<double>(sh.wg_tokens));
  const double stages = keys / kStageKeys;
  const double wgs = gx * static_cast<double>(batch * sh.qblocks);  // absent blocks included
  if (!(wgs > ncu * 9 / 8 && stages >= 4) && !(wgs > ncu * 3 / 4 && stages >= 32)) return 0;
  const double rounds = gx * static_cast<double>(items) / (2 * ncu);
  const bool few_rows = sh.col_blocks == 1;
  const double key_bytes =
      static_cast<double>(batch) * keys * num_kv_heads * (head_size + head_size_v) * elem;
  if (rounds >= 4 && key_bytes > (few_rows ? 32e6 : 256e6)) return static_cast<int>(batch);
  const double load = batch * rounds / stages;  // the search against an item's work
  if (!causal && num_kv_heads * sh.hsplit % 8 == 0 && rounds >= 3 && stages >= 8 &&
      key_bytes > 48e6)
    return static_cast<int>(batch);
  // Keys whose lengths the bounds do not tell.
  const bool cached = causal ? max_seqlen_k >= 2 * max_seqlen_q && stages >= 48
                             : max_seqlen_k > 0 && max_seqlen_k != max_seqlen_q && stages >= 16;
  const int64_t alike = stages >= 30 && load <= 2 ? 96 : 90;  // percent
  if (!cached && total_q > 0 && 100 * total_q > alike * batch * max_seqlen_q) return 0;
  if (few_rows && num_kv_heads * sh.hsplit % 8 != 0 && rounds <= 1 && sh.qblocks <= 2 &&
      stages < 96)
    return 0;
  return load <= 9 ? static_cast<int>(batch) : 0;
}

// Bytes of the work-group key split's partial states (0 without the split).
int64_t prefill_ws_bytes(const PrefillShape& sh, int64_t total_q, int num_heads, int head_size_v) {
  if (sh.xs <= 1) return 0;
  const int64_t bytes = part_ml_offset(sh.xs, total_q, num_heads, head_size_v, sh.part_f32) +
                        static_cast<int64_t>(sh.xs) * total_q * num_heads * kPartMl * 4;
  return (bytes + 255) / 256 * 256;
}

// The merge of a work-group key split: per (row, head), the parts' states
// combined with the log-sum-exp rule (M = max m_p, O = sum O_p 2^(m_p - M),
// l = sum l_p 2^(m_p - M); a part that saw no key has m_p = -inf and weighs 0),
// the sink joined to the sum, O / l written as bf16 (0 for a row with no visible
// key), and the log-sum-exp from the fp32 sums.  A thread takes 8 dims of one
// (row, head); rows past cu_seqlens_q[batch] are left alone.
struct PrefillMergeParams {
  uint16_t* out;
  int64_t out_row_stride;
  const void* part;
  int64_t part_rows;
  int xs;
  int num_heads;
  int dv;
  const int32_t* cu_q;
  int64_t batch;
  const float* sinks;
  float* lse;
  int64_t lse_row_stride;
};

template <bool kF32>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillMergeParams M) {
  const int chunks = M.dv / 8;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t rh = t / chunks;
  const int c8 = static_cast<int>(t - rh * chunks);
  const int64_t rows = M.cu_q[M.batch];
  if (rh >= rows * M.num_heads) return;
  const int64_t row = rh / M.num_heads;
  const int hq = static_cast<int>(rh - row * M.num_heads);
  const int64_t plane = M.part_rows * M.num_heads;  // (row, head) records per part
  const float* const ml = reinterpret_cast<const float*>(
      static_cast<const uint8_t*>(M.part) + part_ml_offset(M.xs, M.part_rows, M.num_heads, M.dv, kF32));
  const uint8_t* const po = static_cast<const uint8_t*>(M.part);
  // Every part's record and O slice (8 values) are loaded before any is used.
  float4 rec[kMaxKeyParts];
  uint4 ov[kMaxKeyParts];
  float4 of[kF32 ? kMaxKeyParts : 1][2];
#pragma unroll
  for (int p = 0; p < kMaxKeyParts; ++p) {
    if (p < M.xs) {
      rec[p] = *reinterpret_cast<const float4*>(ml + (p * plane + rh) * kPartMl);
      const int64_t at = (p * plane + rh) * M.dv + 8 * c8;
      if constexpr (kF32) {
        of[p][0] = *reinterpret_cast<const float4*>(po + at * 4);
        of[p][1] = *reinterpret_cast<const float4*>(po + at * 4 + 16);
      } else {
        ov[p] = *reinterpret_cast<const uint4*>(po + at * 2);
      }
    }
  }
  float mx = kNegInf;
#pragma unroll
  for (int p = 0; p < kMaxKeyParts; ++p)
    if (p < M.xs) mx = fmaxf(mx, rec[p].x);
  float l = 0.f, l32 = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < kMaxKeyParts; ++p) {
    if (p < M.xs) {
      const float w = rec[p].x == kNegInf ? 0.f : __builtin_amdgcn_exp2f(rec[p].x - mx);
      l += w * rec[p].y;
      l32 += w * rec[p].z;
      if constexpr (kF32) {
        const float x[8] = {of[p][0].x, of[p][0].y, of[p][0].z, of[p][0].w,
                            of[p][1].x, of[p][1].y, of[p][1].z, of[p][1].w};
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += w * x[i];
      } else {
        const uint32_t ow[4] = {ov[p].x, ov[p].y, ov[p].z, ov[p].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // dims 2i (low half) and 2i + 1 (high half)
          acc[2 * i] += w * __builtin_bit_cast(float, ow[i] << 16);
          acc[2 * i + 1] += w * __builtin_bit_cast(float, ow[i] & 0xffff0000u);
        }
      }
    }
  }
  const float sink2 = M.sinks ? M.sinks[hq] * kLog2e : kNegInf;
  l = with_sink(l, mx, sink2);
  const float f = l > 0.f ? 1.f / l : 0.f;
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bf16x2_t pk = {static_cast<__bf16>(acc[2 * i] * f), static_cast<__bf16>(acc[2 * i + 1] * f)};
    w[i] = __builtin_bit_cast(uint32_t, pk);
  }
  *reinterpret_cast<uint4*>(M.out + row * M.out_row_stride + static_cast<int64_t>(hq) * M.dv +
                            8 * c8) = make_uint4(w[0], w[1], w[2], w[3]);
  if (M.lse && c8 == 0) {
    l32 = with_sink(l32, mx, sink2);
    M.lse[hq * M.lse_row_stride + row] =
        l32 > 0.f ? (mx + __log2f(l32)) * 0.6931471805599453f : kNegInf;
  }
}

int prefill_entry(const char* name, bool paged, void* out, int64_t out_row_stride, const void* q,
                  int64_t q_row_stride, const void* k, int64_t k_row_bytes, const void* v,
                  int64_t v_row_bytes, int kv_dtype, const float* k_scale, const float* v_scale,
                  const int32_t* block_tables, int64_t bt_row_stride,
                  const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t batch,
                  int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads, int num_kv_heads,
                  int head_size, int head_size_v, int block_size, int64_t num_blocks,
                  float scale, int causal, int window_left, const float* sinks, float* lse,
                  int64_t lse_row_stride, int64_t total_q, void* workspace, int64_t ws_bytes,
                  void* stream) {
  FK_REQUIRE(batch >= 0 && batch <= 65535, "%s: batch %lld out of range [0, 65535]", name,
             (long long)batch);
  FK_REQUIRE(window_left >= -1, "%s: window_left %d must be -1 (no window) or >= 0", name,
             window_left);
  FK_REQUIRE(window_left < 0 || causal,
             "%s: a sliding window needs causal attention (window_size = (left, 0))", name);
  FK_REQUIRE(max_seqlen_q >= 0 && max_seqlen_q <= (int64_t(1) << 30),
             "%s: max_seqlen_q %lld out of range", name, (long long)max_seqlen_q);
  FK_REQUIRE(max_seqlen_k >= 0, "%s: max_seqlen_k %lld must be >= 0 (0: unknown)", name,
             (long long)max_seqlen_k);
  FK_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             "%s: num_heads %d must be a positive multiple of num_kv_heads %d", name, num_heads,
             num_kv_heads);
  if (!prefill_heads_supported(head_size, head_size_v, kv_dtype == FK_DTYPE_FP8_E4M3FN && paged))
    return set_error(FK_ERR_UNSUPPORTED,
                     "%s: head sizes (query/key %d, value %d) unsupported: equal sizes 32, 64, 72, "
                     "80, 96, 128 or 256, or 192 / 128 (fp8 pages: 64, 128 or 256)",
                     name, head_size, head_size_v);
  FK_REQUIRE(num_kv_heads <= 32767, "%s: too many kv heads", name);
  if (paged) {
    FK_REQUIRE(block_size >= kTile && (block_size & (block_size - 1)) == 0,
               "%s: block_size %d must be a power of two >= 16", name, block_size);
    FK_REQUIRE(kv_dtype == FK_DTYPE_BF16 || kv_dtype == FK_DTYPE_FP8_E4M3FN,
               "%s: kv dtype %d unsupported (bf16 or fp8 e4m3fn)", name, kv_dtype);
  }
  FK_REQUIRE(q_row_stride >= static_cast<int64_t>(num_heads) * head_size &&
                 out_row_stride >= static_cast<int64_t>(num_heads) * head_size_v,
             "%s: row stride shorter than num_heads * head_size", name);
  const int64_t elem = kv_dtype == FK_DTYPE_FP8_E4M3FN ? 1 : 2;
  FK_REQUIRE(k_row_bytes >= num_kv_heads * head_size * elem &&
                 v_row_bytes >= num_kv_heads * head_size_v * elem,
             "%s: key/value rows shorter than num_kv_heads * head size", name);
  // The kernel addresses a page's rows (a dense tile's 16 rows) by 32-bit offsets
  // from the page's (tile's) first row.
  FK_REQUIRE((paged ? static_cast<int64_t>(block_size) : int64_t(kTile)) *
                     (k_row_bytes > v_row_bytes ? k_row_bytes : v_row_bytes) <=
                 (int64_t(1) << 32) - 1,
             "%s: a page of key/value rows must span fewer than 2^32 bytes", name);
  FK_REQUIRE(!lse || lse_row_stride >= 0, "%s: lse row stride must be >= 0", name);
  FK_REQUIRE(!lse || !paged, "%s: the log-sum-exp output is built for dense keys only", name);
  if (batch == 0 || max_seqlen_q == 0) return FK_OK;
  FK_REQUIRE(out && q && k && v && cu_seqlens_q && cu_seqlens_k && (!paged || block_tables),
             "%s: null pointer", name);
  FK_REQUIRE(!paged || num_blocks >= 1, "%s: the cache must hold at least one block", name);
  FK_REQUIRE(aligned16(q) && aligned16(out) && aligned16(k) && aligned16(v) &&
                 q_row_stride % 8 == 0 && out_row_stride % 8 == 0 && k_row_bytes % 16 == 0 &&
                 v_row_bytes % 16 == 0,
             "%s: q/out/keys/values must be 16-byte aligned with 16-byte row strides", name);
  const bool fp8 = kv_dtype == FK_DTYPE_FP8_E4M3FN;
  PrefillShape sh = prefill_shape(paged, fp8, batch, workspace ? total_q : 0, max_seqlen_q,
                                  max_seqlen_k, num_heads, num_kv_heads, head_size, head_size_v,
                                  causal);
  if (workspace == nullptr) {
    sh.xs = 1;  // no workspace: the launch without the work-group key split
    sh.ks = sh.ks_plain;
  } else {
    FK_REQUIRE(total_q >= 0, "%s: total_q %lld must be >= 0", name, (long long)total_q);
    const int64_t need = prefill_ws_bytes(sh, total_q, num_heads, head_size_v);
    if (ws_bytes < need)
      return set_error(FK_ERR_WORKSPACE, "%s: workspace of %lld bytes < %lld required", name,
                       (long long)ws_bytes, (long long)need);
    FK_REQUIRE(aligned16(workspace), "%s: workspace must be 16-byte aligned", name);
  }
  const int64_t qblocks = sh.qblocks;
  PrefillParams P;
  P.out = static_cast<uint16_t*>(out);
  P.out_row_stride = out_row_stride;
  P.q = static_cast<const uint16_t*>(q);
  P.q_row_stride = q_row_stride;
  P.k_cache = static_cast<const uint8_t*>(k);
  P.v_cache = static_cast<const uint8_t*>(v);
  P.k_row_bytes = k_row_bytes;
  P.v_row_bytes = v_row_bytes;
  P.k_scale = k_scale;
  P.v_scale = v_scale;
  P.bt_row_stride = paged ? bt_row_stride : 0;
  P.num_kv_heads = num_kv_heads;
  P.gqa = num_heads / num_kv_heads;
  P.block_size_log2 = paged ? __builtin_ctz(static_cast<unsigned>(block_size)) : 0;
  P.num_blocks = paged ? num_blocks : 0;
  FK_REQUIRE(scale > 0.f && scale < __builtin_huge_valf(),
             "%s: softmax scale must be positive and finite (got %g)", name, (double)scale);
  P.scale_log2 = scale * kLog2e;
  P.causal = causal ? 1 : 0;
  P.window_left = window_left;
  P.sinks = sinks;
  P.lse = lse;
  P.lse_row_stride = lse_row_stride;
  P.xs = sh.xs;
  P.part = workspace;
  P.part_rows = total_q;
  P.num_heads = num_heads;
  P.col_blocks = sh.col_blocks;
  FK_REQUIRE(qblocks <= 65535, "%s: max_seqlen_q %lld needs more than 65535 query blocks", name,
             (long long)max_seqlen_q);
  // Items: at most ceil(q_len / block) per sequence, and with a workspace (whose size
  // total_q was already bounded by) no more than total_q rows hold.
  int64_t items = batch * qblocks;
  if (workspace != nullptr && total_q > 0)
    items = std::min(items, total_q / sh.wg_tokens + batch);
  P.lpt = prefill_order(sh, sh.xs, batch, workspace ? total_q : 0, max_seqlen_q, max_seqlen_k,
                        num_kv_heads, head_size, head_size_v, causal, window_left,
                        static_cast<int>(elem), items);
  const dim3 grid =
      P.lpt ? dim3(static_cast<unsigned>(num_kv_heads * sh.hsplit),
                   static_cast<unsigned>(items * sh.xs), 1)
            : dim3(static_cast<unsigned>(num_kv_heads * sh.hsplit), static_cast<unsigned>(batch),
                   static_cast<unsigned>(qblocks * sh.xs));
  hipStream_t s = as_stream(stream);
  const bool split = sh.ks > 1;
  if (head_size == head_size_v && (head_size == 64 || head_size == 128 || head_size == 256)) {
    switch (head_size) {
      case 64: launch_prefill_d<64>(paged, fp8, split, P, grid, block_tables, cu_seqlens_q, cu_seqlens_k, s); break;
      case 256: launch_prefill_d<256>(paged, fp8, split, P, grid, block_tables, cu_seqlens_q, cu_seqlens_k, s); break;
      default: launch_prefill_d<128>(paged, fp8, split, P, grid, block_tables, cu_seqlens_q, cu_seqlens_k, s); break;
    }
  } else if (!launch_prefill_extra(head_size, head_size_v, paged, split, P, grid, block_tables,
                                   cu_seqlens_q, cu_seqlens_k, s)) {
    return set_error(FK_ERR_UNSUPPORTED, "%s: head sizes %d / %d not built", name, head_size,
                     head_size_v);
  }
  if (sh.xs > 1) {
    PrefillMergeParams M;
    M.out = static_cast<uint16_t*>(out);
    M.out_row_stride = out_row_stride;
    M.part = P.part;
    M.part_rows = total_q;
    M.xs = sh.xs;
    M.num_heads = num_heads;
    M.dv = head_size_v;
    M.cu_q = cu_seqlens_q;
    M.batch = batch;
    M.sinks = sinks;
    M.lse = lse;
    M.lse_row_stride = lse_row_stride;
    const int64_t threads = total_q * num_heads * (head_size_v / 8);
    const dim3 mgrid(static_cast<unsigned>((threads + 255) / 256));
    if (threads > 0 && sh.part_f32)
      hipLaunchKernelGGL(prefill_merge_kernel<true>, mgrid, dim3(256), 0, s, M);
    else if (threads > 0)
      hipLaunchKernelGGL(prefill_merge_kernel<false>, mgrid, dim3(256), 0, s, M);
  }
  return check_launch(name);
}

}  // namespace
}  // namespace fk

extern "C" int fk_paged_prefill(void* out, int64_t out_row_stride, const void* q,
                                int64_t q_row_stride, const void* k_cache, const void* v_cache,
                                int kv_dtype, const float* k_scale, const float* v_scale,
                                const int32_t* block_tables, int64_t bt_row_stride,
                                const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                int64_t batch, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                int num_heads, int num_kv_heads, int head_size, int head_size_v,
                                int block_size, int64_t num_blocks, float scale, int causal,
                                int window_left, const float* sinks, void* stream) {
  const int64_t elem = kv_dtype == FK_DTYPE_FP8_E4M3FN ? 1 : 2;
  const int64_t k_row = static_cast<int64_t>(num_kv_heads) * head_size * elem;
  const int64_t v_row = static_cast<int64_t>(num_kv_heads) * head_size_v * elem;
  return fk::prefill_entry("fk_paged_prefill", true, out, out_row_stride, q, q_row_stride,
                           k_cache, k_row, v_cache, v_row, kv_dtype, k_scale, v_scale,
                           block_tables, bt_row_stride, cu_seqlens_q, cu_seqlens_k, batch,
                           max_seqlen_q, max_seqlen_k, num_heads, num_kv_heads, head_size,
                           head_size_v, block_size, num_blocks, scale, causal, window_left,
                           sinks, nullptr, 0, 0, nullptr, 0, stream);
}

extern "C" int fk_varlen_prefill(void* out, int64_t out_row_stride, const void* q,
                                 int64_t q_row_stride, const void* key, int64_t key_row_stride,
                                 const void* value, int64_t value_row_stride,
                                 const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                 int64_t batch, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                 int num_heads, int num_kv_heads, int head_size, int head_size_v,
                                 float scale, int causal, int window_left, const float* sinks,
                                 float* lse, int64_t lse_row_stride, void* stream) {
  return fk::prefill_entry("fk_varlen_prefill", false, out, out_row_stride, q, q_row_stride, key,
                           key_row_stride * 2, value, value_row_stride * 2, FK_DTYPE_BF16,
                           nullptr, nullptr, nullptr, 0, cu_seqlens_q, cu_seqlens_k, batch,
                           max_seqlen_q, max_seqlen_k, num_heads, num_kv_heads, head_size,
                           head_size_v, 16, 0, scale, causal, window_left, sinks, lse,
                           lse_row_stride, 0, nullptr, 0, stream);
}

extern "C" int fk_prefill_split_plan(int paged, int kv_dtype, int64_t batch, int64_t total_q,
                                     int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads,
                                     int num_kv_heads, int head_size, int head_size_v,
                                     int causal, int64_t* workspace_bytes) {
  const char* name = "fk_prefill_split_plan";
  FK_REQUIRE(workspace_bytes != nullptr, "%s: null workspace_bytes", name);
  *workspace_bytes = 0;
  FK_REQUIRE(batch >= 0 && total_q >= 0 && max_seqlen_q >= 0 && max_seqlen_k >= 0,
             "%s: negative size", name);
  FK_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             "%s: num_heads %d must be a positive multiple of num_kv_heads %d", name, num_heads,
             num_kv_heads);
  if (batch == 0 || max_seqlen_q == 0 || total_q == 0) return FK_OK;
  const fk::PrefillShape sh =
      fk::prefill_shape(paged != 0, kv_dtype == FK_DTYPE_FP8_E4M3FN, batch, total_q, max_seqlen_q,
                        max_seqlen_k, num_heads, num_kv_heads, head_size, head_size_v, causal);
  *workspace_bytes = fk::prefill_ws_bytes(sh, total_q, num_heads, head_size_v);
  return FK_OK;
}

extern "C" int fk_prefill_shape(int paged, int kv_dtype, int64_t batch, int64_t total_q,
                                int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads,
                                int num_kv_heads, int head_size, int head_size_v, int causal,
                                int window_left, int with_workspace, int* wg_tokens,
                                int* key_split, int* parts, int* longest_first) {
  const char* name = "fk_prefill_shape";
  FK_REQUIRE(wg_tokens && key_split && parts && longest_first, "%s: null output pointer", name);
  FK_REQUIRE(batch > 0 && total_q >= 0 && max_seqlen_q > 0 && max_seqlen_k >= 0,
             "%s: batch and max_seqlen_q must be positive", name);
  FK_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             "%s: num_heads %d must be a positive multiple of num_kv_heads %d", name, num_heads,
             num_kv_heads);
  const bool fp8 = kv_dtype == FK_DTYPE_FP8_E4M3FN;
  fk::PrefillShape sh =
      fk::prefill_shape(paged != 0, fp8, batch, with_workspace ? total_q : 0, max_seqlen_q,
                        max_seqlen_k, num_heads, num_kv_heads, head_size, head_size_v, causal);
  if (!with_workspace) {
    sh.xs = 1;
    sh.ks = sh.ks_plain;
    total_q = 0;
  }
  int64_t items = batch * sh.qblocks;
  if (total_q > 0) items = std::min(items, total_q / sh.wg_tokens + batch);
  *wg_tokens = static_cast<int>(sh.wg_tokens);
  *key_split = sh.ks;
  *parts = sh.xs;
  *longest_first =
      fk::prefill_order(sh, sh.xs, batch, total_q, max_seqlen_q, max_seqlen_k, num_kv_heads,
                        head_size, head_size_v, causal, window_left, fp8 ? 1 : 2, items);
  return FK_OK;
}

extern "C" int fk_paged_prefill_ws(void* out, int64_t out_row_stride, const void* q,
                                   int64_t q_row_stride, const void* k_cache, const void* v_cache,
                                   int kv_dtype, const float* k_scale, const float* v_scale,
                                   const int32_t* block_tables, int64_t bt_row_stride,
                                   const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                   int64_t batch, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                   int num_heads, int num_kv_heads, int head_size,
                                   int head_size_v, int block_size, int64_t num_blocks,
                                   float scale, int causal, int window_left, const float* sinks,
                                   int64_t total_q, void* workspace, int64_t workspace_bytes,
                                   void* stream) {
  const int64_t elem = kv_dtype == FK_DTYPE_FP8_E4M3FN ? 1 : 2;
  const int64_t k_row = static_cast<int64_t>(num_kv_heads) * head_size * elem;
  const int64_t v_row = static_cast<int64_t>(num_kv_heads) * head_size_v * elem;
  return fk::prefill_entry("fk_paged_prefill_ws", true, out, out_row_stride, q, q_row_stride,
                           k_cache, k_row, v_cache, v_row, kv_dtype, k_scale, v_scale,
                           block_tables, bt_row_stride, cu_seqlens_q, cu_seqlens_k, batch,
                           max_seqlen_q, max_seqlen_k, num_heads, num_kv_heads, head_size,
                           head_size_v, block_size, num_blocks, scale, causal, window_left,
                           sinks, nullptr, 0, total_q, workspace, workspace_bytes, stream);
}

extern "C" int fk_varlen_prefill_ws(void* out, int64_t out_row_stride, const void* q,
                                    int64_t q_row_stride, const void* key, int64_t key_row_stride,
                                    const void* value, int64_t value_row_stride,
                                    const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                    int64_t batch, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                    int num_heads, int num_kv_heads, int head_size,
                                    int head_size_v, float scale, int causal, int window_left,
                                    const float* sinks, float* lse, int64_t lse_row_stride,
                                    int64_t total_q, void* workspace, int64_t workspace_bytes,
                                    void* stream) {
  return fk::prefill_entry("fk_varlen_prefill_ws", false, out, out_row_stride, q, q_row_stride,
                           key, key_row_stride * 2, value, value_row_stride * 2, FK_DTYPE_BF16,
                           nullptr, nullptr, nullptr, 0, cu_seqlens_q, cu_seqlens_k, batch,
                           max_seqlen_q, max_seqlen_k, num_heads, num_kv_heads, head_size,
                           head_size_v, 16, 0, scale, causal, window_left, sinks, lse,
                           lse_row_stride, total_q, workspace, workspace_bytes, stream);
}
