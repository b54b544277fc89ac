// Chunked prefill attention over the paged pool (gfx950, bf16/fp16 MFMA).
//
// Semantics: for sequence b with kv_lens[b] keys resident in pages (the
// prefix plus this chunk) and C_b = cu_q[b+1] - cu_q[b] chunk queries, query i
// sits at absolute position P_b + i, P_b = kv_lens[b] - C_b, and attends to
// keys 0 .. P_b + i (causal, aligned to the bottom right) - what the
// reference's chunked prefill computes through HF attention over the past KV
// (core/engine.py:1826-1854, core/chunked_prefill.py:9-33) and what
// flash_attn_varlen_func(causal=True) computes for a single chunk
// (core/varlen.py:19-42). The reference has no paged prefill; here the keys
// are read from 16-token pages through the block table, and
// ukv_kv_write_varlen first writes the chunk's own K/V into its pages.
//
// Kernel: one workgroup of W waves (W = 8, two per SIMD) takes QW = W * CB *
// (16 / n_rep) consecutive queries of one KV group. Within a wave, an MFMA
// column is a (query, q head) pair: 16 / n_rep queries times the n_rep q heads
// of the group, so one K/V read serves the whole GQA group; a wave holds CB
// 16-column blocks, three or two.
//   * block plan: the chunk of each (sequence, group) is cut from its end down
//     into three-column blocks and then two-column ones (three are cheaper per
//     query, two fill the last round of the launch: the host picks the mix that
//     its model of the dispatch finishes first); each XCD (dispatch is
//     round-robin over the 8 XCDs) runs a contiguous range of (sequence, group)
//     pairs, three-column blocks first: the query blocks of one pair share that
//     XCD's L2 while they stream the same pages;
//   * key tiles of 32 keys (two pages) pass through registers into a 4-slot
//     LDS ring (rows padded to 288 B), written two tiles ahead of their use,
//     with a barrier after every second tile; the loads of tiles t+3 and t+4
//     are in flight while tile t is computed;
//   * S^T = K Q^T on v_mfma_f32_16x16x32 in the input type (A = 16 keys x 32
//     dims from LDS, B = the wave's q columns in registers); lane l ends with
//     keys 4*(l/16) + r of column l % 16;
//   * online softmax per column in log2 units; masks only on tiles that touch
//     the sequence end, an invalid page or the causal diagonal; the running max
//     moves only when a weight reaches 2^8 (wave vote on the packed weights);
//   * P.V on v_mfma_f32_16x16x32_f16: P is rounded to fp16 (11 significant
//     bits, 4x finer than a bf16 P) and, for bf16 pools, the loader converts
//     the V tile to fp16, which is exact for |v| < 65520; a workgroup whose
//     keys hold a larger or non-finite bf16 V recomputes its columns on an
//     fp32 path. The S^T layout is already P's A-operand layout; V's B
//     operands come from ds_read_b64_tr_b16 transpose reads; the softmax
//     denominators come from one more MFMA against a ones operand, so they sum
//     exactly the rounded P;
//   * shapes whose n_rep does not divide 16, and 64-dim heads, run FINE instances: columns are
//     (query, head) pairs laid end to end, so every column of the matrix cores is used, V keeps its
//     type and P goes in as two 16-bit parts (fp32-grade weights, as the scalar kernel they ran on
//     before had): 28 q heads on 4 KV heads, 4 x 512 queries over 5-8K keys in 0.314 ms against
//     72.7 ms; twelve 64-dim prompts of 16-700 tokens in 0.055 ms against 6.4 ms (0.10 ms with one
//     workgroup per CU, three column blocks, 64-key tiles and the pairs' blocks in turn);
//   * key parts: a launch of few query blocks leaves CUs idle however long its prefix. Its keys are
//     then cut into equal parts, each (block, part) a workgroup, and a merge kernel adds the parts
//     up: one 389-query chunk behind 32256 keys (40 blocks) in 0.22 ms against 0.86 ms;
//   * SnapKV row statistics: the blocks holding each sequence's last obs queries
//     also write those rows' running max and denominator; obs_rows_finish_kernel
//     then sums the sink and window keys' weights again from the same scores and
//     takes them off, leaving the middle keys' sum.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "prefill_plan.h"
#include "ukv_common.h"

namespace ukv {

struct PrefillArgs {
  const uint16_t* q;  // [total_q][Hq][D]
  uint16_t* out;      // [total_q][Hq][D] contiguous
  const uint16_t* k;  // one pool layer [N][16][Hkv][D]
  const uint16_t* v;
  int64_t q_st, q_sh;
  int64_t k_sp, k_st, k_sh;
  int64_t v_sp, v_st, v_sh;
  const int32_t* bt;
  const int32_t* cu_q;     // [B+1]
  const int32_t* kv_lens;  // [B] keys per sequence, the chunk included
  int B, Hq, n_rep, n_groups, D, max_blocks, num_pages;
  // Query blocks of every (sequence, KV group), from the end of its chunk down: n3 blocks of three
  // column blocks per wave, then n2 of two. Blocks that reach below the chunk's first query are
  // partial or empty (chunks shorter than the longest). The three-column blocks of every pair are
  // dispatched in a first pass, the two-column ones in a second.
  int n3, n2;
  // Key split (n_parts > 1): the key tiles of a sequence are cut into part_count() <= n_parts equal
  // parts of about part_tiles tiles, each (query block, part) is a work item of its own, and
  // prefill_combine_kernel merges the parts' (m, l, O) from part_o / part_ml, rows
  // [part][query row][q head] of D floats / one float2. A sequence whose keys fill one part takes
  // whole3 + whole2 blocks, the mix of a launch without parts, and writes its rows itself.
  int n_parts, part_tiles, whole3, whole2;
  // Work items in block order (block j of every pair, then block j + 1) instead of pair after pair: for
  // launches whose blocks see very different key counts, longest first.
  int by_block;
  int total_q;
  float* part_o;
  float2* part_ml;
  // The longest chunk the caller declared: the block plan covers that many queries. A chunk
  // longer than it gets NaN in every row of its output (its K/V were not all written either).
  int max_chunk;
  float scale, scale_log2;
  // SnapKV observation statistics (obs > 0): for each of a sequence's last obs queries and q head
  // h, the log2-sum-exp2 of its scaled scores over the middle keys [sink, L - obs) and the zero
  // rows that pad them to a multiple of 16 keys: obs_stats[b * stats_seq_stride + h * obs + i].x
  // (.y = 0, or 1 where the sum lost precision), the row statistics the SnapKV scoring pass takes.
  // The prefill kernel leaves each row's (max, denominator) there and obs_rows_finish_kernel
  // takes the sink and window keys' share off.
  float2* obs_stats;
  int64_t stats_seq_stride;
  int sink, obs;
};

// paged_prefill_kernel's argument (its only one, at the start of the kernel's argument segment), read again
// behind a barrier to the compiler: the fields that only a block's rows need at the end would otherwise be loaded
// at the start and held through the tiles, where the scalar registers they spill cost a v_readlane each (16 a tile in
// the parts' instance for three column blocks, 150 instructions of it against 128).
__device__ __forceinline__ const PrefillArgs& args_again() {
  auto* p = (const __attribute__((address_space(4))) PrefillArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const PrefillArgs*)p;
}

__device__ __forceinline__ int kv_len_of(const PrefillArgs& a, int b) {
  const int cap = a.max_blocks * 16;
  const int L = a.kv_lens[b];
  return L < 0 ? 0 : (L > cap ? cap : L);
}

// Two bf16 values -> two fp16 values (RNE; exact when 2^-14 <= |x| < 65520). A bf16 value
// that fp16 cannot hold (|x| >= 65536, the next bf16 above 65280; inf; NaN) becomes an fp16
// inf or NaN.
__device__ __forceinline__ uint32_t bf16x2_to_f16x2(uint32_t w) {
  return pack_f16(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
}

// Tile loads whose completion the kernel waits for itself. Two register sets
// are in flight while a tile is computed; the compiler's own wait placement
// cannot see which set is older across the unrolled loop and waits for both,
// so the loads are issued here and vm_wait<N>() waits until at most N vector
// memory operations are outstanding. The "+v" operands make every use of the
// loaded registers follow the wait.
__device__ __forceinline__ void gload16(u32x4& r, const void* p) {
  asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(r) : "v"(p));
}
template <int N> __device__ __forceinline__ void vm_wait(u32x4& x) {
  asm volatile("s_waitcnt vmcnt(%1)" : "+v"(x) : "n"(N));
}
template <int N> __device__ __forceinline__ void vm_wait(u32x4& x, u32x4& y) {
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(x), "+v"(y) : "n"(N));
}

// 8-byte LDS transpose read (ds_read_b64_tr_b16).
__device__ __forceinline__ u32x2 ds_read_tr16(const uint16_t* p) {
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  return __builtin_bit_cast(u32x2, v);
}

#ifndef UKV_PREFILL_WAVES
#define UKV_PREFILL_WAVES 8
#endif

// LDS row pitches in 16-bit elements: K and V rows sit 288 B apart, the pitch
// at which SQ_LDS_BANK_CONFLICT reads 0 for the 16-row x 16-byte K reads, the
// 4-row x 32-byte V transpose reads and the 16-byte row stores (272 B leaves
// the K reads conflicting).
#ifndef UKV_PREFILL_KPAD
#define UKV_PREFILL_KPAD 144
#endif
#ifndef UKV_PREFILL_VPAD
#define UKV_PREFILL_VPAD 144
#endif
constexpr int kRowPad = UKV_PREFILL_KPAD;
constexpr int kVRowPad = UKV_PREFILL_VPAD;
constexpr int kStages = 4;  // K/V ring slots: tiles are written two ahead, a barrier every second tile

// Parts the n_tiles key tiles of a sequence are cut into; part s holds tiles
// [s * n_tiles / n, (s + 1) * n_tiles / n).
__device__ __forceinline__ int part_count(const PrefillArgs& a, int n_tiles) {
  return max(1, min(a.n_parts, (n_tiles + a.part_tiles - 1) / a.part_tiles));
}

// Whether any sequence is in more parts than one: the plan knows the table's width alone. (Wave-uniform. The first
// rows are loaded beside the lengths for the reads that follow: first rows are not negative.)
__device__ __forceinline__ bool any_in_parts(const PrefillArgs& a) {
  const int most = a.part_tiles * kTileKeys;  // keys of a sequence in one part
  if (a.B == 1) return kv_len_of(a, 0) > most;  // (scalar loads)
  bool any = false;
  for (int b0 = 0; b0 < a.B && !any; b0 += 64) {
    const int b = min(b0 + (int)(threadIdx.x & 63), a.B - 1);
    any = __any(kv_len_of(a, b) > most || a.cu_q[b + 1] < 0);
  }
  return any;
}

// Fallback for a workgroup whose keys hold a V the matrix cores' P.V would get wrong (a bf16 V of
// magnitude >= 65520, or infinite, which fp16 cannot carry; FINE: an infinite one, which a zero low
// part turns into NaN, or one near the type's end): every column of the workgroup, c0 .. c0 + n_cols - 1,
// is recomputed in fp32 on the vector ALUs, one column per wave at a time, keys in page order (the
// reference's order), natural exp. Lane l owns dims l * D / 64 ... Keys [key_a, key_b) are taken; with
// part >= 0 the column's partial is left for prefill_combine_kernel, its denominator's sign bit set:
// the rows' statistics are then flagged.
template <int DT, int D>
__device__ void prefill_cols_fp32(const PrefillArgs& a, int b, int g, int q_begin, int C, int P0, int Lk, int c0,
                                  int n_cols, int wv, int nwaves, int lane, int part, int key_a, int key_b) {
  constexpr int W = D / 64;  // dims per lane
  const int32_t* btrow = a.bt + (int64_t)b * a.max_blocks;
  for (int c = c0 + wv; c < c0 + n_cols; c += nwaves) {
    if (c < 0) continue;
    const int qi = c / a.n_rep;
    const int h = g * a.n_rep + c % a.n_rep;
    if (qi >= C || h >= a.Hq) continue;
    const int L = min(key_b, max(0, min(Lk, P0 + qi + 1)));
    const uint16_t* qrow = a.q + (int64_t)(q_begin + qi) * a.q_st + (int64_t)h * a.q_sh + W * lane;
    float q[W], acc[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      q[w] = Elem<DT>::one(qrow[w]);
      acc[w] = 0.f;
    }
    float m = kNegFltMax, l = 0.f;
    for (int key = key_a; key < L; ++key) {
      const int id = btrow[key >> 4];
      if ((unsigned)id >= (unsigned)a.num_pages) continue;
      const int64_t slot = key & 15;
      const uint16_t* kr = a.k + (int64_t)id * a.k_sp + slot * a.k_st + (int64_t)g * a.k_sh + W * lane;
      const uint16_t* vr = a.v + (int64_t)id * a.v_sp + slot * a.v_st + (int64_t)g * a.v_sh + W * lane;
      float dot = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) dot += q[w] * Elem<DT>::one(kr[w]);
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) dot += __shfl_xor(dot, off);
      const float sc = dot * a.scale;
      const float mn = fmaxf(m, sc);
      const float alpha = expf(m - mn), pk = expf(sc - mn);
      l = l * alpha + pk;
#pragma unroll
      for (int w = 0; w < W; ++w) acc[w] = acc[w] * alpha + pk * Elem<DT>::one(vr[w]);
      m = mn;
    }
    if (part >= 0) {
      const int64_t row = ((int64_t)part * a.total_q + q_begin + qi) * a.Hq + h;
#pragma unroll
      for (int w = 0; w < W; ++w) a.part_o[row * D + W * lane + w] = acc[w];
      if (lane == 0) a.part_ml[row] = make_float2(m * kLog2e, -l);
      continue;
    }
    uint16_t* orow = a.out + ((int64_t)(q_begin + qi) * a.Hq + h) * D + W * lane;
#pragma unroll
    for (int w = 0; w < W; ++w) orow[w] = Elem<DT>::from_float(acc[w] / l);
  }
}

// Flags (y = 1) the observation rows among queries lo .. hi - 1 of sequence b's chunk (C
// queries), q heads of KV group g, for the scoring pass to recompute from the keys.
template <int WAVES>
__device__ void flag_obs_rows(const PrefillArgs& a, int b, int g, int C, int lo, int hi) {
  lo = max(lo, C - a.obs);
  const int n = max(0, min(hi, C) - lo) * a.n_rep;
  for (int t = threadIdx.x; t < n; t += 64 * WAVES) {
    const int qi = lo + t / a.n_rep, h = g * a.n_rep + t % a.n_rep;
    if (qi >= 0 && h < a.Hq)
      a.obs_stats[(int64_t)b * a.stats_seq_stride + (int64_t)h * a.obs + (qi - (C - a.obs))] = make_float2(NAN, 1.f);
  }
}

// LDS of one workgroup: kStages ring slots of K and V (fp16, or the pool's type) tiles. The 144-byte
// pitch at D = 64 spreads eight rows' 16-byte reads over the banks and lets two workgroups share a CU.
template <int D> struct PrefillLds {
  static constexpr int kPitch = D == 64 ? 72 : kRowPad, kVPitch = D == 64 ? 72 : kVRowPad;
  __attribute__((aligned(16))) uint16_t k_s[kStages][kTileKeys][kPitch];
  __attribute__((aligned(16))) uint16_t v_s[kStages][kTileKeys][kVPitch];
};

// Softmax weights for P.V on 16-bit MFMAs with fp32-grade precision: p ~= hi + lo, both in V's
// type (relative error below 2^-16 in bf16, 2^-21 in fp16). fp16 weights are lifted by 2^7 so
// that small ones stay normal; the tile's vote keeps them below 2^8 (2^15 lifted).
template <int DT> struct PrefillSplit;
template <> struct PrefillSplit<UKV_DTYPE_BF16> {
  static constexpr float kLift = 0.f;
  static constexpr unsigned short kMax = 0x437F;  // bf16 bit pattern just below 2^8
  static constexpr uint32_t kOnes = 0x3F803F80u;
  static __device__ __forceinline__ void split(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    hi = pack_bf16(x0, x1);
    lo = pack_bf16(x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xffff0000u));
  }
};
template <> struct PrefillSplit<UKV_DTYPE_F16> {
  static constexpr float kLift = 7.f;
  static constexpr unsigned short kMax = 0x77FF;  // fp16 bit pattern just below 2^15
  static constexpr uint32_t kOnes = 0x3C003C00u;
  static __device__ __forceinline__ void split(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
    // lo = fp16(x - hi): one mixed-precision FMA per weight (a subtraction of the converted halves
    // and a pack are five instructions; the compiler does not form these two)
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(lo) : "v"(hi), "v"(x0));
    asm("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(lo) : "v"(hi), "v"(x1));
  }
};

// The columns c0 .. c0 + WAVES * CB * 16 - 1 of sequence b, KV group g, with CB 16-column blocks per
// wave. Column c is the pair (query c / n_rep, q head g * n_rep + c % n_rep); c0 may be negative.
//   FINE   the weights keep fp32-grade precision (PrefillSplit) and V its own type: shapes whose
//          n_rep does not divide 16 or whose D is 64. Otherwise n_rep divides 16 (a query's heads
//          lie in one column block) and P and V are fp16.
//   PARTS  part `part` of the sequence's keys (of np = part_count()), left for
//          prefill_combine_kernel; a sequence in one part is written like an undivided one (every row
//          through the partials cost 4 x 512-token prompts in a 2048-page table 53 us against 29). The
//          running max moves to whole powers of two, so that the parts' rounded weights are the ones an
//          undivided pass would have summed.
// With statistics (obs > 0) it also writes, for each of the sequence's last obs queries in the
// block and each q head h, the pair (m, l) of the column's running max m (log2 units) and its
// softmax denominator l (the sum of the rounded weights 2^(s * scale * log2e - m) over every key the
// query sees; FINE: with its lift, taken off m) into obs_stats[b * stats_seq_stride + h * obs + i],
// for obs_rows_finish_kernel.
template <int DT, int D, int WAVES, int CB, bool FINE, bool PARTS>
__device__ __forceinline__ void prefill_tile(const PrefillArgs& a, const int b, const int g, const int c0,
                                             const int part, const int np, PrefillLds<D>& lds) {
  constexpr int STEPS = D / 32;
  constexpr int NE = D / 16;  // output tiles of 16 dims
  constexpr int NT = 64 * WAVES;
  constexpr int TK = kTileKeys;  // keys per tile
  constexpr int PPT = TK / 16;   // pages per tile
  constexpr int CH = D / 8;      // 16-byte chunks per key row
  // A thread loads one 16-byte chunk of K and one of V per tile or, HALF (D = 64), one of either: the
  // lower half of the waves takes K.
  constexpr bool HALF = 2 * TK * CH == NT;
  constexpr int PVT = FINE ? DT : (int)UKV_DTYPE_F16;  // type of the P.V operands
  constexpr float kTau = 8.f;
  constexpr float kLift = FINE ? PrefillSplit<DT>::kLift : 0.f;
  constexpr bool kConvert = DT == UKV_DTYPE_BF16 && !FINE;  // the loader converts V to fp16
  static_assert(HALF || TK * CH == NT, "loader mapping");
  auto& k_s = lds.k_s;
  auto& v_s = lds.v_s;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int i16 = lane & 15;
  const int kg = lane >> 4;

  const int qpb = 16 / a.n_rep;  // queries per column block (not FINE)
  const int q_begin = a.cu_q[b];
  const int C = a.cu_q[b + 1] - q_begin;
  // The block's queries [q0, q1) and the columns' division by n_rep: columns c0 + x of FINE blocks
  // start at remainder rem of query q0, so query and head follow from (rem + x) / n_rep, a
  // multiplication exact below 2^16 / n_rep.
  const int q0 = FINE ? (c0 >= 0 ? c0 / a.n_rep : -((a.n_rep - 1 - c0) / a.n_rep)) : c0 / a.n_rep;
  const int rem = FINE ? c0 - q0 * a.n_rep : 0;
  const uint32_t inv_rep = FINE ? (65535u + a.n_rep) / a.n_rep : 0u;
  const int q1 = FINE ? q0 + (rem + WAVES * CB * 16 + a.n_rep - 1) / a.n_rep : q0 + WAVES * CB * qpb;
  if (q0 >= C || q1 <= 0) return;  // whole workgroup
  int Lk = kv_len_of(a, b);
  int P0 = Lk - C;  // keys before the chunk
  int kend = max(0, min(Lk, P0 + min(C, q1)));
  int key_a = 0;  // PARTS: first key of this part; Lk, P0 and kend count from it below
  bool in_parts = false;  // the sequence's keys are in more parts than one (uniform)
  if constexpr (PARTS) {
    const int nt = (Lk + TK - 1) / TK;
    if (part >= np) return;  // whole workgroup
    in_parts = np > 1;
    key_a = (int)((uint32_t)(part * nt) / (uint32_t)np) * TK;  // (at most kMaxParts * 2^26: 32 bits)
    if (in_parts && key_a >= kend) return;  // no row of the block sees this part (prefill_combine_kernel skips it)
    kend = min(kend, (int)((uint32_t)((part + 1) * nt) / (uint32_t)np) * TK) - key_a;
    Lk -= key_a;
    P0 -= key_a;
  }
  const int n_tiles = (kend + TK - 1) / TK;
  const int n_pg = (kend + 15) >> 4;

  // This wave's queries [wq0, wq1) and this lane's columns.
  const int wx0 = rem + wv * CB * 16;  // the wave's first column, counted from query q0's first
  const int wq0 = FINE ? q0 + (int)(wx0 * inv_rep >> 16) : q0 + wv * CB * qpb;
  const int wq1 = FINE ? q0 + (int)((wx0 + CB * 16 - 1) * inv_rep >> 16) + 1 : wq0 + CB * qpb;
  const bool wave_live = wq0 < C && wq1 > 0;
  const int wpos_min = P0 + wq0;
  // Column x of the wave (x < CB * 16): its query and q head.
  auto col_query = [&](int x) -> int { return FINE ? q0 + (int)((wx0 + x) * inv_rep >> 16) : wq0 + x / a.n_rep; };
  auto col_head = [&](int x) -> int {
    return FINE ? g * a.n_rep + (wx0 + x) - (int)((wx0 + x) * inv_rep >> 16) * a.n_rep : g * a.n_rep + x % a.n_rep;
  };
  const int head = g * a.n_rep + i16 % a.n_rep;  // (not FINE: the same in every column block)
  // the query of this lane's column in column block cb (unused if outside 0 .. C - 1)
  const int qi0 = wq0 + i16 / a.n_rep;
  int qic[FINE ? CB : 1];
  if constexpr (FINE)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) qic[cb] = col_head(cb * 16 + i16) < a.Hq ? col_query(cb * 16 + i16) : -1;
  auto lane_query = [&](int cb) -> int { return FINE ? qic[FINE ? cb : 0] : qi0 + cb * qpb; };
  u32x4 qv[CB][STEPS];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int qi = lane_query(cb);
    const int hh = FINE ? col_head(cb * 16 + i16) : head;
    const bool live = qi >= 0 && qi < C && hh < a.Hq;
    const uint16_t* qp = a.q + (int64_t)(q_begin + (live ? qi : 0)) * a.q_st + (int64_t)(live ? hh : 0) * a.q_sh +
                         8 * kg;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) qv[cb][s] = live ? ld16(qp + 32 * s) : u32x4{0u, 0u, 0u, 0u};
  }

  float m_ref[CB];  // running max of the column (log2 units)
  f32x4 o[CB][NE];
  f32x4 lacc[CB];  // softmax denominators of columns 4*kg + r
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    m_ref[cb] = kNegFltMax;
    lacc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < NE; ++e) o[cb][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // ---- tile loader: thread idx takes 16-byte chunk idx % CH of key row idx / CH.
  // Tile u is loaded into register set u & 1 four tiles ahead, written into
  // ring slot u % 4 two tiles ahead (zeroing rows past the sequence or on an
  // invalid page and converting a bf16 V to fp16), and computed at tile u.
  // The block table is read through the constant address space: the kernel
  // never writes it, and this keeps the wave-uniform page-id loads on the
  // scalar unit (SMEM), apart from the vector-memory count the tile loads use.
  typedef const __attribute__((address_space(4))) int32_t cint32;
  cint32* btrow = (cint32*)(a.bt + (int64_t)b * a.max_blocks + (key_a >> 4));
  auto page_id = [&](int pg) -> int { return pg < n_pg ? btrow[pg] : -1; };
  auto page_ok = [&](int id) -> bool { return (unsigned)id < (unsigned)a.num_pages; };
  // Within a page, this thread's chunk sits at a fixed offset; the page base is wave-uniform.
  const int idx = HALF ? tid & (NT / 2 - 1) : tid;
  const bool half_v = HALF && wv >= WAVES / 2;  // (wave-uniform) this wave loads V
  const int lds_row = idx / CH, lds_ch = idx % CH;
  const int tok = lds_row & 15;
  const uint32_t koff = (uint32_t)(tok * (half_v ? a.v_st : a.k_st) + g * (half_v ? a.v_sh : a.k_sh) + 8 * lds_ch);
  const uint32_t voff = (uint32_t)(tok * a.v_st + g * a.v_sh + 8 * lds_ch);
  const uint16_t* kbase = half_v ? a.v : a.k;
  const uint32_t k_sp = (uint32_t)(half_v ? a.v_sp : a.k_sp);
  u32x4 rk0, rv0, rk1, rv1;
  // the page of this thread's chunk among a tile's two (rows 0-15 and 16-31); wave-uniform
  auto chunk_page = [&](const int (&ids)[PPT]) -> int {
    return __builtin_amdgcn_readfirstlane(idx / (16 * CH)) ? ids[1] : ids[0];
  };
  auto issue = [&](const int (&ids)[PPT], u32x4& rk, u32x4& rv) {
    const int id = chunk_page(ids);
    // page strides fit 32 bits (checked on the host): a 32 x 32 -> 64-bit scalar product
    const uint32_t pg = page_ok(id) ? (uint32_t)id : 0u;
    gload16(rk, kbase + (uint64_t)pg * k_sp + koff);
    if constexpr (!HALF) gload16(rv, a.v + (uint64_t)pg * (uint32_t)a.v_sp + voff);
  };
  // The largest and the smallest fp16 V value this thread stored, over every tile (three-input
  // packed maximum / minimum, which carry a NaN through): checked once after the loop for an
  // inf or NaN, i.e. a bf16 value fp16 cannot hold.
  typedef _Float16 hv2 __attribute__((ext_vector_type(2)));
  hv2 vmax = {0, 0}, vmin = {0, 0};
  auto store = [&](int u, int slot, const int (&ids)[PPT], u32x4& rk, u32x4& rv) {
    const bool full = page_ok(ids[0]) && page_ok(ids[1]) && TK * (u + 1) <= Lk;
    // rows past the sequence or on an invalid page hold junk (wave-uniform: the tile has some)
    auto clear_junk = [&](u32x4& v) {
      if (!full) {
        const bool ok = page_ok(chunk_page(ids)) && TK * u + lds_row < Lk;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = ok ? v[c] : 0u;
      }
    };
    if constexpr (HALF) {
      vm_wait<1>(rk);  // the other register set's load was issued after this one's
      clear_junk(rk);
      uint16_t* dst = half_v ? &v_s[slot][lds_row][8 * lds_ch] : &k_s[slot][lds_row][8 * lds_ch];
      *reinterpret_cast<u32x4*>(dst) = rk;
      return;
    }
    vm_wait<2>(rk, rv);  // the other register set's two loads were issued after this set's
    // (converted before the junk rows are zeroed: the conversion writes new registers, which
    // the zeroing then selects in place, with no copy of the loaded ones)
    u32x4 v;
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = kConvert ? bf16x2_to_f16x2(rv[c]) : rv[c];
    clear_junk(v);
    if constexpr (kConvert) {
      const uint32_t w0 = v[0], w1 = v[1], w2 = v[2], w3 = v[3];
      const hv2 c0 = __builtin_bit_cast(hv2, w0), c1 = __builtin_bit_cast(hv2, w1);
      const hv2 c2 = __builtin_bit_cast(hv2, w2), c3 = __builtin_bit_cast(hv2, w3);
      vmax = __builtin_elementwise_maximum(__builtin_elementwise_maximum(vmax, c0), c1);
      vmax = __builtin_elementwise_maximum(__builtin_elementwise_maximum(vmax, c2), c3);
      vmin = __builtin_elementwise_minimum(__builtin_elementwise_minimum(vmin, c0), c1);
      vmin = __builtin_elementwise_minimum(__builtin_elementwise_minimum(vmin, c2), c3);
    }
    *reinterpret_cast<u32x4*>(&k_s[slot][lds_row][8 * lds_ch]) = rk;
    *reinterpret_cast<u32x4*>(&v_s[slot][lds_row][8 * lds_ch]) = v;
  };

  // Page ids of tiles t .. t+3 (t_id[j] = tile t + j) and of tile t+4.
  int t_id[4][PPT], id_n[PPT];
  auto tile_ids = [&](int t, int (&ids)[PPT]) {
#pragma unroll
    for (int j = 0; j < PPT; ++j) ids[j] = page_id(PPT * t + j);
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) tile_ids(j, t_id[j]);
  // Prologue: tiles 0 and 1 into the ring, tiles 2 and 3 in flight. Loads are issued
  // unconditionally (tiles past the end read page 0 and are never used) so
  // that every wait is on loads of a fixed age: vmcnt(2) on the older set.
  issue(t_id[0], rk0, rv0);
  issue(t_id[1], rk1, rv1);
  store(0, 0, t_id[0], rk0, rv0);
  issue(t_id[2], rk0, rv0);
  store(1, 1, t_id[1], rk1, rv1);
  issue(t_id[3], rk1, rv1);
  tile_ids(4, id_n);
  // Retire every load issued so far (q columns, tiles 2 and 3) once, so that
  // no wait for them is left inside the loop.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();

  // Tiles t < n_full end below the sequence end and below every column's diagonal (key
  // 32t + 31 <= min(Lk - 1, wpos_min)).
  const int n_full = max(0, min(Lk, wpos_min + 1)) / kTileKeys;
  const float sl2 = a.scale_log2;

  auto compute = [&](int t, int slot) {
    const int key0 = t * kTileKeys;
    const bool pg0 = page_ok(t_id[0][0]), pg1 = page_ok(t_id[0][1]);
    const bool full = pg0 && pg1 && t < n_full;
    // S^T[key][column] for the tile's two 16-key blocks and every column block, masked. (As one
    // inlined function the register allocator keeps the three-column loop within 256 VGPRs with
    // no scratch under the iterative-ILP schedule this file is built with; written out in line,
    // that schedule needed 20 bytes per lane of scratch.)
    auto scores = [&](f32x4 (&sacc)[2][CB]) __attribute__((always_inline)) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) sacc[kb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
          const u32x4 ka = *reinterpret_cast<const u32x4*>(&k_s[slot][kb * 16 + i16][32 * s + 8 * kg]);
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) sacc[kb][cb] = mfma16x16x32<DT>(ka, qv[cb][s], sacc[kb][cb]);
        }
      }
      if (!full) {
        // key kb*16 + 4kg + r is visible to a column iff it is below lim[kb]
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const int qi = lane_query(cb);
          const bool live = qi >= 0 && qi < C && (FINE || head < a.Hq);
          const int vis = live ? min(Lk, P0 + qi + 1) - key0 - 4 * kg : -1;  // an unused column sees no key
          const int lim0 = pg0 ? vis : 0, lim1 = pg1 ? vis - 16 : 0;
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) sacc[kb][cb][r] = r < (kb ? lim1 : lim0) ? sacc[kb][cb][r] : -INFINITY;
        }
      }
    };
    f32x4 sacc[2][CB];
    scores(sacc);
    // Softmax: p = 2^(s*scale*log2e - m) as fp16 against the running max m
    // (log2 units) of its column. m moves only when some p of the tile reaches
    // 2^8: the packed fp16 P is checked (non-negative fp16 bit patterns order
    // like their values, and inf and NaN lie above), and a column block whose
    // max moved is rescaled and its P recomputed.
    u32x4 pa[CB], pl[FINE ? CB : 1];  // pl: FINE's low parts
    auto exp_pack = [&](int cb) {
      float p[2][4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p[kb][r] = fast_exp2(__builtin_fmaf(sacc[kb][cb][r], sl2, kLift != 0.f ? kLift - m_ref[cb] : -m_ref[cb]));
      if constexpr (FINE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t hi, lo;
          PrefillSplit<DT>::split(p[i / 2][2 * (i & 1)], p[i / 2][2 * (i & 1) + 1], hi, lo);
          pa[cb][i] = hi;
          pl[cb][i] = lo;
        }
      } else {
        pa[cb] = u32x4{pack_f16(p[0][0], p[0][1]), pack_f16(p[0][2], p[0][3]), pack_f16(p[1][0], p[1][1]),
                       pack_f16(p[1][2], p[1][3])};
      }
    };
    // Moves column block cb's max to the tile's where that lies more than kTau above it,
    // rescaling what was summed under the old one; returns whether it moved.
    auto settle = [&](int cb) -> bool {
      float mloc = sacc[0][cb][0];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, sacc[kb][cb][r]);
      float mcol = fmaxf(mloc, __shfl_xor(mloc, 16));
      mcol = fmaxf(mcol, __shfl_xor(mcol, 32));
      if (!__any(mcol * sl2 > m_ref[cb] + kTau)) return false;
      const float m_new = fmaxf(m_ref[cb], PARTS ? __builtin_ceilf(mcol * sl2) : mcol * sl2);
      const float alpha = fast_exp2(m_ref[cb] - m_new);
      m_ref[cb] = m_new;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ar = __shfl(alpha, 4 * kg + r);
        lacc[cb][r] *= ar;
#pragma unroll
        for (int e = 0; e < NE; ++e) o[cb][e][r] *= ar;
      }
      return true;
    };
    // The weights and the vote run at raised wave priority: when the SIMD's other wave is
    // issuing its MFMAs, this wave's softmax VALU work goes first (4-5 % faster at config 4
    // than without; raising it from the mask check on, to priority 3, or for the loader's
    // stores as well measured slower).
    __builtin_amdgcn_s_setprio(1);
    {  // the tile's weights, then the vote on them
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) exp_pack(cb);
      bool moved;
      if constexpr (FINE) {
        // (non-negative 16-bit float patterns order like their values; inf and NaN lie above)
        u16x2 mx = {0, 0};
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t w = pa[cb][i];
            mx = __builtin_elementwise_max(mx, as_u16x2(w));
          }
        constexpr unsigned short kMax = PrefillSplit<DT>::kMax;
        moved = __any(__builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(mx, u16x2{kMax, kMax})) != 0u);
      } else {
        // The max of the packed weights with three-input fp16 maxima (v_pk_maximum3_f16): a NaN
        // weight makes the maximum NaN, whose pattern, like inf's, lies above the threshold.
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        // (the element is copied out first: clang lowers __builtin_bit_cast of a vector element
        // lvalue to a load of the vector's first element, whatever the index)
        auto hv = [&](int i) {
          const uint32_t w = pa[i / 4][i % 4];
          return __builtin_bit_cast(h2, w);
        };
        h2 mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(hv(0), hv(1)), hv(2));
#pragma unroll
        for (int i = 3; i + 1 < 4 * CB; i += 2)
          mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, hv(i)), hv(i + 1));
        if constexpr ((4 * CB - 3) % 2) mx = __builtin_elementwise_maximum(mx, hv(4 * CB - 1));
        const u16x2 pmax = __builtin_bit_cast(u16x2, mx);
        moved = __any(__builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(pmax, u16x2{0x5BFF, 0x5BFF})) != 0u);
      }
      if (moved) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
          if (settle(cb)) exp_pack(cb);
      }
    }
    // FINE holds it through its twice as many P.V MFMAs: 4 x 512 queries on 28/4 heads 310 against
    // 317 us (313 without it at all).
    if constexpr (!FINE) __builtin_amdgcn_s_setprio(0);
    // P.V: the B operand of output tile e (dims 16e .. 16e + 15) holds, in lane
    // (i16, kg), dim 16e + i16 of keys 4kg..4kg+3 and 16+4kg..16+4kg+3 (the
    // key order of P's A operand). ds_read_b64_tr_b16 builds it from row-major
    // V: within each 16-lane group, lane L names 4 dims 4(L%4).. of key row
    // L/4, and lane j receives dim j of the 4 rows.
    const uint16_t* vlane = &v_s[slot][4 * kg + (i16 >> 2)][4 * (i16 & 3)];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const u32x2 lo = ds_read_tr16(vlane + 16 * e);
      const u32x2 hi = ds_read_tr16(vlane + 16 * PrefillLds<D>::kVPitch + 16 * e);
      const u32x4 bv = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) o[cb][e] = mfma16x16x32<PVT>(pa[cb], bv, o[cb][e]);
      if constexpr (FINE)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) o[cb][e] = mfma16x16x32<PVT>(pl[cb], bv, o[cb][e]);
    }
    if constexpr (FINE) __builtin_amdgcn_s_setprio(0);
    // Denominators: the same P against a ones operand.
    constexpr uint32_t kOnes = FINE ? PrefillSplit<DT>::kOnes : 0x3C003C00u;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      lacc[cb] = mfma16x16x32<PVT>(pa[cb], u32x4{kOnes, kOnes, kOnes, kOnes}, lacc[cb]);
      if constexpr (FINE) lacc[cb] = mfma16x16x32<PVT>(pl[cb], u32x4{kOnes, kOnes, kOnes, kOnes}, lacc[cb]);
    }
  };

  // Tile t: (a) tile t+2 from register set t&1 into ring slot (t+2)%4; (b) tile t+4 into that
  // set; (c) tile t on this wave's columns; (d) after an odd t, a barrier. A slot written at
  // step t is read at step t+2 and written again at step t+4: a barrier after every odd step
  // lies between each write and its reads, and between each read and the next write. The loop
  // is unrolled by the ring's four slots, so slots and register sets are compile-time constants
  // (LDS offsets fold into the instructions; register sets never meet at a runtime join).
  auto step = [&](int t, auto phase, auto do_compute) {
    constexpr int Q = decltype(phase)::value;  // t % 4: the ring slot of tile t
    constexpr int P = Q & 1;                   // register set of tile t+2
    // (a slot written past the last tile is never read)
    if constexpr (P == 0) store(t + 2, (Q + 2) & 3, t_id[2], rk0, rv0);
    else store(t + 2, (Q + 2) & 3, t_id[2], rk1, rv1);
    if constexpr (P == 0) issue(id_n, rk0, rv0);
    else issue(id_n, rk1, rv1);
    do_compute(t, Q);
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
#pragma unroll
      for (int j = 0; j < 3; ++j) t_id[j][i] = t_id[j + 1][i];
      t_id[3][i] = id_n[i];
    }
    tile_ids(t + 5, id_n);
    if constexpr (P == 1) __syncthreads();
  };
  auto run = [&](auto do_compute) {
    for (int t = 0; t < n_tiles; t += 4) {
      step(t, std::integral_constant<int, 0>{}, do_compute);
      if (t + 1 < n_tiles) step(t + 1, std::integral_constant<int, 1>{}, do_compute);
      if (t + 2 < n_tiles) step(t + 2, std::integral_constant<int, 2>{}, do_compute);
      if (t + 3 < n_tiles) step(t + 3, std::integral_constant<int, 3>{}, do_compute);
    }
  };
  if (wave_live) run(compute);
  else run([](int, int) {});
  // Loads of tiles past the end are still in flight: retire them while their
  // registers are still held, so that nothing else is placed in them first.
  vm_wait<0>(rk0);
  vm_wait<0>(rk1);
  if constexpr (!HALF) {
    vm_wait<0>(rv0);
    vm_wait<0>(rv1);
  }

  const PrefillArgs& e = PARTS ? args_again() : a;
  // A V the matrix cores got wrong anywhere in this workgroup's keys: its columns again on the fp32
  // fallback.
  bool redo_mine = false;
  if constexpr (kConvert) {
    // (an fp16 magnitude pattern above 0x7BFF, the largest finite one, is an inf or a NaN)
    const u16x2 mag = __builtin_elementwise_max(as_u16x2(__builtin_bit_cast(uint32_t, vmax) & 0x7fff7fffu),
                                                as_u16x2(__builtin_bit_cast(uint32_t, vmin) & 0x7fff7fffu));
    redo_mine = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(mag, u16x2{0x7BFF, 0x7BFF})) != 0u;
  }
  if constexpr (FINE) {
    // found from the accumulators: one that is not finite times zero is NaN
    float z = 0.f;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int d = 0; d < NE; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) z = __builtin_fmaf(o[cb][d][r], 0.f, z);
    redo_mine = z != 0.f;
  }
  if constexpr (kConvert || FINE) {
    if (__syncthreads_or(redo_mine)) {
      if (!in_parts) flag_obs_rows<WAVES>(e, b, g, C, max(q0, 0), min(C, q1));  // (none without statistics)
      prefill_cols_fp32<DT, D>(e, b, g, q_begin, C, P0 + key_a, Lk + key_a, c0, WAVES * CB * 16, wv, WAVES, lane,
                               in_parts ? part : -1, key_a, key_a + kend);
      return;
    }
  }

  // out[column] = o / l: lane (i16, kg) holds dims 16d + i16 of columns 4*kg + r,
  // and lacc[cb][r] is the denominator of column 4*kg + r (the same in its 16 lanes).
  if (!wave_live) return;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = 4 * kg + r;
      const int qi = FINE ? col_query(cb * 16 + col) : wq0 + cb * qpb + col / e.n_rep;
      const int hh = FINE ? col_head(cb * 16 + col) : g * e.n_rep + col % e.n_rep;
      // the column's running max, held by lane col (column i16 = col)
      const float m_col = __shfl(m_ref[cb], col);
      if (qi >= 0 && qi < C && hh < e.Hq) {
        if (PARTS && in_parts) {
          // (FINE's lift by 2^kLift is in o and l alike: taken off the max)
          const int64_t row = ((int64_t)part * e.total_q + q_begin + qi) * e.Hq + hh;
          float* prow = e.part_o + row * D + i16;
#pragma unroll
          for (int d = 0; d < NE; ++d) prow[16 * d] = o[cb][d][r];
          if (i16 == 0) e.part_ml[row] = make_float2(m_col - kLift, lacc[cb][r]);
          continue;
        }
        const float inv = 1.f / lacc[cb][r];
        uint16_t* orow = e.out + ((int64_t)(q_begin + qi) * e.Hq + hh) * D + i16;
#pragma unroll
        for (int d = 0; d < NE; ++d) orow[16 * d] = Elem<DT>::from_float(o[cb][d][r] * inv);
        if (i16 == 0 && qi >= C - e.obs)  // (never without statistics: obs = 0)
          e.obs_stats[(int64_t)b * e.stats_seq_stride + (int64_t)hh * e.obs + (qi - (C - e.obs))] =
              make_float2(m_col - kLift, lacc[cb][r]);
      }
    }
  }
}

// Merges the parts of each (query, q head) row of the sequences in more parts than one: with M the largest
// of the parts' m, out = sum(2^(m - M) O) / sum(2^(m - M) l). A group of D / 4 lanes takes a row, float4 dims
// 4 * lane ..; its parts' rows are read four at a time. Part s holds a row's keys iff it starts at or below
// the row's position; the others were not written.
template <int DT, int D>
__device__ __forceinline__ void prefill_combine_row(const PrefillArgs& a, const int64_t idx, const int dq) {
  constexpr int TK = kTileKeys;
  const int row = (int)(idx / a.Hq), h = (int)(idx % a.Hq);
  int b = 0, hi = a.B;  // the last sequence starting at or before the row
  while (hi - b > 1) {
    const int mid = (b + hi) >> 1;
    if (a.cu_q[mid] <= row) b = mid;
    else hi = mid;
  }
  const int q_begin = a.cu_q[b], C = a.cu_q[b + 1] - q_begin, qi = row - q_begin;
  if (qi < 0 || qi >= C || C > a.max_chunk) return;
  const int Lk = kv_len_of(a, b);
  const int nt = (Lk + TK - 1) / TK, np = part_count(a, nt);
  if (np == 1) return;  // written whole by its block
  const int pos = Lk - C + qi;
  // Parts that start at or below the row's tile p: s * nt / np <= p iff s < ceil((p + 1) np / nt).
  const int n = pos < 0 ? 0 : min(np, (int)(((uint32_t)(pos / TK + 1) * np + nt - 1) / (uint32_t)nt));
  const int64_t stride = (int64_t)a.total_q * a.Hq;
  float M = kNegFltMax, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  bool flagged = false;
  for (int s0 = 0; s0 < n; s0 += 4) {
    float2 ml[4];
    f32x4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = s0 + u < n;
      const int64_t at = (int64_t)(in ? s0 + u : s0) * stride + idx;
      ml[u] = a.part_ml[at];
      x[u] = *reinterpret_cast<const f32x4*>(a.part_o + at * D + 4 * dq);
      if (!in) ml[u] = make_float2(kNegFltMax, 0.f);
    }
    const float top = fmaxf(M, fmaxf(fmaxf(ml[0].x, ml[1].x), fmaxf(ml[2].x, ml[3].x)));
    const float f = fast_exp2(M - top);
    l *= f;
    acc *= f;
    M = top;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s0 + u >= n) continue;
      const float w = fast_exp2(ml[u].x - M);
      flagged |= __builtin_signbit(ml[u].y);
      l += w * fabsf(ml[u].y);
      acc += w * x[u];
    }
  }
  const float inv = 1.f / l;
  const uint32_t w0 = Elem<DT>::from_float(acc[0] * inv) | (uint32_t)Elem<DT>::from_float(acc[1] * inv) << 16;
  const uint32_t w1 = Elem<DT>::from_float(acc[2] * inv) | (uint32_t)Elem<DT>::from_float(acc[3] * inv) << 16;
  *reinterpret_cast<u32x2*>(a.out + idx * D + 4 * dq) = u32x2{w0, w1};
  if (dq == 0 && qi >= C - a.obs)  // (never without statistics: obs = 0)
    a.obs_stats[(int64_t)b * a.stats_seq_stride + (int64_t)h * a.obs + (qi - (C - a.obs))] =
        flagged ? make_float2(NAN, 1.f) : make_float2(M, l);
}

template <int DT, int D>
__global__ void __launch_bounds__(256) prefill_combine_kernel(const PrefillArgs a) {
  constexpr int LANES = D / 4, ROWS = 256 / LANES;
  const int64_t rows = (int64_t)a.total_q * a.Hq, step = (int64_t)gridDim.x * ROWS;
  if (step < rows) {
    // Several rows a group: a table wider than its sequences may leave nothing to merge, which is then found
    // once, by every wave.
    if (!any_in_parts(a)) return;
  }
  const int dq = threadIdx.x % LANES;
  for (int64_t idx = (int64_t)blockIdx.x * ROWS + threadIdx.x / LANES; idx < rows; idx += step)
    prefill_combine_row<DT, D>(a, idx, dq);
}

// Rows lo .. hi - 1 of sequence b's chunk, the q heads of KV group g, set to NaN (0x7FFF is a
// NaN in fp16 and in bf16). For chunks longer than the declared max_chunk: the block plan does not
// reach their first queries and the chunk write stopped at max_chunk tokens, so every block of
// such a chunk writes NaN into its rows instead of attending, the lowest block also into the rows
// below it.
template <int WAVES>
__device__ void prefill_nan_rows(const PrefillArgs& a, int b, int g, int lo, int hi) {
  const int h0 = g * a.n_rep;
  const int per = min(a.n_rep, a.Hq - h0) * a.D;  // a query row's heads of the group, contiguous
  const int64_t n = (int64_t)max(0, hi - lo) * per;
  uint16_t* base = a.out + ((int64_t)(a.cu_q[b] + lo) * a.Hq + h0) * a.D;
  for (int64_t i = threadIdx.x; i < n; i += 64 * WAVES)
    base[(i / per) * a.Hq * a.D + i % per] = 0x7FFFu;
}

// The s-th work item an XCD dispatches from its range [start, end) of pair-major item numbers
// (item j of pair p is number p * n + j): first the items j < nl of the range's pairs, pair by
// pair, then the items j >= nl. Returns false past the range.
__device__ __forceinline__ bool locate_item(int start, int end, int n, int nl, int s, int& pair, int& j) {
  const int p0 = start / n, p1 = (end - 1) / n;
  for (int pass = 0; pass < 2; ++pass) {
    const int lo = pass ? nl : 0, hi = pass ? n : nl, w = hi - lo;  // the pass's item numbers in a pair
    const int c0 = max(0, min(hi, end - p0 * n) - max(lo, start - p0 * n));  // first pair, cut by start
    if (s < c0) {
      pair = p0;
      j = max(lo, start - p0 * n) + s;
      return true;
    }
    s -= c0;
    if (p1 == p0) continue;
    const int whole = max(0, p1 - p0 - 1);  // pairs wholly in the range
    if (s < whole * w) {
      pair = p0 + 1 + s / w;
      j = lo + s % w;
      return true;
    }
    s -= whole * w;
    const int c1 = max(0, min(hi, end - p1 * n) - lo);  // last pair, cut by end
    if (s < c1) {
      pair = p1;
      j = lo + s;
      return true;
    }
    s -= c1;
  }
  return false;
}

// Column blocks per wave of the wide query blocks (the narrow ones have one fewer): the widest whose
// accumulators, queries and weights (in two parts for FINE) stay in 256 VGPRs. 64-dim heads are FINE, and
// two blocks of theirs fit the 128 VGPRs that paged_prefill_kernel asks for at D = 64: two workgroups
// then share a CU and cover each other's first loads (one 96-token prompt 7.5 us against 11.6).
constexpr int wide_blocks(bool fine) { return fine ? 2 : 3; }

// The range of work items [start, end) of a launch's n_items items that XCD xcd runs: dispatch
// is round-robin over the 8 XCDs, so the workgroups with blockIdx.x % 8 == xcd run there, and
// each XCD takes a contiguous range of the item numbers.
__device__ __forceinline__ void xcd_range(int total, int xcd, int& start, int& end) {
  const int per = total >> 3, rem = total & 7;
  start = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  end = start + per + (xcd < rem ? 1 : 0);
}

// Work items: the n3 + n2 query blocks of each (sequence, KV group) ("pair"), numbered pair
// after pair. Each XCD takes a contiguous range of these numbers, so that the blocks of one pair
// share that XCD's L2 while they stream its pages, and dispatches the three-column blocks of its
// pairs before their two-column blocks: the cheaper blocks then fill the last round of the launch.
// With statistics (obs > 0) the blocks also write the (m, l) pairs of the chunk's last obs queries
// (prefill_tile), which obs_rows_finish_kernel turns into SnapKV row statistics. (Launches without
// statistics run the same instance: compiled with that epilogue, the tile loop's schedule is 0.7 %
// faster at config 4 than without it.)
//
// With PARTS every XCD runs a range of the items for each part, part 0 first: the blocks of one part stay next
// to each other, and where the table is wider than the sequences the workgroups without keys come last.
// (Workgroups that exit at once among those that work, for the larger of two block counts, doubled launches
// of one round: an XCD's shader engines take workgroups in turn, whatever they hold. So did the same four of 28
// items a part on an XCD of 32 slots, nine times.) Where no sequence is in parts the launch runs as one without
// parts, its workgroups past the items exiting at the end: 8 x 512 queries behind 4000 tokens in a 2048-page
// table 292 us, 380 in the order of parts, 284 in a launch without parts. Looking for one costs a launch
// in parts of several sequences a round of loads, ~1.3 us.
template <int DT, int D, int WAVES, bool FINE, bool PARTS>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2)))
paged_prefill_kernel(const PrefillArgs a) {
  __shared__ PrefillLds<D> lds;
  constexpr int CB3 = wide_blocks(FINE), CB2 = CB3 - 1;
  int n3 = a.n3, n2 = a.n2;
  int start, end, pair, j, part = 0, np = 1;
  const bool parts = PARTS && any_in_parts(a);
  if (PARTS && !parts) {
    n3 = a.whole3;
    n2 = a.whole2;
  }
  if (!PARTS && a.by_block) {
    const int pairs = a.n_groups * a.B;
    j = blockIdx.x / pairs;
    pair = blockIdx.x - j * pairs;
  } else {
    const int n = n3 + n2;
    const int total = n * a.n_groups * a.B, xcd = blockIdx.x & 7;
    int s = blockIdx.x >> 3, range = xcd;
    if (parts) {
      // One range for every part; the total & 7 ranges with an item more go round the XCDs. An XCD had
      // floor((xcd + (p - 1) rem) / 8) + (xcd < rem) of those in parts 0 .. p - 1.
      const int per = total >> 3, rem = total & 7, first = xcd < rem ? 1 : 0;
      auto before = [&](int p) -> int { return p == 0 ? 0 : p * per + ((xcd + (p - 1) * rem) >> 3) + first; };
      part = s / (per + 1);  // at least
      while (part < a.n_parts && s >= before(part + 1)) ++part;
      if (part >= a.n_parts) return;
      s -= before(part);
      range = (xcd + part * rem) & 7;
    }
    xcd_range(total, range, start, end);
    if (!locate_item(start, end, n, n3, s, pair, j)) return;  // (only where no sequence is in parts)
  }
  const int g = pair % a.n_groups, b = pair / a.n_groups;
  const int C = a.cu_q[b + 1] - a.cu_q[b];
  if (parts) {
    np = part_count(a, (kv_len_of(a, b) + kTileKeys - 1) / kTileKeys);
    if (np == 1) {
      j += part * (n3 + n2);  // its blocks in the items of every part
      part = 0;
      n3 = a.whole3;
      n2 = a.whole2;
      if (j >= n3 + n2) return;
    }
  }
  constexpr int w2 = WAVES * CB2 * 16, w3 = WAVES * CB3 * 16;
  if (C > a.max_chunk) {
    if (part > 0) return;
    const int cols = a.max_chunk * a.n_rep;  // the plan's columns, counted from the end of the chunk
    const int c1 = cols - (j < n3 ? w3 * j : w3 * n3 + w2 * (j - n3)), c0 = c1 - (j < n3 ? w3 : w2);
    const int skip = C - a.max_chunk;
    const int lo = j == n3 + n2 - 1 ? 0 : max(0, skip + (max(c0, 0) / a.n_rep));
    const int hi = min(C, skip + (max(c1, 0) + a.n_rep - 1) / a.n_rep);
    prefill_nan_rows<WAVES>(a, b, g, lo, hi);
    flag_obs_rows<WAVES>(a, b, g, C, lo, hi);  // (none without statistics)
    return;
  }
  const int cols = C * a.n_rep;
  if (j < n3)
    prefill_tile<DT, D, WAVES, CB3, FINE, PARTS>(a, b, g, cols - w3 * (j + 1), part, np, lds);
  else
    prefill_tile<DT, D, WAVES, CB2, FINE, PARTS>(a, b, g, cols - w3 * n3 - w2 * (j - n3 + 1), part, np, lds);
}

// SnapKV row statistics from the (m, l) pairs paged_prefill_kernel left in obs_stats.
// l sums the weights 2^(s * scale * log2e - m) of every key the query sees, each rounded to fp16;
// the sink keys [0, sink) and the window keys [max(L - obs, sink), the query's own position] are
// summed again here from the same scores (v_mfma_f32_16x16x32 on the same operands, in the same
// order), exp2 and fp16 rounding, and taken off, which leaves the middle keys [sink, L - obs).
// Where the prefill computed those weights against the final m (m moves only when a weight would
// reach 2^8), they cancel exactly and the sum carries only the middle weights' own fp16 rounding;
// weights taken before a later move of m were rescaled in fp32 and leave a residue of at most
// 2^-11 of their share. The row becomes (log2 of that sum and of
// the zero rows padding the middle keys to a multiple of 16, 0) in the units of s * scale * log2e;
// it is flagged (y = 1) for the scoring pass to recompute from the keys where the prefill flagged
// it, where the sink and window hold half of its weight or more (the difference would lose bits),
// or where the middle sum falls below 2^-100 of its max (m is the max over every key the query
// sees: middle weights below 2^-126 of it lose bits). One workgroup per 16 columns (observation query,
// q head of the group) of a (sequence, KV group), its four waves taking every fourth page: a 64-key
// sink and a 128-key window are one round of loads (one wave took them in four, 13.5 us a layer at 2
// x 8 x 32 column blocks). Lane (i16, kg) holds column i16 and keys 4kg .. 4kg + 3 of each 16-key
// page. (The (m, l) pairs exist only where the tiled kernel ran.)
// FINE: the weights as the FINE instances sum them, in two parts.
template <int DT, bool FINE>
__global__ void __launch_bounds__(256) obs_rows_finish_kernel(const PrefillArgs a) {
  __shared__ float wave_part[4][16];
  const int lane = threadIdx.x & 63, i16 = lane & 15, kg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cols = a.obs * a.n_rep;
  const int nblk = (cols + 15) >> 4;
  const int blk = (int)(blockIdx.x % nblk);
  const int64_t pair = blockIdx.x / nblk;
  const int g = (int)(pair % a.n_groups), b = (int)(pair / a.n_groups);
  const int q_begin = a.cu_q[b], C = a.cu_q[b + 1] - q_begin;
  const int L = kv_len_of(a, b);
  const int col = blk * 16 + i16;
  const int i = col / a.n_rep, h = g * a.n_rep + col % a.n_rep;
  const int qi = C - a.obs + i;
  const bool live = col < cols && h < a.Hq && qi >= 0 && C <= a.max_chunk;
  if (!__any(live)) return;  // (workgroup-uniform: a chunk shorter than the window, or too long)
  float2* slot = a.obs_stats + (int64_t)b * a.stats_seq_stride + (int64_t)h * a.obs + i;
  const float2 ml = live ? *slot : make_float2(0.f, 0.f);
  const bool ok = live && __builtin_isfinite(ml.x) && ml.y > 0.f && __builtin_isfinite(ml.y);
  const float m = ok ? ml.x : 0.f;
  // B operand: dims 32s + 8kg .. 32s + 8kg + 7 of column i16's query row
  const uint16_t* qp = a.q + (live ? (int64_t)(q_begin + qi) * a.q_st + (int64_t)h * a.q_sh : 0) + 8 * kg;
  u32x4 qv[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) qv[s] = live ? ld16(qp + 32 * s) : u32x4{0u, 0u, 0u, 0u};
  const int pos = L - C + qi;  // the query's position: it sees keys 0 .. pos
  const float sl2 = a.scale_log2;
  const int32_t* btrow = a.bt + (int64_t)b * a.max_blocks;
  float part = 0.f;
  // The sink's keys [0, s_end) and the window's [w_beg, L), page by page (page pg holds keys 16 pg ..
  // 16 pg + 15): this wave's pages four at a time, their loads issued together. A operand: dims
  // 32s + 8kg .. of key 16 pg + i16.
  const int s_end = min(a.sink, L), w_beg = max(L - a.obs, a.sink);
  const int n_sink = (s_end + 15) >> 4, w_page = w_beg >> 4;
  const int n_all = n_sink + max(0, ((L + 15) >> 4) - w_page);
  for (int t0 = wv; t0 < n_all; t0 += 16) {
    u32x4 ka[4][4];
    int pg[4];
    bool pok[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + 4 * u;
      pg[u] = t < n_sink ? t : w_page + t - n_sink;
      const int id = t < n_all ? btrow[pg[u]] : -1;
      pok[u] = (unsigned)id < (unsigned)a.num_pages;
      const uint16_t* kp =
          a.k + (int64_t)(pok[u] ? id : 0) * a.k_sp + (int64_t)i16 * a.k_st + (int64_t)g * a.k_sh + 8 * kg;
#pragma unroll
      for (int s = 0; s < 4; ++s) ka[u][s] = pok[u] ? ld16(kp + 32 * s) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in_sink = t0 + 4 * u < n_sink;
      const int lo = in_sink ? 0 : w_beg, hi = in_sink ? s_end : L;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = mfma16x16x32<DT>(ka[u][s], qv[s], acc);
      // the weights rounded as the prefill kernel summed them (see above)
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r] = fast_exp2(__builtin_fmaf(acc[r], sl2, -m));
      if constexpr (FINE) {
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          uint32_t h, l;
          PrefillSplit<DT>::split(p[r], p[r + 1], h, l);
          p[r] = Elem<DT>::lo(h) + Elem<DT>::lo(l);
          p[r + 1] = Elem<DT>::hi(h) + Elem<DT>::hi(l);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = (float)(_Float16)p[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = 16 * pg[u] + 4 * kg + r;
        part += (pok[u] && key >= lo && key < hi && key <= pos) ? p[r] : 0.f;
      }
    }
  }
  part += __shfl_xor(part, 16);
  part += __shfl_xor(part, 32);
  if (kg == 0) wave_part[wv][i16] = part;
  __syncthreads();
  if (wv > 0) return;
  part = (wave_part[0][i16] + wave_part[1][i16]) + (wave_part[2][i16] + wave_part[3][i16]);
  if (kg == 0 && live) {
    float2 res = make_float2(0.f, 1.f);
    if (ok) {
      const float l = ml.y - part;
      const int L_mid = L - a.sink - a.obs;
      const int n_pad = ((L_mid + 15) & ~15) - L_mid;
      const float top = n_pad > 0 ? fmaxf(m, 0.f) : m;
      const float lse = top + __log2f(l * exp2f(m - top) + (float)n_pad * exp2f(-top));
      if (l >= 0.5f * ml.y && l >= 0x1p-100f && __builtin_isfinite(lse)) res = make_float2(lse, 0.f);
    }
    *slot = res;
  }
}

// Marks every observation row of the call as recomputed-by-the-scorer: (0, 1) at row
// obs_stats[b * stats_seq_stride + h * obs + i] for b < B, h < Hq, i < obs.
__global__ void __launch_bounds__(256) obs_flag_kernel(const PrefillArgs a, const int64_t rows) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows) return;
  const int64_t per = (int64_t)a.Hq * a.obs;
  a.obs_stats[(idx / per) * a.stats_seq_stride + idx % per] = make_float2(0.f, 1.f);
}

// Reference-order scalar prefill for shapes the MFMA kernel does not cover: one
// workgroup per (q head, query row); natural exp; keys 0 .. P + i in page order.
template <int DT>
__global__ void __launch_bounds__(256) paged_prefill_scalar_kernel(const PrefillArgs a) {
  const int row = blockIdx.x;
  const int h = blockIdx.y;
  // sequence of this query row
  int b = 0;
  while (b + 1 < a.B && a.cu_q[b + 1] <= row) ++b;
  const int C = a.cu_q[b + 1] - a.cu_q[b];
  const int i = row - a.cu_q[b];
  if (i < 0 || i >= C) return;
  if (C > a.max_chunk) {  // longer than declared: its K/V were not all written (see prefill_nan_rows)
    for (int d = threadIdx.x; d < a.D; d += blockDim.x) a.out[((int64_t)row * a.Hq + h) * a.D + d] = 0x7FFFu;
    return;
  }
  const int Lk = kv_len_of(a, b);
  const int L = max(0, min(Lk, Lk - C + i + 1));
  const int g = h / a.n_rep;
  const int tid = threadIdx.x, t = tid >> 4, sub = tid & 15;
  __shared__ float qs[256];
  __shared__ float ss[16];
  const uint16_t* qrow = a.q + (int64_t)row * a.q_st + (int64_t)h * a.q_sh;
  for (int d = tid; d < a.D; d += blockDim.x) qs[d] = Elem<DT>::one(qrow[d]);
  __syncthreads();
  const int n_pages = (L + 15) >> 4;
  const int d = tid;
  float m = kNegFltMax, l = 0.f, acc = 0.f;
  for (int pg = 0; pg < n_pages; ++pg) {
    int bid = a.bt[(int64_t)b * a.max_blocks + pg];
    const bool ok = (unsigned)bid < (unsigned)a.num_pages;
    bid = ok ? bid : 0;
    const int nv = ok ? min(16, L - 16 * pg) : 0;
    float part = 0.f;
    if (t < nv) {
      const uint16_t* krow = a.k + (int64_t)bid * a.k_sp + (int64_t)t * a.k_st + (int64_t)g * a.k_sh;
      for (int dd = sub; dd < a.D; dd += 16) part += Elem<DT>::one(krow[dd]) * qs[dd];
    }
    part = row_sum16(part);
    if (sub == 0) ss[t] = (t < nv) ? part * a.scale : kNegFltMax;
    __syncthreads();
    float mx = kNegFltMax;
    for (int tt = 0; tt < 16; ++tt) mx = fmaxf(mx, ss[tt]);
    const float mn = fmaxf(m, mx);
    const float alpha = expf(m - mn);
    float psum = 0.f, pv = 0.f;
    for (int tt = 0; tt < 16; ++tt) {
      const float pt = (tt < nv) ? expf(ss[tt] - mn) : 0.f;
      psum += pt;
      if (d < a.D && tt < nv)
        pv += pt * Elem<DT>::one(a.v[(int64_t)bid * a.v_sp + (int64_t)tt * a.v_st + (int64_t)g * a.v_sh + d]);
    }
    l = l * alpha + psum;
    acc = acc * alpha + pv;
    m = mn;
    __syncthreads();
  }
  if (d < a.D) a.out[((int64_t)row * a.Hq + h) * a.D + d] = Elem<DT>::from_float(acc / l);
}

// Chunk K/V rows into their pages: row cu_q[b] + i goes to position P_b + i.
struct VarlenWriteArgs {
  uint16_t* k_pool;
  uint16_t* v_pool;
  int64_t k_sp, k_st, k_sh, v_sp, v_st, v_sh;
  const uint16_t* k_new;
  const uint16_t* v_new;
  int64_t n_st, n_sh;  // [total][H][D] strides shared by k_new and v_new
  const int32_t* bt;
  const int32_t* cu_q;
  const int32_t* kv_lens;
  int B, H, D, max_blocks, num_pages, vec;
  int per_shift, h_shift;  // log2(D / 8), log2(H) for the 16-byte path (-1: not powers of two)
};

// 16-byte path for power-of-two heads and D / 8: block (tb, b) writes 16 chunk tokens of
// sequence b; 16-byte chunk `it` = (token, head, chunk) by shifts. The two pages the 16
// positions can touch are read once; each pass issues 8 K and 8 V loads before its stores.
__global__ void __launch_bounds__(256) kv_write_varlen_vec_kernel(const VarlenWriteArgs a) {
  constexpr int J = 8;
  const int b = blockIdx.y;
  const int q_begin = a.cu_q[b];
  const int C = a.cu_q[b + 1] - q_begin;
  const int i0 = blockIdx.x * 16;
  if (i0 >= C) return;
  const int cap = a.max_blocks * 16;
  const int Lk = min(max(a.kv_lens[b], 0), cap);
  const int P0 = Lk - C;
  const int blk0 = (P0 + i0) >> 4;  // first page index these 16 positions touch (P0 + i0 >= 0 when valid)
  const int32_t* btrow = a.bt + (int64_t)b * a.max_blocks;
  const int pg0 = (blk0 >= 0 && blk0 < a.max_blocks) ? btrow[blk0] : -1;
  const int pg1 = (blk0 + 1 >= 0 && blk0 + 1 < a.max_blocks) ? btrow[blk0 + 1] : -1;
  const int per_mask = (1 << a.per_shift) - 1, h_mask = (1 << a.h_shift) - 1;
  const int items = 16 << (a.per_shift + a.h_shift);
  for (int base = 0; base < items; base += J * 256) {
    u32x4 kx[J], vx[J];
    uint16_t* kd[J];
    uint16_t* vd[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int it = base + j * 256 + threadIdx.x;
      const int c = it & per_mask;
      const int h = (it >> a.per_shift) & h_mask;
      const int i = i0 + (it >> (a.per_shift + a.h_shift));
      const int pos = P0 + i;
      const int page = ((pos >> 4) == blk0) ? pg0 : pg1;
      const bool ok = it < items && i < C && pos >= 0 && pos < cap && (unsigned)page < (unsigned)a.num_pages;
      kd[j] = ok ? a.k_pool + (int64_t)page * a.k_sp + (int64_t)(pos & 15) * a.k_st + (int64_t)h * a.k_sh + 8 * c
                 : nullptr;
      vd[j] = ok ? a.v_pool + (int64_t)page * a.v_sp + (int64_t)(pos & 15) * a.v_st + (int64_t)h * a.v_sh + 8 * c
                 : nullptr;
      const int64_t src = (int64_t)(q_begin + (ok ? i : i0)) * a.n_st + (int64_t)h * a.n_sh + 8 * c;
      kx[j] = ok ? *reinterpret_cast<const u32x4*>(a.k_new + src) : u32x4{0u, 0u, 0u, 0u};
      vx[j] = ok ? *reinterpret_cast<const u32x4*>(a.v_new + src) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (kd[j]) {
        *reinterpret_cast<u32x4*>(kd[j]) = kx[j];
        *reinterpret_cast<u32x4*>(vd[j]) = vx[j];
      }
    }
  }
}

// grid (token blocks of 16, B): block (tb, b) writes 16 chunk tokens of sequence b.
__global__ void __launch_bounds__(256) kv_write_varlen_kernel(const VarlenWriteArgs a) {
  const int b = blockIdx.y;
  const int q_begin = a.cu_q[b];
  const int C = a.cu_q[b + 1] - q_begin;
  const int cap = a.max_blocks * 16;
  const int Lk = min(max(a.kv_lens[b], 0), cap);
  const int P0 = Lk - C;
  const int per = a.vec ? a.D / 8 : a.D;
  const int items = 16 * a.H * per;
  for (int it = threadIdx.x; it < items; it += blockDim.x) {
    const int c = it % per;
    const int h = (it / per) % a.H;
    const int i = blockIdx.x * 16 + it / (per * a.H);
    if (i >= C) continue;
    const int pos = P0 + i;
    if (pos < 0 || pos >= cap) continue;
    const int page = a.bt[(int64_t)b * a.max_blocks + (pos >> 4)];
    if ((unsigned)page >= (unsigned)a.num_pages) continue;
    const int64_t e = a.vec ? 8 * c : c;
    const int64_t src = (int64_t)(q_begin + i) * a.n_st + (int64_t)h * a.n_sh + e;
    uint16_t* kd = a.k_pool + (int64_t)page * a.k_sp + (int64_t)(pos & 15) * a.k_st + (int64_t)h * a.k_sh + e;
    uint16_t* vd = a.v_pool + (int64_t)page * a.v_sp + (int64_t)(pos & 15) * a.v_st + (int64_t)h * a.v_sh + e;
    if (a.vec) {
      *reinterpret_cast<u32x4*>(kd) = *reinterpret_cast<const u32x4*>(a.k_new + src);
      *reinterpret_cast<u32x4*>(vd) = *reinterpret_cast<const u32x4*>(a.v_new + src);
    } else {
      *kd = a.k_new[src];
      *vd = a.v_new[src];
    }
  }
}

namespace {
bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool mul8(int64_t x) { return (x & 7) == 0; }

}  // namespace
}  // namespace ukv

using namespace ukv;

extern "C" int ukv_kv_write_varlen(void* k_pool_layer, void* v_pool_layer, const int64_t* k_strides,
                                   const int64_t* v_strides, const void* k_new, const void* v_new,
                                   const int64_t* new_strides, const int32_t* block_table, int max_blocks,
                                   const int32_t* cu_seqlens_q, const int32_t* kv_lens, int batch, int max_chunk,
                                   int num_heads, int head_dim, int num_pages, ukv_stream_t stream) {
  if (batch < 0 || max_chunk < 0 || num_heads <= 0 || head_dim <= 0 || max_blocks < 0) return UKV_ERR_INVALID_ARGUMENT;
  if (batch == 0 || max_chunk == 0) return UKV_OK;
  if (!k_pool_layer || !v_pool_layer || !k_strides || !v_strides || !k_new || !v_new || !new_strides ||
      !block_table || !cu_seqlens_q || !kv_lens)
    return UKV_ERR_INVALID_ARGUMENT;
  VarlenWriteArgs a{};
  a.k_pool = static_cast<uint16_t*>(k_pool_layer);
  a.v_pool = static_cast<uint16_t*>(v_pool_layer);
  a.k_sp = k_strides[0];
  a.k_st = k_strides[1];
  a.k_sh = k_strides[2];
  a.v_sp = v_strides[0];
  a.v_st = v_strides[1];
  a.v_sh = v_strides[2];
  a.k_new = static_cast<const uint16_t*>(k_new);
  a.v_new = static_cast<const uint16_t*>(v_new);
  a.n_st = new_strides[0];
  a.n_sh = new_strides[1];
  a.bt = block_table;
  a.cu_q = cu_seqlens_q;
  a.kv_lens = kv_lens;
  a.B = batch;
  a.H = num_heads;
  a.D = head_dim;
  a.max_blocks = max_blocks;
  a.num_pages = num_pages;
  a.vec = head_dim % 8 == 0 && al16(k_pool_layer) && al16(v_pool_layer) && al16(k_new) && al16(v_new) &&
          mul8(a.k_sp) && mul8(a.k_st) && mul8(a.k_sh) && mul8(a.v_sp) && mul8(a.v_st) && mul8(a.v_sh) &&
          mul8(a.n_st) && mul8(a.n_sh);
  auto log2_exact = [](int x) {
    int s = 0;
    while ((1 << s) < x) ++s;
    return (1 << s) == x ? s : -1;
  };
  a.per_shift = a.vec ? log2_exact(head_dim / 8) : -1;
  a.h_shift = log2_exact(num_heads);
  const dim3 grid((max_chunk + 15) / 16, batch);
  if (a.vec && a.per_shift >= 0 && a.h_shift >= 0)
    hipLaunchKernelGGL(kv_write_varlen_vec_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a);
  else
    hipLaunchKernelGGL(kv_write_varlen_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a);
  return hipGetLastError() == hipSuccess ? UKV_OK : UKV_ERR_LAUNCH;
}

namespace {

// CUs per XCD of the current device (8 XCDs), 0 when unknown.
int cus_per_xcd() {
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int per = cached[dev].load(std::memory_order_relaxed);
  if (per == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    per = n / 8;
    cached[dev].store(per, std::memory_order_relaxed);
  }
  return per;
}

struct ObsStats {
  void* stats;
  int64_t seq_stride;
  int sink, obs;
};

// The tiled kernel's instance for a head shape: FINE where n_rep does not divide 16 (a query's heads
// straddle column blocks) or D is 64, shapes that were computed with fp32 weights before it and keep
// that precision.
bool tiled_shape(int head_dim, int n_rep) { return (head_dim == 128 || head_dim == 64) && n_rep <= 64; }
bool fine_shape(int head_dim, int n_rep) { return head_dim != 128 || 16 % n_rep != 0; }

BlockPlan plan_for(int batch, int64_t rows, int max_chunk, int n_groups, int head_dim, int n_rep, int max_blocks,
                   bool parts) {
  constexpr int W = UKV_PREFILL_WAVES, tile_pages = kTileKeys / 16;
  const int cb3 = wide_blocks(fine_shape(head_dim, n_rep));
  PlanShape f{};
  f.max_cols = (int64_t)max_chunk * n_rep;
  f.pairs = (int64_t)n_groups * batch;
  f.part_row_bytes = rows * head_dim * (int64_t)sizeof(float);
  f.w2 = W * (cb3 - 1) * 16;
  f.w3 = W * cb3 * 16;
  f.n_rep = n_rep;
  f.slots_per_xcd = cus_per_xcd() * (head_dim == 64 ? 2 : 1);  // (two 64-dim workgroups share a CU)
  f.tiles = (max_blocks + tile_pages - 1) / tile_pages;
  f.narrow = cb3 == 2 ? kNarrowCostFine : kNarrowCost;
  f.allow_parts = parts;
  return choose_plan(f);
}

size_t up256(size_t x) { return (x + 255) & ~size_t(255); }
size_t part_o_bytes(int parts, int64_t rows, int head_dim) {
  return up256((size_t)parts * rows * head_dim * sizeof(float));
}
size_t part_bytes(int parts, int64_t rows, int head_dim) {
  return part_o_bytes(parts, rows, head_dim) + up256((size_t)parts * rows * sizeof(float2));
}
// Partials above this are not worth their traffic: the launch is large enough without parts.
constexpr size_t kMaxPartBytes = size_t(512) << 20;

constexpr int kMergeWgs = 2048;

template <int DT, int D, bool FINE, bool PARTS>
void launch_tiled(const PrefillArgs& a, unsigned tile_wgs, hipStream_t stream) {
  constexpr int W = UKV_PREFILL_WAVES;
  hipLaunchKernelGGL((paged_prefill_kernel<DT, D, W, FINE, PARTS>), dim3(tile_wgs), dim3(64 * W), 0, stream, a);
  if constexpr (PARTS) {
    constexpr int ROWS = 256 / (D / 4);
    const int64_t rows = (int64_t)a.total_q * a.Hq;
    // (eight workgroups a CU at once; rows beyond them are taken in turn)
    const int64_t wgs = std::min<int64_t>((rows + ROWS - 1) / ROWS, kMergeWgs);
    hipLaunchKernelGGL((prefill_combine_kernel<DT, D>), dim3((unsigned)wgs), dim3(256), 0, stream, a);
  }
}

template <int DT, bool PARTS>
void launch_tiled_dt(const PrefillArgs& a, bool fine, unsigned wgs, hipStream_t stream) {
  if (a.D == 64)
    launch_tiled<DT, 64, true, PARTS>(a, wgs, stream);
  else if (fine)
    launch_tiled<DT, 128, true, PARTS>(a, wgs, stream);
  else
    launch_tiled<DT, 128, false, PARTS>(a, wgs, stream);
}

template <int DT>
void launch_finish(const PrefillArgs& a, bool fine, dim3 grid, hipStream_t stream) {
  if (fine)
    hipLaunchKernelGGL((obs_rows_finish_kernel<DT, true>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((obs_rows_finish_kernel<DT, false>), grid, dim3(256), 0, stream, a);
}

void launch_tiled_any(const PrefillArgs& a, int dtype, bool fine, unsigned wgs, hipStream_t stream) {
  const bool parts = a.n_parts > 1;
  if (dtype == UKV_DTYPE_BF16)
    parts ? launch_tiled_dt<UKV_DTYPE_BF16, true>(a, fine, wgs, stream)
          : launch_tiled_dt<UKV_DTYPE_BF16, false>(a, fine, wgs, stream);
  else
    parts ? launch_tiled_dt<UKV_DTYPE_F16, true>(a, fine, wgs, stream)
          : launch_tiled_dt<UKV_DTYPE_F16, false>(a, fine, wgs, stream);
}

int prefill_impl(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table,
                 const int32_t* cu_seqlens_q, const int32_t* kv_lens, void* out, int batch, int total_q, int max_chunk,
                 int num_q_heads, int num_kv_heads, int head_dim, int n_rep, int max_blocks, int num_pages,
                 const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides, float softmax_scale,
                 int dtype, void* workspace, size_t workspace_bytes, ukv_stream_t stream_handle, const ObsStats* obs) {
  if (batch <= 0 || num_q_heads <= 0 || head_dim <= 0) return UKV_ERR_EMPTY;
  if (head_dim > 256) return UKV_ERR_HEAD_DIM;
  if (dtype != UKV_DTYPE_F16 && dtype != UKV_DTYPE_BF16) return UKV_ERR_DTYPE;
  if (num_kv_heads <= 0 || n_rep < 1) return UKV_ERR_GQA;
  const int n_groups = (num_q_heads + n_rep - 1) / n_rep;
  if (n_groups > num_kv_heads) return UKV_ERR_GQA;
  if (total_q < 0 || max_chunk < 0 || max_blocks < 0 || num_pages < 0) return UKV_ERR_INVALID_ARGUMENT;
  if (total_q == 0) return UKV_OK;
  // The chunks hold total_q queries, so the longest holds at least total_q / batch of them.
  if ((int64_t)max_chunk * batch < total_q) return UKV_ERR_INVALID_ARGUMENT;
  if (!q || !out || !cu_seqlens_q || !kv_lens || !q_strides || !k_strides || !v_strides)
    return UKV_ERR_INVALID_ARGUMENT;
  if (max_blocks > 0 && (!block_table || !k_cache || !v_cache || num_pages <= 0)) return UKV_ERR_INVALID_ARGUMENT;
  PrefillArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.out = static_cast<uint16_t*>(out);
  a.k = static_cast<const uint16_t*>(k_cache);
  a.v = static_cast<const uint16_t*>(v_cache);
  a.q_st = q_strides[0];
  a.q_sh = q_strides[1];
  a.k_sp = k_strides[0];
  a.k_st = k_strides[1];
  a.k_sh = k_strides[2];
  a.v_sp = v_strides[0];
  a.v_st = v_strides[1];
  a.v_sh = v_strides[2];
  a.bt = block_table;
  a.cu_q = cu_seqlens_q;
  a.kv_lens = kv_lens;
  a.B = batch;
  a.Hq = num_q_heads;
  a.n_rep = n_rep;
  a.n_groups = n_groups;
  a.D = head_dim;
  a.max_blocks = max_blocks;
  a.num_pages = num_pages;
  a.max_chunk = max_chunk;
  a.scale = softmax_scale;
  a.scale_log2 = softmax_scale * kLog2e;
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_handle);
  // The tiled kernel keeps a row's offset within its page in 32 bits.
  auto in_page_ok = [&](int64_t st, int64_t sh) {
    return st >= 0 && sh >= 0 && 15 * st + (int64_t)(num_kv_heads - 1) * sh + head_dim <= (int64_t)UINT32_MAX;
  };
  auto page_stride_ok = [](int64_t sp) { return sp >= 0 && sp <= (int64_t)UINT32_MAX; };
  const bool strides_ok = mul8(a.q_st) && mul8(a.q_sh) && mul8(a.k_sp) && mul8(a.k_st) && mul8(a.k_sh) &&
                          mul8(a.v_sp) && mul8(a.v_st) && mul8(a.v_sh) && in_page_ok(a.k_st, a.k_sh) &&
                          in_page_ok(a.v_st, a.v_sh) && page_stride_ok(a.k_sp) && page_stride_ok(a.v_sp);
  const bool fast = tiled_shape(head_dim, n_rep) && softmax_scale > 0.f && std::isfinite(softmax_scale) && strides_ok &&
                    al16(q) && al16(out) && al16(k_cache) && al16(v_cache) && max_blocks > 0;
  if (obs) {
    a.obs_stats = static_cast<float2*>(obs->stats);
    a.stats_seq_stride = obs->seq_stride;
    a.sink = obs->sink;
    a.obs = obs->obs;
  }
  if (fast) {
    const bool fine = fine_shape(head_dim, n_rep);
    const int64_t pairs = (int64_t)n_groups * batch, rows = (int64_t)total_q * num_q_heads;
    BlockPlan plan = plan_for(batch, rows, max_chunk, n_groups, head_dim, n_rep, max_blocks, workspace != nullptr);
    // (the caller sizes the workspace by the same plan; a smaller one runs without parts)
    if (plan.parts > 1 && (part_bytes(plan.parts, rows, head_dim) > workspace_bytes ||
                           (rows + 7) / 8 > INT32_MAX || (reinterpret_cast<uintptr_t>(workspace) & 15u)))
      plan = plan_for(batch, rows, max_chunk, n_groups, head_dim, n_rep, max_blocks, false);
    a.n3 = plan.n3;
    a.n2 = plan.n2;
    a.n_parts = plan.parts;
    a.part_tiles = plan.part_tiles;
    a.whole3 = plan.whole3;
    a.whole2 = plan.whole2;
    // No more keys than twice the chunk's: the blocks' key counts differ by a factor of two or more, and
    // every pair's longest blocks go first. (With a long prefix they are alike, and the blocks of one
    // pair stay together for their XCD's L2.)
    a.by_block = (int64_t)max_blocks * 16 <= 2 * (int64_t)max_chunk;
    a.total_q = total_q;
    if (plan.parts > 1) {
      a.part_o = static_cast<float*>(workspace);
      a.part_ml = reinterpret_cast<float2*>(static_cast<char*>(workspace) + part_o_bytes(plan.parts, rows, head_dim));
    }
    // Parts: eight times what an XCD runs at most. (Two parts' items hold a pair's whole blocks: narrow ones are
    // at least half as wide as wide ones.)
    const int64_t items = pairs * (a.n3 + a.n2);
    const int64_t wgs = plan.parts > 1 ? 8 * ((items * plan.parts + 7) / 8) : items;
    // The 64-dim instances write no statistics: every row is flagged, and the scoring pass recomputes
    // them from the keys.
    const int obs_rows = obs && head_dim == 64 ? a.obs : 0;
    if (obs_rows > 0) a.obs = 0;
    const int64_t finish_wgs = obs && obs_rows == 0 ? (int64_t)batch * n_groups * ((a.obs * n_rep + 15) / 16) : 0;
    if (wgs > INT32_MAX || finish_wgs > INT32_MAX) return UKV_ERR_INVALID_ARGUMENT;
    if (wgs > 0) {
      // With statistics, the prefill kernel writes the observation rows' (m, l) pairs and
      // obs_rows_finish_kernel, next on the same stream, turns them into the rows.
      launch_tiled_any(a, dtype, fine, (unsigned)wgs, stream);
    }
    if (obs_rows > 0) {
      a.obs = obs_rows;
      const int64_t flags = (int64_t)batch * num_q_heads * a.obs;
      hipLaunchKernelGGL(obs_flag_kernel, dim3((unsigned)((flags + 255) / 256)), dim3(256), 0, stream, a, flags);
    }
    if (finish_wgs > 0) {
      const dim3 fgrid((unsigned)finish_wgs);
      if (dtype == UKV_DTYPE_BF16)
        launch_finish<UKV_DTYPE_BF16>(a, fine, fgrid, stream);
      else
        launch_finish<UKV_DTYPE_F16>(a, fine, fgrid, stream);
    }
  } else {
    const dim3 grid(total_q, num_q_heads);
    if (dtype == UKV_DTYPE_BF16)
      hipLaunchKernelGGL(paged_prefill_scalar_kernel<UKV_DTYPE_BF16>, grid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL(paged_prefill_scalar_kernel<UKV_DTYPE_F16>, grid, dim3(256), 0, stream, a);
    // The statistics come from the tiled kernel only: here every row is flagged, and the
    // scoring pass recomputes them from the keys.
    if (obs) {
      const int64_t rows = (int64_t)batch * num_q_heads * a.obs;
      if (rows > 0)
        hipLaunchKernelGGL(obs_flag_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, stream, a, rows);
    }
  }
  return hipGetLastError() == hipSuccess ? UKV_OK : UKV_ERR_LAUNCH;
}

}  // namespace

extern "C" int ukv_paged_prefill(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                 const int32_t* cu_seqlens_q, const int32_t* kv_lens, void* out, int batch,
                                 int total_q, int max_chunk, int num_q_heads, int num_kv_heads, int head_dim,
                                 int n_rep, int max_blocks, int num_pages, const int64_t* q_strides,
                                 const int64_t* k_strides, const int64_t* v_strides, float softmax_scale,
                                 int dtype, ukv_stream_t stream_handle) {
  return prefill_impl(q, k_cache, v_cache, block_table, cu_seqlens_q, kv_lens, out, batch, total_q, max_chunk,
                      num_q_heads, num_kv_heads, head_dim, n_rep, max_blocks, num_pages, q_strides, k_strides,
                      v_strides, softmax_scale, dtype, nullptr, 0, stream_handle, nullptr);
}

extern "C" int ukv_paged_prefill_obs_stats(const void* q, const void* k_cache, const void* v_cache,
                                           const int32_t* block_table, const int32_t* cu_seqlens_q,
                                           const int32_t* kv_lens, void* out, int batch, int total_q, int max_chunk,
                                           int num_q_heads, int num_kv_heads, int head_dim, int n_rep,
                                           int max_blocks, int num_pages, const int64_t* q_strides,
                                           const int64_t* k_strides, const int64_t* v_strides,
                                           float softmax_scale, int dtype, int sink_len, int obs_len,
                                           float* obs_stats, int64_t stats_seq_stride, ukv_stream_t stream_handle) {
  if (sink_len < 0 || obs_len <= 0 || !obs_stats || (reinterpret_cast<uintptr_t>(obs_stats) & 7u) ||
      stats_seq_stride < (int64_t)num_q_heads * obs_len)
    return UKV_ERR_INVALID_ARGUMENT;
  const ObsStats st{obs_stats, stats_seq_stride, sink_len, obs_len};
  return prefill_impl(q, k_cache, v_cache, block_table, cu_seqlens_q, kv_lens, out, batch, total_q, max_chunk,
                      num_q_heads, num_kv_heads, head_dim, n_rep, max_blocks, num_pages, q_strides, k_strides,
                      v_strides, softmax_scale, dtype, nullptr, 0, stream_handle, &st);
}

extern "C" size_t ukv_paged_prefill_workspace_bytes(int batch, int total_q, int max_chunk, int num_q_heads,
                                                    int num_kv_heads, int head_dim, int n_rep, int max_blocks) {
  if (batch <= 0 || total_q <= 0 || max_chunk <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || n_rep < 1 ||
      max_blocks <= 0 || !tiled_shape(head_dim, n_rep))
    return 0;
  const int n_groups = (num_q_heads + n_rep - 1) / n_rep;
  const int64_t rows = (int64_t)total_q * num_q_heads;
  const BlockPlan plan = plan_for(batch, rows, max_chunk, n_groups, head_dim, n_rep, max_blocks, true);
  if (plan.parts <= 1) return 0;
  const size_t bytes = part_bytes(plan.parts, rows, head_dim);
  return bytes > kMaxPartBytes ? 0 : bytes;
}

extern "C" int ukv_paged_prefill_parts(const void* q, const void* k_cache, const void* v_cache,
                                       const int32_t* block_table, const int32_t* cu_seqlens_q,
                                       const int32_t* kv_lens, void* out, int batch, int total_q, int max_chunk,
                                       int num_q_heads, int num_kv_heads, int head_dim, int n_rep, int max_blocks,
                                       int num_pages, const int64_t* q_strides, const int64_t* k_strides,
                                       const int64_t* v_strides, float softmax_scale, int dtype, int sink_len,
                                       int obs_len, float* obs_stats, int64_t stats_seq_stride, void* workspace,
                                       size_t workspace_bytes, ukv_stream_t stream_handle) {
  if (obs_stats && (sink_len < 0 || obs_len <= 0 || (reinterpret_cast<uintptr_t>(obs_stats) & 7u) ||
                    stats_seq_stride < (int64_t)num_q_heads * obs_len))
    return UKV_ERR_INVALID_ARGUMENT;
  const ObsStats st{obs_stats, stats_seq_stride, sink_len, obs_len};
  return prefill_impl(q, k_cache, v_cache, block_table, cu_seqlens_q, kv_lens, out, batch, total_q, max_chunk,
                      num_q_heads, num_kv_heads, head_dim, n_rep, max_blocks, num_pages, q_strides, k_strides,
                      v_strides, softmax_scale, dtype, workspace, workspace_bytes, stream_handle,
                      obs_stats ? &st : nullptr);
}
