// Attention for many queries (prefill / prompt chunk) on the MFMA matrix cores:
// flash-style, causal / windowed, grouped-query, the queries being the last rows
// of the keys.
//
// grid = ceil(seq/128) * heads; a block of 4 waves takes 128 query rows of one
// head, a wave 32 of them.  Keys and values stream through LDS in tiles of 64
// rows.  The wave computes the TRANSPOSED score tile S^T = K Q^T (M = keys,
// N = queries): a lane then owns one query column, so the row max / row sum of
// the online softmax are in-lane reductions plus one exchange with lane^32, and
// the probabilities are already laid out as the B operand of O^T = V^T P^T.  V^T
// fragments come from the transposing LDS read.  All softmax state is f32 in the
// exp2 domain; the reference the exponents are taken against follows the maxima
// lazily, and a tile whose sums of exponentials stay in range never takes its
// maximum (tile_step below).
#include "../../include/iron_hip.h"
#include "common.h"

#include <type_traits>

namespace iron {

// max(x, x of the lane 32 away) without a trip through LDS: the two halves of the wave swapped
// between two copies (v_permlane32_swap), then one maximum.  The wait states between a vector
// write and the swap that reads it, and between the swap and what reads its results, are in the
// statement, since the compiler does not look inside it.
__device__ __forceinline__ float max_with_other_half(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

constexpr int BQ = 128;   // query rows per block (four waves of 32; 64 where a block is two)
constexpr int BKV = 64;   // key rows per tile
constexpr float kLazyBits = 8.f;        // how far a maximum may run ahead of the reference the exponents are taken against
constexpr float kSumLow = 0x1p-60f, kSumHigh = 0x1p24f;   // a tile's sum of exponentials outside this range: take its maximum and redo it
// 128-wide heads of up to 1024 blocks by four waves (calls without bounds): how many of a block's first tiles have their weights in two terms of bf16.  A weight rounds to bf16 against its
// reference, and only the largest, exactly 1 against a reference that is its maximum, comes through whole; eight waves a block have a reference for each half
// of the tiles and so two such weights.  Two terms in the first two tiles, all that the first 128 queries have, are nearer than that
// (relative error against 64 bits, 32 heads, 3001 queries: eight waves 0.00209, four with one term 0.00212, so 0.00188, of which 0.00166 are the output's own rounding; window of
// 1024 0.00211 / 0.00213 / 0.00192; 2500 queries, window of 129 0.00211 / 0.00222 / 0.00196) and cost 2 us (four tiles: 4).
constexpr int kFineTiles = 2;
constexpr int kCUs = 256;                // compute units the block orders below assume
// Which 16-byte chunk of a key's (value's) row in LDS holds its first one: the others are XORed by it.  A row of 64 elements is half the banks, so sixteen
// rows' fragments at one chunk, and four rows' at four, meet no bank twice by these; a row of 128 is all of them and takes the row itself
// (with the narrow rows' swizzle its reads took every bank twice: 32 heads of 128, 3001 queries 100.3 -> 94.6 us, 8192 542 -> 523).
template <int D>
__device__ __forceinline__ int k_swizzle(int row) { return D == 64 ? (row >> 1) & 7 : row & 15; }
template <int D>
__device__ __forceinline__ int v_swizzle(int row) { return (row & 3) << (D == 64 ? 1 : 2); }
// Whether `groups` blocks of 32 queries and a head, the keys dealt over a block's waves (prefill_few_rows), take the place of a launch's
// blocks of 32 W queries.  Each of them reads all the keys, so it pays while the chip has CUs for them (at d = 64 with eight waves, where
// a CU holds two blocks, twice as many), and from a few tiles a wave on.  us, 32 / 8 heads, tiles against few rows: 40 queries, d = 64, 512 / 2048 / 12043
// keys 11.2 / 9.7, 23.8 / 14.5, 103 / 44; 512 queries 11.5 / 11.0, 25.3 / 22.0, 112 / 83; d = 128, 8000 keys, 256 queries 121 / 56, 512 queries over
// 512 keys 18.3 / 21.8.
template <int D, int W>
__host__ __device__ __forceinline__ bool few_rows_pay(int groups, int keys) { return groups <= (D == 64 && W == 4 ? 512 : 256) && keys >= 512; }
constexpr int kFewBlocks = 512;          // launches of fewer blocks than this halve their blocks' queries (S = 1024 at 32 heads: 18.5 -> 13.9 us)
constexpr int kWideBigBlocks = 512;     // wide heads: launches of at least this many 128-query blocks keep that size
// Launches of few blocks split each block's tiles over two halves of eight waves, which halves a block's chain of tiles; more fill the chip better
// four waves each.  64-wide heads (two eight-wave blocks share a CU): S = 8192 at 32 heads 365 -> 353-360 us split, past S = 16384 not.  128-wide ones: see
// split_128.
constexpr int kSplitMaxBlocks64 = 4096;

// Few live queries over many keys (a turn late in a conversation: 40 rows of a 2048-row launch, 12 000 keys): by the
// tiles below, a block a head and 128 queries, most of the chip would idle behind a block's chain
// of tiles.  Here a block takes 32 queries of one head and its NW waves deal the keys among them, wave w the 32-key
// tiles w, w + NW, ...; their (max, sum, O) meet in LDS.  No wave waits for another before that: a
// wave has a K and a V tile of its own in LDS, takes both into registers and sends for the next ones before it
// computes.  S^T, the lanes' queries and O^T lie as in the
// kernel below.
template <int D, int NW>
__device__ __forceinline__ void prefill_few_rows(
    char* smem, const bf16_t* __restrict__ Qh, const bf16_t* __restrict__ Kh, const bf16_t* __restrict__ Vh,
    bf16_t* __restrict__ Oh, int q0, int seq, int q_tokens, int kv_tokens, int offset, float scale_log2, int causal, int window,
    long q_row_stride, long kv_row_stride) {
  constexpr int ROWB = D * 2, KS = D / 16, DT = D / 32, CPR = D / 8;
  constexpr int TK = 32, TILE = TK * ROWB, VINST = TILE / 1024, RPI = 1024 / ROWB;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (what depends on the lane is made here: shared with the caller's, a value of it spilled)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, g = lane >> 5;
  const int my_q = q0 + col;
  const bool q_live = my_q < q_tokens;
  const int qpos = offset + my_q, wq_lo = offset + q0, wq_hi = offset + min(q0 + 31, q_tokens - 1);

  // Keys the block's live queries can see, in tiles; this wave's are wave, wave + NW, ...
  int kv_hi = kv_tokens;
  if (causal) kv_hi = min(kv_hi, wq_hi + 1);
  else if (window >= 0) kv_hi = min(kv_hi, wq_hi + window + 1);
  const int kv_lo = window >= 0 ? max(0, wq_lo - window) / TK * TK : 0;
  const int ntiles = (kv_hi - kv_lo + TK - 1) / TK;
  const int steps = ntiles > wave ? (ntiles - wave + NW - 1) / NW : 0;

  // The head's keys (values) from kv_lo's row to the last key's end are one buffer: rows past it read as zeros.
  const int row_bytes = (int)kv_row_stride * 2;
  const int reach = kv_hi > kv_lo ? (kv_tokens - kv_lo - 1) * row_bytes + ROWB : 0;
  const __amdgpu_buffer_rsrc_t k_rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(Kh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(Vh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
  // Load i covers tile rows i RPI + l.  A row starts on a multiple of its head's bytes, so the part of K's
  // swizzle that is the load's own is an XOR of the lane's offset.
  static_assert(RPI % 4 == 0, "V's swizzle is by row % 4: the lane's alone");
  const int l = lane / CPR;
  const int k_lane = l * row_bytes + (((lane % CPR) ^ k_swizzle<D>(l)) << 4), v_lane = l * row_bytes + (((lane % CPR) ^ v_swizzle<D>(l)) << 4);
  char* stage = smem + wave * (2 * TILE);   // the wave's K tile, then its V tile
  auto issue = [&](int step) {
    const int at = (wave + step * NW) * TK * row_bytes;
#pragma unroll
    for (int i = 0; i < VINST; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rows, IRON_LDS_PTR(stage + i * 1024), 16,
                                               (int)(k_lane ^ (k_swizzle<D>(i * RPI) << 4)) + at + i * RPI * row_bytes, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rows, IRON_LDS_PTR(stage + TILE + i * 1024), 16,
                                               (int)v_lane + at + i * RPI * row_bytes, 0, 0, 0);
    }
  };
  if (steps > 0) issue(0);

  bf16x8 qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (q_live) v = *reinterpret_cast<const uint4*>(Qh + (size_t)my_q * q_row_stride + 8 * g + 16 * s);
    qf[s] = __builtin_bit_cast(bf16x8, v);
  }
  const int v_key = 4 * g + ((lane & 15) >> 2), v_swz = v_swizzle<D>(lane >> 2);
  unsigned v_frag[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int chunk = dt * 4 + (((lane >> 4) & 1) << 1) + ((lane & 3) >> 1);
    v_frag[dt] = (unsigned)(size_t)IRON_LDS_PTR(stage) + TILE + v_key * ROWB + ((chunk ^ v_swz) << 4) + ((lane & 1) << 3);
  }
  int see_hi = kv_tokens - 1, see_lo = 0;
  if (causal) see_hi = min(see_hi, qpos);
  else if (window >= 0) see_hi = min(see_hi, qpos + window);
  if (window >= 0) see_lo = max(0, qpos - window);
  const unsigned see_span = see_hi >= see_lo ? (unsigned)(see_hi - see_lo) : 0u;
  if (see_hi < see_lo) see_lo = 1 << 30;

  f32x16 oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[t][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const unsigned k_frag = (unsigned)(size_t)IRON_LDS_PTR(stage) + col * ROWB;
  const int k_swz = k_swizzle<D>(col);
  for (int step = 0; step < steps; ++step) {
    const int kv0 = kv_lo + (wave + step * NW) * TK;
    wait_vmcnt<0>();   // the wave's own tiles: nobody else's wait, no barrier
    bf16x8 kf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) kf[s] = lds_read_b128_at<0>(k_frag + (((2 * s + g) ^ k_swz) << 4));
    TrFrag vf[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      vf[dt][0].lo = lds_read_tr16_at<0>(v_frag[dt]);
      vf[dt][0].hi = lds_read_tr16_at<8 * ROWB>(v_frag[dt]);
      vf[dt][1].lo = lds_read_tr16_at<16 * ROWB>(v_frag[dt]);
      vf[dt][1].hi = lds_read_tr16_at<24 * ROWB>(v_frag[dt]);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) lds_wait_for<0>(kf[s]);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) lds_tr_wait(vf[dt][0], vf[dt][1]);
    if (step + 1 < steps) issue(step + 1);   // the tiles are in registers: their buffers take the next ones
    f32x16 sacc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sacc[e] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], sacc, 0, 0, 0);
    // Element e is key kv0 + 8 (e / 4) + 4 g + e % 4, query `col`.
    bool edge = kv0 + TK > kv_tokens;
    if (causal) edge |= kv0 + TK - 1 > wq_lo;
    else if (window >= 0) edge |= kv0 + TK - 1 > wq_lo + window;
    if (window >= 0) edge |= kv0 < wq_hi - window;
    if (edge) {
      const int rel = kv0 + 4 * g - see_lo;
#pragma unroll
      for (int e = 0; e < 16; ++e) sacc[e] = (unsigned)(rel + 8 * (e >> 2) + (e & 3)) > see_span ? -INFINITY : sacc[e];
    }
    // The reference follows the maxima lazily, as below.
    float rmax = sacc[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) rmax = fmaxf(rmax, sacc[e]);
    if (__builtin_amdgcn_ballot_w64((rmax - m_run) * scale_log2 > kLazyBits || (m_run == -INFINITY && rmax != -INFINITY)) != 0) {
      const float m_new = fmaxf(m_run, max_with_other_half(rmax));
      const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);
      l_run *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[t][e] *= alpha;
      m_run = m_new;
    }
    const float mc = m_run == -INFINITY ? 0.f : m_run * scale_log2;
    bf16x8 pf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float e = __builtin_amdgcn_exp2f(fmaf(sacc[8 * h + j], scale_log2, -mc));
        if (edge && sacc[8 * h + j] == -INFINITY) e = 0.f;   // also where the scale is 0 and -inf * 0 is no number
        p[j] = e;
        l_run += e;
      }
      pf[h] = __builtin_bit_cast(bf16x8, pack8(p));
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int h = 0; h < 2; ++h) oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_join(vf[dt][h]), pf[h], oacc[dt], 0, 0, 0);
  }

  // The upper half of the waves hands over to the lower, until one is left: a value a lane a row.
  constexpr int FIELDS = 2 + 16 * DT;
  float* hand = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int left = NW / 2; left >= 1; left >>= 1) {
    __syncthreads();   // every wave is done with the stages, or with what the round before handed over
    if (wave >= left && wave < 2 * left) {
      float* to = hand + (wave - left) * FIELDS * 64 + lane;
      to[0] = m_run;
      to[64] = l_run;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) to[(2 + 16 * t + e) * 64] = oacc[t][e];
    }
    __syncthreads();
    if (wave < left) {
      const float* from = hand + wave * FIELDS * 64 + lane;
      const float m_other = from[0], l_other = from[64];
      const float m_new = fmaxf(m_run, m_other);
      const float mc = (m_new == -INFINITY) ? 0.f : m_new * scale_log2;
      const float a_mine = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fmaf(m_run, scale_log2, -mc));   // a wave
      const float a_other = m_other == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fmaf(m_other, scale_log2, -mc));   // may have seen no key
      m_run = m_new;
      l_run = l_run * a_mine + l_other * a_other;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[t][e] = oacc[t][e] * a_mine + from[(2 + 16 * t + e) * 64] * a_other;
    }
  }
  if (wave != 0 || my_q >= seq) return;
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = (q_live && l_tot > 0.f) ? 1.0f / l_tot : 0.f;
  bf16_t* op = Oh + (size_t)my_q * q_row_stride;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<uint2*>(op + 32 * dt + 8 * q + 4 * g) =
          make_uint2(pack_bf16(oacc[dt][4 * q + 0] * inv, oacc[dt][4 * q + 1] * inv),
                     pack_bf16(oacc[dt][4 * q + 2] * inv, oacc[dt][4 * q + 3] * inv));
}

// How a launch deals keys over blocks (DEALT below): a block has 128 queries of one KV head, those of all its query heads in turn, and one of `slices` slices of the
// key tiles that they see.  `blocks`: a KV head's, by queries.  The launch is for few queries over many keys, whose blocks leave CUs without one: as many slices as
// give each CU one block, or two where that is the less by what was measured, a step of a block's two tiles 1.2 us, of two on a CU 2.05, and a block's part out and
// back 0.017; no slice of fewer tiles than kSliceTiles.  Us, 32 / 8 heads of 64, a block a CU and two (or as many of them as there are): 200 queries, 7000 keys 27.6 / 29.5,
// 12043 42.9 / 38.4; 450, 4500 32.9 / 35.7, 12043 71.2 / 62; 600, 7000 64 / 51; 1000, 7000 69.5 / 71.5, 12043 127 / 114; 40 queries, slices of 6 tiles and of 12 at the least,
// 3000 keys 15.4 / 18.1.
struct PrefillDeal {
  int blocks, slices;
};
constexpr int kSliceTiles = 6;
constexpr int kDealtBlocks64 = 512, kDealtBlocks128 = 256;   // eight-wave blocks the chip holds at once
template <int D>
__device__ __forceinline__ PrefillDeal prefill_deal(int q_tokens, int kv_tokens, int heads, int group, int window) {
  const int blocks = (q_tokens * group + BQ - 1) / BQ, all = max(1, blocks * (heads / group));
  const int seen = window < 0 ? kv_tokens : min(kv_tokens, window + q_tokens), tiles = (seen + BKV - 1) / BKV, most = max(1, tiles / kSliceTiles);
  const int one = max(1, min(kCUs / all, most)), two = D == 64 ? max(1, min(2 * kCUs / all, most)) : one;
  const int some = min(tiles, 1 << 20);   // (in ns, whole numbers: both kernels have to come to the same)
  const int ns1 = 600 * some / one + (one > 1 ? 17 * all * one : 0), ns2 = 1025 * some / two + (two > 1 ? 17 * all * two : 0);
  return PrefillDeal{blocks, two > one && all * two > kCUs && ns2 < ns1 ? two : one};
}

// ... and the slices' parts of each query together.  Items: (KV head and query block, four columns, query).
template <int D>
__global__ __launch_bounds__(256) void mha_prefill_merge_kernel(const float* __restrict__ part, bf16_t* __restrict__ O, int heads, int group, int seq,
                                                                int seq_len, int kv_len, float scale_log2, int masked, int window, long q_row_stride, long q_head_stride,
                                                                const int* __restrict__ valid, const int* __restrict__ kv_valid) {
  const int q_tokens = valid ? bound_or(valid, seq) : seq_len;
  const int kv_tokens = kv_valid ? bound_or(kv_valid, kv_len) : (kv_len - seq + q_tokens);
  const PrefillDeal deal = prefill_deal<D>(q_tokens, kv_tokens, heads, group, window);
  if (deal.slices <= 1 || (masked && kv_tokens < q_tokens)) return;
  constexpr int QUADS = D / 4, AHEAD = 4;
  const int items = heads / group * deal.blocks * QUADS * BQ;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < items; i += gridDim.x * 256) {
    const int in_block = i % BQ, quad = i / BQ % QUADS, unit = i / (BQ * QUADS), kvh = unit / deal.blocks;
    const int nth = (unit - kvh * deal.blocks) * BQ + in_block, row = nth / group;
    const float* from = part + (size_t)unit * deal.slices * (BQ * (D + 2)) + in_block;
    float top = -INFINITY, sum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < deal.slices; s0 += AHEAD) {
      float m[AHEAD], l[AHEAD];
      f32x4 o[AHEAD];
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {   // (past the last: the last again, without weight)
        const float* p = from + (size_t)min(s0 + s, deal.slices - 1) * (BQ * (D + 2));
        m[s] = p[0];
        l[s] = p[BQ];
        o[s] = *reinterpret_cast<const f32x4*>(p - in_block + 2 * BQ + (quad * BQ + in_block) * 4);
      }
      float now = top;
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) now = fmaxf(now, m[s]);
      const float ref = now == -INFINITY ? 0.f : now * scale_log2, fade = top == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fmaf(top, scale_log2, -ref));
      sum *= fade;
      acc *= fade;
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {
        const float w = s0 + s < deal.slices && m[s] != -INFINITY ? __builtin_amdgcn_exp2f(fmaf(m[s], scale_log2, -ref)) : 0.f;
        sum = fmaf(l[s], w, sum);
        acc += o[s] * w;
      }
      top = now;
    }
    if (row >= q_tokens) continue;
    const float inv = sum > 0.f ? 1.0f / sum : 0.f;
    *reinterpret_cast<uint2*>(O + (size_t)(kvh * group + nth - row * group) * q_head_stride + (size_t)row * q_row_stride + quad * 4) =
        make_uint2(pack_bf16(acc[0] * inv, acc[1] * inv), pack_bf16(acc[2] * inv, acc[3] * inv));
  }
}

// K and V tiles go straight from global memory into LDS (buffer loads with the LDS bit, no register staging), as
// stored: [64 keys][D], STAGES tiles deep.  16-byte chunks of a row are XOR-swizzled so unpadded
// rows read without bank conflicts: K by k_swizzle for its 16-byte fragment reads, V by
// v_swizzle for the transposing reads (ds_read_b64_tr_b16) that deliver V^T fragments.  A bare
// s_barrier and counted s_waitcnt vmcnt keep the younger tiles' loads in flight across the barrier.
//
// At least two waves a SIMD caps the register budget at 256, which makes the compiler keep MFMA
// accumulators in ordinary VGPRs: the softmax reads S and rescales O in place instead of copying
// every value out of (and back into) accumulation registers.  The eight-wave form at d = 64 is held
// to 128 registers and two stages (64 KB), so that a CU holds two blocks at different places of their
// loops (S = 4096: 118 -> 95 us; the 64-query blocks of short prompts likewise); three four-wave blocks a CU measured slower than two (S = 8192:
// 382 against 365 us).
//
// SPLIT = 2: eight waves; waves 4..7 serve the same four groups of 32 queries as waves 0..3 but take
// the odd key tiles (their own loads, their own stage buffers), and the two halves' (max, sum, O)
// are merged through LDS at the end.  A query block's chain of tiles is half as long, which is what
// bounds a short sequence: its blocks are few and the one that sees every key finishes last.
//
// W: the waves that share a tile's loads, each with 32 of the block's 32 W queries.  Four; two
// where four would leave CUs without a block (a short prompt), so that twice as many blocks go out.
template <int D, int SPLIT, int W, bool FEW, bool FINE, bool DEALT>
__global__ __launch_bounds__(64 * W * SPLIT) __attribute__((amdgpu_waves_per_eu(W == 4 ? (D == 64 && SPLIT == 2 ? 4 : 2) : 2))) void mha_prefill_kernel(
    const bf16_t* __restrict__ Q, const bf16_t* __restrict__ K, const bf16_t* __restrict__ V,
    bf16_t* __restrict__ O, int heads, int group, int seq, int seq_len, int kv_len, float scale_log2,
    int causal, int window, long q_row_stride, long q_head_stride, long kv_row_stride,
    long kv_head_stride, const int* __restrict__ valid, const int* __restrict__ kv_valid,
    const int* __restrict__ kv_first, int kv_rows, float* __restrict__ part) {
  constexpr int ROWB = D * 2;            // bytes of a tile row
  constexpr int KS = D / 16;             // k16 steps of S^T
  constexpr int DT = D / 32;             // 32-row tiles of O^T
  constexpr int CPR = D / 8;             // 16-byte chunks a row has
  constexpr int STAGES = D == 64 && SPLIT == 1 ? 3 : 2;
  // 128-wide heads by four waves: a tile's K fragments are read under the softmax of the tile before, and a tile's loads have a whole step to land (one
  // barrier a step as without; 8192 queries 521 -> 501 us).  Not with eight waves, one block
  // a CU, where the 32 more registers bought nothing (3001 queries 93.9 / 95.2; halves half a step apart, one's products under the
  // other's softmax, 102), nor with 64-wide heads, whose four waves a SIMD cover the reads.
  constexpr bool PIPED = D == 128 && SPLIT == 1;
  constexpr int TILE = BKV * ROWB;       // bytes of a K (or V) tile
  constexpr int STAGE = 2 * TILE;
  constexpr int BQW = 32 * W;            // query rows of this block
  constexpr int INST = TILE / 1024 / W;  // 1 KB loads of K (and of V) a wave issues per tile
  constexpr int RPI = 1024 / ROWB;       // rows one load covers
  extern __shared__ __align__(1024) char smem_all[];   // SPLIT * STAGES * STAGE bytes

  const int tid = threadIdx.x, lane = tid & 63;
  // Which tiles, and which 32 queries -- uniform over the wave, so what depends on them (LDS
  // destinations, the rows a wave loads) stays in scalar registers.
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = wave_id / W, wave = wave_id % W;
  char* smem = smem_all + half * (STAGES * STAGE);            // this half's stage buffers
  const int col = lane & 31, g = lane >> 5;
  // Blocks are dispatched in id order, so the id runs over the query blocks from the last (under a
  // causal mask the heaviest: it sees the most keys) to the first, all heads of one query block
  // together: the long blocks start first and the short ones fill the tail.  Within a query block
  // the heads are dealt so that an XCD (block id mod 8) serves the heads of one KV group, whose
  // K and V it then reads from its own L2.
  // (DEALT: a block's queries are those of all a KV head's heads, and its keys a slice of what they see, see prefill_deal.)
  const int columns = DEALT ? __builtin_amdgcn_readfirstlane(heads / group) : heads, j = DEALT ? __builtin_amdgcn_readfirstlane(blockIdx.x % columns) : blockIdx.x % columns;
  const int head_of_block = DEALT ? 0 : ((heads % 8 == 0) ? (j % 8) * (heads / 8) + j / 8 : j);
  const int kvh = DEALT ? j : head_of_block / group;
  // A launch whose blocks are all resident two a CU (more blocks than CUs, no more than twice as
  // many): the second half of the ids runs from the lightest query block up, so the two blocks a CU
  // holds -- ids i and i + 256 -- are a heavy one and a light one, and every CU has the same work.
  const int nqb = (int)(gridDim.x / columns), at = DEALT ? __builtin_amdgcn_readfirstlane(blockIdx.x / columns) : (int)(blockIdx.x / columns);
  const bool folded = causal && gridDim.x > kCUs && gridDim.x <= 2 * kCUs && SPLIT == 2 && W == 4 && D == 64;
  const int q_tokens = valid ? bound_or(valid, seq) : seq_len;
  const int kv_tokens = kv_valid ? bound_or(kv_valid, kv_len) : (kv_len - seq + q_tokens);
  const bool masked_any = causal || window >= 0;
  const int offset = masked_any ? (kv_tokens - q_tokens) : 0;
  // (what a division makes is made in vector registers: brought back, or each holds one through the whole loop)
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  PrefillDeal deal{nqb, 1};
  int qb = folded && at >= (nqb + 1) / 2 ? at - (nqb + 1) / 2 : nqb - 1 - at, slice = 0;
  if constexpr (DEALT) {
    deal = prefill_deal<D>(q_tokens, kv_tokens, heads, group, window);
    deal = PrefillDeal{uniform(deal.blocks), uniform(deal.slices)};
    qb = uniform(at / deal.slices);
    slice = at - qb * deal.slices;
    qb = deal.blocks - 1 - qb;
  }

  // Few live queries (FEW: the launch may have them; the code beside the tiles' costs those 1.5 to 2.5 % at d = 128): groups of 32 take the first blocks, all blocks the zeros of the rows past them.
  const int groups = FEW ? (q_tokens + 31) >> 5 : 0;
  if (FEW && groups > 0 && groups <= nqb && offset >= 0 &&
      few_rows_pay<D, W>(heads * groups, window < 0 ? kv_tokens : min(kv_tokens, window + q_tokens))) {
    const int all = (seq + 31) >> 5;
    for (int unit = blockIdx.x; unit < heads * (all - groups); unit += gridDim.x) {
      const int h = unit % heads, r0 = (groups + unit / heads) * 32;
      bf16_t* to = O + (size_t)h * q_head_stride;
      for (int i = tid; i < 32 * CPR; i += 64 * W * SPLIT) {
        const int r = r0 + i / CPR, c = (i % CPR) * 8;
        if (r < seq) *reinterpret_cast<uint4*>(to + (size_t)r * q_row_stride + c) = make_uint4(0, 0, 0, 0);
      }
    }
    if (at >= groups) return;
    const long first_row = kv_first ? max(0, min(*kv_first, kv_rows - kv_len)) : 0;
    const size_t kv_at = (size_t)kvh * kv_head_stride + first_row * kv_row_stride;
    prefill_few_rows<D, W * SPLIT>(smem_all, Q + (size_t)head_of_block * q_head_stride, K + kv_at, V + kv_at, O + (size_t)head_of_block * q_head_stride,
                                   (groups - 1 - at) * 32, seq, q_tokens, kv_tokens, offset, scale_log2, causal, window,
                                   q_row_stride, kv_row_stride);
    return;
  }

  // This lane's query row and head, and the first rows of the block and of the wave (DEALT: query `nth` of a KV head is head nth % group's of row nth / group).
  const int nth = qb * BQW + wave * 32 + col;
  const int my_q = DEALT ? nth / group : nth;
  const int head = DEALT ? kvh * group + nth - my_q * group : head_of_block;
  const int q0 = DEALT ? uniform(qb * BQW / group) : qb * BQW, wq0 = DEALT ? uniform((qb * BQW + wave * 32) / group) : q0 + wave * 32;
  const int q_last = min(DEALT ? uniform((qb * BQW + BQW - 1) / group) : q0 + BQW - 1, q_tokens - 1);
  const int wq_last = min(DEALT ? uniform((qb * BQW + wave * 32 + 31) / group) : wq0 + 31, q_tokens - 1);
  const bool q_live = my_q < q_tokens;
  const int qpos = offset + my_q;
  const int wq_lo = offset + wq0;        // positions of the wave's first and last live query
  const int wq_hi = offset + wq_last;

  bf16_t* Oh = O + (size_t)head * q_head_stride;
  // Rows past the bound: zeros.  A block wholly past it does only that.
  if constexpr (DEALT) {
    const int from = offset < 0 ? 0 : q_tokens, all = (seq - from) * heads * CPR;
    for (int i = blockIdx.x * (64 * W * SPLIT) + tid; i < all; i += gridDim.x * (64 * W * SPLIT)) {
      const int r = i / (heads * CPR), c = i - r * (heads * CPR), h = c / CPR;
      *reinterpret_cast<uint4*>(O + (size_t)h * q_head_stride + (size_t)(from + r) * q_row_stride + (c - h * CPR) * 8) = make_uint4(0, 0, 0, 0);
    }
    if (offset < 0 || at >= deal.blocks * deal.slices) return;
  } else if (q0 >= q_tokens || offset < 0) {
    for (int i = tid; i < BQW * CPR; i += 64 * W * SPLIT) {
      const int r = q0 + i / CPR, c = (i % CPR) * 8;
      if (r < seq) *reinterpret_cast<uint4*>(Oh + (size_t)r * q_row_stride + c) = make_uint4(0, 0, 0, 0);
    }
    return;
  }

  // Q^T fragments (B operand): lane holds query `col`, d = 16*s + 8*g .. +7.
  bf16x8 qf[KS];
  {
    const bf16_t* qp = Q + (size_t)head * q_head_stride + (size_t)my_q * q_row_stride + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (q_live) v = *reinterpret_cast<const uint4*>(qp + 16 * s);
      qf[s] = __builtin_bit_cast(bf16x8, v);
    }
  }

  f32x16 oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[t][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;   // the reference maximum (of the raw, unscaled scores) and the sum against it
  float mc = 0.f;                         // the reference in the exp2 domain, 0 while it is -inf

  // Keys this block's live queries can see.
  int kv_hi = kv_tokens;
  if (causal) kv_hi = min(kv_hi, offset + q_last + 1);
  else if (window >= 0) kv_hi = min(kv_hi, offset + q_last + window + 1);
  int kv_lo = 0;
  if (window >= 0) kv_lo = max(0, offset + q0 - window) / BKV * BKV;
  int ntiles = (kv_hi - kv_lo + BKV - 1) / BKV;
  if constexpr (DEALT) {   // ... of which the block has a slice
    const int from = uniform(slice * ntiles / deal.slices), to = uniform((slice + 1) * ntiles / deal.slices);
    kv_lo += from * BKV;
    ntiles = to - from;
  }
  // This half's tiles are half, half + SPLIT, ...; both halves make the same number of steps (a
  // block's waves share its barriers), the last of which may be past this half's last tile: it
  // then loads the last tile again and computes nothing.
  const int steps = (ntiles + SPLIT - 1) / SPLIT;

  if (ntiles > 0) {
    // The keys may be a window of a longer buffer, rows *kv_first on (held inside the buffer).
    const long first_row = kv_first ? max(0, min(*kv_first, kv_rows - kv_len)) : 0;
    const bf16_t* Kh = K + (size_t)kvh * kv_head_stride + first_row * kv_row_stride;
    const bf16_t* Vh = V + (size_t)kvh * kv_head_stride + first_row * kv_row_stride;

    // Loader: buffer loads straight into LDS.  Load i of a wave covers tile rows
    // (wave*INST + i)*RPI .. ; lane -> (row, physical chunk), and fetches the logical chunk that
    // the row's swizzle maps there.  The buffer is the tile's rows of this head up to the last key
    // (rebuilt per tile with scalar instructions): a lane's place in it is a constant 32-bit
    // offset, and rows past the last key -- only the last tile can hold any -- lie outside the
    // buffer and read as zeros, which the mask below turns into zero weights.
    const int l_row = lane / CPR, l_pch = lane % CPR;
    const int row_bytes = (int)kv_row_stride * 2;
    int k_voff[INST], v_voff[INST];
#pragma unroll
    for (int i = 0; i < INST; ++i) {
      const int r = (wave * INST + i) * RPI + l_row;
      k_voff[i] = r * row_bytes + (l_pch ^ k_swizzle<D>(r)) * 16;
      v_voff[i] = r * row_bytes + (l_pch ^ v_swizzle<D>(r)) * 16;
    }
    // The keys (and values) of the head that this block can see, from row kv_lo's start to the
    // last key's row end, are one buffer for the whole loop; a tile's place in it goes into the
    // lanes' offsets, the part of the address the bounds check sees.
    const int reach = (kv_tokens - kv_lo - 1) * row_bytes + ROWB;
    const __amdgpu_buffer_rsrc_t k_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(Kh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(Vh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
    const int tile_bytes = BKV * row_bytes;
    auto issue_k = [&](int tile, int buf) {
      char* st = smem + buf * STAGE;
      const int at = tile * tile_bytes;
#pragma unroll
      for (int i = 0; i < INST; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rows, IRON_LDS_PTR(st + (wave * INST + i) * 1024), 16, (int)k_voff[i] + at, 0, 0, 0);
    };
    auto issue_v = [&](int tile, int buf) {
      char* st = smem + buf * STAGE;
      const int at = tile * tile_bytes;
#pragma unroll
      for (int i = 0; i < INST; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rows, IRON_LDS_PTR(st + TILE + (wave * INST + i) * 1024), 16, (int)v_voff[i] + at, 0, 0, 0);
    };
    auto issue = [&](int tile, int buf) {
      issue_k(tile, buf);
      issue_v(tile, buf);
    };
    auto tile_of = [&](int step) { return min(step * SPLIT + half, ntiles - 1); };
    // Always STAGES-1 tiles in flight before the loop and one more each iteration (past the end
    // the last tile again, into a buffer nobody reads), so the wait counts below are exact.
    if constexpr (PIPED) {
      issue_k(tile_of(0), 0);
      issue_v(tile_of(0), 0);
      issue_k(tile_of(1), 1);
    } else {
#pragma unroll
      for (int s = 0; s < STAGES - 1; ++s) issue(tile_of(s), s);
    }

    // Fragment addressing.  K (A operand of S^T): lane reads key t*32 + col, chunk 2s + g.
    const int k_frag = col * ROWB, k_swz = k_swizzle<D>(col);
    // V^T (A operand of O^T): for (t, h) a lane group g needs keys 32t + 16h + 4g + 0..3 (low
    // half of its k slots) and the same + 8 (high half) of column d = 32 dt + col.  In the
    // transposing read a lane points at 4 consecutive d of the key row 4g + (lane & 15) / 4 ...
    const int v_key = 4 * g + ((lane & 15) >> 2);
    const int v_swz = v_swizzle<D>(lane >> 2);           // the same for every (t, h)
    int v_frag[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int chunk = dt * 4 + (((lane >> 4) & 1) << 1) + ((lane & 3) >> 1);
      v_frag[dt] = v_key * ROWB + ((chunk ^ v_swz) << 4) + ((lane & 1) << 3);
    }
    const unsigned lds_base = (unsigned)(size_t)IRON_LDS_PTR(smem);
    // The keys this lane's query may see are one range of positions for the whole loop: key kpos
    // is masked out iff (unsigned)(kpos - see_lo) > see_span (an empty range lets nothing pass).
    int see_hi = kv_tokens - 1, see_lo = 0;
    if (causal) see_hi = min(see_hi, qpos);
    else if (window >= 0) see_hi = min(see_hi, qpos + window);
    if (window >= 0) see_lo = max(0, qpos - window);
    const unsigned see_span = see_hi >= see_lo ? (unsigned)(see_hi - see_lo) : 0u;
    if (see_hi < see_lo) see_lo = 1 << 30;

    // A tile's K fragments, a 32-key half's all requested together (one wait, not one a fragment).
    auto k_half = [&](int buf, int t, bf16x8 (&kf)[KS]) {
      const char* kt = smem + buf * STAGE + t * 32 * ROWB;
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(kt + k_frag + (((2 * s + g) ^ k_swz) << 4));
      __builtin_amdgcn_sched_barrier(0);
    };
    // S^T = K Q^T for the two 32-key halves of the tile.
    auto scores = [&](const bf16x8 (&kf)[2][KS], f32x16 (&sacc)[2]) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[t][e] = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s)
          sacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t][s], qf[s], sacc[t], 0, 0, 0);
      }
    };
    // The softmax and O^T += V^T P^T of a tile on stage buffer `buf`.
    auto rest = [&](int tile, int buf, f32x16 (&sacc)[2]) __attribute__((always_inline)) {
      const int kv0 = kv_lo + tile * BKV;
      const unsigned vt = lds_base + buf * STAGE + TILE;
      {
        // Only tiles that touch a bound or the mask's edge pay for masking.  Element e of half t
        // is key kv0 + 32 t + 8 (e/4) + 4 g + e%4, query `col`.
        bool edge = kv0 + BKV > kv_tokens;
        if (causal) edge |= kv0 + BKV - 1 > wq_lo;
        else if (window >= 0) edge |= kv0 + BKV - 1 > wq_lo + window;
        if (window >= 0) edge |= kv0 < wq_hi - window;
        if (edge) {
          const int rel = kv0 + 4 * g - see_lo;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              sacc[t][e] = (unsigned)(rel + 32 * t + 8 * (e >> 2) + (e & 3)) > see_span ? -INFINITY : sacc[t][e];
        }
        // The reference the exponents are taken against follows the maxima lazily: it moves, and
        // the sums so far are rescaled, only when some query's maximum has left it more than
        // kLazyBits doublings behind (moving on every new maximum rescaled two tiles in three at
        // S = 8192: any of a wave's 32 queries decides).  And a tile is first tried WITHOUT its
        // maximum: the exponentials against the reference as it stands, and only if some query's
        // sum of them is out of a wide range (a score far above the reference, or all of them
        // so far below it that the sum vanishes) is the maximum taken and the tile redone -- the
        // arithmetic is floating point throughout, so any reference that neither overflows nor
        // underflows gives the same quotient.  Edge tiles and queries that have no reference yet
        // take the maximum at once.
        bool careful = edge || __builtin_amdgcn_ballot_w64(m_run == -INFINITY) != 0;
        bool moves = false;
        float alpha = 1.f, rsum;
        bf16x8 pf[2][2];
        for (;;) {
          if (careful) {
            float rmax = sacc[0][0];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int e = 0; e < 16; ++e) rmax = fmaxf(rmax, sacc[t][e]);
            rmax = max_with_other_half(rmax);
            moves = __builtin_amdgcn_ballot_w64((rmax - m_run) * scale_log2 > kLazyBits) != 0;   // -inf - -inf: no
            if (moves) {
              const float m_new = fmaxf(m_run, rmax);
              const float mc_new = (m_new == -INFINITY) ? 0.f : m_new * scale_log2;
              alpha = __builtin_amdgcn_exp2f(fmaf(m_run, scale_log2, -mc_new));  // exp2(-inf) = 0 at the start
              m_run = m_new;
              mc = mc_new;
            }
          }
          rsum = 0.f;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              float p[8];
#pragma unroll
              for (int j = 0; j < 8; ++j) {
                p[j] = __builtin_amdgcn_exp2f(fmaf(sacc[t][8 * h + j], scale_log2, -mc));
                rsum += p[j];
              }
              pf[t][h] = __builtin_bit_cast(bf16x8, pack8(p));
            }
          if (careful) break;
          if (__builtin_amdgcn_ballot_w64(!(rsum >= kSumLow && rsum <= kSumHigh)) == 0) break;
          careful = true;
        }
        l_run = l_run * alpha + rsum;
        // What rounding to bf16 leaves of the first tiles' weights (see kFineTiles).
        const bool fine = FINE && tile < kFineTiles;
        bf16x8 lo[2][2];
        if (fine) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              float p[8], hi[8];
              unpack8(__builtin_bit_cast(uint4, pf[t][h]), hi);
#pragma unroll
              for (int j = 0; j < 8; ++j) p[j] = __builtin_amdgcn_exp2f(fmaf(sacc[t][8 * h + j], scale_log2, -mc)) - hi[j];
              lo[t][h] = __builtin_bit_cast(bf16x8, pack8(p));
            }
        }
        if (moves) {   // the output sums follow the reference (here, where the scores' registers are free again)
#pragma unroll
          for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) oacc[t][e] *= alpha;
        }

        // O^T += V^T P^T, a 32-key half at a time so one wait covers a batch of reads; the key
        // offsets ride in the reads' offset fields.
        auto pv_half = [&](auto half, const bf16x8 (&weights)[2][2]) {
          constexpr int t = decltype(half)::value;
          TrFrag vf[DT][2];
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const unsigned a = vt + v_frag[dt];
            vf[dt][0].lo = lds_read_tr16_at<(32 * t) * ROWB>(a);
            vf[dt][0].hi = lds_read_tr16_at<(32 * t + 8) * ROWB>(a);
            vf[dt][1].lo = lds_read_tr16_at<(32 * t + 16) * ROWB>(a);
            vf[dt][1].hi = lds_read_tr16_at<(32 * t + 24) * ROWB>(a);
          }
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            lds_tr_wait(vf[dt][0], vf[dt][1]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
              oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_join(vf[dt][h]), weights[t][h], oacc[dt], 0, 0, 0);
          }
        };
        pv_half(std::integral_constant<int, 0>{}, pf);
        pv_half(std::integral_constant<int, 1>{}, pf);
        if (fine) {
          pv_half(std::integral_constant<int, 0>{}, lo);
          pv_half(std::integral_constant<int, 1>{}, lo);
        }
      }
    };
    // A step of the loop on stage buffer `buf`.
    auto tile_step = [&](int step, const int buf) {
      const int ahead_buf = (buf + STAGES - 1) % STAGES;
      const int tile = step * SPLIT + half;
      wait_vmcnt<(STAGES - 2) * 2 * INST>();   // this wave's share of the tile has landed
      block_barrier();                          // everyone's has; everyone is done with the step before
      if constexpr (SPLIT > 1) {
        if (tile >= ntiles) {   // past this half's last tile: keep the loads (and the wait counts) going
          issue(ntiles - 1, ahead_buf);
          return;
        }
      }
      bf16x8 kf[2][KS];
      f32x16 sacc[2];
      k_half(buf, 0, kf[0]);
      k_half(buf, 1, kf[1]);   // (while the first half's MFMAs run)
      scores(kf, sacc);
      // The prefetch goes out while the score MFMAs run (its buffer, tile - 1's, is free since
      // the barrier above).
      issue(tile_of(step + STAGES - 1), ahead_buf);
      rest(tile, buf, sacc);
    };
    if constexpr (PIPED) {
      bf16x8 kf[2][KS];
      wait_vmcnt<2 * INST>();   // the first tile's keys have landed
      block_barrier();
      k_half(0, 0, kf[0]);
      k_half(0, 1, kf[1]);
      // The first tile's keys are in registers before this wave meets the barrier behind which their place is refilled: the products, which would wait for
      // them, may be scheduled past it.  (Every later tile's are there once the values read behind them are, which `rest` waits for.)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      auto piped_step = [&](int step, const int buf) {
        f32x16 sacc[2];
        scores(kf, sacc);
        wait_vmcnt<0>();   // this tile's values and the next one's keys: sent for a step ago
        block_barrier();   // everyone's have landed; everyone has this tile's keys in registers and is done with the values before
        k_half(buf ^ 1, 0, kf[0]);
        k_half(buf ^ 1, 1, kf[1]);
        issue_k(tile_of(step + 2), buf);
        issue_v(tile_of(step + 1), buf ^ 1);
        if (step < ntiles) rest(step, buf, sacc);
      };
      for (int step = 0; step < steps; step += 2) {
        piped_step(step, 0);
        piped_step(step + 1, 1);
      }
    } else if constexpr (SPLIT > 1) {
      // Few, long blocks (a short sequence): the loop unrolled over the stage buffers, so that a
      // fragment's place in its stage is an immediate of the read and the buffer arithmetic goes
      // (S = 2048: 3.5 % faster).  Where a CU holds several blocks at different places of the loop
      // the three-fold code measured 2.4 % slower (S = 8192), so there the loop stays rolled.
      // An odd count of steps is rounded up: the added step is past every half's last tile and, like
      // the odd half's own last step may be, only keeps the loads and the wait counts going (a tail
      // of single steps would be two more copies of the body, whose registers spilled).
      static_assert(STAGES == 2, "the loop below names the buffers");
      for (int step = 0; step < steps; step += STAGES) {
        tile_step(step, 0);
        tile_step(step + 1, 1);
      }
    } else {
      for (int step = 0; step < steps; ++step) tile_step(step, step % STAGES);
    }
    wait_vmcnt<0>();   // the idle fetches of the last iterations land before the block's LDS is released
  }

  if constexpr (SPLIT == 2) {
    // The odd tiles' half hands its (max, sum, O) over through LDS, a value a lane a row (no bank
    // conflicts); the even tiles' half folds it in by the usual rule and stores.
    constexpr int FIELDS = 2 + 16 * DT;
    static_assert(W * FIELDS * 64 * 4 <= SPLIT * STAGES * STAGE, "the hand-over fits the stage buffers");
    float* hand = reinterpret_cast<float*>(smem_all) + wave * FIELDS * 64 + lane;
    block_barrier();   // every wave is out of the tile loop: the stage buffers are free
    if (half == 1) {
      hand[0] = m_run;
      hand[64] = l_run;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) hand[(2 + 16 * t + e) * 64] = oacc[t][e];
    }
    __syncthreads();
    if (half == 1) return;
    const float m_other = hand[0], l_other = hand[64];
    const float m_new = fmaxf(m_run, m_other);
    const float mc = (m_new == -INFINITY) ? 0.f : m_new * scale_log2;
    const float a_mine = __builtin_amdgcn_exp2f(fmaf(m_run, scale_log2, -mc));      // exp2(-inf) = 0: a half
    const float a_other = __builtin_amdgcn_exp2f(fmaf(m_other, scale_log2, -mc));   // that saw no key
    if (DEALT) m_run = m_new;
    l_run = l_run * a_mine + l_other * a_other;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[t][e] = oacc[t][e] * a_mine + hand[(2 + 16 * t + e) * 64] * a_other;
  }

  // Normalize and store: lane holds query `col`, columns 32 dt + 8 q + 4 g + 0..3.
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (DEALT) {
    // (What depends on the lane is made again: held through the loop, some of it spilled.)
    int l = threadIdx.x;
    asm volatile("" : "+v"(l));
    const int gl = (l >> 5) & 1, in_block = wave * 32 + (l & 31);
    if (deal.slices > 1) {   // the merge's part: the queries' references and sums, then four columns of each
      float* to = part + ((size_t)(kvh * deal.blocks + qb) * deal.slices + slice) * (BQW * (D + 2));
      if (gl == 0) {
        to[in_block] = m_run;
        to[BQW + in_block] = l_tot;
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(to + 2 * BQW + ((8 * dt + 2 * q + gl) * BQW + in_block) * 4) =
              make_float4(oacc[dt][4 * q], oacc[dt][4 * q + 1], oacc[dt][4 * q + 2], oacc[dt][4 * q + 3]);
      return;
    }
    const int at_query = qb * BQW + in_block, row = at_query / group;
    if (row >= q_tokens) return;   // (zeroed above)
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    bf16_t* op = O + (size_t)(kvh * group + at_query - row * group) * q_head_stride + (size_t)row * q_row_stride;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint2*>(op + 32 * dt + 8 * q + 4 * gl) =
            make_uint2(pack_bf16(oacc[dt][4 * q] * inv, oacc[dt][4 * q + 1] * inv), pack_bf16(oacc[dt][4 * q + 2] * inv, oacc[dt][4 * q + 3] * inv));
    return;
  }
  const float inv = (q_live && l_tot > 0.f) ? 1.0f / l_tot : 0.f;
  if (my_q < seq) {
    // (The row's address is made here: computed where its inputs first are, it is 64 bits a lane held
    // -- at eight waves a block, spilled -- through the whole loop.)
    int row = my_q;
    asm volatile("" : "+v"(row));
    bf16_t* op = Oh + (size_t)row * q_row_stride;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v0 = oacc[dt][4 * q + 0] * inv, v1 = oacc[dt][4 * q + 1] * inv,
                    v2 = oacc[dt][4 * q + 2] * inv, v3 = oacc[dt][4 * q + 3] * inv;
        *reinterpret_cast<uint2*>(op + 32 * dt + 8 * q + 4 * g) =
            make_uint2(pack_bf16(v0, v1), pack_bf16(v2, v3));
      }
  }
}

// ---- 256- and 512-wide heads (Gemma's)
//
// A 64-key tile pair of 512-wide rows, or a wave's 32 queries of 512-wide output, fit neither the
// stages nor the registers of the kernel above (and at 256 it is down to one wave a SIMD).  Here a
// wave owns QN groups of 16 queries, each the columns of a 16-wide MFMA tile
// (v_mfma_f32_16x16x32_bf16), as the heads of a KV group are in decode attention: S^T = K Q^T over
// 32-key tiles (two 16-key MFMA tiles, the D columns in D / 32 k-steps, Q^T held in registers), a
// lane then owns one query column a group, its four lanes exchanging their maximum only when one
// passes the column's reference; the probabilities, rounded to bf16, are the B operand of
// O^T = V^T P^T as they stand, and O^T is D / 16 tiles of 16 output columns a group.  One group at
// 512 and two at 256 are the same 128 accumulator and 64 Q^T registers a lane; with two, every K and
// V^T fragment read out of LDS serves two MFMAs (the LDS reads are what bounds the kernel).  W waves
// (16 QN W queries of one head; two waves a SIMD, which holds a wave to 256 registers, all of them
// ordinary -- given 512 the compiler kept the accumulators in accumulation registers and copied all
// 128 around the conditional rescale on every tile) share the K and V tiles: 32 keys each, two
// stages, sent from global memory straight into LDS 1 KB an instruction; a row's 16-byte chunks are
// XORed by key & 15 in K (a fragment read is 16 keys at one chunk: all banks once) and by
// 2 (key & 3) in V (the transposing read).  Masks, bounds and the block order are the kernel's above.
template <int D, int QN, int W>
__global__ __launch_bounds__(64 * W, 2) void mha_prefill_wide_kernel(
    const bf16_t* __restrict__ Q, const bf16_t* __restrict__ K, const bf16_t* __restrict__ V,
    bf16_t* __restrict__ O, int heads, int group, int seq, int seq_len, int kv_len, float scale_log2,
    int causal, int window, long q_row_stride, long q_head_stride, long kv_row_stride,
    long kv_head_stride, const int* __restrict__ valid, const int* __restrict__ kv_valid,
    const int* __restrict__ kv_first, int kv_rows) {
  constexpr int ROWB = D * 2;            // bytes of a tile row
  constexpr int KS = D / 32;             // 32-wide k-steps of S^T
  constexpr int DT = D / 16;             // 16-row tiles of O^T
  constexpr int CPR = D / 8;             // 16-byte chunks a row has
  constexpr int TK = 32;                 // keys a tile
  constexpr int WQ = 16 * QN;            // queries of a wave
  constexpr int BQW = WQ * W;            // and of a block
  constexpr int TILE = TK * ROWB;
  constexpr int STAGE = 2 * TILE;
  constexpr int RPI = 1024 / ROWB;       // rows a 1 KB load covers
  constexpr int INST = TK / RPI / W;     // loads of K (and of V) a wave issues per tile
  static_assert(CPR * RPI == 64 && INST >= 1 && KS % 4 == 0 && DT % 4 == 0, "the tile splits into whole 1 KB loads a wave");
  extern __shared__ __align__(1024) char smem_wide[];   // 2 * STAGE bytes

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, q = lane >> 4;   // query column, quarter of the k slots
  const int j = blockIdx.x % heads;
  const int head = (heads % 8 == 0) ? (j % 8) * (heads / 8) + j / 8 : j;
  const int kvh = head / group;
  // (Two four-wave blocks a CU where the stages are 64 KB: a heavy and a light query block, as above.)
  const int nqb = (int)(gridDim.x / heads), at = (int)(blockIdx.x / heads);
  const bool folded = causal && D == 256 && W == 4 && gridDim.x > kCUs && gridDim.x <= 2 * kCUs;
  const int qb = folded && at >= (nqb + 1) / 2 ? at - (nqb + 1) / 2 : nqb - 1 - at;
  const int q0 = qb * BQW;

  const int q_tokens = valid ? bound_or(valid, seq) : seq_len;
  const int kv_tokens = kv_valid ? bound_or(kv_valid, kv_len) : (kv_len - seq + q_tokens);
  const bool masked_any = causal || window >= 0;
  const int offset = masked_any ? (kv_tokens - q_tokens) : 0;

  int my_q[QN], qpos[QN];
  bool q_live[QN];
#pragma unroll
  for (int u = 0; u < QN; ++u) {
    my_q[u] = q0 + wave * WQ + 16 * u + n;
    q_live[u] = my_q[u] < q_tokens;
    qpos[u] = offset + my_q[u];
  }
  const int wq_lo = offset + q0 + wave * WQ;
  const int wq_hi = offset + min(q0 + wave * WQ + WQ - 1, q_tokens - 1);

  bf16_t* Oh = O + (size_t)head * q_head_stride;
  if (q0 >= q_tokens || offset < 0) {   // rows of this block past the bound: zeros
    for (int i = tid; i < BQW * CPR; i += 64 * W) {
      const int r = q0 + i / CPR, c = (i % CPR) * 8;
      if (r < seq) *reinterpret_cast<uint4*>(Oh + (size_t)r * q_row_stride + c) = make_uint4(0, 0, 0, 0);
    }
    return;
  }

  // Q^T fragments (B operand): lane holds query n of its group, d = 32 s + 8 q .. + 7.
  bf16x8 qf[QN][KS];
#pragma unroll
  for (int u = 0; u < QN; ++u) {
    const bf16_t* qp = Q + (size_t)head * q_head_stride + (size_t)my_q[u] * q_row_stride + 8 * q;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (q_live[u]) v = *reinterpret_cast<const uint4*>(qp + 32 * s);
      qf[u][s] = __builtin_bit_cast(bf16x8, v);
    }
  }
  f32x4 oacc[QN][DT];
  float m_ref[QN], l_run[QN];   // a column's reference maximum (raw scores), this lane's sum
  const float lazy_raw = scale_log2 > 0.f ? kLazyBits / scale_log2 : INFINITY;   // kLazyBits doublings, in raw scores
#pragma unroll
  for (int u = 0; u < QN; ++u) {
    m_ref[u] = -INFINITY;
    l_run[u] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[u][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int q_last = min(q0 + BQW, q_tokens) - 1;
  int kv_hi = kv_tokens;
  if (causal) kv_hi = min(kv_hi, offset + q_last + 1);
  else if (window >= 0) kv_hi = min(kv_hi, offset + q_last + window + 1);
  int kv_lo = 0;
  if (window >= 0) kv_lo = max(0, offset + q0 - window) / TK * TK;
  const int ntiles = (kv_hi - kv_lo + TK - 1) / TK;

  if (ntiles > 0) {
    const long first_row = kv_first ? max(0, min(*kv_first, kv_rows - kv_len)) : 0;
    const bf16_t* Kh = K + (size_t)kvh * kv_head_stride + first_row * kv_row_stride;
    const bf16_t* Vh = V + (size_t)kvh * kv_head_stride + first_row * kv_row_stride;
    const int row_bytes = (int)kv_row_stride * 2;
    // Load i of a wave covers tile rows (wave INST + i) RPI + lane / CPR: a lane lands at physical
    // chunk lane % CPR of its row and fetches the logical chunk the row's swizzle maps there.  The
    // first row of a load is even where a load has two, so the row's low bit is the lane's own and
    // the rest of the swizzle is the load's (a scalar): two vector instructions a load, made where
    // they are used, against sixteen registers held through the loop.
    const int l_row = lane / CPR, l_ch = lane % CPR;
    const int k_lane = l_row * row_bytes + ((l_ch ^ l_row) << 4);
    const int v_lane = l_row * row_bytes + ((l_ch ^ (l_row << 1)) << 4);
    const int reach = (kv_tokens - kv_lo - 1) * row_bytes + ROWB;
    const __amdgpu_buffer_rsrc_t k_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(Kh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(Vh + (long)kv_lo * kv_row_stride), 0, reach, 0x00020000);
    const int tile_bytes = TK * row_bytes;
    auto issue = [&](int tile, int buf) {
      char* st = smem_wide + buf * STAGE;
      const int at = tile * tile_bytes;
#pragma unroll
      for (int i = 0; i < INST; ++i) {
        const int piece = wave * INST + i, r = piece * RPI, row_at = at + r * row_bytes;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rows, IRON_LDS_PTR(st + piece * 1024), 16,
                                                 (int)(k_lane ^ ((r & 15) << 4)) + row_at, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rows, IRON_LDS_PTR(st + TILE + piece * 1024), 16,
                                                 (int)(v_lane ^ ((r & 3) << 5)) + row_at, 0, 0, 0);
      }
    };
    issue(0, 0);

    // K fragment (tile t, k-step s): key 16 t + n, logical chunk 4 s + q, physical (4 s + q) ^ n: with
    // s = 4 a + b that is 16 a + (4 (b ^ (n >> 2)) | (q ^ (n & 3))) -- four bases a lane, the rest immediates.
    int k_frag[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) k_frag[b] = n * ROWB + (((4 * (b ^ (n >> 2))) | (q ^ (n & 3))) << 4);
    // V^T fragment (output tile dt): the lanes of quarter q point at key rows 4 q + 0..3 (k slots
    // 8 q + 0..3; the same 16 rows on for slots 8 q + 4..7, as S^T's second tile lies in P), 4 of the
    // tile's 16 columns each; chunk 2 dt + (lane & 3) / 2, swizzled.  dt = 4 k + r: four bases, 128 k on.
    const int v_swz = ((lane >> 2) & 3) << 1;
    const unsigned lds_base = (unsigned)(size_t)IRON_LDS_PTR(smem_wide);
    unsigned v_frag[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      v_frag[r] = lds_base + TILE + (4 * q + ((lane & 15) >> 2)) * ROWB +
                  (((2 * r + ((lane & 3) >> 1)) ^ v_swz) << 4) + ((lane & 1) << 3);

    // The keys a lane's query may see: one range of positions for the whole loop.
    int see_lo[QN];
    unsigned see_span[QN];
#pragma unroll
    for (int u = 0; u < QN; ++u) {
      int see_hi = kv_tokens - 1;
      see_lo[u] = 0;
      if (causal) see_hi = min(see_hi, qpos[u]);
      else if (window >= 0) see_hi = min(see_hi, qpos[u] + window);
      if (window >= 0) see_lo[u] = max(0, qpos[u] - window);
      see_span[u] = see_hi >= see_lo[u] ? (unsigned)(see_hi - see_lo[u]) : 0u;
      if (see_hi < see_lo[u]) see_lo[u] = 1 << 30;
    }

    auto tile_step = [&](int tile, auto buf_c) {
      constexpr int buf = decltype(buf_c)::value;
      const int kv0 = kv_lo + tile * TK;
      wait_vmcnt<0>();    // this wave's share of the tile has landed
      block_barrier();    // everyone's has; everyone is done with the tile before
      issue(min(tile + 1, ntiles - 1), buf ^ 1);
      if (causal && kv0 > wq_hi) return;   // the tile lies past every query of this wave
      const char* kt = smem_wide + buf * STAGE;
      // S^T = K Q^T for the tile's two 16-key halves, every K fragment for all the wave's groups.
      f32x4 sacc[QN][2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int u = 0; u < QN; ++u) sacc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int a = 0; a < KS / 4; ++a) {
          bf16x8 kf[4];
#pragma unroll
          for (int b = 0; b < 4; ++b)
            kf[b] = *reinterpret_cast<const bf16x8*>(kt + k_frag[b] + t * 16 * ROWB + a * 256);
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int u = 0; u < QN; ++u)
              sacc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[b], qf[u][4 * a + b], sacc[u][t], 0, 0, 0);
        }
      }
      // Element i of half t is key kv0 + 16 t + 4 q + i, query n of the group.
      bool edge = kv0 + TK > kv_tokens;
      if (causal) edge |= kv0 + TK - 1 > wq_lo;
      else if (window >= 0) edge |= kv0 + TK - 1 > wq_lo + window;
      if (window >= 0) edge |= kv0 < wq_hi - window;
      bf16x8 pf[QN];
#pragma unroll
      for (int u = 0; u < QN; ++u) {
        bool out[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            out[t][i] = edge && (unsigned)(kv0 + 16 * t + 4 * q + i - see_lo[u]) > see_span[u];
            if (out[t][i]) sacc[u][t][i] = -INFINITY;
          }
        float lm = sacc[u][0][0];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) lm = fmaxf(lm, sacc[u][t][i]);
        // The reference follows the maxima lazily: it moves (and the 16 DT sums a lane holds are
        // rescaled) only when some lane of the wave has left it more than kLazyBits doublings behind
        // or has none yet, so a probability is at most 2^kLazyBits -- nothing to float32 sums or to
        // bf16's exponent.  Moving on every new maximum rescaled on a third of the tiles and more (a
        // wave's 16 queries share the decision): 32 heads at S = 4096, d = 256: 375 -> 324 us.
        if (__builtin_amdgcn_ballot_w64(lm > m_ref[u] + lazy_raw) != 0) {
          float mx = fmaxf(lm, __shfl_xor(lm, 16, 64));
          mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
          const float m_new = fmaxf(m_ref[u], mx);
          // A column that had seen no key has zero sums to rescale; one that still has none keeps -inf.
          const float alpha = (m_ref[u] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m_ref[u] - m_new) * scale_log2);
          l_run[u] *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) oacc[u][dt][i] *= alpha;
          m_ref[u] = m_new;
        }
        const float mc = (m_ref[u] == -INFINITY) ? 0.f : m_ref[u] * scale_log2;
        float p[8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float e = __builtin_amdgcn_exp2f(fmaf(sacc[u][t][i], scale_log2, -mc));
            if (out[t][i]) e = 0.f;   // also where the scale is 0 and -inf * 0 is no number
            p[4 * t + i] = e;
            l_run[u] += e;
          }
        pf[u] = __builtin_bit_cast(bf16x8, pack8(p));
      }
      // O^T += V^T P^T, four output tiles' fragments requested at a time, each for all the groups.
#pragma unroll
      for (int k = 0; k < DT / 4; ++k) {
        TrFrag vf[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const unsigned at = v_frag[r] + (buf * STAGE + 128 * k);
          vf[r].lo = lds_read_tr16_at<0>(at);
          vf[r].hi = lds_read_tr16_at<16 * ROWB>(at);
        }
        lds_tr_wait(vf[0], vf[1]);
        lds_tr_wait(vf[2], vf[3]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < QN; ++u)
            oacc[u][4 * k + r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tr_join(vf[r]), pf[u], oacc[u][4 * k + r], 0, 0, 0);
      }
    };
    using buf0 = std::integral_constant<int, 0>;
    using buf1 = std::integral_constant<int, 1>;
    for (int tile = 0; tile < ntiles; tile += 2) {
      tile_step(tile, buf0{});
      if (tile + 1 < ntiles) tile_step(tile + 1, buf1{});
    }
    wait_vmcnt<0>();   // the idle fetch of the last iteration lands before the block's LDS is released
  }

  // The lane's sum over its own keys -> the column's; normalize and store: lane holds query n of the
  // group, columns 16 dt + 4 q + 0..3.
#pragma unroll
  for (int u = 0; u < QN; ++u) {
    float l_tot = l_run[u] + __shfl_xor(l_run[u], 16, 64);
    l_tot += __shfl_xor(l_tot, 32, 64);
    const float inv = (q_live[u] && l_tot > 0.f) ? 1.0f / l_tot : 0.f;
    if (my_q[u] < seq) {
      int row = my_q[u];   // (the address made here, as in the kernel above)
      asm volatile("" : "+v"(row));
      bf16_t* op = Oh + (size_t)row * q_row_stride + 4 * q;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<uint2*>(op + 16 * dt) = make_uint2(pack_bf16(oacc[u][dt][0] * inv, oacc[u][dt][1] * inv),
                                                             pack_bf16(oacc[u][dt][2] * inv, oacc[u][dt][3] * inv));
    }
  }
}

struct PrefillArgs {
  const uint16_t *Q, *K, *V;
  uint16_t* O;
  int heads, group, seq, seq_len, kv_len;
  float scale_log2;
  int causal, window;
  long q_row, q_head, kv_row, kv_head;
  const int *valid, *kv_valid;
  const int* kv_first;
  int kv_rows;
};

// The stage buffers are dynamic LDS (more than the 64 KB a kernel may declare statically).
template <int D, int SPLIT, int W, bool FEW, bool FINE, bool DEALT = false>
static int launch_prefill_as(const PrefillArgs& a, int blocks, void* stream, float* part = nullptr) {
  constexpr int STAGES = D == 64 && SPLIT == 1 ? 3 : 2;
  constexpr size_t lds = (size_t)SPLIT * STAGES * 2 * BKV * D * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&mha_prefill_kernel<D, SPLIT, W, FEW, FINE, DEALT>), lds); e != hipSuccess) {
    set_error("mha_prefill: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL((mha_prefill_kernel<D, SPLIT, W, FEW, FINE, DEALT>), dim3(blocks), dim3(64 * W * SPLIT), lds, (hipStream_t)stream, a.Q,
                     a.K, a.V, a.O, a.heads, a.group, a.seq, a.seq_len, a.kv_len, a.scale_log2, a.causal, a.window,
                     a.q_row, a.q_head, a.kv_row, a.kv_head, a.valid, a.kv_valid, a.kv_first, a.kv_rows, part);
  return 0;
}

// Bounds read on the device may leave few queries; else the sizes say whether there are.
template <int D, int SPLIT, int W = 4>
static int launch_prefill(const PrefillArgs& a, int blocks, void* stream) {
  const bool bounded = a.valid != nullptr || a.kv_valid != nullptr || a.seq_len != a.seq;
  // (a launch so short that all its queries may go 32 to a block has a block for each 32)
  const int groups = ((a.seq + 31) / 32) * a.heads;
  const bool few = few_rows_pay<D, W>(groups, a.kv_len);
  if (a.kv_len < 512 || (!bounded && !few)) return launch_prefill_as<D, SPLIT, W, false, false>(a, blocks, stream);
  return launch_prefill_as<D, SPLIT, W, true, false>(a, few && groups > blocks ? groups : blocks, stream);
}

// Whether a launch of 128-wide heads takes blocks of 64 queries (one a CU) and not of 128.  One round of them does: it is the shorter
// for every length (32 heads, us by 128 and by 64: 512 queries 14.3 / 11.4, 300 over 4096 keys 60 / 52).  A second round as long as the first does not
// (640 queries over 4000 keys 60 / 90), but under a causal mask over the queries' own keys the blocks go out longest first, so the second round's meet the
// first's shortest: with L blocks a head, 256 / heads of them in the first round, those two in line, each with about 5 blocks' time of its start and end,
// end before a longest one while 2 (L - 256 / heads) + 5 <= L.  Both sides of that line: 8 heads 3001 queries 46.1 / 39.8, 16 heads 1650 30.2 / 26.7,
// 24 heads 1024 21.7 / 20.6, 32 heads 704 17.1 / 16.8; past it 24 heads 1100 22.7 / 23.5, 32 heads 777 18.3 / 19.6, 40 heads 576 15.3 / 17.0.
static bool half_blocks_128(const PrefillArgs& a) {
  const long levels = (a.seq + 63) / 64;
  if (a.heads * levels <= kCUs) return true;
  return a.causal && (a.window < 0 || a.window >= a.kv_len) && a.heads * (levels + 5 + (a.kv_len - a.seq) / 64) <= 2 * kCUs;
}

// Whether a launch of 128-wide heads by blocks of 128 queries takes eight waves a block, one block a CU, or four, two blocks a CU, which read a tile's keys
// ahead (kFineTiles).  Up to 512 blocks of four waves are one round, in which a block takes longer than of eight.  Past 832 blocks four are the faster (us, eight / four: 32
// heads, 3400 queries behind 4000 keys 339 / 324, without a mask 217 / 203, 3780 behind 4000 366 / 361; 8 heads 13500 queries 372 / 359; but windows of 2048 keys 16 heads 6724 queries
// 118 / 122, from 896 blocks on 127 / 125).  Between the two it is how the blocks' lengths differ.  As long as each other, they make a round more or less: eight waves stay (2500 queries
// without a mask 123 / 132, behind 4000 keys 236 / 249).  Queries over their own keys: four where there are heads enough for the blocks that go out last to fill in behind the longest (32
// heads 2500 queries 72.5 / 70.4, 3012 94.0 / 86.7, 24 heads 3780 106 / 103, 16 heads 6340 177 / 171, 64 heads 1092 41.5 / 35.2; short of the line 24 heads 3268 85.7 / 86.4,
// 16 heads 5572 142 / 144, 8 heads 9200 185 / 211), and behind short windows (2116 queries, windows of 301 and 1024 34.7 / 30.2 and 47.4 / 42.7; 3012 queries 44.1 / 42.1 and
// 70.9 / 68.9; window of 1401, 24 heads 3268 queries 65.0 / 62.6, 4164 86.8 / 89.7).  Bounds on the device may leave fewer: eight waves up to 1024
// blocks, so a decoder's prompt, whose launches all have bounds, takes none of this.
static bool split_128(const PrefillArgs& a, int blocks) {
  if (a.valid != nullptr || a.kv_valid != nullptr || a.seq_len != a.seq) return blocks <= 4 * kCUs;
  if (blocks <= 2 * kCUs) return true;
  const bool windowed = a.window >= 0 && a.window < a.kv_len;
  if (blocks > 832) return windowed && a.window >= 1536 && blocks < 896;
  if (!a.causal || a.kv_len >= a.seq + BQ) return true;
  if (windowed) return a.window >= (blocks <= 640 ? 1536 : 1024);
  return 2 * blocks < 1000 + 13 * (blocks / a.heads);
}

template <int D>
static int launch_prefill_dealt(const PrefillArgs& a, float* part, void* stream) {
  const int columns = a.heads / a.group, blocks = ((int)(((long)a.seq * a.group + BQ - 1) / BQ)) * columns, room = (D == 64 ? kDealtBlocks64 : kDealtBlocks128) / columns * columns;   // (slices are dealt only where they fit)
  const int rc = launch_prefill_as<D, 2, 4, false, false, true>(a, blocks > room ? blocks : room, stream, part);
  if (rc != 0) return rc;
  hipLaunchKernelGGL(mha_prefill_merge_kernel<D>, dim3(512), dim3(256), 0, (hipStream_t)stream, part, a.O, a.heads, a.group, a.seq, a.seq_len, a.kv_len, a.scale_log2,
                     a.causal || a.window >= 0, a.window, a.q_row, a.q_head, a.valid, a.kv_valid);
  return 0;
}

template <int D, int QN, int W>
static int launch_prefill_wide(const PrefillArgs& a, void* stream) {
  constexpr size_t lds = (size_t)2 * 2 * 32 * D * 2;   // two stages of a 32-key K tile and V tile
  constexpr int block_queries = 16 * QN * W;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&mha_prefill_wide_kernel<D, QN, W>), lds); e != hipSuccess) {
    set_error("mha_prefill: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL((mha_prefill_wide_kernel<D, QN, W>), dim3(((a.seq + block_queries - 1) / block_queries) * a.heads),
                     dim3(64 * W), lds, (hipStream_t)stream, a.Q, a.K, a.V, a.O, a.heads, a.group, a.seq, a.seq_len, a.kv_len,
                     a.scale_log2, a.causal, a.window, a.q_row, a.q_head, a.kv_row, a.kv_head, a.valid, a.kv_valid,
                     a.kv_first, a.kv_rows);
  return 0;
}

}  // namespace iron

using namespace iron;

static int mha_prefill(const uint16_t* Q, const uint16_t* K, const uint16_t* V, uint16_t* O, int heads, int kv_heads,
                       int d, int seq, int seq_len, int kv_len, float scale, int causal, int window, int q_interleaved,
                       int kv_interleaved, const int* valid, const int* kv_valid, const int* kv_first, int kv_rows,
                       void* stream, float* part = nullptr) {
  IRON_REQUIRE(Q && K && V && O, "mha_prefill: null operand");
  IRON_REQUIRE(kv_first == nullptr || (kv_interleaved && kv_rows >= kv_len),
               "mha_prefill: a window of the keys takes them row by row (kv_interleaved) out of kv_rows (%d) >= kv_len (%d)",
               kv_rows, kv_len);
  IRON_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
               "mha_prefill: heads (%d) must be a positive multiple of kv_heads (%d)", heads, kv_heads);
  IRON_REQUIRE(d == 64 || d == 128 || d == 256 || d == 512, "mha_prefill: d (%d) must be 64, 128, 256 or 512", d);
  IRON_REQUIRE(seq > 0 && seq_len > 0 && seq_len <= seq,
               "mha_prefill: seq_len (%d) must be in [1, seq (%d)]", seq_len, seq);
  IRON_REQUIRE(kv_len >= seq, "mha_prefill: kv_len (%d) must be at least seq (%d): the queries are its last rows",
               kv_len, seq);
  IRON_REQUIRE(scale >= 0.f && scale < INFINITY, "mha_prefill: scale must be finite and not negative");
  IRON_REQUIRE((((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)O) & 15) == 0,
               "mha_prefill: operands must be 16-byte aligned");
  const long q_row = q_interleaved ? (long)heads * d : d;
  const long q_head = q_interleaved ? d : (long)seq * d;
  const long kv_row = kv_interleaved ? (long)kv_heads * d : d;
  const long kv_head = kv_interleaved ? d : (long)kv_len * d;
  IRON_REQUIRE(kv_row <= (1L << 20), "mha_prefill: a key row spans %ld values, more than the 2^20 a tile's 32-bit offsets reach", kv_row);
  IRON_REQUIRE((long)kv_len * kv_row * 2 < (1L << 31),
               "mha_prefill: the keys of a head span %ld bytes, more than the 2^31 its loads' 32-bit offsets reach",
               (long)kv_len * kv_row * 2);
  const float scale_log2 = scale * 1.4426950408889634f;
  const int blocks = ((seq + BQ - 1) / BQ) * heads;
  PrefillArgs a{Q, K, V, O, heads, heads / kv_heads, seq, seq_len, kv_len, scale_log2, causal, window,
                q_row, q_head, kv_row, kv_head, valid, kv_valid, kv_first, kv_rows};
  int rc;
  if (part != nullptr) {
    rc = d == 64 ? launch_prefill_dealt<64>(a, part, stream) : launch_prefill_dealt<128>(a, part, stream);
    if (rc != 0) return rc;
    IRON_LAUNCH_CHECK();
  }
  // Wide heads: 16-query groups on 16x16x32 tiles.  Blocks of 128 queries (eight waves) once those
  // fill the chip twice over, of 64 (four waves) below that; at 256, where two groups a wave fit the
  // registers, launches of a thousand blocks and more take two (half the LDS reads a flop: 32 heads at
  // S = 4096 382 against 424 us; at 2048 it is the other way round, 154 against 119).
  if (d == 512) rc = blocks >= kWideBigBlocks ? launch_prefill_wide<512, 1, 8>(a, stream) : launch_prefill_wide<512, 1, 4>(a, stream);
  else if (d == 256)
    rc = blocks >= 2 * kWideBigBlocks ? launch_prefill_wide<256, 2, 4>(a, stream)
         : blocks >= kWideBigBlocks   ? launch_prefill_wide<256, 1, 8>(a, stream)
                                      : launch_prefill_wide<256, 1, 4>(a, stream);
  // Fewer blocks of 128 queries than two a CU (a short prompt): blocks of 64, two waves a part.
  else if (d == 64 && blocks < kFewBlocks) rc = launch_prefill<64, 2, 2>(a, ((seq + 63) / 64) * heads, stream);
  else if (d == 64) rc = blocks <= kSplitMaxBlocks64 ? launch_prefill<64, 2>(a, blocks, stream) : launch_prefill<64, 1>(a, blocks, stream);
  // (where the few-row form takes the whole launch, and the keys are many, its blocks have eight waves: 40 queries over 512 / 1024 / 2000 / 12043 keys
  // with four 9.5 / 12.8 / 19.0 / 87 us, with eight 10.9 / 13.3 / 18.0 / 69)
  else if (half_blocks_128(a) && !(kv_len >= 1536 && few_rows_pay<128, 4>(((seq + 31) / 32) * heads, kv_len)))
    rc = launch_prefill<128, 2, 2>(a, ((seq + 63) / 64) * heads, stream);
  else if (split_128(a, blocks)) rc = launch_prefill<128, 2>(a, blocks, stream);
  // (those that eight waves would be as near for; without bounds, so no queries are few, see split_128)
  else if (blocks <= 4 * kCUs) rc = launch_prefill_as<128, 1, 4, false, true>(a, blocks, stream);
  else rc = launch_prefill<128, 1>(a, blocks, stream);
  if (rc != 0) return rc;
  IRON_LAUNCH_CHECK();
}

extern "C" int iron_mha_prefill_bf16(const uint16_t* Q, const uint16_t* K, const uint16_t* V,
                                     uint16_t* O, int heads, int kv_heads, int d, int seq,
                                     int seq_len, int kv_len, float scale, int causal, int window,
                                     int q_interleaved, int kv_interleaved, const int* valid,
                                     const int* kv_valid, void* stream) {
  return mha_prefill(Q, K, V, O, heads, kv_heads, d, seq, seq_len, kv_len, scale, causal, window, q_interleaved,
                     kv_interleaved, valid, kv_valid, nullptr, 0, stream);
}

extern "C" int iron_mha_prefill_at_bf16(const uint16_t* Q, const uint16_t* K, const uint16_t* V,
                                        uint16_t* O, int heads, int kv_heads, int d, int seq,
                                        int seq_len, int kv_len, float scale, int causal, int window,
                                        int q_interleaved, const int* valid, const int* kv_valid,
                                        const int* kv_first, int kv_rows, void* stream) {
  IRON_REQUIRE(kv_first != nullptr, "mha_prefill_at: null kv_first");
  return mha_prefill(Q, K, V, O, heads, kv_heads, d, seq, seq_len, kv_len, scale, causal, window, q_interleaved, 1,
                     valid, kv_valid, kv_first, kv_rows, stream);
}

extern "C" int64_t iron_mha_prefill_dealt_workspace_bytes(int heads, int kv_heads, int d) {
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || (d != 64 && d != 128)) return 0;
  return (int64_t)(d == 64 ? kDealtBlocks64 : kDealtBlocks128) * BQ * (d + 2) * sizeof(float);
}

extern "C" int iron_mha_prefill_dealt_bf16(const uint16_t* Q, const uint16_t* K, const uint16_t* V, uint16_t* O, int heads, int kv_heads, int d, int seq, int seq_len,
                                           int kv_len, float scale, int causal, int window, int q_interleaved, int kv_interleaved, const int* valid,
                                           const int* kv_valid, void* workspace, void* stream) {
  IRON_REQUIRE(workspace != nullptr && ((uintptr_t)workspace & 15) == 0, "mha_prefill_dealt: a workspace, 16-byte aligned");
  IRON_REQUIRE(iron_mha_prefill_dealt_workspace_bytes(heads, kv_heads, d) > 0, "mha_prefill_dealt: d (%d) is 64 or 128, heads (%d) a multiple of kv_heads (%d)", d, heads, kv_heads);
  IRON_REQUIRE(seq > 0 && (int64_t)seq * heads * (d / 8) < (1L << 31), "mha_prefill_dealt: %d rows of %d heads are more than its counters hold", seq, heads);
  return mha_prefill(Q, K, V, O, heads, kv_heads, d, seq, seq_len, kv_len, scale, causal, window, q_interleaved, kv_interleaved, valid, kv_valid, nullptr, 0, stream,
                     (float*)workspace);
}
