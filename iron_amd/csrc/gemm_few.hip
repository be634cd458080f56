// C = A B^T for a few rows of A (a batch's decode step): bound by streaming B, (N, K), once.
//
// Two kernels.  `gemm_strips_kernel` takes B eight rows at a time through LDS; `gemm_few_kernel` takes sixteen straight into the
// MFMA's registers and stands where the first's operands do not fit.  With GATED a second matrix is streamed beside the first and
// the output is act(A B^T) * (A B2^T), rounded where the separate steps round.
//
// Around a float32 stream A may be its normed rows (iron_norm_strips_bf16), and C may join it through a gate (iron_gated_strips_bf16); or A is
// the query latents of rows whose other latents go into caches (iron_latent_strips_bf16).
#include "../../include/iron_hip.h"
#include "latent.h"

#include <type_traits>

namespace iron {

// A block's eight waves deal K in strips of 256 columns: a strip of a tile's eight rows of B is 4 KB, sent from memory into the wave's own
// part of LDS as 512-byte runs (16-byte pieces XORed by the row, so that the MFMA's fragments read back without bank conflicts), STAGES - 1
// strips ahead; no wave waits for another until a tile's sums meet.  With SINGLE (K up to eight strips) a wave keeps its strip of A in
// registers over all of a block's tiles; else a strip of A is fetched with each of B.
//
// What bounds it is the way to the memory, so the shape follows that: eight rows a tile and not the MFMA's sixteen (half of each product is
// dropped; the matrix cores idle anyway), because 2048 rows of B then occupy all 256 CUs; up to sixteen rows of A as contiguous runs, because
// rows a power of two apart, read a fragment at a time by every block, meet on one L2 channel.  Eight rows of A over cold weights, us with
// gemm_few_kernel and with this: 2048 x 2048 5.2 / 3.9, 2048 x 8192 13.5 / 8.6, 4160 x 2048 7.9 / 5.4, 8192 x 2048 9.5 / 7.6,
// 10240 x 2048 13.8 / 9.1, 128256 x 2048 95 / 77 (6.8 TB/s); thirty-two rows: 4160 x 2048 13.7 / 9.4, 128256 x 2048 148 / 87.
constexpr int STRIP = 256, STRIP_BYTES = 512, STRIP_WAVES = 8, STRIP_ROWS = 8;
constexpr unsigned STRIP_BLOCKS = 256;   // one a CU; fewer tiles: a block each
// The blocks take rounds of 256 neighbouring tiles, so that all of them together read one run of B at a time; the blocks of a chiplet (every eighth) have
// eight neighbours, whose columns make a line of C in its L2.  Where a block's own tiles were neighbours the blocks read 256 places that are the same
// power of two apart, and a stream alone took 6.6 us for 33 MB and 12.1 for 67 that takes 6.4 and 11.4 so (weights out of memory, us: 8 rows of 3072 x 1536 4.75 -> 4.1,
// 4160 x 2048 5.95 -> 5.5, 8192 x 2048 8.0 -> 7.7, 50257 x 768 19.4 -> 15.9, 128256 x 2048 81.5 -> 79; 16 rows of 32000 x 1024 14.6 -> 12.5).  But rows of B that
// are 8192 columns or a multiple, give or take a line, put a round's tiles themselves a power of two apart: up to eight rows keep neighbours there (one row, 28672 x 8192 73.6, in
// rounds 80.5; 28672 x 16384 143 and 148).  More than sixteen rows keep
// neighbours, and STRIP_OUT columns of C leave as whole lines: a C that its chiplets do not hold until its lines are whole costs more than that (32 rows of
// 128256 x 2048 90, in rounds 104).
constexpr int STRIP_OUT = 64;
__device__ __forceinline__ unsigned strip_place(unsigned block) { return (block >> 6 << 6) + ((block & 7) << 3) + (block >> 3 & 7); }

__device__ __forceinline__ void lds_write_b128(unsigned addr, const f32x4& v) { asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
// A barrier behind the wave's own LDS accesses that leaves its loads from memory in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// MT: tiles of sixteen rows of A; one of them has MA rows at the most and comes by LDS, more come straight into registers.
// MEET: tiles whose sums meet at one barrier, instead of one a tile at which every wave waited for the slowest (with the same weights out of the last-level
// cache, where that is most of it: 8 rows of 4096 x 2048 4.55 -> 3.95 us, 16000 x 600 7.0 -> 6.0).
template <int MT, int MA, bool SINGLE, int STAGES, int MEET = 1>
struct Strips {
  static constexpr bool A_BY_LDS = MT == 1;
  static constexpr int A_BYTES = A_BY_LDS ? MA * STRIP_BYTES : 0, B_BYTES = STRIP_ROWS * STRIP_BYTES;
  static constexpr int ITEM = (SINGLE ? 0 : A_BYTES) + B_BYTES, WAVE = ITEM * STAGES + (SINGLE ? A_BYTES : 0);
  static constexpr int PART = STRIP_WAVES * MT * 1024;
  // LDS: the waves' strips (with MEET A's strips first, whose place every other meeting's sums take: A is in registers by then), one
  // meeting's sums or two, a norm's, columns of C.
  static constexpr bool OVER_A = MEET > 1;
  static constexpr int SUMS = STRIP_WAVES * WAVE, NORM = SUMS + (OVER_A ? 1 : 2) * MEET * PART, OUT0 = NORM + 512, OUT = MT * 16 * STRIP_OUT * 2;
  static constexpr int LDS = OUT0 + (MT > 1 ? 2 * OUT : 0);
  static_assert(!OVER_A || (SINGLE && MT == 1 && MEET * PART <= STRIP_WAVES * A_BYTES), "the sums fit where A's strips were");
  static constexpr int A_INST = A_BYTES / 1024, B_INST = B_BYTES / 1024, INST = ITEM / 1024;
};

// A's rows are rows of the stream, RMS-normed (as in stream.hip), up to eight of them and K up to eight strips: every block makes all of A for
// its own tiles, a wave its strip of K while the first of B is on its way.  The launch of a norm between two of 256 blocks takes 2.2 us, and making
// the rows here 1.0: twice A's bytes out of L2, and a chain of sums, root and scale.  Eight rows over K = 2048, weights out of memory, a norm and a
// product against both here: 2048 columns 6.1 / 5.0 us, 4160 7.95 / 6.6, 10240 11.45 / 10.0, 128256 82.0 / 80.7.  (A recurrence's step made the same
// way ahead of the product behind it was not the faster one, 8.9 / 9.3: three exponentials an element, 8 x 2048 of them a block.)
struct StripsNorm {
  const bf16_t* gain;
  float eps, unit;
};
// C joins the stream: stream += (C + y_bias) * sigmoid(gate + gate_bias), C rounded as it would be stored, by the lanes that hold its sums, which ask
// for what they add them to ahead of everything else: 0.4 us where a launch for it took 2.9 with the next norm (2048 columns: K = 2048 6.9 / 4.4,
// K = 8192 12.4 / 9.5).
struct StripsOut {
  float* stream;              // rows of N
  const bf16_t *y_bias, *gate, *gate_bias;   // y_bias may be null
  int gate_stride;
};
// C's columns are [zx | ux | gx | gate] of N / 4 each and the first three a gated recurrence's (min_gru.hip), its spans of one row at the most: a block has
// the same eight columns of each, and a row's step and state are the lanes' that hold their sums; y gets its output, C the gates alone.
// The launch of eight blocks that this was took 2.1 us behind the product, and costs 0.1 here (8192 columns over 2048, with the norm: 2 rows 11.0 -> 8.8
// us, 8 rows 11.25 -> 9.3).
struct StripsGru {
  const bf16_t *z_bias, *x_bias;
  float* state;
  const int* spans;
  bf16_t* y;
  int slots;
};
// A's rows are the query latents at the head of rows [query latent | latent | shared key part | ..] (mha_latent.hip), over their root mean squares as
// in NORMED; the rest of row i goes into the caches by block i, a 16-byte piece a thread.
// The launch of a block a row that this was takes 2.7 us between two others; here the norm costs 1.2 and the rest 0.3, because all of a block's waves
// share it (by one wave 0.9: cold code for several pieces, which the norm's barrier waits for).  Behind another product, weights out of memory: 2048
// columns over 1536, latents of 512, 2 rows 5.7 -> 4.6 us, 8 rows 6.4 -> 4.9; 3072 columns, 512 + 64, 8 rows 7.4 -> 5.75.
struct StripsLatent {
  LatentRow row;
  LatentShape a;
  const int* spans;
  bf16_t *latents, *shared_keys;
  int stride;
};
struct Joined {   // ... what four columns of it need
  float4 held;
  uint2 gate, gate_bias, y_bias;
};

// A lane's eight columns of rows 2 i + lane / 32 of the stream, normed.  `sums`: LDS, 64 floats.  LATENT: rounded as latent_row does.
template <bool LATENT>
__device__ __forceinline__ void norm_strips(const StripsNorm& norm, int K, int lane, int wave, unsigned sums, const float4 (&f)[4][2], const uint4& gain,
                                            uint4 (&out)[4]) {
  float ss[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 a = f[i][0], b = f[i][1];
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    ss[i] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) ss[i] = fmaf(x[j], x[j], ss[i]);
    ss[i] = half_wave_sum(ss[i]);
  }
  if ((lane & 31) == 31) {
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("ds_write_b32 %0, %1" ::"v"(sums + ((2 * i + (lane >> 5)) * STRIP_WAVES + wave) * 4), "v"(ss[i]) : "memory");
  }
  lds_barrier();
  // Lane l has row l % 8's: a root and a quotient a lane, and not one a lane and row.
  bf16x8 part[2];
  part[0] = lds_read_b128_at<0>(sums + (lane & 7) * STRIP_WAVES * 4);
  part[1] = lds_read_b128_at<16>(sums + (lane & 7) * STRIP_WAVES * 4);
  float total = 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    lds_wait_for<0>(part[h]);
    const f32x4 p = __builtin_bit_cast(f32x4, part[h]);
    total += p[0] + p[1] + p[2] + p[3];
  }
  const int inverse = __builtin_bit_cast(int, 1.0f / sqrtf(total / (float)K + norm.eps));
  float g[8];
  unpack8(gain, g);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int even = __builtin_amdgcn_readlane(inverse, 2 * i), odd = __builtin_amdgcn_readlane(inverse, 2 * i + 1);
    const float inv = __builtin_bit_cast(float, lane < 32 ? even : odd);
    const float4 a = f[i][0], b = f[i][1];
    float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = LATENT ? x[j] * (inv * g[j]) : x[j] * inv * (norm.unit + g[j]);
    out[i] = pack8(x);
  }
}

// A lane's 16-byte piece of a row's latent and shared key part.
struct LatentPiece {
  uint4 x, gain;
  Span span;   // lane s: slot s's
  float f[8];
  __device__ __forceinline__ void ask(const StripsLatent& o, const bf16_t* __restrict__ rows, int row, int M, int piece) {
    const int cn = o.a.rank >> 3, e = min(piece, cn + (o.a.rot >> 3) - 1);   // (the last again past the end)
    x = reinterpret_cast<const uint4*>(rows + (size_t)row * o.stride + o.row.q_rank)[e];
    gain = reinterpret_cast<const uint4*>(o.row.c_gain)[min(e, cn - 1)];
    span = span_of(o.spans, min((int)threadIdx.x & 63, o.a.slots - 1), M);
  }
  // The wave's part of the latent's sum of squares.
  __device__ __forceinline__ float squares(const StripsLatent& o, int piece) {
    unpack8(x, f);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) sum = fmaf(f[j], f[j], sum);
    return wave_sum(piece < o.a.rank >> 3 ? sum : 0.f);
  }
  __device__ __forceinline__ void store(const StripsLatent& o, int row, int piece, float squares) {
    const int cn = o.a.rank >> 3, n = cn + (o.a.rot >> 3), c = (piece - cn) * 8;
    const unsigned long long holds = __builtin_amdgcn_ballot_w64(((int)threadIdx.x & 63) < o.a.slots && row >= span.row0 && row < span.row0 + span.rows);
    if (holds == 0) return;
    const int slot = __builtin_ctzll(holds), pos = __builtin_amdgcn_readlane(span.start, slot) + row - __builtin_amdgcn_readlane(span.row0, slot);
    const size_t at = (size_t)slot * o.a.ring + pos % o.a.ring;
    if (piece < cn) {
      const float inv = 1.0f / sqrtf(squares / (float)o.a.rank + o.row.eps);
      float g[8];
      unpack8(gain, g);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] *= inv * g[j];
      *reinterpret_cast<uint4*>(o.latents + at * o.a.rank + piece * 8) = pack8(f);
    } else if (piece < n) {
      if (c < o.a.turned) {
        const float4* turn = reinterpret_cast<const float4*>(o.row.angles + (size_t)min(pos, o.a.angle_rows - 1) * o.a.turned + c);
        const float4 a = turn[0], b = turn[1];
        const float by[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const float u = f[j], v = f[j + 1];
          f[j] = u * by[j] - v * by[j + 1];
          f[j + 1] = v * by[j] + u * by[j + 1];
        }
      }
      *reinterpret_cast<uint4*>(o.shared_keys + at * o.a.rot + c) = pack8(f);
    }
  }
};

template <int MT, int MA, bool SINGLE, bool JOINS, bool GRU>   // (what LDS has room for)
__host__ __device__ constexpr int strips_meet() { return MT > 1 || !SINGLE || JOINS || GRU ? 1 : (MA == 8 ? 4 : 2); }

template <int MT, int MA, bool SINGLE, int STAGES, bool STREAM, bool NORMED = false, bool JOINS = false, bool GRU = false, bool LATENT = false,
          bool MANY = false>
__global__ __launch_bounds__(STRIP_WAVES * 64) void gemm_strips_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                                       bf16_t* __restrict__ C, int M, int N, int K, StripsNorm norm, StripsOut out, StripsGru gru,
                                                                       StripsLatent latent) {
  constexpr int MEET = strips_meet<MT, MA, SINGLE, JOINS, GRU>();
  typedef Strips<MT, MA, SINGLE, STAGES, MEET> S;
  static_assert(!GRU || (MT == 1 && MA == 8 && !JOINS), "one lane a row and four columns");
  static_assert(!NORMED || (SINGLE && MT == 1 && MA == 8), "a wave norms its own strip of eight rows");
  static_assert(!MANY || (SINGLE && STAGES == 2 && MT == 1 && !JOINS && !GRU && !LATENT), "a block's tiles follow each other strip by strip");
  static_assert(!LATENT || (NORMED && !JOINS && !GRU), "the query latents are normed rows");
  constexpr int W = STRIP_WAVES, R = STRIP_ROWS;
  constexpr bool LINED = MT > 1 && !JOINS && !GRU;   // the columns of GROUP of a block's tiles are stored together
  constexpr int GROUP = STRIP_OUT / R;
  static_assert(STAGES <= 2, "the last item's wait is for all that is out");
  constexpr int NOWHERE = 0x7ffffff0;   // an offset past the end of every run of rows (64 rows of at most 2^22, the entry point's bound, are 2^29 bytes)
  extern __shared__ __align__(1024) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l16 = lane & 15, quad = lane >> 4;
  const int strips = (K + STRIP - 1) / STRIP, mine = SINGLE ? wave < strips : (strips - wave + W - 1) / W, most = SINGLE ? 1 : (strips + W - 1) / W;
  const unsigned tiles = ((unsigned)N + R - 1) / R;
  // (64 bits: 256 times the tiles of an N of 2^27 pass 32)
  auto neighbours = [&](unsigned block) { return (unsigned)((unsigned long long)block * tiles / STRIP_BLOCKS); };
  const bool next = LINED || (!SINGLE && MA == 8 && ((K + 64) & 8191) <= 128);   // a block's tiles are neighbours
  const unsigned first = GRU || tiles <= STRIP_BLOCKS ? blockIdx.x : (next ? neighbours(blockIdx.x) : strip_place(blockIdx.x));
  const unsigned end = next && tiles > STRIP_BLOCKS ? neighbours(blockIdx.x + 1) : tiles;
  const int step = next ? 1 : (int)STRIP_BLOCKS;
  const bool idle = LATENT && blockIdx.x >= tiles;   // (a block for its row's latent alone; the tile that it fetches all the same is the first)
  const int tile0 = GRU || idle ? 0 : (int)first;
  const int my_tiles = GRU ? 4 : (idle ? 0 : (tiles <= STRIP_BLOCKS ? 1 : (int)((end - first + step - 1) / step))), items = my_tiles * mine;
  auto column_of = [&](int t) { return GRU ? t * (N >> 2) + (int)blockIdx.x * R : (tile0 + t * step) * R; };   // tile t's first
  char* const own = lds + wave * (S::OVER_A ? S::A_BYTES : S::WAVE);   // (with SINGLE A's strip)
  char* const held = S::OVER_A ? lds + W * S::A_BYTES + wave * (STAGES * S::ITEM) : own + (SINGLE ? S::A_BYTES : 0);
  const unsigned lds0 = (unsigned)(uintptr_t)IRON_LDS_PTR(lds), part0 = lds0 + S::SUMS;
  const unsigned norm_sums = lds0 + S::NORM, rest_sums = norm_sums + 64 * 4;

  // `count` loads of two rows each, `past` the caches or not: a lane's place in LDS is fixed, so the row's pieces are chosen by it.  Past the
  // rows or K: zeros.
  auto fetch_rows = [&](const bf16_t* base, int rows, int strip, char* to, auto count, auto past, int most_rows = 64) {
    const __amdgpu_buffer_rsrc_t run = bounded_bytes(base, rows * K * 2);
#pragma unroll
    for (int i = 0; i < decltype(count)::value; ++i) {
      if (2 * i >= most_rows) break;
      const int r = 2 * i + (lane >> 5), col = strip * STRIP + (((lane & 31) ^ (r & 15)) << 3);
      const int offset = col < K && r < rows ? (r * K + col) * 2 : NOWHERE;
      if (decltype(past)::value) __builtin_amdgcn_raw_ptr_buffer_load_lds(run, IRON_LDS_PTR(to + i * 1024), 16, offset, 0, 0, 2);   // non-temporal
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(run, IRON_LDS_PTR(to + i * 1024), 16, offset, 0, 0, 0);
    }
  };
  auto fetch = [&](int item) {
    char* to = held + item % STAGES * S::ITEM;
    const int t = SINGLE ? item : item / max(mine, 1), strip = wave + W * (SINGLE ? 0 : item - t * mine);
    const int row0 = column_of(t), rows = min(R, N - row0);
    if (!SINGLE && S::A_BY_LDS) {
      fetch_rows(A, M, strip, to, std::integral_constant<int, S::A_INST>(), std::false_type());
      to += S::A_BYTES;
    }
    fetch_rows(B + (size_t)row0 * K, rows, strip, to, std::integral_constant<int, S::B_INST>(), std::integral_constant<bool, STREAM>());
  };
  // Fragments: lane (quad, l16) has columns 32 k + 8 quad .. + 7 of row l16 (of B's eight rows l16 % 8; of a row of A past the last whatever
  // is there, for columns of the product that are not stored).
  const int ar = l16 & (MA - 1), br = l16 & (R - 1);
  const unsigned a_at = ar * STRIP_BYTES + ((quad ^ ar) << 4), b_at = br * STRIP_BYTES + ((quad ^ br) << 4);
  bf16x8 af[MT][8];
  auto a_from_memory = [&](int strip) {
    const __amdgpu_buffer_rsrc_t run = bounded_bytes(A, M * K * 2);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int col = strip * STRIP + k * 32 + quad * 8, r = m * 16 + l16;
        af[m][k] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(run, r < M && col < K ? (r * K + col) * 2 : NOWHERE, 0, 0));
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto a_from_lds = [&](unsigned at) {
#pragma unroll
    for (int k = 0; k < 8; ++k) af[0][k] = lds_read_b128_at<0>((at + a_at) ^ (k << 6));
  };
  // What the stream's columns need of a tile, asked for ahead of everything for the first.
  const bool joins = JOINS && lane < 32 && l16 < M;
  auto join_loads = [&](int t) {
    Joined j{};
    const int n = column_of(t) + quad * 4;
    if (joins && n < N) {
      j.held = *reinterpret_cast<const float4*>(out.stream + (size_t)l16 * N + n);
      j.gate = *reinterpret_cast<const uint2*>(out.gate + (size_t)l16 * out.gate_stride + n);
      j.gate_bias = *reinterpret_cast<const uint2*>(out.gate_bias + n);
      if (out.y_bias != nullptr) j.y_bias = *reinterpret_cast<const uint2*>(out.y_bias + n);
    }
    return j;
  };
  // ... and what a recurrence's step needs: lane (quad, l16) of the first wave's first two quads, four columns of row l16.
  int start = -1, state_at = 0;   // the row's position (none: no span has it), and its slot's first state
  float4 old_state = make_float4(0.f, 0.f, 0.f, 0.f);
  uint2 z_bias = make_uint2(0, 0), x_bias = make_uint2(0, 0);
  float gru_z[4] = {}, gru_u[4] = {};
  const int gru_col = (int)blockIdx.x * R + (quad & 1) * 4;
  Span mine_span{};
  if (GRU && wave == 0) {
    const int col = gru_col;
    z_bias = *reinterpret_cast<const uint2*>(gru.z_bias + col);
    x_bias = *reinterpret_cast<const uint2*>(gru.x_bias + col);
    mine_span = span_of(gru.spans, min(lane, gru.slots - 1), M);
  }
  // ... and a row's latent (the first blocks' waves, as many as its pieces fill).
  const int piece = (int)threadIdx.x;
  const bool rest_here = LATENT && (int)blockIdx.x < M && wave * 64 < (latent.a.rank + latent.a.rot) >> 3;
  LatentPiece rest;
  if constexpr (LATENT) {
    if (rest_here) rest.ask(latent, A, blockIdx.x, M, piece);
  }
  Joined first_joined{};
  if (JOINS && wave == 0) first_joined = join_loads(0);
  if (!NORMED && SINGLE && items > 0) {
    if (S::A_BY_LDS) fetch_rows(A, M, wave, own, std::integral_constant<int, S::A_INST>(), std::false_type(), M);
    else a_from_memory(wave);
  }
  if constexpr (!NORMED) {
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
      if (i < items) fetch(i);
  } else {
    // Rows as they are fetched: row 2 i + lane / 32, eight columns a lane (past the rows or K: zeros).
    const int col = wave * STRIP + ((lane & 31) << 3), hi = lane >> 5;
    const __amdgpu_buffer_rsrc_t rows = bounded_bytes(A, LATENT ? M * latent.stride * 2 : M * K * 4);
    float4 f[4][2];
    uint4 made[4], halves[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 2 * i + hi;
      if (LATENT) {
        halves[i] = load_bounded(rows, col < K && r < M ? (r * latent.stride + col) * 2 : NOWHERE);
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) f[i][h] = __builtin_bit_cast(float4, load_bounded(rows, col < K && r < M ? (r * K + col) * 4 + 16 * h : NOWHERE));
      }
    }
    const uint4 gain = load_bounded(bounded_bytes(norm.gain, K * 2), col * 2);
    __builtin_amdgcn_sched_barrier(0);
    // (of a wave without a strip too, for whom it is nothing: behind a branch the compiler, which then counts none of its loads, would wait for B
    // before the norm)
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i) fetch(i);
    __builtin_amdgcn_sched_barrier(0);
    if (LATENT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x[8];
        unpack8(halves[i], x);
        f[i][0] = make_float4(x[0], x[1], x[2], x[3]);
        f[i][1] = make_float4(x[4], x[5], x[6], x[7]);
      }
    }
    if constexpr (LATENT) {   // (the norm's barrier is this sum's too)
      if (rest_here) {
        const float sum = rest.squares(latent, piece);
        if (lane == 0) asm volatile("ds_write_b32 %0, %1" ::"v"(rest_sums + wave * 4), "v"(sum) : "memory");
      }
    }
    norm_strips<LATENT>(norm, K, lane, wave, norm_sums, f, gain, made);
    // (the strip is the wave's alone: no barrier)
    const unsigned mine_at = lds0 + (unsigned)(own - lds);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 2 * i + hi;
      lds_write_b128(mine_at + r * STRIP_BYTES + (((lane & 31) ^ r) << 4), __builtin_bit_cast(f32x4, made[i]));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    a_from_lds(mine_at);
#pragma unroll
    for (int k = 0; k < 8; ++k) lds_wait_for<0>(af[0][k]);
  }
  if (!NORMED && SINGLE && S::A_BY_LDS && items > 0) {
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<(STAGES - 1) * S::INST>();   // (the first item's loads stay out)
    a_from_lds(lds0 + (unsigned)(own - lds));
#pragma unroll
    for (int k = 0; k < 8; ++k) lds_wait_for<0>(af[0][k]);
  }
  if constexpr (LATENT) {
    if (rest_here) {
      bf16x8 part[2];
      part[0] = lds_read_b128_at<0>(rest_sums);
      part[1] = lds_read_b128_at<16>(rest_sums);
      float total = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        lds_wait_for<0>(part[h]);
        const f32x4 p = __builtin_bit_cast(f32x4, part[h]);
#pragma unroll
        for (int q = 0; q < 4; ++q) total += (4 * h + q) * 64 < latent.a.rank >> 3 ? p[q] : 0.f;   // (waves that have none left nothing)
      }
      rest.store(latent, blockIdx.x, piece, total);
    }
  }
  if (GRU && wave == 0) {   // (the spans' trip passed under the norm, this one passes under the products)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const unsigned long long holds = __builtin_amdgcn_ballot_w64(lane < gru.slots && mine_span.rows > 0 && mine_span.row0 == r);
      if (holds == 0) continue;
      const int slot = __builtin_ctzll(holds), at = __builtin_amdgcn_readlane(mine_span.start, slot);
      if (l16 == r) start = at, state_at = slot * (N >> 1) + gru_col;
    }
    if (lane < 32 && start > 0) old_state = *reinterpret_cast<const float4*>(gru.state + state_at + ((start - 1) & 1) * (N >> 2));
  }
  const bool staged = LINED && my_tiles > 1;
  // The columns of `count` tiles from `from` on, from half `half` of the out stage, by one wave.
  auto flush = [&](int from, int count, int half) {
    for (int e = lane; e < M * count; e += 64) {
      const int r = e / count, p = e - r * count, n = (tile0 + from + p) * R;
      bf16x8 v = lds_read_b128_at<0>(lds0 + S::OUT0 + half * S::OUT + (r * STRIP_OUT + p * R) * 2);
      lds_wait_for<0>(v);
      if (n < N) store_ragged(C + (size_t)r * N + n, __builtin_bit_cast(uint4, v), N - n);
    }
  };
  int item = 0;
  for (int t = 0; t < my_tiles; ++t) {
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < most; ++s) {
      if (s >= mine) continue;   // (the other waves' last strips)
      if (!SINGLE && !S::A_BY_LDS) a_from_memory(wave + W * s);
      if (STAGES == 1 || item + STAGES - 1 < items) {
        if (!MANY || item == 0) fetch(item + STAGES - 1);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<(STAGES - 1) * S::INST>();
      } else {
        wait_vmcnt<0>();
      }
      __builtin_amdgcn_sched_barrier(0);
      const unsigned at = lds0 + (unsigned)(held - lds) + item % STAGES * S::ITEM;
      if (!SINGLE && S::A_BY_LDS) a_from_lds(at);
      bf16x8 bf[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) bf[k] = lds_read_b128_at<0>((at + (SINGLE ? 0 : S::A_BYTES) + b_at) ^ (k << 6));
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (!SINGLE && S::A_BY_LDS) lds_wait_for<0>(af[0][k]);
        lds_wait_for<0>(bf[k]);
      }
      if (MANY && item + STAGES < items) {
        asm volatile("" ::: "memory");   // (behind the reads)
        __builtin_amdgcn_sched_barrier(0);
        fetch(item + STAGES);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[k], af[m][k], acc[m], 0, 0, 0);
      ++item;
    }
    // The waves' sums meet, through assembly: the compiler would wait for every strip in flight before each access to LDS.
    const int meeting = t / MEET;
    const unsigned sums0 = S::OVER_A ? (meeting & 1 ? lds0 : part0) : part0 + (meeting & 1) * S::PART;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      f32x4 v = acc[m];
      asm volatile("s_nop 15\n\ts_nop 3" : "+v"(v));   // (the matrix cores' results, which assembly is not waited for with)
      lds_write_b128(sums0 + t % MEET * S::PART + ((wave * MT + m) * 64 + lane) * 16, v);
    }
    if (MEET > 1 && (t + 1) % MEET != 0 && t + 1 < my_tiles) continue;
    lds_barrier();
    const int met = meeting * MEET;   // the first tile of this meeting; tile met + i's sums by wave (met + i) % 8
    if (LINED && t > 0 && t % GROUP == 0 && wave == (t + W / 2) % W) flush(t - GROUP, GROUP, (t / GROUP - 1) & 1);
    const int u = GRU ? t : met + ((wave - met) & (W - 1));
    const unsigned pa = sums0 + (u - met) * S::PART;
    // Lane (quad, l16) of the first two quads has columns 4 quad .. + 3 of row l16.
    const Joined joined = JOINS ? (t == 0 ? first_joined : (wave == t % W ? join_loads(t) : Joined{})) : Joined{};
    if ((GRU ? wave == 0 : u <= t) && lane < 32) {
      const int n = column_of(u) + quad * 4;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        bf16x8 p[W];
#pragma unroll
        for (int q = 0; q < W; ++q) p[q] = lds_read_b128_at<0>(pa + ((q * MT + m) * 64 + lane) * 16);
#pragma unroll
        for (int q = 0; q < W; ++q) lds_wait_for<0>(p[q]);
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < W; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] += __builtin_bit_cast(f32x4, p[q])[j];
        const int r = m * 16 + l16;
        if (JOINS) {
          if (r < M && n < N) {
            float h[4] = {joined.held.x, joined.held.y, joined.held.z, joined.held.w};
            const float g[4] = {bf16_lo(joined.gate.x), bf16_hi(joined.gate.x), bf16_lo(joined.gate.y), bf16_hi(joined.gate.y)};
            const float gb[4] = {bf16_lo(joined.gate_bias.x), bf16_hi(joined.gate_bias.x), bf16_lo(joined.gate_bias.y), bf16_hi(joined.gate_bias.y)};
            const float yb[4] = {bf16_lo(joined.y_bias.x), bf16_hi(joined.y_bias.x), bf16_lo(joined.y_bias.y), bf16_hi(joined.y_bias.y)};
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] += (round_bf16(v[j]) + yb[j]) * (1.0f / (1.0f + expf(-(g[j] + gb[j]))));
            *reinterpret_cast<float4*>(out.stream + (size_t)r * N + n) = make_float4(h[0], h[1], h[2], h[3]);
          }
        } else if (GRU && t < 3) {
          // (zx and ux are kept, rounded as they would be stored, until gx is there)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float rounded = round_bf16(v[j]);
            if (t == 0) gru_z[j] = rounded;
            else if (t == 1) gru_u[j] = rounded;
            else v[j] = rounded;
          }
          if (t == 2 && r < M && start >= 0) {
            const float zb[4] = {bf16_lo(z_bias.x), bf16_hi(z_bias.x), bf16_lo(z_bias.y), bf16_hi(z_bias.y)};
            const float ub[4] = {bf16_lo(x_bias.x), bf16_hi(x_bias.x), bf16_lo(x_bias.y), bf16_hi(x_bias.y)};
            float S[4] = {old_state.x, old_state.y, old_state.z, old_state.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float share = __builtin_amdgcn_rcpf(1.0f + __expf(-(gru_z[j] + zb[j]))), u = gru_u[j] + ub[j];
              const float c = u >= 0.f ? u + 0.5f : __builtin_amdgcn_rcpf(1.0f + __expf(-u));
              S[j] = fmaf(1.0f - share, S[j], share * c);
              v[j] = S[j] * (v[j] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[j])));
            }
            const int width = N >> 2, col = (int)blockIdx.x * R + quad * 4;
            *reinterpret_cast<float4*>(gru.state + state_at + (start & 1) * width) = make_float4(S[0], S[1], S[2], S[3]);
            *reinterpret_cast<uint2*>(gru.y + (size_t)r * width + col) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
          }
        } else if (staged) {
          const unsigned to = lds0 + S::OUT0 + (u / GROUP & 1) * S::OUT + (r * STRIP_OUT + u % GROUP * R + quad * 4) * 2;
          const uint64_t four = (uint64_t)pack_bf16(v[2], v[3]) << 32 | pack_bf16(v[0], v[1]);
          asm volatile("ds_write_b64 %0, %1" ::"v"(to), "v"(four) : "memory");
        } else if (r < M && n < N) {
          bf16_t* to = C + (size_t)r * N + n;
          if (n + 4 <= N) {
            store_loose(to, pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
          } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
              if (n + j < N) to[j] = f32_to_bf16(v[j]);
          }
        }
      }
    }
  }
  if (staged) {
    lds_barrier();
    const int from = (my_tiles - 1) / GROUP * GROUP;
    if (wave == 0) flush(from, my_tiles - from, from / GROUP & 1);
  }
  wait_vmcnt<0>();   // (loads of nothing may still be on their way into LDS)
}

constexpr int FEW_WAVES = 8, FEW_STEP = 64;   // K columns a wave takes at a time

// MODE: one tile of 16 rows of B a block, two of them (a tall B), or one of each of two matrices.
enum { FEW_ONE = 0, FEW_TWO = 1, FEW_GATED = 2 };
template <int MT, int MODE>
__global__ __launch_bounds__(FEW_WAVES * 64) void gemm_few_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                                  const bf16_t* __restrict__ B2, bf16_t* __restrict__ C, int M,
                                                                  int N, int K, int activation) {
  constexpr int MATS = MODE == FEW_ONE ? 1 : 2, DEPTH = MT == 1 ? 4 : (MT == 2 ? 2 : 1);
  constexpr bool GATED = MODE == FEW_GATED;
  __shared__ float4 part[FEW_WAVES][MATS][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, quad = lane >> 4;
  const int n0 = blockIdx.x * (MODE == FEW_TWO ? 32 : 16), steps = (K + FEW_WAVES * FEW_STEP - 1) / (FEW_WAVES * FEW_STEP);
  // Bounded buffers: a piece past K reads as zeros (of a row's own end, whatever follows it meets zeros of A).
  const __amdgpu_buffer_rsrc_t ab = bounded_bytes(A, M * K * 2);
  const size_t row = (size_t)min(n0 + l16, N - 1) * K;
  const bf16_t* w[MATS] = {B + row};
  if (MODE != FEW_ONE) w[MATS - 1] = GATED ? B2 + row : B + (size_t)min(n0 + 16 + l16, N - 1) * K;
  int a_row[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) a_row[m] = min(m * 16 + l16, M - 1) * K * 2;
  f32x4 acc[MATS][MT];
#pragma unroll
  for (int x = 0; x < MATS; ++x)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[x][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Piece {
    u32x4 b[MATS][2], a[MT][2];
  } held[DEPTH];
  auto fetch = [&](Piece& p, int step) {
    // (a lane takes 32 consecutive bytes of its row: which of the 64 columns meet in which product is free)
    const int k = (step * FEW_WAVES + wave) * FEW_STEP + quad * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kh = k + h * 8, in = min(kh, K - 8);   // past K: B's last piece, against zeros of A
#pragma unroll
      for (int x = 0; x < MATS; ++x) p.b[x][h] = *reinterpret_cast<const u32x4*>(w[x] + in);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        // A row past the last reads the last again (its results are not stored).
        const int past = (K - 1 - kh) >> 31 & 0x40000000;   // past K: outside the buffer
        p.a[m][h] = __builtin_amdgcn_raw_buffer_load_b128(ab, a_row[m] + 2 * kh + past, 0, 0);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    fetch(held[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  auto add = [&](const Piece& p) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int x = 0; x < MATS; ++x)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[x][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, p.b[x][h]), __builtin_bit_cast(bf16x8, p.a[m][h]), acc[x][m], 0, 0, 0);
  };
  for (int s = 0; s + DEPTH < steps; s += DEPTH) {   // (a step past the last adds zeros)
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      add(held[d]);
      fetch(held[d], s + d + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) add(held[d]);
#pragma unroll
  for (int x = 0; x < MATS; ++x)
#pragma unroll
    for (int m = 0; m < MT; ++m) part[wave][x][m][lane] = make_float4(acc[x][m][0], acc[x][m][1], acc[x][m][2], acc[x][m][3]);
  __syncthreads();
  // Lane (quad, l16) of a tile: columns n0 + quad * 4 .. + 3 of row m * 16 + l16.
  for (int e = threadIdx.x; e < MT * 64; e += FEW_WAVES * 64) {
    const int m = e >> 6, l = e & 63, r = m * 16 + (l & 15), n = n0 + (l >> 4) * 4;
    if (r >= M) continue;
    float v[MATS][4];
#pragma unroll
    for (int x = 0; x < MATS; ++x) {
      float4 sum = part[0][x][m][l];
#pragma unroll
      for (int q = 1; q < FEW_WAVES; ++q) {
        const float4 o = part[q][x][m][l];
        sum.x += o.x; sum.y += o.y; sum.z += o.z; sum.w += o.w;
      }
      v[x][0] = sum.x; v[x][1] = sum.y; v[x][2] = sum.z; v[x][3] = sum.w;
    }
    if (GATED) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[0][j] = round_bf16(gate_of(activation, round_bf16(v[0][j]))) * round_bf16(v[MATS - 1][j]);
    }
    bf16_t* to = C + (size_t)r * N + n;
#pragma unroll
    for (int x = 0; x < (MODE == FEW_TWO ? 2 : 1); ++x) {
      if (n + 16 * x + 4 <= N) {
        store_loose(to + 16 * x, pack_bf16(v[x][0], v[x][1]), pack_bf16(v[x][2], v[x][3]));
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (n + 16 * x + j < N) to[16 * x + j] = f32_to_bf16(v[x][j]);
      }
    }
  }
}

template <int MODE>
static int launch_gemm_few(const bf16_t* A, const bf16_t* B, const bf16_t* B2, bf16_t* C, int M, int N, int K, int activation, hipStream_t s) {
  const int per = MODE == FEW_TWO ? 32 : 16;
  const dim3 grid((N + per - 1) / per);
#define IRON_FEW(MT) \
  hipLaunchKernelGGL((gemm_few_kernel<MT, MODE>), grid, dim3(FEW_WAVES * 64), 0, s, A, B, B2, C, M, N, K, activation)
  if (M <= 16) IRON_FEW(1);
  else if (M <= 32) IRON_FEW(2);
  else IRON_FEW(4);
#undef IRON_FEW
  IRON_LAUNCH_CHECK();
}

template <int MT, int MA, bool SINGLE, int STAGES, bool STREAM, bool NORMED = false, bool JOINS = false, bool GRU = false,
          bool LATENT = false, bool MANY = false>
static int launch_gemm_strips(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, hipStream_t s, const StripsNorm& norm = {},
                              const StripsOut& out = {}, const StripsGru& gru = {}, const StripsLatent& latent = {}) {
  typedef Strips<MT, MA, SINGLE, STAGES, strips_meet<MT, MA, SINGLE, JOINS, GRU>()> S;
  static_assert(S::LDS <= 163840, "a CU's LDS");
  static LdsOptIn opt;
  auto kernel = &gemm_strips_kernel<MT, MA, SINGLE, STAGES, STREAM, NORMED, JOINS, GRU, LATENT, MANY>;
  const hipError_t e = opt.ensure(reinterpret_cast<const void*>(kernel), S::LDS);
  if (e != hipSuccess) {
    set_error("gemm_few: %s", hipGetErrorString(e));
    return (int)e;
  }
  const unsigned tiles = ((unsigned)N + STRIP_ROWS - 1) / STRIP_ROWS;
  unsigned blocks = GRU ? tiles / 4 : (tiles < STRIP_BLOCKS ? tiles : STRIP_BLOCKS);
  if (LATENT && blocks < (unsigned)M) blocks = M;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(STRIP_WAVES * 64), S::LDS, s, A, B, C, M, N, K, norm, out, gru, latent);
  IRON_LAUNCH_CHECK();
}

// Eight tiles a block and more: a stage is filled again as soon as it is in registers, not behind its tile's sums (8 rows, weights out of memory: 128256 x 2048
// 79.6 -> 78.6 us, 32000 x 1024 12.8 -> 12.5; but 10240 x 2048 with the norm 9.9 -> 10.4: there is little to overlap, and the memory takes longer with
// more out).
static bool strips_many(int N) { return N >= 8 * (int)STRIP_BLOCKS * STRIP_ROWS; }

// Which products go by strips, by what both kernels took over three hundred shapes with weights out of memory (us, gemm_few_kernel against strips).
// K up to eight strips: up to 16 rows of A (8 rows: 64 x 384 3.9 / 2.6, 1024 x 1024 4.7 / 2.9, 8192 x 2048 9.5 / 7.5, 16000 x 600 8.9 / 6.5, 128256 x 2048
// 95 / 77; one row: 2048 x 2048 4.4 / 3.5, 7159 x 2048 7.4 / 6.8), but not many rows of B that are a cache line or less (6 rows: 3440 x 40 2.95 / 3.15)
// nor, where they make two tiles a block of gemm_few_kernel's one round, rows of 1024 columns and more that straddle lines (of 120 shapes of K to 1280 strips take 0.86 of the other's
// time, and the same weights again 0.99, of 120 to 2047 0.85 and 1.04; 480 shapes short of 1024 0.81 to 0.95 and 0.88 to 0.96, none of them slower); up to 32 rows, whose
// sums take a second set of registers, over long rows
// that keep to their lines (32 rows: 1024 x 2048 7.9 / 6.3, 4160 x 2048 13.7 / 9.4; but 2400 x 192 3.9 / 5.3) or a B of 64 MB (20 rows: 128256 x 2048 128 / 82).
// A longer K: the strips of A that come with every tile cost as much as B's own.  Up to eight rows (2048 x 8192 13.5 / 8.6, 6000 x 6000 20.3 / 15.8,
// 4096 x 14336 24.7 / 22.7, 4560 x 4416 18.2 / 10.9; two tiles a block of one round too: 3904 x 3072 7.9 / 6.5, 3656 x 4160 10.4 / 8.2, and the same weights
// again, out of the last-level cache, 7.1 / 6.4 and 9.8 / 7.9; there rows that straddle lines from K = 8192 on: of 60 shapes of K to 4096 strips take 0.99 of the
// other's time, a third of them more, of 60 to 8192 0.95, and through the caches, as past it, the same weights again no less);
// up to 16 where a block has one tile (2048 x 8192 16.1 / 10.1) or three and more (4788 x 6848 28.9 / 20.1, 9762 x 9056 60.8 / 47.7).  With
// two tiles a block, or three and a half whose rows straddle lines, strips take the less of weights out of memory, but of the same weights again that is the other for
// a quarter of the sizes (on lines: K to 3072 0.82 and 0.95, to 4096 0.89 and 1.04, to 6144 0.87 and 0.97, past it 0.88 and 0.96; rows that straddle them 1.00 and 0.97, three and
// a half tiles 1.03 and 1.04): that kernel; more rows where that one's rows keep to their cache lines or are few (32 rows: 2048 x 4096
// 13.6 / 12.2, 1024 x 8192 24.7 / 19.2; 20 rows of 1960 x 6512 18.8 / 15.2, but the same weights again 12.1 / 13.7), and are not three or less (22 rows of 2 x 2688 5.9 / 6.6), past
// 32 rows from K = 2560 on, or 3072 of rows that straddle lines (38 rows of 9 x 2200 6.7 / 8.6, 51 of 32 x 2080 7.6 / 9.3; of 110 drawn ones short of there strips take 1.05 to 1.29 of
// the other's time).  The loads go past the caches except where a block has
// one tile over a long K (2048 x 8192, 8 rows: 9.3, past them 10.5; 4096 x 4096 10.1 and 9.4), or two of rows that straddle lines, or of more
// than eight rows any number of these (309 drawn ones: through them 0.93 of gemm_few_kernel's time and 0.91 with the same weights again, past them 0.92 and 1.15).
// Returns -1 where it is not for them.
static int strips_for(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, hipStream_t s) {
  const bool one_tile = N <= 256 * STRIP_ROWS, two_tiles = !one_tile && N <= 512 * STRIP_ROWS, on_lines = K % 64 == 0;
  if (K <= STRIP * STRIP_WAVES) {
    const bool long_rows = K >= 1600 && on_lines && !two_tiles, large = (long long)N * K >= (1 << 25) && (on_lines || K >= 1024);
    if (M > 32 || (M > 16 && !long_rows && !large)) return -1;
    if (M > 16) return launch_gemm_strips<2, 16, true, 2, true>(A, B, C, M, N, K, s);
    if (!one_tile && K < 64) return -1;
    if (two_tiles && !on_lines && K >= 1024) return -1;
    if (strips_many(N)) {
      if (M <= 8) return launch_gemm_strips<1, 8, true, 2, true, false, false, false, false, true>(A, B, C, M, N, K, s);
      return launch_gemm_strips<1, 16, true, 2, true, false, false, false, false, true>(A, B, C, M, N, K, s);
    }
    if (M <= 8) return launch_gemm_strips<1, 8, true, 2, true>(A, B, C, M, N, K, s);
    return launch_gemm_strips<1, 16, true, 2, true>(A, B, C, M, N, K, s);
  }
  if (M <= 8) {
    if (two_tiles && !on_lines && K < 8192) return -1;
    if (one_tile || (two_tiles && !on_lines)) return launch_gemm_strips<1, 8, false, 2, false>(A, B, C, M, N, K, s);
    return launch_gemm_strips<1, 8, false, 2, true>(A, B, C, M, N, K, s);
  }
  if (M <= 16) {
    if (one_tile) return launch_gemm_strips<1, 16, false, 1, false>(A, B, C, M, N, K, s);
    if (two_tiles || (!on_lines && N > 6144 && N < 8192 && K < 5632)) return -1;
    if (!on_lines) return launch_gemm_strips<1, 16, false, 1, false>(A, B, C, M, N, K, s);
    return launch_gemm_strips<1, 16, false, 1, true>(A, B, C, M, N, K, s);
  }
  if (!one_tile || N < STRIP_ROWS / 2 || (M > 32 && K < (on_lines ? 2560 : 3072))) return -1;
  if (!on_lines && N > 1280) return -1;
  return M <= 32 ? launch_gemm_strips<2, 16, false, 2, false>(A, B, C, M, N, K, s) : launch_gemm_strips<4, 16, false, 2, false>(A, B, C, M, N, K, s);
}

}  // namespace iron

using namespace iron;

extern "C" int iron_gemm_few_bf16(const uint16_t* A, const uint16_t* B, const uint16_t* B2, uint16_t* C, int M, int N, int K,
                                  int activation, void* stream) {
  IRON_REQUIRE(A && B && C, "gemm_few: null operand");
  IRON_REQUIRE(M > 0 && M <= 64 && N > 0, "gemm_few: M (%d) from 1 to 64, N (%d) positive", M, N);
  IRON_REQUIRE(K >= 8 && K % 8 == 0 && K <= (1 << 22), "gemm_few: K (%d) is a positive multiple of 8 up to 2^22", K);
  IRON_REQUIRE((((uintptr_t)A | (uintptr_t)B | (uintptr_t)B2) & 15) == 0, "gemm_few: operands must be 16-byte aligned");
  IRON_REQUIRE(B2 == nullptr || (activation >= 1 && activation <= 3), "gemm_few: activation (%d) is 1 (SiLU), 2 (GELU, tanh form) or 3 (ReLU)",
               activation);
  hipStream_t s = (hipStream_t)stream;
  if (B2 == nullptr) {
    const int done = strips_for(A, B, C, M, N, K, s);
    if (done >= 0) return done;
  }
  if (B2 != nullptr) return launch_gemm_few<FEW_GATED>(A, B, B2, C, M, N, K, activation, s);
  if (N >= 8192) return launch_gemm_few<FEW_TWO>(A, B, nullptr, C, M, N, K, 0, s);
  return launch_gemm_few<FEW_ONE>(A, B, nullptr, C, M, N, K, 0, s);
}

// x of a norm: float rows.
extern "C" int iron_norm_strips_bf16(const float* x, const uint16_t* gain, float eps, float unit, const uint16_t* W, uint16_t* y, int rows, int N, int K,
                                     void* stream) {
  IRON_REQUIRE(x && gain && W && y, "norm_strips: null operand");
  IRON_REQUIRE(rows > 0 && rows <= 8 && N > 0, "norm_strips: rows (%d) from 1 to 8, N (%d) positive", rows, N);
  IRON_REQUIRE(K >= 8 && K % 8 == 0 && K <= STRIP * STRIP_WAVES, "norm_strips: K (%d) is a positive multiple of 8 up to %d", K, STRIP * STRIP_WAVES);
  IRON_REQUIRE((((uintptr_t)x | (uintptr_t)gain | (uintptr_t)W) & 15) == 0, "norm_strips: operands must be 16-byte aligned");
  const StripsNorm norm{gain, eps, unit};
  if (strips_many(N))
    return launch_gemm_strips<1, 8, true, 2, true, true, false, false, false, true>(reinterpret_cast<const bf16_t*>(x), W, y, rows, N, K, (hipStream_t)stream, norm);
  return launch_gemm_strips<1, 8, true, 2, true, true>(reinterpret_cast<const bf16_t*>(x), W, y, rows, N, K, (hipStream_t)stream, norm);
}

extern "C" int iron_norm_gru_strips_bf16(const float* x, const uint16_t* gain, float eps, float unit, const uint16_t* W, const uint16_t* z_bias,
                                         const uint16_t* x_bias, float* state, const int* spans, uint16_t* packed, uint16_t* y, int slots, int rows,
                                         int width, int K, void* stream) {
  IRON_REQUIRE(x && gain && W && z_bias && x_bias && state && spans && packed && y, "norm_gru_strips: null operand");
  IRON_REQUIRE(rows > 0 && rows <= 8 && slots > 0 && slots <= 64, "norm_gru_strips: rows (%d) from 1 to 8, slots (%d) from 1 to 64", rows, slots);
  IRON_REQUIRE(width > 0 && width % 8 == 0 && width <= 8 * (int)STRIP_BLOCKS, "norm_gru_strips: width (%d) is a positive multiple of 8 up to %d", width,
               8 * (int)STRIP_BLOCKS);
  IRON_REQUIRE(K >= 8 && K % 8 == 0 && K <= STRIP * STRIP_WAVES, "norm_gru_strips: K (%d) is a positive multiple of 8 up to %d", K, STRIP * STRIP_WAVES);
  IRON_REQUIRE((((uintptr_t)x | (uintptr_t)gain | (uintptr_t)W | (uintptr_t)z_bias | (uintptr_t)x_bias | (uintptr_t)state | (uintptr_t)spans |
                 (uintptr_t)packed | (uintptr_t)y) & 15) == 0, "norm_gru_strips: operands must be 16-byte aligned");
  const StripsGru gru{z_bias, x_bias, state, spans, y, slots};
  return launch_gemm_strips<1, 8, true, 2, true, true, false, true>(reinterpret_cast<const bf16_t*>(x), W, packed, rows, 4 * width, K, (hipStream_t)stream,
                                                                    StripsNorm{gain, eps, unit}, {}, gru);
}

extern "C" int iron_latent_strips_bf16(const uint16_t* x, const uint16_t* q_gain, const uint16_t* c_gain, const float* angles, const int* spans,
                                       const uint16_t* W, uint16_t* q, uint16_t* latents, uint16_t* shared_keys, int slots, int rows, int N, int stride,
                                       int q_rank, int rank, int rot, int turned, int angle_rows, int ring, float eps, void* stream) {
  IRON_REQUIRE(x && q_gain && c_gain && spans && W && q && latents && (rot == 0 || shared_keys), "latent_strips: null operand");
  IRON_REQUIRE(rows > 0 && rows <= 8 && slots > 0 && slots <= 64 && N > 0, "latent_strips: rows (%d) from 1 to 8, slots (%d) from 1 to 64, N (%d) positive",
               rows, slots, N);
  IRON_REQUIRE(q_rank >= 8 && q_rank % 8 == 0 && q_rank <= STRIP * STRIP_WAVES, "latent_strips: the query latent (%d) is a positive multiple of 8 up to %d",
               q_rank, STRIP * STRIP_WAVES);
  IRON_REQUIRE(rank > 0 && rot >= 0 && ring > 0 && (rank | rot | stride) % 8 == 0 && rank <= 4096 && rot <= 4096 - rank,
               "latent_strips: latents of %d + %d columns, whole 16-byte pieces and 4096 together at the most, a ring (%d) of at least 1", rank, rot, ring);
  IRON_REQUIRE(stride >= q_rank + rank + rot && stride <= (1 << 22), "latent_strips: a row of %d holds no latents of %d and %d + %d", stride, q_rank, rank, rot);
  IRON_REQUIRE(turned >= 0 && turned <= rot && turned % 8 == 0 && (turned == 0 || (angles && angle_rows > 0)),
               "latent_strips: %d of %d shared columns turn, whole 16-byte pieces, by a table of %d rows", turned, rot, angle_rows);
  IRON_REQUIRE((((uintptr_t)x | (uintptr_t)q_gain | (uintptr_t)c_gain | (uintptr_t)angles | (uintptr_t)spans | (uintptr_t)W | (uintptr_t)latents |
                 (uintptr_t)shared_keys) & 15) == 0, "latent_strips: operands must be 16-byte aligned");
  const StripsLatent latent{LatentRow{q_gain, c_gain, angles, q_rank, eps}, LatentShape{slots, rows, 1, 1, rot, 1, rank, turned, angle_rows, 1, ring, 0, 1.f},
                            spans, latents, shared_keys, stride};
  return launch_gemm_strips<1, 8, true, 2, true, true, false, false, true>(x, W, q, rows, N, q_rank, (hipStream_t)stream, StripsNorm{q_gain, eps, 0.f}, {}, {},
                                                                           latent);
}

extern "C" int iron_gated_strips_bf16(const uint16_t* x, const uint16_t* W, const uint16_t* y_bias, const uint16_t* gate, int gate_stride,
                                      const uint16_t* gate_bias, float* stream_rows, int rows, int N, int K, void* stream) {
  IRON_REQUIRE(x && W && gate && gate_bias && stream_rows, "gated_strips: null operand");
  IRON_REQUIRE(rows > 0 && rows <= 8 && N > 0 && N % 4 == 0, "gated_strips: rows (%d) from 1 to 8, N (%d) a positive multiple of 4", rows, N);
  IRON_REQUIRE(K >= 8 && K % 8 == 0 && K <= (1 << 22), "gated_strips: K (%d) is a positive multiple of 8 up to 2^22", K);
  IRON_REQUIRE(gate_stride >= N && gate_stride % 4 == 0, "gated_strips: gates %d apart, a multiple of 4, for N (%d)", gate_stride, N);
  IRON_REQUIRE((((uintptr_t)x | (uintptr_t)W | (uintptr_t)stream_rows) & 15) == 0 && (((uintptr_t)y_bias | (uintptr_t)gate | (uintptr_t)gate_bias) & 7) == 0,
               "gated_strips: operands must be 16-byte aligned, a gate and the output's biases 8-byte");
  const StripsOut out{stream_rows, y_bias, gate, gate_bias, gate_stride};
  hipStream_t s = (hipStream_t)stream;
  if (K <= STRIP * STRIP_WAVES) return launch_gemm_strips<1, 8, true, 2, true, false, true>(x, W, nullptr, rows, N, K, s, {}, out);
  return launch_gemm_strips<1, 8, false, 2, false, false, true>(x, W, nullptr, rows, N, K, s, {}, out);
}
