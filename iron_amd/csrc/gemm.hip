// GEMM: C = A @ B in bf16 on the MFMA matrix cores, f32 accumulation, one rounding.
//
// Two families of kernels.  The general one (gemm_kernel, first below) takes every shape and
// option: a block of 4 waves computes a BM x BN tile of C; per 64-wide K step it stages a BM x 64
// tile of A and a BN x 64 tile of B in LDS through registers (both K-contiguous, rows padded to
// 72 elements so the 16-byte fragment reads of 32 consecutive rows fall in distinct banks),
// double-buffered; a wave owns a (BM/WM) x (BN/WN) sub-tile as 32x32x16 MFMA tiles; B as (K,N) is
// transposed on its way into LDS (a thread loads a 4(k) x 8(n) patch and writes eight 8-byte
// k-runs).  The fast ones (K at least 64, no bound on K) feed LDS straight from global memory
// and come in tiles from 32 x 32 to 256 x 256, each described where it stands: gemm_plan says which a product takes,
// by small_tiles' and BIG_PRICES; a launch under a row bound chooses by ROWS_PRICES, a gated pair by PAIR_PRICES.
//
// For a row-major C the MFMA is issued with the operands swapped (B tile as the "A" operand), so a
// lane ends up holding 4 consecutive columns of one row of C and stores them as 8 bytes.
#include "../../include/iron_hip.h"
#include "common.h"
#include "grouped.h"

#include <type_traits>


namespace iron {

constexpr int BK = 64;
constexpr int LDK = BK + 8;  // padded LDS row, in elements

// Zero the elements of an 8-element piece from index keep on.
__device__ __forceinline__ uint4 keep_first(uint4 v, int keep) {
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (2 * i >= keep) w[i] = 0;
    else if (2 * i + 1 >= keep) w[i] &= 0xffffu;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

template <int BM, int BN, int WM, int WN, bool B_NK, bool C_NM>
__global__ __launch_bounds__(256) void gemm_kernel(const bf16_t* __restrict__ A,
                                                   const bf16_t* __restrict__ B,
                                                   bf16_t* __restrict__ C, int M, int N, int K,
                                                   const int* __restrict__ valid,
                                                   const int* __restrict__ valid_k, int tiles_m,
                                                   int tiles_n) {
  static_assert(WM * WN == 4, "4 waves");
  constexpr int TM = BM / WM / 32;  // MFMA tiles per wave along M
  constexpr int TN = BN / WN / 32;
  constexpr int A_PIECES = BM * (BK / 8) / 256;  // 16-byte pieces a thread loads of A
  constexpr int B_PIECES = BN * (BK / 8) / 256;

  extern __shared__ __align__(16) bf16_t smem[];
  bf16_t* As = smem;                  // [2][BM][LDK]
  bf16_t* Bs = smem + 2 * BM * LDK;   // [2][BN][LDK]

  const int Mv = bound_or(valid, M);
  const int Kv = bound_or(valid_k, K);

  // Tile order: consecutive blocks share a band of 8 tile rows, so the blocks
  // resident together re-read few panels of A and B from L2.
  int tm, tn;
  {
    const int bid = blockIdx.x;
    constexpr int BAND = 8;
    const int per_band = BAND * tiles_n;
    const int band = bid / per_band;
    const int first = band * BAND;
    const int height = min(BAND, tiles_m - first);
    const int in_band = bid - band * per_band;
    tm = first + in_band % height;
    tn = in_band / height;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  if (m0 >= Mv) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;

  // (K,N) B: a pass covers 256/(BN/8) groups of 4 k rows; BK/4 groups make a tile.
  constexpr int B_NC = BN / 8;
  constexpr int B_KG = 256 / B_NC;
  constexpr int B_PASSES = (BK / 4 + B_KG - 1) / B_KG;
  uint4 a_reg[A_PIECES];
  uint4 b_reg[B_NK ? B_PIECES : 4 * B_PASSES];

  auto load_a = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_PIECES; ++i) {
      const int p = tid + i * 256;
      const int row = p >> 3, kc = (p & 7) * 8;
      const int gm = m0 + row, gk = k0 + kc;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (gm < Mv && gk < Kv) {
        v = *reinterpret_cast<const uint4*>(A + (size_t)gm * K + gk);
        if (gk + 8 > Kv) v = keep_first(v, Kv - gk);
      }
      a_reg[i] = v;
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_PIECES; ++i) {
      const int p = tid + i * 256;
      const int row = p >> 3, kc = (p & 7) * 8;
      *reinterpret_cast<uint4*>(As + (buf * BM + row) * LDK + kc) = a_reg[i];
    }
  };
  auto load_b = [&](int k0) {
    if constexpr (B_NK) {
#pragma unroll
      for (int i = 0; i < B_PIECES; ++i) {
        const int p = tid + i * 256;
        const int row = p >> 3, kc = (p & 7) * 8;
        const int gn = n0 + row, gk = k0 + kc;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (gn < N && gk < Kv) {
          v = *reinterpret_cast<const uint4*>(B + (size_t)gn * K + gk);
          if (gk + 8 > Kv) v = keep_first(v, Kv - gk);
        }
        b_reg[i] = v;
      }
    } else {
      // A thread takes 4 consecutive k rows of one 8-column strip per pass.
#pragma unroll
      for (int j = 0; j < B_PASSES; ++j) {
        const int strip = tid % B_NC;
        const int kg = tid / B_NC + j * B_KG;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gk = k0 + kg * 4 + r, gn = n0 + strip * 8;
          uint4 v = make_uint4(0, 0, 0, 0);
          if (kg < BK / 4 && gk < Kv && gn < N) {
            if (gn + 8 <= N) {
              v = *reinterpret_cast<const uint4*>(B + (size_t)gk * N + gn);
            } else {
              // N is not a multiple of 8 here only if the caller passed such an N;
              // read the columns that exist one by one.
              uint32_t w[4] = {0, 0, 0, 0};
              for (int c = 0; c < N - gn; ++c)
                w[c >> 1] |= (uint32_t)B[(size_t)gk * N + gn + c] << (16 * (c & 1));
              v = make_uint4(w[0], w[1], w[2], w[3]);
            }
          }
          b_reg[j * 4 + r] = v;
        }
      }
    }
  };
  auto store_b = [&](int buf) {
    if constexpr (B_NK) {
#pragma unroll
      for (int i = 0; i < B_PIECES; ++i) {
        const int p = tid + i * 256;
        const int row = p >> 3, kc = (p & 7) * 8;
        *reinterpret_cast<uint4*>(Bs + (buf * BN + row) * LDK + kc) = b_reg[i];
      }
    } else {
#pragma unroll
      for (int j = 0; j < B_PASSES; ++j) {
        const int strip = tid % B_NC;
        const int kg = tid / B_NC + j * B_KG;
        if (kg >= BK / 4) continue;
        const uint4 r0 = b_reg[j * 4 + 0], r1 = b_reg[j * 4 + 1], r2 = b_reg[j * 4 + 2],
                    r3 = b_reg[j * 4 + 3];
        const uint32_t w0[4] = {r0.x, r0.y, r0.z, r0.w}, w1[4] = {r1.x, r1.y, r1.z, r1.w},
                       w2[4] = {r2.x, r2.y, r2.z, r2.w}, w3[4] = {r3.x, r3.y, r3.z, r3.w};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          // Column c of the strip: its 4 k values, k ascending.
          const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
          uint2 out;
          out.x = __builtin_amdgcn_perm(w1[c >> 1], w0[c >> 1], sel);
          out.y = __builtin_amdgcn_perm(w3[c >> 1], w2[c >> 1], sel);
          *reinterpret_cast<uint2*>(Bs + (buf * BN + strip * 8 + c) * LDK + kg * 4) = out;
        }
      }
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int nk = (Kv + BK - 1) / BK;
  if (nk > 0) {
    load_a(0);
    load_b(0);
    store_a(0);
    store_b(0);
  }
  __syncthreads();

  const int frag_row = lane & 31;
  const int frag_k = (lane >> 5) * 8;

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) {
      load_a((kt + 1) * BK);
      load_b((kt + 1) * BK);
    }
    const bf16_t* Ab = As + (cur * BM + wm * (BM / WM) + frag_row) * LDK + frag_k;
    const bf16_t* Bb = Bs + (cur * BN + wn * (BN / WN) + frag_row) * LDK + frag_k;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *reinterpret_cast<const bf16x8*>(Ab + i * 32 * LDK + ks * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bfr[j] = *reinterpret_cast<const bf16x8*>(Bb + j * 32 * LDK + ks * 16);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (C_NM)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
        }
    }
    if (kt + 1 < nk) {
      store_a(cur ^ 1);
      store_b(cur ^ 1);
    }
    __syncthreads();
  }

  // Epilogue.  Swapped operands (row-major C): lane holds row m = lane%32 and the
  // 4-column runs n = 8*q + 4*(lane/32) + 0..3, q = 0..3.  Unswapped (C as (N,M)):
  // lane holds column n = lane%32 and the 4-row runs of m.
  const int hi = (lane >> 5) * 4;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int mb = m0 + wm * (BM / WM) + i * 32;
      const int nb = n0 + wn * (BN / WN) + j * 32;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v0 = acc[i][j][4 * q + 0], v1 = acc[i][j][4 * q + 1],
                    v2 = acc[i][j][4 * q + 2], v3 = acc[i][j][4 * q + 3];
        if constexpr (!C_NM) {
          const int m = mb + frag_row, n = nb + 8 * q + hi;
          if (m >= Mv || n >= N) continue;
          bf16_t* p = C + (size_t)m * N + n;
          if (n + 4 <= N) {
            store_loose(p, pack_bf16(v0, v1), pack_bf16(v2, v3));
          } else {
            const float v[4] = {v0, v1, v2, v3};
#pragma unroll
            for (int e = 0; e < 4; ++e)   // (constant indices: a runtime trip count puts the array in scratch memory)
              if (n + e < N) p[e] = f32_to_bf16(v[e]);
          }
        } else {
          const int n = nb + frag_row, m = mb + 8 * q + hi;
          if (n >= N || m >= Mv) continue;
          bf16_t* p = C + (size_t)n * M + m;
          if (m + 4 <= Mv) {
            store_loose(p, pack_bf16(v0, v1), pack_bf16(v2, v3));
          } else {
            const float v[4] = {v0, v1, v2, v3};
            for (int e = 0; e < 4 && m + e < Mv; ++e) p[e] = f32_to_bf16(v[e]);
          }
        }
      }
    }
}


// ---------------------------------------------------------------------------
// Fast paths: A (M,K) K-contiguous, K a multiple of 8 from 64 on, C (M,N) or, of B (K,N), (N,M).
//
// Tiles stream global -> LDS directly (buffer loads with the LDS bit: no VGPR staging, and the
// L2 -> CU path delivers more per clock to LDS than to registers), several stages deep.  A wave
// instruction moves 8 rows x 128 B; the 16-byte chunk a lane fetches is XOR-swizzled by its row
// ((row >> 1) & 7) so the fragment reads of 16 consecutive rows fall in distinct bank groups
// although LDS rows are unpadded.  The stage barrier is a bare s_barrier: the fence
// __syncthreads() carries would wait for every outstanding load (vmcnt(0)) and drain the
// prefetch; each wave instead waits until only the younger stages are in flight.
constexpr int NT_STAGES = 4;
constexpr int PAIR_STAGES = 3;   // of the two-product body: 48 KB each

// B_KN (128 x 128 and 256 x 256 tiles): B is (K,N) row-major.  Its tile lands in LDS as stored, a
// row a k (a wave instruction moves 4 k-rows x 256 B, or 2 x 512 B; chunks swizzled by the row so
// that the four rows of a 16-lane group, and the groups of a pass, lie in different banks), and
// the fragments are fetched with the transposing LDS read (ds_read_b64_tr_b16): within 16 lanes,
// lane i points at 4 consecutive n of row k0 + i/4 and receives k0..k0+3 of column n0 + i%16.
// QKV: one launch for a prompt chunk's three projections and the rotation of two of them.  B, C and
// N then stand for q's weight (N,K), output and width; `qkv` brings k's and v's (each kv_n wide,
// widths multiples of the 128-column tile) and the chunk's angle rows (M, 64; cos and sin
// interleaved).  A block's tile column picks its matrix.  With 64-wide heads a wave's 64 columns are
// one head whose two halves are its two accumulator tiles, so q and k are rotated in registers:
// rounded to bf16 as the projection would store them, turned (two halves), rounded again.
struct QkvTail {
  const bf16_t* Bk;
  const bf16_t* Bv;
  bf16_t* Ck;
  bf16_t* Cv;
  const bf16_t* angles;
  int kv_n;
  // Not of the fused projections: a plain product's epilogue, C = bf16(residual_scale * bf16(A B) + residual)
  // (one fused multiply-add; residual (M, N) like C), when residual is not NULL.
  const bf16_t* residual;
  float residual_scale;
  // ... or, with gated set, C = bf16(bf16(act(residual)) * bf16(A B)): `residual` then holds a gated
  // feed-forward's other product, and this one leaves as the activated gate times it (1: SiLU,
  // 2: GELU by its tanh form).
  int gated;
  // Of the fused projections again: Ck and Cv are KV caches of kv_rows rows (a row kv_n wide, as the
  // projections write one), and the chunk's rows go to rows *kv_row0 on, when kv_row0 is not NULL.
  const int* kv_row0;
  int kv_rows;
  // Of a plain product on the 128 x 128 tiles, one block of several that share a tile's K: columns
  // k_begin .. k_begin + k_len of A and B (k_len 0: all of them), the float32 sums left at `partial`
  // (an (M, N) array of this slice's) instead of C; tile_plus1: the tile's number + 1 where the
  // kernel deals tiles itself instead of by the block's id.
  int k_begin, k_len, tile_plus1;
  float* partial;
  // ... or the block's 128 x 128 float32 sums whole, as C's rows lie, at `tile_sums` (with C (N,M): C's).
  float* tile_sums;
};


// The k and v outputs moved to the chunk's rows of their caches.  The first row is held where the
// rows under the bound still end inside the cache, whatever the word holds.
__device__ __forceinline__ void to_cache_rows(QkvTail& t, const int* __restrict__ valid, int M) {
  if (t.kv_row0 == nullptr) return;
  const int rows = bound_or(valid, M);
  const int first = max(0, min(*t.kv_row0, t.kv_rows - rows));
  t.Ck += (size_t)first * t.kv_n;
  t.Cv += (size_t)first * t.kv_n;
}

// Which tile a block computes.  Blocks are dispatched in id order and dealt round-robin over the 8
// XCDs, each with an L2 of its own, so the order is chosen for what an XCD's blocks share:
// `patched` (whole 8 x 4-tile patches, a multiple of 8 of them): an XCD owns patches, whose A and B
// panels it re-reads from its own L2.  Otherwise the tiles in bands of 8 tile rows, a band's columns one after the other, and an XCD
// owns an eighth of that order in one piece: the weight tile that its blocks share crosses HBM once instead of once an XCD
// (against tile rows dealt round-robin: 7058 x 12872 x 792 174 -> 157 us, 941 x 9386 x 5296 121 -> 112, 181 x 10780 x 272 8.5 -> 7.5).  A matrix more than
// twice as tall as wide goes by columns for rows (2056 x 713 x 1136 12.9 -> 11.5), and so does one of two bands or more that is more than a round of tiles: the tiles of
// the last round, which few CUs share, then meet weights that the round before has read, where by rows they are the first to ask memory for theirs (K from 1024 on, weights out of
// memory, 300 to 420 tiles: 2048 x 2560 x 8448 with the next norm dealt round-robin 142 us, by rows 163, by columns 140; over 870 drawn products of 128 x 128 tiles by columns 0.96
// of by rows, with the same weights again 1.00).
__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n, int patched, int& tm, int& tn) {
  const int xcd = bid & 7, loc = bid >> 3;
  if (patched) {
    const int patch = (loc >> 5) * 8 + xcd, within = loc & 31;
    const int patches_n = tiles_n >> 2;
    tm = (patch / patches_n) * 8 + (within & 7);
    tn = (patch % patches_n) * 4 + (within >> 3);
  } else {
    const int tiles = tiles_m * tiles_n, at = xcd * (tiles >> 3) + min(xcd, tiles & 7) + loc;
    const bool tall = tiles_m > 2 * tiles_n || (tiles_m >= 12 && tiles > 288);
    const int across = tall ? tiles_n : tiles_m, along = tall ? tiles_m : tiles_n;
    // (eight by four tiles are an XCD's CUs; up to three left over join the last band)
    const int band = min(at / (8 * along), max(1, (across + 4) >> 3) - 1), first = band * 8;
    const int width = first + 12 > across ? across - first : 8, in_band = at - first * along;
    const int l = in_band / width, c = first + in_band - l * width;
    tm = tall ? l : c;
    tn = tall ? c : l;
  }
}

// The same under a row bound read on the device: an order that is not patched is that of the live tile rows alone, or the few
// there are would be a few XCDs'; so is one whose patches of eight tile rows would be cut (3072 x 3072 columns and K, 300 rows 33.4 -> 18.6 us).
// False: the block has none.
__device__ __forceinline__ bool live_tile(int bid, int tiles_m, int tiles_n, int patched, int live_m, int& tm, int& tn) {
  if (live_m < 8) patched = 0;
  if (!patched) {
    tiles_m = min(tiles_m, live_m);
    if (bid >= tiles_m * tiles_n) return false;
  }
  tile_of_block(bid, tiles_m, tiles_n, patched, tm, tn);
  return true;
}

// The epilogue over a piece of a row: x, the product as it would be stored, and r, the second operand's piece, become
// scale * x + r, or bf16(act(r)) * x.  The kind is asked once a piece: asked an element, every branch was
// a wait (gated product 2048 x 2048 x 2048 27.9 -> 22.7 us, residual sum 23.0 -> 21.8).
template <int COUNT>
__device__ __forceinline__ void tail_of(const QkvTail& qkv, float (&x)[COUNT], const float (&r)[COUNT]) {
  auto gate = [&](auto kind) {
#pragma unroll
    for (int e = 0; e < COUNT; ++e) x[e] = round_bf16(gate_of(decltype(kind)::value, r[e])) * x[e];
  };
  if (qkv.gated == 0) {
#pragma unroll
    for (int e = 0; e < COUNT; ++e) x[e] = fmaf(qkv.residual_scale, x[e], r[e]);
  } else if (qkv.gated == 1) {
    gate(std::integral_constant<int, 1>{});
  } else if (qkv.gated == 2) {
    gate(std::integral_constant<int, 2>{});
  } else {
    gate(std::integral_constant<int, 3>{});
  }
}

// A K that is no whole number of stages: the FIRST stage is the short one.  Stage kt covers k from kt BK
// - pad, so the loop and its wait counts are the same for every K, and only the loads of stage 0, before
// the loop, ask where a lane's piece lies: those below k = 0 go to an offset past every buffer's
// end, for which the load brings zeros into LDS, for A and B alike (0 x 0 adds nothing, whatever lies
// before the row).  K a multiple of 8, at least BK.
__host__ __device__ __forceinline__ int k_pad(int K) { return (BK - K % BK) % BK; }
constexpr int NOWHERE = (int)0x80000000u;   // past stage_rows' 2^31 - 1 bytes, whatever scalar offset is added

// 64 x 64 tiles, B as (N,K), for problems -- or row bounds -- whose 128 x 128 tiles would leave CUs
// idle (k/v projections, short chunks): the direct-to-LDS pipeline of the 128 x 128 kernel below
// (buffer loads, XOR-swizzled chunks) with a wave owning 2 x 2 tiles of 16x16x32 MFMAs.  A stage is eight
// MFMAs of a wave, far less than an LDS read takes to return, so the fragments of a WHOLE stage
// are read one stage ahead into a second register set: at the top of stage kt the stage's one
// barrier (stage kt+1 has landed in every wave, and nobody reads stage kt-1 any more) behind its first two
// MFMAs, then, between the others, the eight fragment reads of stage kt+1 and the loads of stage kt+STAGES-1 into stage
// kt-1's buffer.  Reading a k-step ahead, as the larger tiles do, left every MFMA
// waiting for its operands: 600 cycles a stage.  STAGES = 4 (64 KB: a CU holds two blocks) where
// the tiles outnumber the CUs, 8 (128 KB, more loads in flight) where a CU has one block anyway.
// An element's sum is the same chain of 32-wide k-steps as in the 128 x 128 and the 256 x 256 tiles: where a row bound chooses
// the tile, a row's products are the same bits whatever rows share the launch.
// `qkv` carries only the optional residual epilogue here, or (QKV) the fused projections'.  WM x 4 / WM waves of MI x NJ tiles: <2, 2, 2> are 64 x 64, <4>
// 128 x 64.  PAIR: both first products of a gated feed-forward, 32 columns of each (`qkv` says the gate's kind).  B_KN: B is (K,N), 64 columns a tile; C_NM: and C (N,M).
// A few rows' tiles wait for what a CU can draw of operands that are 128 bytes of a row here and there, some 60 GB/s of weights out of memory, whatever the
// stages in flight (8 or 10 of 16 KB the same): where the tiles leave CUs without one, smaller tiles have more CUs draw less each.  2048 columns over 2048
// with a residual, us by 64 x 64 tiles, 64 x 32 <1, 4, 2> and 32 x 32 <1, 2, 1>: 12.5 / 10.4 / 8.6 (256 blocks: up to 640, 256 and 128 rows); over 8192
// 36 / 28.7 / 21.3.
template <int STAGES, bool PAIR = false, int MI = 2, int WM = 2, int NJ = 2, bool QKV = false, bool B_KN = false, bool C_NM = false>
__device__ __forceinline__ void gemm_nt64_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                               bf16_t* __restrict__ C, int M, int N, int K,
                                               int Mv, int tiles_m, int tiles_n,
                                               int patched, const QkvTail& qkv,
                                               const bf16_t* __restrict__ up = nullptr, bf16_t* __restrict__ gate_out = nullptr) {
  constexpr int NT_BM = 16 * MI * WM, NT_BN = 16 * NJ * (4 / WM);
  constexpr int NT_A_BYTES = NT_BM * BK * 2, NT_STAGE_BYTES = (NT_BM + NT_BN) * BK * 2;
  constexpr int INST = NT_BM / 8 / 4, B_INST = NT_BN / 8 / 4;  // 1 KB loads of A and of B a wave issues per stage
  constexpr int LOADS = INST + B_INST, PER = (LOADS + 2 * MI - 1) / (2 * MI);   // PER: loads behind every second MFMA
  static_assert(BK == 64 && STAGES >= 4 && ((MI == 2 && WM == 2 && NJ == 2) || !PAIR) && (!QKV || (NJ == 2 && NT_BN <= 64)) &&
                    (!B_KN || (NT_BN == 64 && NJ == 2 && !PAIR && !QKV)) && (B_KN || !C_NM),
                "two 32-wide k-steps a stage");
  extern __shared__ __align__(16) char smem_nt[];

  int tm, tn;
  if (!live_tile(blockIdx.x, tiles_m, tiles_n, patched, (Mv + NT_BM - 1) / NT_BM, tm, tn)) return;
  const int m0 = tm * NT_BM, n0 = QKV ? 0 : (B_KN ? max(min(tn * NT_BN, N - NT_BN), 0) : tn * (PAIR ? NT_BN / 2 : NT_BN));
  if (m0 >= Mv) return;
  // QKV: a tile is columns first .. + NT_BN / 2 and 32 + first .. of one 64-wide head of the list q | k | v (C's rows of N columns hold q), a wave's two
  // accumulators the two halves that RoPE turns.
  const int q_heads = N >> 6, kv_heads = QKV ? qkv.kv_n >> 6 : 0, head = tn / (64 / NT_BN), first = tn % (64 / NT_BN) * (NT_BN / 2);
  const int which = !QKV || head < q_heads ? 0 : (head < q_heads + kv_heads ? 1 : 2), own = head - (which == 0 ? 0 : q_heads + (which - 1) * kv_heads);
  if constexpr (QKV) B = (which == 0 ? B : (which == 1 ? qkv.Bk : qkv.Bv)) + (size_t)own * 64 * K;

  // The wave's number is uniform, so what depends on it (LDS destinations, the rows it loads) stays
  // in scalar registers.
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / (4 / WM), wn = wave % (4 / WM);
  const int lrow = lane >> 3, pch = lane & 7;
  int a_voff[4], b_voff[2], a_head[4], b_head[2];
  // (K,N): a row of 64 columns is half the banks; what sixteen lanes' transposing read takes, four rows of 32 bytes, and its neighbours' eight rows on meet none twice.
  auto kn_swizzle = [](int k) { return (k & 2) | ((k >> 1) & 4); };
#pragma unroll
  for (int i = 0; i < INST; ++i) {
    const int r = (wave * INST + i) * 8 + lrow;
    const int lch = pch ^ ((r >> 1) & 7);
    a_head[i] = lch * 8;
    // Rows past the last live one bring zeros, without traffic (what they produce is never stored): a CU's few rows wait for what it draws, and a tile's dead rows
    // were as much of that as live ones.  A 1B decoder's prompt, us, by dead rows read and not: 2 rows 1286 / 1208, 29 1306 / 1243, 513 2511 / 2281, 900 3034 / 2807.
    a_voff[i] = m0 + r < Mv ? (r * K + lch * 8) * 2 : NOWHERE;
  }
#pragma unroll
  for (int i = 0; i < B_INST; ++i) {
    const int r = (wave * B_INST + i) * 8 + lrow;
    if constexpr (B_KN) {   // as stored, a row a k: 64 columns, the last tile moved back to end at N
      b_head[i] = r;
      b_voff[i] = (int)(((size_t)r * N + min((pch ^ kn_swizzle(r)) * 8, N - 8 - n0)) * 2);
      continue;
    }
    b_head[i] = (pch ^ ((r >> 1) & 7)) * 8;
    b_voff[i] = (int)(((size_t)(QKV ? first + (r >> 4 & 1) * 32 + (r >> 5) * 16 + (r & 15) : min(n0 + (PAIR ? r % (NT_BN / 2) : r), N - 1) - n0) * K + b_head[i]) * 2);
  }
  const int pad = k_pad(K);
  const bf16_t* a_tile = A + (size_t)m0 * K - pad;
  // (PAIR: the tile's first 32 columns are the gate's, which waves 0 and 1 load and the waves wn = 0 compute, the rest the up projection's)
  const bf16_t* b_tile = B_KN ? B + n0 - (ptrdiff_t)pad * N : (PAIR && wave >= 2 ? up : B) + (size_t)n0 * K - pad;
  const int b_first = NT_A_BYTES + wave * B_INST * 1024;   // where a wave's part of B begins in a stage
  // One load of the 2*INST a wave issues per stage (A's first, then B's).
  auto issue_one = [&](char* st, int kt, int idx, bool head) {
    const int k0 = kt * BK;
    if (idx < INST) {
      const __amdgpu_buffer_rsrc_t rows = stage_rows(a_tile + k0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, IRON_LDS_PTR(st + (wave * INST + idx) * 1024), 16,
                                               head && a_head[idx] < pad ? NOWHERE : a_voff[idx], 0, 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t rows = stage_rows(b_tile + (B_KN ? (size_t)k0 * N : (size_t)k0));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, IRON_LDS_PTR(st + b_first + (idx - INST) * 1024),
                                               16, head && b_head[idx - INST] < pad ? NOWHERE : b_voff[idx - INST], 0, 0, 0);
    }
  };

  f32x4 acc[MI][NJ];
#pragma unroll
  for (int t = 0; t < NJ * MI; ++t) acc[t / NJ][t % NJ] = f32x4{0.f, 0.f, 0.f, 0.f};

  // acc[i][j][e]: row 16 i + fr of the wave's 16 MI x 16 NJ, column 16 j + 4 kq + e.
  const int fr = lane & 15, kq = lane >> 4;
  const int mb = m0 + wm * (16 * MI) + fr, nb = n0 + (PAIR ? 0 : wn * (16 * NJ)) + 4 * kq;
  // A residual's pieces this lane will add in the epilogue are requested now, so that their
  // latency passes under the whole product instead of at its end (N a multiple of 4: 8-byte pieces).
  uint2 res[MI][NJ];
  const bool res_ahead = !PAIR && !QKV && qkv.residual != nullptr && (N & 3) == 0;
  if (res_ahead) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        res[i][j] = *reinterpret_cast<const uint2*>(qkv.residual + (size_t)min(mb + 16 * i, M - 1) * N + min(nb + 16 * j, N - 4));
  }

  const int nk = (K + pad) / BK;
  // Always STAGES-1 stages in flight before the loop (short K repeats its last stage), so the
  // loop's wait counts hold from the first iteration.
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
    for (int idx = 0; idx < LOADS; ++idx) issue_one(smem_nt + s * NT_STAGE_BYTES, min(s, nk - 1), idx, s == 0);

  // Fragments: lane -> row fr of a 16-row tile, 16-byte chunk kq of the k-step's four.
  const int a_off = (wm * (16 * MI) + fr) * 128, b_off = NT_A_BYTES + (wn * (16 * NJ) + fr) * 128, swz = (fr >> 1) & 7;
  auto a_frag = [&](const char* st, int ks, int i) {
    return *reinterpret_cast<const bf16x8*>(st + a_off + i * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };
  auto b_frag = [&](const char* st, int ks, int j) {
    return *reinterpret_cast<const bf16x8*>(st + b_off + j * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };

  wait_vmcnt<(STAGES - 2) * LOADS>();   // stage 0 has landed once only the younger ones are out
  block_barrier();
  bf16x8 af[2][2][MI], bfr[2][2][NJ];   // [stage parity][k-step][tile]
  // (K,N): reads that the compiler does not count, A's too, so that every wait is this code's own (as in the 128 x 128 tiles).
  TrFrag tfb[2][2][NJ];
  const unsigned lds_base = (unsigned)(size_t)IRON_LDS_PTR(smem_nt);
  unsigned a_lane[2], kn_lane[NJ];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a_lane[ks] = lds_base + a_off + (((ks * 4 + kq) ^ swz) << 4);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int k = 8 * kq + ((lane & 15) >> 2), n = wn * (16 * NJ) + j * 16 + 4 * (lane & 3);
    kn_lane[j] = lds_base + NT_A_BYTES + k * 128 + (((n >> 3) ^ kn_swizzle(k)) << 4) + ((n & 4) << 1);
  }
  auto kn_reads = [&](unsigned at, int parity, int ks, int i) {   // at: the stage's place; what slot (ks, i) reads
    if (i == 0) af[parity][ks][0] = lds_read_b128_at<0>(a_lane[ks] + at);
    else af[parity][ks][MI - 1] = lds_read_b128_at<(MI - 1) * 16 * 128>(a_lane[ks] + at);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (j % MI == i) {
        TrFrag& t = tfb[parity][ks][j];
        if (ks == 0) {
          t.lo = lds_read_tr16_at<0>(kn_lane[j] + at);
          t.hi = lds_read_tr16_at<4 * 128>(kn_lane[j] + at);
        } else {
          t.lo = lds_read_tr16_at<32 * 128>(kn_lane[j] + at);
          t.hi = lds_read_tr16_at<36 * 128>(kn_lane[j] + at);
        }
      }
  };
  // A k-step's fragments are there once at most the next k-step's are outstanding.
  auto kn_wait = [&](int parity, int ks) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(tfb[parity][ks][0].lo), "+v"(tfb[parity][ks][0].hi), "+v"(tfb[parity][ks][NJ - 1].lo), "+v"(tfb[parity][ks][NJ - 1].hi) : "n"(MI + 2 * NJ));
#pragma unroll
    for (int i = 0; i < MI; ++i) lds_wait_for<MI + 2 * NJ>(af[parity][ks][i]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) bfr[parity][ks][j] = tr_join(tfb[parity][ks][j]);
  };
  static_assert(!B_KN || MI <= 2, "two rows of tiles a wave");
#pragma unroll
  for (int t = 0; t < 2 * MI; ++t) {
    if constexpr (B_KN) {
      kn_reads(0, 0, t / MI, t % MI);
      continue;
    }
    af[0][t / MI][t % MI] = a_frag(smem_nt, t / MI, t % MI);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (j % MI == t % MI) bfr[0][t / MI][j] = b_frag(smem_nt, t / MI, j);
  }
  // Two stages an iteration, so that the register sets are named at compile time.
  auto stage = [&](int kt, auto parity) {
    constexpr int P = decltype(parity)::value;
    const char* st1 = smem_nt + ((kt + 1) % STAGES) * NT_STAGE_BYTES;     // past the end: a stage nobody needs
    char* nst = smem_nt + ((kt + STAGES - 1) % STAGES) * NT_STAGE_BYTES;  // stage kt-1's buffer
    const int kn = min(kt + STAGES - 1, nk - 1);   // past the end the last stage again: the wait counts stay exact
#pragma unroll
    for (int t = 0; t < 2 * MI; ++t) {
      const int ks = t / MI, i = t % MI;
      if constexpr (B_KN) {
        if (i == 0) kn_wait(P, ks);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        // (the operands' order decides whether a lane owns four columns of a row or four rows of a column)
        if constexpr (C_NM) mfma_16x16x32_in_place(acc[i][j], af[P][ks][i], bfr[P][ks][j]);
        else mfma_16x16x32_in_place(acc[i][j], bfr[P][ks][j], af[P][ks][i]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (t == 0) {   // (behind the first products, which the waves wait under: 300 x 512 x 2048 8.1 -> 7.8 us)
        // Of this wave's loads in flight the oldest LOADS are stage kt+1's; the STAGES-3 stages after it may stay out.
        wait_vmcnt<(STAGES - 3) * LOADS>();
        block_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (B_KN) {
        kn_reads((unsigned)(st1 - smem_nt), P ^ 1, ks, i);
        __builtin_amdgcn_sched_barrier(0);
      } else {
        af[P ^ 1][ks][i] = a_frag(st1, ks, i);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (j % MI == i) bfr[P ^ 1][ks][j] = b_frag(st1, ks, j);
      }
#pragma unroll
      for (int idx = t * PER; idx < t * PER + PER && idx < LOADS; ++idx) issue_one(nst, kn, idx, false);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // (Unrolled over all its stage buffers, so that a fragment's stage rides in its read's offset
  // field as in the 128 x 128 loop, this loop measured the same: it waits for L2, not for issue slots.)
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    stage(kt, std::integral_constant<int, 0>{});
    stage(kt + 1, std::integral_constant<int, 1>{});
  }
  if (kt < nk) stage(kt, std::integral_constant<int, 0>{});

  if constexpr (B_KN) {   // the fragments read past the end, before their registers are given away
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        lds_tr_wait(tfb[p][ks][0], tfb[p][ks][NJ - 1]);
#pragma unroll
        for (int i = 0; i < MI; ++i) lds_wait_for<0>(af[p][ks][i]);
      }
  }
  wait_vmcnt<0>();  // the idle fetches of the last iterations land before the block's LDS is released
  // (the matrix cores' last results: the compiler does not know what the assembly's are)
  asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
#pragma unroll
  for (int t = 0; t < NJ * MI; ++t) asm volatile("" : "+a"(acc[t / NJ][t % NJ]));
  if constexpr (C_NM) {   // C (N,M), no bound: acc[i][j][e] is row 16 i + 4 kq + e, column 16 j + fr of the wave's
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int m = m0 + wm * (16 * MI) + 16 * i + 4 * kq, n = n0 + wn * (16 * NJ) + 16 * j + fr;
        if (n >= N || m >= M) continue;
        bf16_t* to = C + (size_t)n * M + m;
        if (m + 4 <= M) {
          store_loose(to, pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (m + e < M) to[e] = f32_to_bf16(acc[i][j][e]);
        }
      }
    return;
  }
  if constexpr (QKV) {
    const int row_len = which == 0 ? N : qkv.kv_n, c = first + wn * 16 + 4 * kq;   // ... of the head's first half
    bf16_t* to = (which == 0 ? C : (which == 1 ? qkv.Ck : qkv.Cv)) + own * 64 + c;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = mb + 16 * i;
      if (m >= Mv) continue;
      if (which < 2) {   // rounded as the projection would store them, turned, rounded again
        float cs[8];
        unpack8(*reinterpret_cast<const uint4*>(qkv.angles + (size_t)m * 64 + 2 * c), cs);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x1 = round_bf16(acc[i][0][e]), x2 = round_bf16(acc[i][NJ - 1][e]);
          acc[i][0][e] = x1 * cs[2 * e] - x2 * cs[2 * e + 1];
          acc[i][NJ - 1][e] = x2 * cs[2 * e] + x1 * cs[2 * e + 1];
        }
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        store_loose(to + (size_t)m * row_len + 32 * j, pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
    }
    return;
  }
  if constexpr (PAIR) {
    // The gate's waves leave their product, rounded as it is stored, in LDS for the others and store it where it is asked for; those make
    // bf16(bf16(act(bf16 g)) * bf16 u) of it.
    float* gates = reinterpret_cast<float*>(smem_nt) + (wm * 64 + lane) * 17;
    block_barrier();   // every wave is done with the stages
    if (wn == 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e) gates[e] = acc[e >> 3][(e >> 2) & 1][e & 3] = round_bf16(acc[e >> 3][(e >> 2) & 1][e & 3]);
    }
    __syncthreads();
    if (wn == 0) {
      if (gate_out == nullptr) return;
      C = gate_out;
    } else {
      float x[16], g[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) x[e] = round_bf16(acc[e >> 3][(e >> 2) & 1][e & 3]), g[e] = gates[e];
      tail_of(qkv, x, g);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e >> 3][(e >> 2) & 1][e & 3] = x[e];
    }
  }
  const bool vec = (N & 3) == 0;   // rows of 8-byte pieces
  auto pieces = [&](auto residual) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = mb + 16 * i;
      if (m >= Mv) continue;
      bf16_t* row = C + (size_t)m * N;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int n = nb + 16 * j;
        if (n >= N) continue;
        if constexpr (decltype(residual)::value) {   // the product rounded as it would be stored, then scale * it + residual
          float rf[4] = {0.f, 0.f, 0.f, 0.f}, prod[4];
          if (vec) {
            rf[0] = __uint_as_float(res[i][j].x << 16); rf[1] = __uint_as_float(res[i][j].x & 0xffff0000u);
            rf[2] = __uint_as_float(res[i][j].y << 16); rf[3] = __uint_as_float(res[i][j].y & 0xffff0000u);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < N) rf[e] = bf16_to_f32(qkv.residual[(size_t)m * N + n + e]);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) prod[e] = round_bf16(acc[i][j][e]);
          tail_of(qkv, prod, rf);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] = prod[e];
        }
        if (n + 4 <= N) {
          store_loose(row + n, pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) row[n + e] = f32_to_bf16(acc[i][j][e]);
        }
      }
    }
  };
  if (!PAIR && qkv.residual != nullptr) pieces(std::true_type());
  else pieces(std::false_type());
}

// Up to LONG_ROWS rows, one row of tiles, over a K of whole LONG_K, where the tiles are one round over the chip: few rows wait for what a CU draws, so as many CUs
// as there are draw as little as there is to draw, and in long pieces: stages of LONG_K columns are runs of 512 bytes and eight k-steps between two barriers; B,
// of which every block reads rows of its own once, goes past the caches.  A group is sixteen rows of B, an MFMA's: LONG_PAIR: eight of
// the gate's and eight of the up projection's, four groups a block, a wave a group; LONG_QKV: eight of each half of a head, one group; LONG_PLAIN: eight rows, read
// twice over.  Of the last two a block has one group, a wave sixteen rows of A each, and waves past those only fetch.  An element's sum is the chain of
// 32-wide k-steps that it is in every other tile: the same bits.
// us, 29 rows, weights out of memory, by the tiles of 32 and 64 rows below and by this: 2048 columns over 2048 with a residual 8.6 / 6.4, over 8192 20.9 / 13.4, over 14336
// 37.3 / 22.0, 256 over 512 4.2 / 3.8; 48 heads of q, k and v over 2048 8.6 / 7.2 (64 rows 10.4 / 8.8); both of 8192 over 2048 18.9 / 15.8, of 1024 over 4096 17.9 / 16.1.  With
// more than a round of them 1.01 to 1.08 of the others' time (2560 columns over 2048 8.95 / 9.4); 64 rows of a plain product 0.9 to 1.1, of a pair 18.5 / 19.5: those stay.
constexpr int LONG_K = 256, LONG_ROW = LONG_K * 2;
enum LongKind { LONG_PLAIN, LONG_PAIR, LONG_QKV };
constexpr int long_b_rows(LongKind kind) { return kind == LONG_PAIR ? 64 : (kind == LONG_QKV ? 16 : 8); }
constexpr int long_lds(int rows, int b_rows, int stages) { return (rows + b_rows) * LONG_ROW * stages; }
template <LongKind KIND, int LONG_ROWS, int STAGES, int B_ROWS = long_b_rows(KIND), bool RAGGED = false>
__device__ __forceinline__ void gemm_long_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, bf16_t* __restrict__ C, int N, int K, int Mv,
                                               const QkvTail& qkv, const bf16_t* __restrict__ up = nullptr, bf16_t* __restrict__ gate_out = nullptr) {
  constexpr int STAGE = long_lds(LONG_ROWS, B_ROWS, 1), GROUPS = B_ROWS < 16 ? 1 : B_ROWS / 16, WM = 4 / GROUPS;   // WM: waves a group
  constexpr int MI = LONG_ROWS / 16 > WM ? LONG_ROWS / 16 / WM : 1;                                // tiles of A's rows a wave
  constexpr int A_INST = LONG_ROWS / 8, B_INST = B_ROWS / 8, LOADS = A_INST + B_INST;   // loads of two rows each, a wave's share
  static_assert(LONG_K == 256 && (LONG_ROWS == 32 || LONG_ROWS == 64), "two rows a load of 1 KB");
  extern __shared__ __align__(16) char smem_nt[];
  const int tile = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), fr = lane & 15, kq = lane >> 4;
  const int group = wave / WM, wm = wave % WM;
  const bool computes = wm * MI < LONG_ROWS / 16;
  // QKV: a tile is columns first .. + 7 and 32 + first .. of a 64-wide head of the list q | k | v.
  const int q_heads = N >> 6, kv_heads = KIND == LONG_QKV ? qkv.kv_n >> 6 : 0, head = tile >> 2, first = (tile & 3) * 8;
  const int which = KIND != LONG_QKV || head < q_heads ? 0 : (head < q_heads + kv_heads ? 1 : 2), own = head - (which == 0 ? 0 : q_heads + (which - 1) * kv_heads);
  const int n0 = KIND == LONG_QKV ? first : tile * (KIND == LONG_PAIR ? B_ROWS / 2 : B_ROWS);
  if (KIND == LONG_QKV ? head >= q_heads + 2 * kv_heads : n0 >= N) return;
  if constexpr (KIND == LONG_QKV) B = (which == 0 ? B : (which == 1 ? qkv.Bk : qkv.Bv)) + (size_t)own * 64 * K;
  else B += (size_t)n0 * K;
  if (KIND == LONG_PAIR) up += (size_t)n0 * K;
  int a_voff[A_INST], b_voff[B_INST];
#pragma unroll
  for (int i = 0; i < A_INST; ++i) {
    const int r = (wave * A_INST + i) * 2 + (lane >> 5);
    a_voff[i] = r < Mv ? (r * K + (((lane & 31) ^ (r & 15)) << 3)) * 2 : NOWHERE;
  }
#pragma unroll
  for (int i = 0; i < B_INST; ++i) {
    const int r = (wave * B_INST + i) * 2 + (lane >> 5);
    if (RAGGED && n0 + r >= N) {
      b_voff[i] = NOWHERE;
      continue;
    }
    const int row = KIND == LONG_PAIR ? (r >> 4) * 8 + (r & 7) : (KIND == LONG_QKV ? first + (r >> 3) * 32 + (r & 7) : r);
    b_voff[i] = (row * K + (((lane & 31) ^ (r & 15)) << 3)) * 2;
  }
  const int nk = RAGGED ? (K + LONG_K - 1) / LONG_K : K / LONG_K;
  // (RAGGED: of the last stage what lies past K comes from nowhere, for A and B alike)
  auto at = [&](int voff, int r, int kt) { return RAGGED && kt == nk - 1 && (((lane & 31) ^ (r & 15)) << 3) >= K - kt * LONG_K ? NOWHERE : voff; };
  auto issue = [&](int buffer, int kt) {   // (a stage past the last: zeros out of empty buffers, so that the waits can count)
    char* st = smem_nt + buffer * STAGE;
    const int k0 = kt * LONG_K, room = kt < nk ? 0x7fffffff : 0;
#pragma unroll
    for (int i = 0; i < B_INST; ++i) {
      const bool second = KIND == LONG_PAIR && ((wave * B_INST + i) * 2 & 15) >= 8;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(bounded_bytes((second ? up : B) + k0, room), IRON_LDS_PTR(st + LONG_ROWS * LONG_ROW + (wave * B_INST + i) * 1024), 16,
                                               (int)at(b_voff[i], (wave * B_INST + i) * 2 + (lane >> 5), kt), 0, 0, 2);   // non-temporal
    }
#pragma unroll
    for (int i = 0; i < A_INST; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(bounded_bytes(A + k0, room), IRON_LDS_PTR(st + (wave * A_INST + i) * 1024), 16, (int)at(a_voff[i], (wave * A_INST + i) * 2 + (lane >> 5), kt), 0, 0, 0);
  };
  f32x4 acc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // acc[i][e]: row fr of the wave's i-th sixteen, row 4 kq + e of the group's of B.
  const int m_own = wm * MI * 16 + fr, n_own = KIND == LONG_PLAIN && B_ROWS > 8 ? n0 + group * 16 + 4 * kq : n0 + group * 8 + 4 * (kq & 1);
  uint2 res = make_uint2(0, 0);   // a residual's piece this lane will add
  if (KIND == LONG_PLAIN && qkv.residual != nullptr && m_own < Mv) res = *reinterpret_cast<const uint2*>(qkv.residual + (size_t)m_own * N + n_own);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) issue(s, s);
  const int a_off = (wm * MI * 16 + fr) * LONG_ROW, b_row = B_ROWS == 8 ? fr & 7 : group * 16 + fr, b_off = (LONG_ROWS + b_row) * LONG_ROW, b_swz = b_row & 15;
  for (int kt = 0, buffer = 0; kt < nk; ++kt) {
    wait_vmcnt<(STAGES - 2) * LOADS>();   // stage kt has landed once only the younger ones are out
    block_barrier();                      // ... in every wave, and nobody reads stage kt - 1 any more
    issue(buffer == 0 ? STAGES - 1 : buffer - 1, kt + STAGES - 1);
    if (computes) {
      const char* st = smem_nt + buffer * STAGE;
      bf16x8 bf[LONG_K / 32], af[MI][LONG_K / 32];
#pragma unroll
      for (int ks = 0; ks < LONG_K / 32; ++ks) {
        bf[ks] = *reinterpret_cast<const bf16x8*>(st + b_off + (((ks * 4 + kq) ^ b_swz) << 4));
#pragma unroll
        for (int i = 0; i < MI; ++i) af[i][ks] = *reinterpret_cast<const bf16x8*>(st + a_off + i * 16 * LONG_ROW + (((ks * 4 + kq) ^ fr) << 4));
      }
#pragma unroll
      for (int ks = 0; ks < LONG_K / 32; ++ks)
#pragma unroll
        for (int i = 0; i < MI; ++i) mfma_16x16x32_in_place(acc[i], bf[ks], af[i][ks]);
    }
    buffer = buffer == STAGES - 1 ? 0 : buffer + 1;
  }
  wait_vmcnt<0>();   // the empty fetches land before the block's LDS is released
  if (!computes) return;
  asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");   // (the matrix cores' last results)
#pragma unroll
  for (int i = 0; i < MI; ++i) asm volatile("" : "+a"(acc[i]));
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m_own + i * 16;
    float x[4], other[4];   // rounded as the product would be stored; the group's other eight rows'
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = acc[i][e];
      if (KIND != LONG_PLAIN || qkv.residual != nullptr) x[e] = round_bf16(x[e]);
      other[e] = KIND == LONG_PLAIN ? 0.f : __shfl_xor(x[e], 32, 64);
    }
    if (m >= Mv) continue;
    bf16_t* to = C + (size_t)m * N + n_own;
    if constexpr (KIND == LONG_PAIR) {
      if (kq >= 2) tail_of(qkv, x, other);
      else if (gate_out == nullptr) continue;
      else to = gate_out + (size_t)m * N + n_own;
    } else if constexpr (KIND == LONG_QKV) {
      const int c = first + 4 * (kq & 1), row_len = which == 0 ? N : qkv.kv_n;   // ... of the head's half
      to = (which == 0 ? C : (which == 1 ? qkv.Ck : qkv.Cv)) + (size_t)m * row_len + own * 64 + c + (kq >> 1) * 32;
      if (which < 2) {
        float cs[8];
        unpack8(*reinterpret_cast<const uint4*>(qkv.angles + (size_t)m * 64 + 2 * c), cs);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x1 = kq < 2 ? x[e] : other[e], x2 = kq < 2 ? other[e] : x[e];
          x[e] = kq < 2 ? x1 * cs[2 * e] - x2 * cs[2 * e + 1] : x2 * cs[2 * e] + x1 * cs[2 * e + 1];
        }
      }
    } else {
      if (B_ROWS == 8 && kq >= 2) continue;
      if (RAGGED && n_own + 4 > N) {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (n_own + e < N) to[e] = f32_to_bf16(x[e]);
        continue;
      }
      if (qkv.residual != nullptr) {
        const float rf[4] = {__uint_as_float(res.x << 16), __uint_as_float(res.x & 0xffff0000u), __uint_as_float(res.y << 16), __uint_as_float(res.y & 0xffff0000u)};
        tail_of(qkv, x, rf);
      }
    }
    store_loose(to, pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]));
  }
}

// 128 x 128 x 64 tiles, four stages of 32 KB fed straight from global memory into LDS (buffer loads:
// the tile's rows from the stage's k on are the buffer, rebuilt per stage with scalar instructions,
// a lane's place in it a constant 32-bit offset, so a load costs one scalar add for its LDS
// destination and no vector ALU work between two MFMAs); 16-byte chunks XOR-swizzled by the row so
// unpadded rows read conflict-free; a bare s_barrier and counted s_waitcnt vmcnt(N).  Four waves, a
// wave's 64 x 64 as 4 x 4 tiles of 16x16x32 MFMAs (two 32-wide k-steps a stage; the part sustains
// more of these under its power limit than of the 32x32x16 form), accumulators tied in place.  A
// wave is alone on its SIMD, so its own instruction stream interleaves: after an MFMA one fragment
// read of the next k-step or one prefetch load goes out, and the stage's one barrier sits before
// its second k-step, whose fragments are in registers by then.  B as (N,K), or as (K,N): then the
// stage lands as stored and the B operands come from transposing reads.  The output is staged
// through LDS so that it leaves as whole 128-byte row segments (16 bytes a lane).  QKV: the fused
// projections' per-tile choice of weight and output, RoPE on the accumulators.  Otherwise `qkv`
// carries the optional residual epilogue.
template <bool QKV, bool B_KN = false, bool C_NM = false, bool SHARED = false>
__device__ __forceinline__ void gemm_nt16_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B_,
                                               bf16_t* __restrict__ C_, int M, int N_, int K,
                                               int Mv, int tiles_m, int tiles_n,
                                               int patched, const QkvTail& qkv) {
  constexpr int NT_BM = 128, NT_BN = 128;
  constexpr int NT_A_BYTES = NT_BM * BK * 2, NT_STAGE_BYTES = (NT_BM + NT_BN) * BK * 2;
  constexpr int INST = NT_BM / 8 / 4;  // 1 KB loads of A (and of B) a wave issues per stage
  constexpr int LOADS = 2 * INST;
  static_assert(BK == 64 && INST == 4, "two 32-wide k-steps a stage, eight loads a wave");
  static_assert(!(B_KN && QKV), "the fused projections read weights as stored, (N,K)");
  static_assert(B_KN || !C_NM, "with B (N,K) the (N,M) output is the product of B and A");
  extern __shared__ __align__(16) char smem_nt[];

  int tm, tn;
  const bool given = !QKV && qkv.tile_plus1 > 0;
  if (given) {
    tm = (qkv.tile_plus1 - 1) / tiles_n;
    tn = (qkv.tile_plus1 - 1) % tiles_n;
  } else if (!live_tile(blockIdx.x, tiles_m, tiles_n, patched, (Mv + NT_BM - 1) / NT_BM, tm, tn)) {
    return;
  }
  const int m0 = tm * NT_BM;
  if (m0 >= Mv) return;
  const bf16_t* B = B_;
  bf16_t* C = C_;
  int N = N_, which = 0;
  if constexpr (QKV) {
    const int q_tiles = N_ / NT_BN, kv_tiles = qkv.kv_n / NT_BN;
    if (tn >= q_tiles) {
      which = tn < q_tiles + kv_tiles ? 1 : 2;
      tn -= q_tiles + (which - 1) * kv_tiles;
      B = which == 1 ? qkv.Bk : qkv.Bv;
      C = which == 1 ? qkv.Ck : qkv.Cv;
      N = qkv.kv_n;
    }
  }
  // (K,N): B's columns are read in whole tiles, so the last tile is moved back to end at N (what two
  // tiles both cover comes out the same from both).  A matrix narrower than a tile is read to its last piece again.
  const int n0 = B_KN ? max(min(tn * NT_BN, N - NT_BN), 0) : tn * NT_BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int lrow = lane >> 3, pch = lane & 7;
  auto kn_swizzle = [](int k) { return ((k & 3) << 1) | (((k >> 3) & 1) << 3); };
  int a_voff[INST], b_voff[INST], a_head[INST], b_head[INST];   // *_head: the k of a stage the lane's piece begins at
#pragma unroll
  for (int i = 0; i < INST; ++i) {
    const int r = (wave * INST + i) * 8 + lrow;
    const int lch = pch ^ ((r >> 1) & 7);
    a_voff[i] = m0 + r < Mv ? (r * K + lch * 8) * 2 : NOWHERE;
    a_head[i] = b_head[i] = lch * 8;
    if constexpr (!B_KN) {
      b_voff[i] = (int)(((size_t)(min(n0 + r, N - 1) - n0) * K + lch * 8) * 2);
    } else {
      // B (K,N) lands as stored: 64 k-rows of 128 columns (256 bytes a row, four rows an
      // instruction), a row's 16 chunks XORed with kn_swizzle(row) for the transposing reads below.
      const int kr = (wave * INST + i) * 4 + (lane >> 4);
      b_voff[i] = (int)(((size_t)kr * N + min(((lane & 15) ^ kn_swizzle(kr)) * 8, N - 8 - n0)) * 2);
      b_head[i] = kr;
    }
  }
  const int k_first = QKV || (B_KN && !SHARED) ? 0 : qkv.k_begin;
  const int pad = QKV ? 0 : k_pad(K);
  const bf16_t* a_tile = A + (size_t)m0 * K + k_first - pad;
  const bf16_t* b_tile = B_KN ? B + n0 + ((ptrdiff_t)k_first - pad) * N : B + (size_t)n0 * K + k_first - pad;
  auto issue_one = [&](char* st, int kt, int idx, bool head) {
    const int k0 = kt * BK;
    if (idx < INST) {
      const __amdgpu_buffer_rsrc_t rows = stage_rows(a_tile + k0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, IRON_LDS_PTR(st + (wave * INST + idx) * 1024), 16,
                                               head && a_head[idx] < pad ? NOWHERE : a_voff[idx], 0, 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t rows = stage_rows(b_tile + (B_KN ? (size_t)k0 * N : (size_t)k0));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, IRON_LDS_PTR(st + NT_A_BYTES + (wave * INST + idx - INST) * 1024),
                                               16, head && b_head[idx - INST] < pad ? NOWHERE : b_voff[idx - INST], 0, 0, 0);
    }
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;

  // Where this lane stores: rows r0 + lane / 8 of the wave's 64 (r0 = 0, 8, ..), 8 columns from 8 (lane % 8).
  const int out_row = lane >> 3, out_col = (lane & 7) * 8;
  const int out_n = n0 + wn * 64 + out_col;
  // A residual's pieces this lane will add in the epilogue are requested now, so that their
  // latency passes under the whole product instead of at its end (N a multiple of 8: 16-byte pieces).
  uint4 res[8];
  const bool res_ahead = !QKV && qkv.residual != nullptr && (N & 7) == 0;
  if constexpr (!QKV) {
    if (res_ahead) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int m = min(m0 + wm * 64 + r * 8 + out_row, M - 1);
        res[r] = *reinterpret_cast<const uint4*>(qkv.residual + (size_t)m * N + min(out_n, N - 8));
      }
    }
  }

  const int nk = (!QKV && (!B_KN || SHARED) && qkv.k_len > 0 ? qkv.k_len : K + pad) / BK;
#pragma unroll
  for (int s = 0; s < NT_STAGES - 1; ++s)
#pragma unroll
    for (int idx = 0; idx < LOADS; ++idx) issue_one(smem_nt + s * NT_STAGE_BYTES, min(s, nk - 1), idx, s == 0 && (!SHARED || k_first == 0));

  // Fragments: lane -> row fr of a 16-row tile, 16-byte chunk kq of the k-step's four.
  const int fr = lane & 15, kq = lane >> 4;
  const int swz = (fr >> 1) & 7;   // tile rows are multiples of 16 apart: one swizzle for all
  const int a_row = (wm * 64 + fr) * 128, b_row = NT_A_BYTES + (wn * 64 + fr) * 128;
  auto a_frag = [&](const char* st, int ks, int i) {
    return *reinterpret_cast<const bf16x8*>(st + a_row + i * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };
  auto b_frag = [&](const char* st, int ks, int j) {
    return *reinterpret_cast<const bf16x8*>(st + b_row + j * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };

  // (K,N): the B operand of tile j wants, for column n = 16 j + fr, the k-step's k = 8 kq .. + 7; a
  // transposing read hands a 16-lane group the 4 k-rows x 16 columns its lanes point at, turned
  // round (a lane gets 4 k of one column): rows 8 kq .. + 3, then 8 kq + 4 .. + 7.
  const int tr_k = 8 * kq + ((lane & 15) >> 2), tr_n = wn * 64 + 4 * (lane & 3);
  const unsigned lds_base_nt = (unsigned)(size_t)IRON_LDS_PTR(smem_nt);
  const unsigned kn_base = lds_base_nt + NT_A_BYTES;
  // The lane's place in a stage's B tile for tile j (k-step 0, low half) is fixed for the whole loop;
  // the k-step (32 rows on) and the high half (4 rows on) leave the swizzle as it is -- kn_swizzle(k +
  // 4) = kn_swizzle(k) for k % 8 < 4, and k + 32 keeps the bits it reads -- and the (K,N) loop is
  // unrolled over the four stage buffers, so k-step, half and stage all ride in the reads' offset
  // fields (16 bits: a second set of lane addresses two stages on) and a fragment read costs no
  // vector arithmetic at all: with one wave a SIMD every vector instruction between two MFMAs is
  // time off the matrix pipe (sixteen adds a k-step, then four, then none: 2048^3 25.0 -> 23.5 -> 22.7 us).
  unsigned kn_lane[2][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = tr_n + j * 16;
    kn_lane[0][j] = kn_base + (((n >> 3) ^ kn_swizzle(tr_k)) << 4) + ((n & 4) << 1) + tr_k * 256;
    kn_lane[1][j] = kn_lane[0][j] + 2 * NT_STAGE_BYTES;
  }
  auto b_frag_kn = [&](auto stage_c, int ks, int j, TrFrag& t) {
    constexpr int STAGE = decltype(stage_c)::value, OFF = (STAGE & 1) * NT_STAGE_BYTES;
    const unsigned at = kn_lane[STAGE >> 1][j];
    if (ks == 0) {
      t.lo = lds_read_tr16_at<OFF>(at);
      t.hi = lds_read_tr16_at<OFF + 4 * 256>(at);
    } else {
      t.lo = lds_read_tr16_at<OFF + 32 * 256>(at);
      t.hi = lds_read_tr16_at<OFF + 36 * 256>(at);
    }
  };
  TrFrag tfb[2][4];
  // The compiler does not count the transposing reads: a k-step's B fragments pass through this
  // wait before they are joined into operands.  LDS reads return in order and the only reads
  // issued after a k-step's B fragments are its four A fragments, so "at most four outstanding"
  // is "B has arrived".
  auto join_b = [&](int ks, bf16x8 (&b)[4]) {
    asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(tfb[ks][0].lo), "+v"(tfb[ks][0].hi), "+v"(tfb[ks][1].lo), "+v"(tfb[ks][1].hi),
                                           "+v"(tfb[ks][2].lo), "+v"(tfb[ks][2].hi), "+v"(tfb[ks][3].lo), "+v"(tfb[ks][3].hi));
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = tr_join(tfb[ks][j]);
  };
  // (K,N): the A fragments are read by uncounted reads as well, so that every wait of the loop is
  // this code's own.  With counted A reads the compiler's waits for them took no account of the
  // transposing reads issued in between and came out as "all but two outstanding" where eleven
  // were in flight: each k-step waited an LDS trip for fragments of the NEXT one (a quarter of
  // the loop's time).  The lane's place in a stage for k-step ks; tile row i is the read's offset.
  unsigned a_lane[2][2];   // [stage / 2][k-step]
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_lane[0][ks] = lds_base_nt + a_row + (((ks * 4 + kq) ^ swz) << 4);
    a_lane[1][ks] = a_lane[0][ks] + 2 * NT_STAGE_BYTES;
  }
  auto a_frags_kn = [&](auto stage_c, int ks, int i, bf16x8& out) {
    constexpr int STAGE = decltype(stage_c)::value, OFF = (STAGE & 1) * NT_STAGE_BYTES;
    const unsigned at = a_lane[STAGE >> 1][ks];
    if (i == 0) out = lds_read_b128_at<OFF + 0 * 16 * 128>(at);
    else if (i == 1) out = lds_read_b128_at<OFF + 1 * 16 * 128>(at);
    else if (i == 2) out = lds_read_b128_at<OFF + 2 * 16 * 128>(at);
    else out = lds_read_b128_at<OFF + 3 * 16 * 128>(at);
  };

  wait_vmcnt<(NT_STAGES - 2) * LOADS>();   // stage 0 has landed once only the two younger ones are out
  block_barrier();
  bf16x8 af[2][4], bfr[2][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (B_KN) b_frag_kn(std::integral_constant<int, 0>{}, 0, i, tfb[0][i]);
    else bfr[0][i] = b_frag(smem_nt, 0, i);
  }
  __builtin_amdgcn_sched_barrier(0);   // B's reads first, then A's: join_b counts on that order
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (B_KN) a_frags_kn(std::integral_constant<int, 0>{}, 0, i, af[0][i]);
    else af[0][i] = a_frag(smem_nt, 0, i);
  }
  // One stage of the loop, which is unrolled over the four stage buffers: stage_c = kt % NT_STAGES,
  // so a fragment's place in LDS is a lane address fixed before the loop plus an offset field, and
  // nothing is computed for it between two MFMAs ((N,K) at 2048^3: 20.7 -> 20.0 us; (K,N) above).
  auto stage_step = [&](int kt, auto stage_c) {
    constexpr int STAGE = decltype(stage_c)::value;
    static_assert(STAGE >= 0 && STAGE < NT_STAGES, "a stage buffer");
    // Prefetch goes into the buffer of stage kt-1.  Past the end the last stage is fetched again
    // (into buffers nobody reads any more) rather than branch: every iteration issues the same
    // loads, which keeps the wait counts exact and the scheduling region whole.
    const int kn = min(kt + NT_STAGES - 1, nk - 1);
    constexpr int STAGE_NEXT = (STAGE + 1) % NT_STAGES;
    char* nst = smem_nt + ((STAGE + NT_STAGES - 1) % NT_STAGES) * NT_STAGE_BYTES;
    const char* st = smem_nt + STAGE * NT_STAGE_BYTES;
    const char* st1 = smem_nt + STAGE_NEXT * NT_STAGE_BYTES;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks == 1) {
        // The stage's one barrier, before its second k-step (whose fragments are in registers): of
        // the loads in flight the oldest LOADS are stage kt+1's (then stage kt+2's, and the 4 issued
        // so far for stage kt+3); after it nobody reads stage kt any more.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vmcnt<LOADS + 4>();
        block_barrier();
      }
      const char* from = ks == 0 ? st : st1;
      const int nks = ks ^ 1;
      if constexpr (B_KN) join_b(ks, bfr[ks]);
      // Source order is issue order (nothing crosses a sched_barrier): after an MFMA one fragment
      // read of the next k-step (B's first: its first MFMAs need all of them) or one load goes out.
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (B_KN) {
          // Reads in flight when tile row i starts, in issue order: this k-step's A fragments from
          // i on, then what this k-step has issued for the next one (8 transposing reads during
          // row 0, 4 A reads during row 1): fragment i has arrived once all but those after it have.
          if (i == 0) lds_wait_for<3>(af[ks][0]);         // after join_b: a1 a2 a3 may be out
          else if (i == 1) lds_wait_for<10>(af[ks][1]);   // a2 a3 + 8
          else if (i == 2) lds_wait_for<13>(af[ks][2]);   // a3 + 8 + 4
          else lds_wait_for<12>(af[ks][3]);               // 8 + 4
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // (the operands' order decides whether a lane owns four columns of a row or four rows of a column)
          if constexpr (C_NM) mfma_16x16x32_in_place(acc[i][j], af[ks][i], bfr[ks][j]);
          else mfma_16x16x32_in_place(acc[i][j], bfr[ks][j], af[ks][i]);
          __builtin_amdgcn_sched_barrier(0);
          const int slot = i * 4 + j;
          if (slot < 4) {
            if constexpr (B_KN) {
              if (ks == 0) b_frag_kn(stage_c, nks, slot, tfb[nks][slot]);
              else b_frag_kn(std::integral_constant<int, STAGE_NEXT>{}, nks, slot, tfb[nks][slot]);
            } else {
              bfr[nks][slot] = b_frag(from, nks, slot);
            }
          } else if (slot < 8) {
            if constexpr (B_KN) {
              if (ks == 0) a_frags_kn(stage_c, nks, slot - 4, af[nks][slot - 4]);
              else a_frags_kn(std::integral_constant<int, STAGE_NEXT>{}, nks, slot - 4, af[nks][slot - 4]);
            } else {
              af[nks][slot - 4] = a_frag(from, nks, slot - 4);
            }
          } else if (slot & 1) issue_one(nst, kn, ks * 4 + (slot - 9) / 2, false);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  static_assert(NT_STAGES == 4, "the loop below names the four stage buffers");
  for (int kt0 = 0; kt0 < nk; kt0 += NT_STAGES) {
    stage_step(kt0, std::integral_constant<int, 0>{});
    if (kt0 + 1 < nk) stage_step(kt0 + 1, std::integral_constant<int, 1>{});
    if (kt0 + 2 < nk) stage_step(kt0 + 2, std::integral_constant<int, 2>{});
    if (kt0 + 3 < nk) stage_step(kt0 + 3, std::integral_constant<int, 3>{});
  }

  wait_vmcnt<0>();   // the idle fetches of the last iterations land ...
  block_barrier();   // ... in every wave, and every wave is done with the stages, before LDS is reused

  if constexpr (QKV) {
    if (which < 2) {
      // acc[i][j][e] and acc[i][j + 2][e] are columns c and c + 32 of the wave's head, c = 16 j + 4 kq + e,
      // of row m = 16 i + fr: the pair RoPE turns by the angle row's (cos, sin) number c.
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = min(m0 + wm * 64 + i * 16 + fr, M - 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float cs[8];
          unpack8(*reinterpret_cast<const uint4*>(qkv.angles + (size_t)m * 64 + 2 * (16 * j + 4 * kq)), cs);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x1 = round_bf16(acc[i][j][e]), x2 = round_bf16(acc[i][j + 2][e]);
            const float c = cs[2 * e], sn = cs[2 * e + 1];
            acc[i][j][e] = x1 * c - x2 * sn;
            acc[i][j + 2][e] = x2 * c + x1 * sn;
          }
        }
      }
    }
  }

  if constexpr (SHARED) {
    if (qkv.tile_sums != nullptr) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int row = C_NM ? wn * 64 + j * 16 + fr : wm * 64 + i * 16 + fr;
          const int at = C_NM ? wm * 64 + i * 16 + 4 * kq : wn * 64 + j * 16 + 4 * kq;
          *reinterpret_cast<f32x4*>(qkv.tile_sums + row * NT_BN + at) = acc[i][j];
        }
      return;
    }
  }
  if constexpr (!QKV && !B_KN) {
    if (qkv.partial != nullptr) {
      // A slice of K: the float32 sums as they are, four columns of a row a lane and tile.
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + wm * 64 + i * 16 + fr;
        if (m >= Mv) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = n0 + wn * 64 + j * 16 + 4 * kq;
          if (n + 4 <= N) *reinterpret_cast<f32x4*>(qkv.partial + (size_t)m * N + n) = acc[i][j];
        }
      }
      return;
    }
  }
  // Output through LDS: the wave lays its 64 x 64 out row-major (rows padded by 16 bytes, which
  // spreads the 8-byte writes and the 16-byte reads over the banks) and each lane then owns 8
  // consecutive columns of a row: a row of the tile leaves as one 128-byte segment.
  constexpr int OROWB = 64 * 2 + 16;
  char* ot = smem_nt + wave * (64 * OROWB);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<uint2*>(ot + ((C_NM ? j : i) * 16 + fr) * OROWB + ((C_NM ? i : j) * 16 + 4 * kq) * 2) =
          make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
  // The tile is private to the wave, whose LDS operations execute in order: no block barrier,
  // only a fence to keep the compiler from moving the reads above other lanes' writes.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // Rows of whole pieces and a half begin on a half: two stores of one, which a launch of one round ends on sooner than on a store across (us, across / halves: (N,M) of
  // 348 x 464 x 168 5.88 / 5.42, 132 x 4096 x 64 5.32 / 4.86, (M,N) of 8192 x 140 x 192 6.33 / 5.90); larger outputs are bound by what they write, 4100 x 4096 x 512 33.6 / 35.0.
  const bool halves = ((C_NM ? M : N) & 3) == 0 && tiles_m * tiles_n <= 256;
  auto store_halves = [](bf16_t* p, const uint4& v, int left) {
    *reinterpret_cast<uint2*>(p) = make_uint2(v.x, v.y);
    if (left > 4) *reinterpret_cast<uint2*>(p + 4) = make_uint2(v.z, v.w);
  };
  if constexpr (C_NM) {   // the tile's rows are C's columns n, 8 consecutive m of each a lane
    const int out_m = m0 + wm * 64 + out_col;
    const bool whole_m = (M & 7) == 0 && out_m + 8 <= M;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int row = r * 8 + out_row;
      const uint4 v = *reinterpret_cast<const uint4*>(ot + row * OROWB + out_col * 2);
      if (out_m >= M || n0 + wn * 64 + row >= N) continue;
      bf16_t* p = C + (size_t)(n0 + wn * 64 + row) * M + out_m;
      if (whole_m) *reinterpret_cast<uint4*>(p) = v;
      else if (halves) store_halves(p, v, M - out_m);
      else store_ragged(p, v, M - out_m);
    }
    return;
  }
  const bool whole = (N & 7) == 0 && out_n + 8 <= N;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int row = r * 8 + out_row, m = m0 + wm * 64 + row;
    uint4 v = *reinterpret_cast<const uint4*>(ot + row * OROWB + out_col * 2);
    if (m >= Mv || out_n >= N) continue;
    bf16_t* p = C + (size_t)m * N + out_n;
    if constexpr (!QKV) {
      if (qkv.residual != nullptr) {   // the product rounded as it would be stored, then scale * it + residual
        float x[8], rf[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        unpack8(v, x);
        if (whole) {
          unpack8(res_ahead ? res[r] : *reinterpret_cast<const uint4*>(qkv.residual + (size_t)m * N + out_n), rf);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)   // (constant indices: a runtime trip count puts the array in scratch memory)
            if (out_n + e < N) rf[e] = bf16_to_f32(qkv.residual[(size_t)m * N + out_n + e]);
        }
        tail_of(qkv, x, rf);
        v = pack8(x);
      }
    }
    if (whole) *reinterpret_cast<uint4*>(p) = v;
    else if (halves) store_halves(p, v, N - out_n);
    else store_ragged(p, v, N - out_n);
  }
}


template <bool B_KN, bool QKV, int T, int STAGES64 = 4, bool C_NM = false>
__global__ __launch_bounds__(256) void gemm_nt_kernel(const bf16_t* __restrict__ A,
                                                      const bf16_t* __restrict__ B,
                                                      bf16_t* __restrict__ C, int M, int N, int K,
                                                      const int* __restrict__ valid, int tiles_m,
                                                      int tiles_n, int patched, QkvTail qkv) {
  if constexpr (QKV) to_cache_rows(qkv, valid, M);
  static_assert(T == 2 || (T == 1 && !B_KN && !QKV), "64x64 tiles: B (N,K), plain or residual output");
  if constexpr (T == 2)
    gemm_nt16_body<QKV, B_KN, C_NM>(A, B, C, M, N, K, bound_or(valid, M), tiles_m, tiles_n, patched, qkv);
  else
    gemm_nt64_body<STAGES64>(A, B, C, M, N, K, bound_or(valid, M), tiles_m, tiles_n, patched, qkv);
}

template <bool B_KN, bool QKV = false, int T = 2, int STAGES64 = 4, bool C_NM = false>
static int launch_gemm_nt(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K,
                          const int* valid, hipStream_t s, QkvTail qkv = QkvTail{}) {
  constexpr int BM = 64 * T, BN = 64 * T;
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = QKV ? (N + 2 * qkv.kv_n) / BN : (N + BN - 1) / BN;
  if constexpr (T == 1 && STAGES64 == 4) {
    // No more 64 x 64 tiles than CUs: a CU has one block whatever its LDS, so the deeper pipeline.
    if ((long)tiles_m * tiles_n <= 256)
      return launch_gemm_nt<B_KN, QKV, 1, 8>(A, B, C, M, N, K, valid, s, qkv);
  }
  const size_t lds = (size_t)(T == 1 ? STAGES64 : NT_STAGES) * (BM + BN) * BK * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_nt_kernel<B_KN, QKV, T, STAGES64, C_NM>), lds); e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  const int patched = (tiles_m % 8 == 0 && tiles_n % 4 == 0 && ((tiles_m / 8) * (tiles_n / 4)) % 8 == 0) ? 1 : 0;
  hipLaunchKernelGGL((gemm_nt_kernel<B_KN, QKV, T, STAGES64, C_NM>), dim3(tiles_m * tiles_n), dim3(256), lds, s, A, B, C, M, N, K,
                     valid, tiles_m, tiles_n, patched, qkv);
  IRON_LAUNCH_CHECK();
}

template <int STAGES, int MI, int WM, int NJ, bool B_KN = false, bool C_NM = false>
__global__ __launch_bounds__(256) void gemm_small_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, bf16_t* __restrict__ C, int M, int N,
                                                         int K, int tiles_m, int tiles_n) {
  gemm_nt64_body<STAGES, false, MI, WM, NJ, false, B_KN, C_NM>(A, B, C, M, N, K, M, tiles_m, tiles_n, 0, QkvTail{});
}
template <int STAGES, int MI, int WM, int NJ, bool B_KN = false, bool C_NM = false>
static int launch_gemm_small(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, hipStream_t s) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NJ * (4 / WM);
  constexpr size_t lds = (size_t)STAGES * (BM + BN) * BK * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_small_kernel<STAGES, MI, WM, NJ, B_KN, C_NM>), lds); e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_small_kernel<STAGES, MI, WM, NJ, B_KN, C_NM>), dim3(tiles_m * tiles_n), dim3(256), lds, s, A, B, C, M, N, K, tiles_m, tiles_n);
  IRON_LAUNCH_CHECK();
}

// The fused projections at 128 x 192 tiles: three 64-wide heads of the concatenated q | k | v head
// list a tile, so a 2048-row chunk of a 32 + 8 + 8-head layer is 16 x 16 = 256 tiles -- one a CU in
// one round, where 128 x 128 tiles make 384 (a round and a half, run as two).  Four waves stacked
// along m: a wave owns 32 rows x 192 columns (6 accumulator tiles), so every head's two halves sit
// in one wave and RoPE stays in registers.  Three stages of 40 KB; the loop is the 128 x 128
// kernel's (direct-to-LDS loads, pinned interleave, the stage's barrier before its last k-step).
// HPT = heads a tile: 3 as above, or 1 -- 128 x 64 tiles, for a row bound so short that wider
// tiles leave most CUs idle (512 rows of that layer: 192 tiles of one head against 64 of three).
constexpr int Q3_BM = 128, Q3_BN = 192, Q3_STAGES = 3;
constexpr int Q3_A_BYTES = Q3_BM * BK * 2, Q3_STAGE_BYTES = (Q3_BM + Q3_BN) * BK * 2;
constexpr int Q1_STAGE_BYTES = (Q3_BM + 64) * BK * 2, Q1_STAGES = 5;   // one head a tile: five 24 KB stages

template <int HPT>
__device__ __forceinline__ void qkv_heads_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bq,
                                               bf16_t* __restrict__ Cq, int M, int heads, int kv_heads, int K,
                                               const int* __restrict__ valid, int tiles_m, int tiles_n,
                                               int patched, const QkvTail& qkv) {
  constexpr int Q3_BN = 64 * HPT, Q3_STAGE_BYTES = (Q3_BM + Q3_BN) * BK * 2, NACC = 2 * HPT;
  constexpr int A_INST = Q3_BM / 8 / 4, B_INST = Q3_BN / 8 / 4, LOADS = A_INST + B_INST;   // 4 + 6 (or 2) a wave
  constexpr int PER = LOADS / 3, REST = LOADS - 3 * PER;   // loads issued under each of a stage's first three k-steps, and its last
  static_assert(PER <= NACC && REST <= NACC, "a load rides an MFMA");
  extern __shared__ __align__(16) char smem_q3[];
  const int Mv = bound_or(valid, M);

  int tm, tn;
  tile_of_block(blockIdx.x, tiles_m, tiles_n, patched, tm, tn);
  const int m0 = tm * Q3_BM;
  if (m0 >= Mv) return;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane >> 3, pch = lane & 7;
  // Head g of the concatenated list: its weight rows and where its 64 columns go.
  auto head_weight = [&](int g) {
    if (g < heads) return Bq + (size_t)g * 64 * K;
    if (g < heads + kv_heads) return qkv.Bk + (size_t)(g - heads) * 64 * K;
    return qkv.Bv + (size_t)(g - heads - kv_heads) * 64 * K;
  };
  // Buffer loads straight into LDS (see gemm_nt16_body): the activations' tile rows are one buffer;
  // the eight weight rows of an instruction lie in one head, so each of a wave's weight
  // instructions has its own buffer, which starts at its first row.  The stage's k is the scalar
  // offset, a lane's place the constant vector offset.
  const __amdgpu_buffer_rsrc_t a_rows = stage_rows(A + (size_t)m0 * K);
  __amdgpu_buffer_rsrc_t b_rows[B_INST];
  int a_voff[A_INST], b_voff[B_INST];
#pragma unroll
  for (int i = 0; i < A_INST; ++i) {
    const int r = (wave * A_INST + i) * 8 + lrow;
    a_voff[i] = m0 + r < Mv ? (r * K + (pch ^ ((r >> 1) & 7)) * 8) * 2 : NOWHERE;
  }
#pragma unroll
  for (int i = 0; i < B_INST; ++i) {
    const int r0 = (wave * B_INST + i) * 8;   // first of the instruction's rows among the tile's weight rows: head r0 / 64, its row r0 % 64
    const int r = r0 + lrow;
    b_rows[i] = stage_rows(head_weight(tn * HPT + r0 / 64) + (size_t)(r0 % 64) * K);
    b_voff[i] = (int)(((size_t)lrow * K + (pch ^ ((r >> 1) & 7)) * 8) * 2);
  }
  auto issue_one = [&](char* st, int kt, int idx) {
    const int k_off = kt * BK * 2;
    if (idx < A_INST)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rows, IRON_LDS_PTR(st + (wave * A_INST + idx) * 1024), 16,
                                               (int)a_voff[idx], k_off, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rows[idx - A_INST],
                                               IRON_LDS_PTR(st + Q3_A_BYTES + (wave * B_INST + idx - A_INST) * 1024), 16,
                                               (int)b_voff[idx - A_INST], k_off, 0, 0);
  };

  f32x16 acc[NACC];
#pragma unroll
  for (int j = 0; j < NACC; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;

  const int nk = K / BK;
  const int fr = lane & 31, kh = lane >> 5;
  const int swz = (fr >> 1) & 7;   // tile rows are multiples of 32 apart: one swizzle for all
  const int a_off = (wave * 32 + fr) * 128, b_off = Q3_A_BYTES + fr * 128;
  auto frag = [&](const char* st, int off, int ks) {
    return *reinterpret_cast<const bf16x8*>(st + off + (((ks * 2 + kh) ^ swz) << 4));
  };
  if constexpr (HPT == 1) {
    // One head a tile: a k-step is two MFMAs of a wave, far less than an LDS read takes to return,
    // so -- as in gemm_nt64_body -- the fragments of a whole stage are read one stage ahead into a
    // second register set.  At the top of stage kt the one barrier (stage kt+1 has landed in every
    // wave, nobody reads stage kt-1 any more), then stage kt's eight MFMAs out of registers with
    // the twelve fragment reads of stage kt+1 and the six loads of stage kt+STAGES-1 between them.
    constexpr int STAGES = Q1_STAGES, KSTEPS = BK / 16;
    static_assert(LOADS == 6 && KSTEPS == 4, "six loads and twelve reads ride eight MFMAs");
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
      for (int idx = 0; idx < LOADS; ++idx) issue_one(smem_q3 + s * Q3_STAGE_BYTES, min(s, nk - 1), idx);
    wait_vmcnt<(STAGES - 2) * LOADS>();   // stage 0 has landed once only the younger ones are out
    block_barrier();
    bf16x8 af[2][KSTEPS], bfr[2][KSTEPS][2];   // [stage parity][k-step]([column half])
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      af[0][ks] = frag(smem_q3, a_off, ks);
      bfr[0][ks][0] = frag(smem_q3, b_off, ks);
      bfr[0][ks][1] = frag(smem_q3, b_off + 32 * 128, ks);
    }
    auto stage = [&](int kt, auto parity) {
      constexpr int P = decltype(parity)::value;
      // Of this wave's loads in flight the oldest LOADS are stage kt+1's; the STAGES-3 stages after it may stay out.
      wait_vmcnt<(STAGES - 3) * LOADS>();
      block_barrier();
      const char* st1 = smem_q3 + ((kt + 1) % STAGES) * Q3_STAGE_BYTES;     // past the end: a stage nobody needs
      char* nst = smem_q3 + ((kt + STAGES - 1) % STAGES) * Q3_STAGE_BYTES;  // stage kt-1's buffer
      const int kn = min(kt + STAGES - 1, nk - 1);   // past the end the last stage again: the wait counts stay exact
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[P][ks][0], af[P][ks], acc[0], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        af[P ^ 1][ks] = frag(st1, a_off, ks);
        bfr[P ^ 1][ks][0] = frag(st1, b_off, ks);
        if (ks < 2) issue_one(nst, kn, ks);
        __builtin_amdgcn_sched_barrier(0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[P][ks][1], af[P][ks], acc[1], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        bfr[P ^ 1][ks][1] = frag(st1, b_off + 32 * 128, ks);
        issue_one(nst, kn, 2 + ks);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      stage(kt, std::integral_constant<int, 0>{});
      stage(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) stage(kt, std::integral_constant<int, 0>{});
  } else {
#pragma unroll
  for (int s = 0; s < Q3_STAGES - 1; ++s)
#pragma unroll
    for (int idx = 0; idx < LOADS; ++idx) issue_one(smem_q3 + s * Q3_STAGE_BYTES, min(s, nk - 1), idx);

  wait_vmcnt<LOADS>();   // stage 0 has landed once only stage 1's loads are out
  block_barrier();
  bf16x8 af[2], bfr[2][NACC];
  af[0] = frag(smem_q3, a_off, 0);
#pragma unroll
  for (int j = 0; j < NACC; ++j) bfr[0][j] = frag(smem_q3, b_off + j * 32 * 128, 0);
  // One stage of the loop, which is unrolled over the three stage buffers (stage_c = kt % Q3_STAGES):
  // a fragment's stage then rides in its read's offset field instead of a vector add a read.
  auto stage_step = [&](int kt, auto stage_c) {
    constexpr int S = decltype(stage_c)::value;
    const int kn = min(kt + Q3_STAGES - 1, nk - 1);
    char* nst = smem_q3 + ((S + Q3_STAGES - 1) % Q3_STAGES) * Q3_STAGE_BYTES;
    const char* st = smem_q3 + S * Q3_STAGE_BYTES;
    const char* st1 = smem_q3 + ((S + 1) % Q3_STAGES) * Q3_STAGE_BYTES;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int cur = ks & 1, nxt = cur ^ 1;
      const bool last = ks == BK / 16 - 1;
      if (last) {
        // Of the loads in flight the oldest LOADS are stage kt+1's; the 3 PER issued so far for stage
        // kt+2 may stay out.  After the barrier nobody reads stage kt any more.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vmcnt<3 * PER>();
        block_barrier();
      }
      const char* from = last ? st1 : st;
      const int nks = last ? 0 : ks + 1;
#pragma unroll
      for (int j = 0; j < NACC; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][j], af[cur], acc[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (j == 0) af[nxt] = frag(from, a_off, nks);
        bfr[nxt][j] = frag(from, b_off + j * 32 * 128, nks);
        // A stage's loads (ten, or six): PER under each of the first three k-steps, the rest under the last.
        if (!last && j < PER) issue_one(nst, kn, ks * PER + j);
        if (last && j < REST) issue_one(nst, kn, 3 * PER + j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  static_assert(Q3_STAGES == 3, "the loop below names the three stage buffers");
  for (int kt0 = 0; kt0 < nk; kt0 += Q3_STAGES) {
    stage_step(kt0, std::integral_constant<int, 0>{});
    if (kt0 + 1 < nk) stage_step(kt0 + 1, std::integral_constant<int, 1>{});
    if (kt0 + 2 < nk) stage_step(kt0 + 2, std::integral_constant<int, 2>{});
  }
  }
  wait_vmcnt<0>();   // the idle fetches of the last iterations land before the block's LDS is released

  // acc[2h][e] and acc[2h+1][e] are columns c and c + 32 of head h of the tile, c = 8 (e/4) + 4 kh + e%4,
  // of row fr of the wave's 32: the pair RoPE turns by the angle row's (cos, sin) number c.
  const int m = m0 + wave * 32 + fr;
  const bf16_t* ang = qkv.angles + (size_t)min(m, M - 1) * 64 + 8 * kh;
#pragma unroll
  for (int h = 0; h < HPT; ++h) {
    const int g = tn * HPT + h;
    bf16_t* C;
    int N, col;
    if (g < heads) { C = Cq; N = heads * 64; col = g * 64; }
    else if (g < heads + kv_heads) { C = qkv.Ck; N = kv_heads * 64; col = (g - heads) * 64; }
    else { C = qkv.Cv; N = kv_heads * 64; col = (g - heads - kv_heads) * 64; }
    if (g < heads + kv_heads) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float cs[8];
        unpack8(*reinterpret_cast<const uint4*>(ang + 16 * q), cs);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x1 = round_bf16(acc[2 * h][4 * q + e]), x2 = round_bf16(acc[2 * h + 1][4 * q + e]);
          const float c = cs[2 * e], sn = cs[2 * e + 1];
          acc[2 * h][4 * q + e] = x1 * c - x2 * sn;
          acc[2 * h + 1][4 * q + e] = x2 * c + x1 * sn;
        }
      }
    }
    if (m < Mv) {
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          bf16_t* p = C + (size_t)m * N + col + 32 * half + 8 * q + 4 * kh;
          const f32x16& a = acc[2 * h + half];
          *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(a[4 * q], a[4 * q + 1]), pack_bf16(a[4 * q + 2], a[4 * q + 3]));
        }
    }
  }
}

__global__ __launch_bounds__(256) void qkv192_kernel(const bf16_t* __restrict__ A,
                                                     const bf16_t* __restrict__ Bq, bf16_t* __restrict__ Cq,
                                                     int M, int heads, int kv_heads, int K,
                                                     const int* __restrict__ valid, int tiles_m, int tiles_n,
                                                     int patched, QkvTail qkv) {
  to_cache_rows(qkv, valid, M);
  qkv_heads_body<3>(A, Bq, Cq, M, heads, kv_heads, K, valid, tiles_m, tiles_n, patched, qkv);
}

__global__ __launch_bounds__(256) void qkv64_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bq,
                                                    bf16_t* __restrict__ Cq, int M, int heads, int kv_heads, int K,
                                                    const int* __restrict__ valid, int tiles_m, int tiles_n,
                                                    int patched, QkvTail qkv) {
  to_cache_rows(qkv, valid, M);
  qkv_heads_body<1>(A, Bq, Cq, M, heads, kv_heads, K, valid, tiles_m, tiles_n, patched, qkv);
}

// Both tilings in one launch: the row bound is read on the device, and which tiling makes fewer
// rounds over the chip depends on it, so the blocks choose -- the 192-wide tiles when the bound is
// past `above` (if wide_top, else when it is not), the 128-wide ones otherwise.  The grid is the
// larger of the two; a block past its tiling's tiles leaves at once.
struct Tiling {
  int tiles_m, tiles_n, patched;
};
__global__ __launch_bounds__(256) void qkv_either_kernel(const bf16_t* __restrict__ A,
                                                         const bf16_t* __restrict__ Bq, bf16_t* __restrict__ Cq,
                                                         int M, int heads, int kv_heads, int K,
                                                         const int* __restrict__ valid, Tiling narrow, Tiling wide,
                                                         Tiling thin, int above, int wide_top, int thin_upto,
                                                         int half_upto, int low_upto, QkvTail qkv) {
  const int Mv = bound_or(valid, M);
  const bool past = Mv > above;
  to_cache_rows(qkv, valid, M);
  const bool longs = K % LONG_K == 0 && (heads + 2 * kv_heads) * 4 <= min(256, (int)gridDim.x);
  if (longs && Mv <= 32) {
    gemm_long_body<LONG_QKV, 32, 5>(A, Bq, Cq, heads * 64, K, Mv, qkv);
  } else if (longs && Mv <= 64) {
    gemm_long_body<LONG_QKV, 64, 3>(A, Bq, Cq, heads * 64, K, Mv, qkv);
  } else if (Mv <= half_upto) {   // ... or half-head ones of 64 rows
    gemm_nt64_body<10, false, 1, 4, 2, true>(A, Bq, Cq, M, heads * 64, K, Mv, (M + 63) / 64, (heads + 2 * kv_heads) * 2, 0, qkv);
  } else if (Mv <= low_upto) {
    gemm_nt64_body<8, false, 2, 2, 2, true>(A, Bq, Cq, M, heads * 64, K, Mv, (M + 63) / 64, heads + 2 * kv_heads, 0, qkv);
  } else if (Mv <= thin_upto) {   // so few rows that one-head tiles still fit one round over the chip
    if ((int)blockIdx.x < thin.tiles_m * thin.tiles_n)
      qkv_heads_body<1>(A, Bq, Cq, M, heads, kv_heads, K, valid, thin.tiles_m, thin.tiles_n, thin.patched, qkv);
  } else if (wide.tiles_n > 0 && past == (wide_top != 0)) {
    if ((int)blockIdx.x < wide.tiles_m * wide.tiles_n)
      qkv_heads_body<3>(A, Bq, Cq, M, heads, kv_heads, K, valid, wide.tiles_m, wide.tiles_n, wide.patched, qkv);
  } else {
    if ((int)blockIdx.x < narrow.tiles_m * narrow.tiles_n)
      gemm_nt16_body<true>(A, Bq, Cq, M, heads * 64, K, Mv, narrow.tiles_m, narrow.tiles_n, narrow.patched, qkv);
  }
}

static int patched_order(int tiles_m, int tiles_n) {
  return (tiles_m % 8 == 0 && tiles_n % 4 == 0 && ((tiles_m / 8) * (tiles_n / 4)) % 8 == 0) ? 1 : 0;
}

// The rows up to which 64-row tiles of `columns` (a whole head's 64 or 32, q | k | v of `total` heads) are one round over the chip: few rows wait
// for what a CU draws, so a tile of fewer operand rows is the faster one as long as each has a CU of its own.  Hidden 2048, 32 + 8 + 8 heads,
// weights out of memory, us by 128 x 64 tiles and by these (up to 64 rows gemm_long_body's are the faster): 8 rows 15.8 / 10.0, 45 15.9 / 10.1, 128 16.5 / 10.2, 200 16.2 / 12.4, 320 16.4 / 13.0.
static int few_qkv_rows(int total, int K, int columns) { return K < 8 * BK ? 0 : 256 / (total * 64 / columns) * 64; }
// wide_ok: the head count comes in threes (else the 192-wide tiling is never chosen).  thin_upto: the
// row bound up to which the one-head tiles run (0: never).
static int launch_qkv_either(const bf16_t* A, const bf16_t* Bq, bf16_t* Cq, int M, int heads, int kv_heads, int K,
                             const int* valid, hipStream_t s, QkvTail qkv, int above, bool wide_top, bool wide_ok,
                             int thin_upto) {
  const int tiles_m = (M + 127) / 128, total = heads + 2 * kv_heads;
  const Tiling narrow{tiles_m, total / 2, patched_order(tiles_m, total / 2)};
  const Tiling wide{wide_ok ? tiles_m : 0, wide_ok ? total / 3 : 0, wide_ok ? patched_order(tiles_m, total / 3) : 0};
  const int thin_m = (thin_upto + 127) / 128;
  const Tiling thin{thin_m, total, patched_order(thin_m, total)};
  constexpr size_t lds_narrow = (size_t)NT_STAGES * 256 * BK * 2, lds_wide = (size_t)Q3_STAGES * Q3_STAGE_BYTES;
  constexpr size_t lds = lds_narrow > lds_wide ? lds_narrow : lds_wide;
  static_assert(lds >= (size_t)long_lds(32, 16, 5) && lds >= (size_t)long_lds(64, 16, 3), "the few rows' stages fit too");
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&qkv_either_kernel), lds); e != hipSuccess) {
    set_error("prefill_qkv: %s", hipGetErrorString(e));
    return (int)e;
  }
  int blocks = tiles_m * (narrow.tiles_n > wide.tiles_n ? narrow.tiles_n : wide.tiles_n);
  if (thin.tiles_m * thin.tiles_n > blocks) blocks = thin.tiles_m * thin.tiles_n;
  const int half_upto = few_qkv_rows(total, K, 32), low_upto = few_qkv_rows(total, K, 64);
  if (blocks < 256 && low_upto > 0) blocks = 256;
  hipLaunchKernelGGL(qkv_either_kernel, dim3(blocks), dim3(256), lds, s, A, Bq, Cq, M, heads, kv_heads, K, valid, narrow,
                     wide, thin, above, wide_top ? 1 : 0, thin_upto, half_upto, low_upto, qkv);
  IRON_LAUNCH_CHECK();
}

static int launch_qkv64(const bf16_t* A, const bf16_t* Bq, bf16_t* Cq, int M, int heads, int kv_heads, int K,
                        const int* valid, hipStream_t s, QkvTail qkv) {
  const int tiles_m = (M + Q3_BM - 1) / Q3_BM, tiles_n = heads + 2 * kv_heads;
  const size_t lds = (size_t)Q1_STAGES * Q1_STAGE_BYTES;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&qkv64_kernel), lds); e != hipSuccess) {
    set_error("prefill_qkv: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(qkv64_kernel, dim3(tiles_m * tiles_n), dim3(256), lds, s, A, Bq, Cq, M, heads, kv_heads, K, valid,
                     tiles_m, tiles_n, patched_order(tiles_m, tiles_n), qkv);
  IRON_LAUNCH_CHECK();
}

static int launch_qkv192(const bf16_t* A, const bf16_t* Bq, bf16_t* Cq, int M, int heads, int kv_heads, int K,
                         const int* valid, hipStream_t s, QkvTail qkv) {
  const int tiles_m = (M + Q3_BM - 1) / Q3_BM, tiles_n = (heads + 2 * kv_heads) / 3;
  const size_t lds = (size_t)Q3_STAGES * Q3_STAGE_BYTES;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&qkv192_kernel), lds); e != hipSuccess) {
    set_error("prefill_qkv: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(qkv192_kernel, dim3(tiles_m * tiles_n), dim3(256), lds, s, A, Bq, Cq, M, heads, kv_heads, K, valid,
                     tiles_m, tiles_n, patched_order(tiles_m, tiles_n), qkv);
  IRON_LAUNCH_CHECK();
}

template <int BM, int BN, int WM, int WN>
static int launch_gemm(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, int b_nk,
                       int c_nm, const int* valid, const int* valid_k, hipStream_t s) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const size_t lds = (size_t)2 * (BM + BN) * LDK * sizeof(bf16_t);
  dim3 grid(tiles_m * tiles_n), block(256);
#define IRON_GEMM_LAUNCH(BNK, CNM)                                                          \
  do {                                                                                      \
    auto kern = gemm_kernel<BM, BN, WM, WN, BNK, CNM>;                                      \
    static LdsOptIn opt_in;                                                               \
    if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(kern), lds); e != hipSuccess) { \
      set_error("gemm: %s", hipGetErrorString(e));                                        \
      return (int)e;                                                                      \
    }                                                                                       \
    hipLaunchKernelGGL(kern, grid, block, lds, s, A, B, C, M, N, K, valid, valid_k, tiles_m, \
                       tiles_n);                                                            \
  } while (0)
  if (b_nk && c_nm) IRON_GEMM_LAUNCH(true, true);
  else if (b_nk) IRON_GEMM_LAUNCH(true, false);
  else if (c_nm) IRON_GEMM_LAUNCH(false, true);
  else IRON_GEMM_LAUNCH(false, false);
#undef IRON_GEMM_LAUNCH
  IRON_LAUNCH_CHECK();
}


// Large problems: whole tiles of up to 256 x 256 outputs on eight waves (two a SIMD: one's loads and fragment reads issue under the
// other's MFMAs; 2048 x 8192 x 2048 60.5 -> 56.5 us, 4096^3 111 -> 107.5 against four waves of 128 x 128; 8192^3 the same), stages of 64
// k fed straight into LDS.  Against the 128x128 kernel a CU pulls half as many global bytes per flop -- the 64 B/clk a CU can move
// from L2 into LDS is what bounds the smaller tile.  WM x WN waves, each owning MI x NT accumulator tiles of 16 x 16: the
// tile's height and width are then chosen by how the product's rounds over the chip come out (see big_tiling).  Within a wave
// the instruction stream still interleaves the next k-step's fragment reads and the next stages' loads with the MFMAs.  Where the
// blocks of one launch choose their tile size by a row bound (gemm_rows_kernel) the large tile is four waves of
// 128 x 128, as every other tiling of that launch is four waves.

// The operands of a gated feed-forward's two first projections beyond the gate's own.
struct GatedPair {
  const bf16_t* up;      // the up projection's weights, (N,K) as the gate's
  bf16_t* gate_out;      // where the gate's product goes, if anywhere
  int activation;
};

template <int WM_, int WN_, int MI_, int NT_>
struct BigTile {
  static constexpr int WM = WM_, WN = WN_, MI = MI_, NT = NT_, WAVES = WM * WN, BM = WM * MI * 16, BN = WN * NT * 16;
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, LDS_MOST = 160 * 1024;
  // B, which comes from memory where a weight is used once, is held three stages deep, A too where that fits, else two (weights out of memory,
  // us with two and with three stages of B: 2048 x 16384 x 2048 120 / 109, 2048 x 8192 x 2048 60.4 / 54.9, 4096^3 105 / 98; the same weights
  // again 105 either way, 8192^3 733 / 729).  Where the waves' loads do not come out even, those without rows go to 1 KB behind the stages.
  static constexpr int SPARE = BM / 8 % WAVES == 0 && BN / 8 % WAVES == 0 ? 0 : 1024;
  static constexpr int FIT = (LDS_MOST - SPARE) / (A_BYTES + B_BYTES);   // (tiles of four waves with room for more take four)
  static constexpr int B_STAGES = FIT >= 4 ? 4 : 3, A_STAGES = FIT >= 3 ? B_STAGES : 2, STAGES_BYTES = A_STAGES * A_BYTES + B_STAGES * B_BYTES;
  static constexpr int OUT_ROW_BYTES = NT * 32 + 16, OUT_BYTES = WAVES * MI * 16 * OUT_ROW_BYTES;
  static constexpr int LDS_BYTES = STAGES_BYTES + SPARE > OUT_BYTES ? STAGES_BYTES + SPARE : OUT_BYTES;
  static_assert(LDS_BYTES <= LDS_MOST, "a CU's LDS");
};

// PAIR: both first products of a gated feed-forward.  TAIL: a residual sum or a gate in the epilogue (N a multiple of 8).
template <class T, bool B_KN = false, bool STREAM_OUT = false, bool PAIR = false, bool TAIL = false>
__device__ __forceinline__ void gemm_big_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                              bf16_t* __restrict__ C, int M, int N, int K,
                                              int Mv, int tiles_m, int tiles_n,
                                              int patched, const GatedPair& pair = GatedPair{}, const QkvTail& tail = QkvTail{}) {
  constexpr int WAVES = T::WAVES, MI = T::MI, NT = T::NT, A_STAGES = T::A_STAGES, B_STAGES = T::B_STAGES;
  constexpr int ROWB = BK * 2;                                        // bytes of a tile row in LDS, eight 16-byte chunks
  constexpr int A_BYTES = T::A_BYTES, B_BYTES = T::B_BYTES, B_BASE = A_STAGES * A_BYTES;   // A's stages, then B's
  constexpr int A_INST = T::BM / 8, B_INST = T::BN / 8;               // 1 KB loads of a stage: eight rows each
  constexpr int A_EACH = (A_INST + WAVES - 1) / WAVES, B_EACH = (B_INST + WAVES - 1) / WAVES, LOADS = A_EACH + B_EACH;   // ... a wave's
  constexpr int A_LAST = A_INST % WAVES, B_LAST = B_INST % WAVES;     // waves that have a last one (0: all)
  extern __shared__ __align__(16) char smem_big[];

  int tm, tn;
  if (!live_tile(blockIdx.x, tiles_m, tiles_n, patched, (Mv + T::BM - 1) / T::BM, tm, tn)) return;
  if (tm * T::BM >= Mv) return;
  // The last tile of each direction is moved back to end at the matrix's edge, so that every tile is
  // whole; what two tiles both cover comes out the same from both.
  const int m0 = min(tm * T::BM, M - T::BM), n0 = PAIR ? tn * (T::BN / 2) : min(tn * T::BN, N - T::BN);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: LDS and global bases stay in scalar registers
  const int wm = wave / T::WN, wn = wave % T::WN;
  // Loader: a wave's instruction i moves rows 8 (i WAVES + wave) .. + 7; lane -> (row, physical chunk); the logical chunk it
  // fetches is the physical one swizzled by the row.  Loads go out as buffer loads straight into LDS: the lane's
  // place within an instruction's rows is the (constant) vector offset, the instruction's rows and the
  // stage's k are the scalar offset, so a load costs two scalar adds and no vector ALU work between two MFMAs.
  const int lrow = lane >> 3, ld_head = ((lane & 7) ^ ((wave & 1) * 4 + (lrow >> 1))) * 8;   // ld_head: the k of a stage at which the lane's piece begins
  static_assert(WAVES % 2 == 0, "a wave's instructions all begin on an even eight rows, or all on an odd");
  const int ld_off = (int)(((size_t)lrow * K + ld_head) * 2);
  const int pad = k_pad(K);
  // (A ends at its last live row: a load past it brings zeros and costs no traffic.)
  const __amdgpu_buffer_rsrc_t a_rows = bounded_bytes(A + (size_t)(m0 + wave * 8) * K - pad, (int)max(0L, min(0x7fffffffL, 2 * ((long)(Mv - m0 - wave * 8) * K + pad))));
  // B as (K,N) lands as stored: the stage's 64 k-rows of BN columns, a row's chunks XORed with kn_swizzle(row) so that the
  // transposing reads below find the four rows of a 16-lane group, and the groups of a pass, in different banks.
  constexpr int KN_CHUNKS = T::BN / 8, KN_ROWS = 64 / KN_CHUNKS;   // chunks of a k-row, k-rows of an instruction
  static_assert(!B_KN || KN_CHUNKS == 32, "(K,N): rows of 256 columns");
  auto kn_swizzle = [](int k) { return ((k & 3) << 1) | (((k >> 3) & 3) << 3); };
  // (PAIR: 8 NT rows of the gate's weights, as many of the up projection's, and so on.)
  const __amdgpu_buffer_rsrc_t b_rows = stage_rows(B_KN ? B + n0 + ((ptrdiff_t)(wave * KN_ROWS) - pad) * N : B + (size_t)(n0 + wave * 8) * K - pad);
  const __amdgpu_buffer_rsrc_t up_rows = PAIR ? stage_rows(pair.up + (size_t)(n0 + wave * 8) * K - pad) : b_rows;
  int kn_off[B_EACH], kn_row[B_EACH];   // (K,N): this lane's 16 bytes within instruction idx's k-rows, and the k-row
#pragma unroll
  for (int i = 0; i < B_EACH; ++i) {
    kn_row[i] = (i * WAVES + wave) * KN_ROWS + lane / KN_CHUNKS;
    kn_off[i] = (int)(((size_t)(lane / KN_CHUNKS) * N + ((lane % KN_CHUNKS) ^ kn_swizzle(kn_row[i])) * 8) * 2);
  }
  const int inst_stride = WAVES * 8 * K * 2;
  static_assert(!PAIR || (WAVES == 4 && NT % 4 == 0), "PAIR: the rows of an instruction below are four waves'");
  auto issue_one = [&](int a_at, int b_at, int kt, int idx, bool head) {
    const int k_off = kt * ROWB;
    const bool is_a = idx < A_EACH;
    const int i = is_a ? idx : idx - A_EACH;
    const int last = is_a ? A_LAST : B_LAST;
    // A wave without a last instruction issues it all the same, from past the buffer's end and to where nobody reads: every wave's
    // loads are then as many, which the waits count.
    const bool none = last != 0 && i == (is_a ? A_EACH : B_EACH) - 1 && wave >= last;
    char* to = smem_big + (none ? T::STAGES_BYTES : (is_a ? a_at : B_BASE + b_at) + (i * WAVES + wave) * 1024);
    if (is_a)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rows, IRON_LDS_PTR(to), 16, none || (head && ld_head < pad) ? NOWHERE : ld_off,
                                               i * inst_stride + k_off, 0, 0);
    else if constexpr (PAIR)   // (NT / 4 of four waves' instructions are a wave's columns of one weight)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i / (NT / 4) % 2 ? up_rows : b_rows, IRON_LDS_PTR(to), 16, head && ld_head < pad ? NOWHERE : ld_off,
                                               (i / (NT / 2) * (NT / 4) + i % (NT / 4)) * inst_stride + k_off, 0, 0);
    else if constexpr (!B_KN)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rows, IRON_LDS_PTR(to), 16, none || (head && ld_head < pad) ? NOWHERE : ld_off,
                                               i * inst_stride + k_off, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rows, IRON_LDS_PTR(to), 16, head && kn_row[i] < pad ? NOWHERE : kn_off[i],
                                               (i * WAVES * KN_ROWS + kt * BK) * N * 2, 0, 0);
  };

  // The product runs on 16x16x32 MFMAs (a k-step is 32 wide, two a stage): on random operands the
  // part sustains about a sixth more of them than of the 32x32x16 form, at the same registers and
  // the same LDS reads per flop.
  f32x4 acc[MI][NT];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;

  // Where a lane stores: lanes of 16 bytes a tile row, rows an instruction (of 96-byte rows ten: four lanes idle).
  constexpr int LPRW = NT * 2, ORPI = 64 / LPRW, PIECES = (MI * 16 + ORPI - 1) / ORPI;
  const int lr = lane / LPRW, lc = lane % LPRW;
  const int row0 = m0 + wm * MI * 16;
  // A residual's pieces this lane will add in the epilogue are requested now, so that their latency passes under the product.
  uint4 res[TAIL ? PIECES : 1];
  if constexpr (TAIL) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      res[i] = *reinterpret_cast<const uint4*>(tail.residual + (size_t)min(row0 + i * ORPI + lr, M - 1) * N + n0 + wn * NT * 16 + lc * 8);
  }

  const int nk = (K + pad) / BK;
  // A stage is two k-steps of MI NT MFMAs; source order is issue order (nothing crosses a sched_barrier): after an MFMA one
  // fragment read or one load goes out.  A k-step's first MFMAs need all of its B fragments and its first A fragment, so
  // B's are read first.
  //   first k-step: the second's B fragments from the start and its A fragments from the middle; loads in the slots between (EARLY of them)
  //   second k-step: up to slot BARRIER nothing -- then the stage's one barrier: every wave's loads of stage kt + 1 have landed and
  //     nobody reads stage kt any more (this k-step's fragments are in registers) -- then stage kt + 1's first fragments and LATE loads
  // B's loads, and with as many stages A's, are stage kt + B_STAGES - 1's and begin in the first k-step: the last barrier freed their buffer.  A's,
  // with two stages, are stage kt + 2's and the late ones, into this stage's buffer.
  static_assert(A_STAGES == B_STAGES || (A_STAGES == 2 && B_STAGES == 3), "stages alike, or two of A and three of B");
  constexpr int SLOTS = MI * NT, A_FROM = NT > SLOTS / 2 ? NT : SLOTS / 2, FREE = SLOTS - NT - MI;
  constexpr int EARLY = A_STAGES == 2 ? B_EACH : (LOADS < FREE ? LOADS : FREE), LATE = LOADS - EARLY;
  constexpr int EARLY_FROM = A_STAGES == 2 ? A_EACH : 0, LATE_FROM = A_STAGES == 2 ? 0 : EARLY;   // their numbers
  constexpr int BARRIER = SLOTS - NT - MI - LATE < SLOTS / 2 ? SLOTS - NT - MI - LATE : SLOTS / 2;
  static_assert(A_FROM + MI <= SLOTS && EARLY <= FREE && BARRIER >= 0, "a k-step has a slot for each of its reads and loads");
  constexpr int GAP = A_FROM - NT, APART = EARLY > 0 && GAP / EARLY > 1 ? GAP / EARLY : 1;   // slots between the B and the A reads
  constexpr int IN_GAP = EARLY < GAP / APART ? EARLY : GAP / APART;
  constexpr int Q3_FIRST = BARRIER + NT + MI, Q3_EVERY = SLOTS - Q3_FIRST > 2 * LATE && LATE > 0 ? (SLOTS - Q3_FIRST) / (LATE > 0 ? LATE : 1) : 1;
#pragma unroll
  for (int st = 0; st < B_STAGES - 1; ++st)
#pragma unroll
    for (int idx = 0; idx < LOADS; ++idx) issue_one(st * A_BYTES, st * B_BYTES, min(st, nk - 1), idx, st == 0);

  // Fragments: lane -> row fr of a 16-row tile, 16-byte chunk kq of the k-step's four.
  const int fr = lane & 15, kq = lane >> 4;
  const int swz = fr >> 1;   // tile rows are multiples of 16 apart: one swizzle for all
  const int a_row = (wm * MI * 16 + fr) * ROWB, b_row = B_BASE + (wn * NT * 16 + fr) * ROWB;
  auto a_frag = [&](int at, int ks, int i) {
    return *reinterpret_cast<const bf16x8*>(smem_big + at + a_row + i * 16 * ROWB + (((ks * 4 + kq) ^ swz) << 4));
  };
  auto b_frag = [&](int at, int ks, int j) {
    return *reinterpret_cast<const bf16x8*>(smem_big + at + b_row + j * 16 * ROWB + (((ks * 4 + kq) ^ swz) << 4));
  };
  // (K,N): the B operand of tile j wants, for column n = 16 j + fr, the k-step's k = 8 kq .. + 7.  A
  // transposing read hands a 16-lane group the 4 x 16 block its lanes point at (4 k-rows, each
  // lane 4 columns) turned round: the lane gets 4 k of one column.  Rows 8 kq .. + 3 and 8 kq + 4 .. + 7.
  const int tr_k = 8 * kq + ((lane & 15) >> 2), tr_n = wn * NT * 16 + 4 * (lane & 3);
  const unsigned lds_base_big = (unsigned)(size_t)IRON_LDS_PTR(smem_big);
  const unsigned kn_base = lds_base_big + B_BASE;
  // The lane's place in a stage's B tile for tile j (k-step 0, low half) is fixed before the loop; the
  // k-step (32 rows on) and the high half (4 rows on) leave the swizzle as it is and ride in the
  // reads' offset fields, so a k-step's reads cost one vector add a tile (the stage) and no more.
  // (Unrolled over its two stage buffers so that the stage too is an offset field, as the 128 x 128
  // loop is, this kernel spilled a hundred registers: two waves a SIMD leave it 256.)
  unsigned kn_lane[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = tr_n + j * 16;
    kn_lane[j] = kn_base + (((n >> 3) ^ kn_swizzle(tr_k)) << 4) + ((n & 4) << 1) + tr_k * (T::BN * 2);
  }
  auto b_frag_kn = [&](int stage_bytes, int ks, int j, TrFrag& t) {
    const unsigned at = kn_lane[j] + stage_bytes;
    if (ks == 0) {
      t.lo = lds_read_tr16_at<0>(at);
      t.hi = lds_read_tr16_at<4 * T::BN * 2>(at);
    } else {
      t.lo = lds_read_tr16_at<32 * T::BN * 2>(at);
      t.hi = lds_read_tr16_at<36 * T::BN * 2>(at);
    }
  };
  // (K,N): the A fragments are read by uncounted reads as well, so that every wait of the loop is
  // this code's own (the compiler's waits for counted A reads take no account of the transposing
  // reads issued in between and come out far too strict).  A k-step's fragments, A's and B's, are
  // all issued before join_b's wait at its start, which they pass through.
  const unsigned a_lane[2] = {lds_base_big + a_row + (((0 * 4 + kq) ^ swz) << 4), lds_base_big + a_row + (((1 * 4 + kq) ^ swz) << 4)};
  auto a_frag_kn = [&](int stage_bytes, int ks, int i, bf16x8& out) {
    const unsigned at = a_lane[ks] + stage_bytes;
    if (i == 0) out = lds_read_b128_at<0 * 16 * ROWB>(at);
    else if (i == 1) out = lds_read_b128_at<1 * 16 * ROWB>(at);
    else if (i == 2) out = lds_read_b128_at<2 * 16 * ROWB>(at);
    else if (i == 3) out = lds_read_b128_at<3 * 16 * ROWB>(at);
    else if (i == 4) out = lds_read_b128_at<4 * 16 * ROWB>(at);
    else if (i == 5) out = lds_read_b128_at<5 * 16 * ROWB>(at);
    else if (i == 6) out = lds_read_b128_at<6 * 16 * ROWB>(at);
    else out = lds_read_b128_at<7 * 16 * ROWB>(at);
  };
  TrFrag tfb[2][NT];
  bf16x8 af[2][MI], bfr[2][NT];
  // The compiler does not count these reads: a k-step's fragments pass through this wait (every LDS
  // read issued so far) before they are used.
  auto join_kn = [&](int ks) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < NT; ++j) asm volatile("" : "+v"(tfb[ks][j].lo), "+v"(tfb[ks][j].hi));
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      i32x4 a = __builtin_bit_cast(i32x4, af[ks][i]);
      asm volatile("" : "+v"(a));
      af[ks][i] = __builtin_bit_cast(bf16x8, a);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) bfr[ks][j] = tr_join(tfb[ks][j]);
  };

  wait_vmcnt<(B_STAGES - 2) * LOADS>();   // stage 0 has landed once only the younger ones are out
  block_barrier();
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if constexpr (B_KN) a_frag_kn(0, 0, i, af[0][i]);
    else af[0][i] = a_frag(0, 0, i);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if constexpr (B_KN) b_frag_kn(0, 0, j, tfb[0][j]);
    else bfr[0][j] = b_frag(0, 0, j);
  }
  // Where this stage's A and B lie, the next one's, and what the loads fill.
  int a_now = 0, a_next = A_BYTES, a_fill = A_STAGES == 2 ? 0 : (A_STAGES - 1) * A_BYTES, b_now = 0, b_next = B_BYTES, b_fill = (B_STAGES - 1) * B_BYTES;
  for (int kt = 0; kt < nk; ++kt) {
    // Past the end the last stage is fetched again (into buffers nobody reads any more) rather than
    // branch: a branch would end the scheduling region and undo the interleaving below.
    const int k2 = min(kt + B_STAGES - 1, nk - 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if constexpr (B_KN) join_kn(ks);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int slot = i * NT + j;
          if (ks == 1 && slot == BARRIER) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            wait_vmcnt<(B_STAGES - 3) * LOADS + EARLY>();   // all but the stages behind the next one
            block_barrier();
          }
          mfma_16x16x32_in_place(acc[i][j], bfr[ks][j], af[ks][i]);
          __builtin_amdgcn_sched_barrier(0);
          if (ks == 0) {
            if (slot < NT) {
              if constexpr (B_KN) b_frag_kn(b_now, 1, slot, tfb[1][slot]);
              else bfr[1][slot] = b_frag(b_now, 1, slot);
            } else if (slot >= A_FROM && slot < A_FROM + MI) {
              if constexpr (B_KN) a_frag_kn(a_now, 1, slot - A_FROM, af[1][slot - A_FROM]);
              else af[1][slot - A_FROM] = a_frag(a_now, 1, slot - A_FROM);
            } else {
              const int nth = slot < A_FROM ? ((slot - NT) % APART == 0 && (slot - NT) / APART < IN_GAP ? (slot - NT) / APART : EARLY)
                                            : IN_GAP + slot - A_FROM - MI;
              if (nth < EARLY) issue_one(a_fill, b_fill, k2, EARLY_FROM + nth, false);
            }
          } else if (slot >= BARRIER) {
            if (slot < BARRIER + NT) {
              if constexpr (B_KN) b_frag_kn(b_next, 0, slot - BARRIER, tfb[0][slot - BARRIER]);
              else bfr[0][slot - BARRIER] = b_frag(b_next, 0, slot - BARRIER);
            } else if (slot < Q3_FIRST) {
              if constexpr (B_KN) a_frag_kn(a_next, 0, slot - BARRIER - NT, af[0][slot - BARRIER - NT]);
              else af[0][slot - BARRIER - NT] = a_frag(a_next, 0, slot - BARRIER - NT);
            } else if ((slot - Q3_FIRST) % Q3_EVERY == 0 && (slot - Q3_FIRST) / Q3_EVERY < LATE) {
              issue_one(a_fill, b_fill, k2, LATE_FROM + (slot - Q3_FIRST) / Q3_EVERY, false);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    b_fill = b_now;
    a_fill = A_STAGES == 2 ? a_next : a_now;
    a_now = a_next;
    b_now = b_next;
    a_next = a_now == (A_STAGES - 1) * A_BYTES ? 0 : a_now + A_BYTES;
    b_next = b_now == (B_STAGES - 1) * B_BYTES ? 0 : b_now + B_BYTES;
  }

  if constexpr (B_KN) join_kn(0);   // the idle reads of the last iteration land while their registers are still theirs
  wait_vmcnt<0>();   // ... and its idle fetch before LDS is reused
  block_barrier();   // every wave is done reading the stages

  if constexpr (PAIR) {
    // Columns 0 .. NT / 2 - 1 of the wave's tiles are the gate's product, the rest the up projection's, of
    // the same 8 NT columns of the output: the gate's product leaves as it is stored, where it is asked for, then, made in the
    // accumulators' own layout, bf16(bf16(act(bf16 g)) * bf16 u).
    constexpr int HT = NT / 2, OROWB = HT * 32 + 16, LPRW = HT * 2, ORPI = 64 / LPRW;   // (half a tile's columns at a time)
    constexpr int ROWS = MI * 16;   // of a wave
    char* ot = smem_big + wave * (ROWS * OROWB);
    const int lr = lane / LPRW, lc = lane % LPRW;
    const size_t first = (size_t)(m0 + wm * ROWS) * N + n0 + wn * HT * 16 + lc * 8;
    auto leave = [&](bf16_t* to) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 4
      for (int r0 = 0; r0 < ROWS; r0 += ORPI) {
        const int r = r0 + lr;
        const uint4 v = *reinterpret_cast<const uint4*>(ot + r * OROWB + lc * 16);
        if (m0 + wm * ROWS + r < Mv) *reinterpret_cast<uint4*>(to + first + (size_t)r * N) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();   // the rows are read before the next product overwrites them
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // (The kind of gate is chosen once: asked an element, its branches made the lone wave of a SIMD wait 128 times over, and a
    // 2048 x 8192 x 2048 pair take 143 us instead of 130.)
    if (pair.gate_out != nullptr) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < HT; ++j)
          *reinterpret_cast<uint2*>(ot + (i * 16 + fr) * OROWB + (j * 16 + 4 * kq) * 2) =
              make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
      leave(pair.gate_out);
    }
    auto gated = [&](auto kind) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      // A tile row at a time leaves the accumulation registers: all at once they would not fit.
#pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        float c[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          c[e] = round_bf16(gate_of(decltype(kind)::value, round_bf16(acc[i][j][e]))) * round_bf16(acc[i][j + HT][e]);
        *reinterpret_cast<uint2*>(ot + (i * 16 + fr) * OROWB + (j * 16 + 4 * kq) * 2) =
            make_uint2(pack_bf16(c[0], c[1]), pack_bf16(c[2], c[3]));
      }
    }
    };
    if (pair.activation == 1) gated(std::integral_constant<int, 1>{});
    else if (pair.activation == 2) gated(std::integral_constant<int, 2>{});
    else gated(std::integral_constant<int, 3>{});
    leave(C);
    return;
  }
  // Output through LDS: a wave lays its (16 MI) x (16 NT) tile out row-major (rows padded by 16 bytes,
  // which spreads both the 8-byte writes below and the 16-byte reads over all banks) and stores
  // whole 16-byte pieces, so a row of the tile leaves as one contiguous segment.
  // acc[i][j][e]: row fr of A tile i, column 4*kq + e of B tile j.
  constexpr int OROWB = T::OUT_ROW_BYTES;
  char* ot = smem_big + wave * (MI * 16 * OROWB);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *reinterpret_cast<uint2*>(ot + (i * 16 + fr) * OROWB + (j * 16 + 4 * kq) * 2) =
          make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
  // The tile is private to the wave, whose LDS operations execute in order: no block barrier,
  // only a fence to keep the compiler from moving the reads above other lanes' writes.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  bf16_t* cbase = C + (size_t)row0 * N + n0 + wn * NT * 16 + lc * 8;
  // STREAM_OUT (the launch sets it over a long K): the tile leaves by non-temporal stores, so C's
  // lines do not stay in the XCD's L2 among the A and B panels its blocks re-read (8192^3: 790 ->
  // 750 us; 1 to 5 % from K = 4096 on, and 1.5 % slower at K = 2048, where a tile's stores are a
  // larger part of its time).  A template argument: as a branch on K the compiler merged the two
  // stores into one plain one.
  typedef unsigned int u32x4_t __attribute__((ext_vector_type(4), aligned(2)));   // (rows begin where they begin, see store_loose)
#pragma unroll TAIL ? PIECES : 4
  for (int r0 = 0; r0 < MI * 16; r0 += ORPI) {
    const int r = r0 + lr;
    if (64 % LPRW != 0 && (lr >= ORPI || r >= MI * 16)) continue;
    uint4 v = *reinterpret_cast<const uint4*>(ot + r * OROWB + lc * 16);
    if constexpr (TAIL) {   // the product rounded as it would be stored, then scale * it + residual, or its gate
      float x[8], rf[8];
      unpack8(v, x);
      unpack8(res[r0 / ORPI], rf);
      tail_of(tail, x, rf);
      v = pack8(x);
    }
    // (TAIL: C may be the residual itself, so what two tiles both cover is one's to store)
    if (row0 + r < Mv && (!TAIL || (row0 + r >= tm * T::BM && n0 + wn * NT * 16 + lc * 8 >= tn * T::BN))) {
      if constexpr (STREAM_OUT)
        __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, v), reinterpret_cast<u32x4_t*>(cbase + (size_t)r * N));
      else
        store_loose(cbase + (size_t)r * N, v);
    }
  }
}

typedef BigTile<2, 4, 8, 4> Tile256;       // 256 x 256, eight waves
typedef BigTile<2, 4, 7, 4> Tile224x256;
typedef BigTile<2, 4, 6, 4> Tile192x256;
typedef BigTile<2, 4, 5, 4> Tile160x256;
typedef BigTile<2, 4, 4, 4> Tile128x256;
typedef BigTile<2, 4, 4, 3> Tile128x192;   // B (N,K) only, and the following
typedef BigTile<2, 2, 3, 4> Tile96x128;    // four waves
typedef BigTile<2, 2, 8, 8> Tile256Four;   // 256 x 256 by four waves, for launches whose other tilings are four waves

template <class T, bool B_KN = false, bool STREAM_OUT = false>
__global__ __launch_bounds__(T::WAVES * 64) void gemm_big_kernel(const bf16_t* __restrict__ A,
                                                                 const bf16_t* __restrict__ B,
                                                                 bf16_t* __restrict__ C, int M, int N, int K,
                                                                 const int* __restrict__ valid, int tiles_m,
                                                                 int tiles_n, int patched) {
  gemm_big_body<T, B_KN, STREAM_OUT>(A, B, C, M, N, K, bound_or(valid, M), tiles_m, tiles_n, patched);
}

// Which form a launch under a row bound takes: the price list's, read by the bound where it is known, on the device.  Four bits for each run of
// 64 << shift rows (the words are chosen by tests, not by an index: that would be another trip to memory behind the bound's), and a bit for each
// form whose tiles come in patches.
struct FormTable {
  uint64_t w[4];
  int shift, patched;
};
struct FormOfRows {
  int rows, form, patched;
};
__device__ __forceinline__ FormOfRows form_of_rows(const FormTable& t, const int* __restrict__ valid, int M) {
  uint64_t w0 = t.w[0], w1 = t.w[1], w2 = t.w[2], w3 = t.w[3];
  int shift = t.shift, patched = t.patched, bound = valid == nullptr ? M : *valid;
  asm volatile("" : "+s"(w0), "+s"(w1), "+s"(w2), "+s"(w3), "+s"(shift), "+s"(patched), "+s"(bound));   // (one wait for the bound and the table)
  const int rows = max(0, min(bound, M)), run = max(rows - 1, 0) >> (6 + shift);
  const uint64_t w = run < 32 ? (run < 16 ? w0 : w1) : (run < 48 ? w2 : w3);
  const int form = (int)(w >> ((run & 15) * 4)) & 15;
  return FormOfRows{rows, form, patched >> form & 1};
}
static int form_of_rows(const FormTable& t, int rows) {
  const int run = (rows < 1 ? 0 : rows - 1) >> (6 + t.shift);
  return (int)(t.w[run >> 4] >> ((run & 15) * 4)) & 15;
}
// `best(rows)` for the most rows of every run up to M, without a bound for M alone; `upto[form]`: the most rows a form is taken for.
template <class Best>
static FormTable form_table(int M, bool bounded, Best best, int* upto) {
  FormTable t{};
  while ((64L << t.shift) * 64 < M) ++t.shift;
  const long run = 64L << t.shift;
  for (long rows = bounded ? run : M, i = 0; rows < M + run; rows += run, ++i) {
    const int r = rows < M ? (int)rows : M, form = best(r);
    if (bounded) t.w[i >> 4] |= (uint64_t)form << ((i & 15) * 4);
    else for (uint64_t& w : t.w) w = (uint64_t)form * 0x1111111111111111u;
    if (r > upto[form]) upto[form] = r;
  }
  return t;
}

// Whether a launch of `blocks` blocks that has chosen its tiles of 32 x 32 (64 x (32 + 32) of a gated pair) makes up to 32 rows by long stages instead.  The blocks
// are as many as the chosen tiles need, at most for all rows of the bound's buffer, so a buffer of few rows may have too few for a tile of eight columns a block
// (64 rows of 2048 columns over 2048 are 128 tiles of 32 x 32): those keep the tiles.
__device__ __host__ inline bool rows_by_long_stages(int rows, int N, int K, int blocks) {
  return rows <= 32 && K % LONG_K == 0 && N % 8 == 0 && N / 8 <= (blocks < 256 ? blocks : 256);
}
__device__ __host__ inline bool pair_by_long_stages(int rows, int N, int K) { return rows <= 32 && K % LONG_K == 0 && N % 32 == 0; }

// A product under a row bound that is read on the device: the blocks of ONE launch take the form that is the cheapest at the bound (512 valid rows of
// 2048 leave 64 of 256 large tiles).  Each form's grid covers only the rows it can be chosen for; the launch's grid is the largest of
// them and a block past its tiling's tiles leaves at once.  LDS is the largest tiling's, so a CU
// holds one block whatever the choice, and four waves are a block whatever the stand-alone launch of a form uses.
// The prices: rounds of blocks, as big_form, at what a round was measured to take with weights out of memory behind the launch's own 4.5 us (by 64 x 64,
// 128 x 128 and 256 x 256 tiles alone and by all these, us: 2048 columns over 2048 with a residual, 640 rows 19.9 / 17.7, 1024 23.7 / 18.4; over 8192, 900
// rows 68 / 52; 8192 over 2048, 256 rows 22.9 / 18.6, 640 42 / 26, 1024 43 / 34, 1280 50 / 39; 6144 over 2048, 1200 rows 54 / 32).
// Up to K = 1536 a round is mostly its start and its end, which tiles with a second operand pay twice: prices of their own, [0] without one and [1] with, fitted to 1800
// launches of every form up to 1024, of which the cheapest by them takes 1.0002 of the best on average and 1.03 at the most (by the long K's prices 1.08 below
// K = 512, 1.02 from there on, and up to 2.1: 2048 x 2560 x 64 by 64 x 64 tiles 15.5, by 192 x 128 7.2; 2048 x 6144 x 512 27.3 / 20.0; from 1088 to 1536
// 87 launches of few rows by many columns 1.002 and 1.11: 3 rows of 64 x 26574 x 1152 with a second operand by two rounds of 64 x 64 tiles 21.2, by one of 128 x 128 15.9).
enum RowsForm { ROWS_32X32, ROWS_64X32, ROWS_64X64, ROWS_128X64, ROWS_128X128, ROWS_96X128, ROWS_160X128, ROWS_192X128, ROWS_224X128, ROWS_256X128, ROWS_160X256, ROWS_192X256, ROWS_224X256,
                ROWS_256X256, ROWS_FORMS };
constexpr int SHORT_STAGES = 24;
struct RoundPrice {
  float start, stage;
};
struct RowsPrice {
  int bm, bn;
  RoundPrice long_k, short_k[2];
};
constexpr RowsPrice ROWS_PRICES[ROWS_FORMS] = {
    {32, 32, {0.8f, 0.15f}, {{2.f, 0.142f}, {2.2f, 0.146f}}},     {64, 32, {0.8f, 0.2f}, {{2.45f, 0.171f}, {2.85f, 0.17f}}},
    {64, 64, {0.8f, 0.28f}, {{2.5f, 0.235f}, {3.3f, 0.235f}}},    {128, 64, {2.f, 0.34f}, {{3.05f, 0.357f}, {4.55f, 0.362f}}},
    {128, 128, {4.f, 0.45f}, {{3.4f, 0.515f}, {5.1f, 0.53f}}},    {96, 128, {3.4f, 0.39f}, {{3.3f, 0.46f}, {4.8f, 0.47f}}},
    {160, 128, {3.4f, 0.52f}, {{3.4f, 0.583f}, {5.4f, 0.6f}}},
    {192, 128, {5.f, 0.57f}, {{3.9f, 0.645f}, {6.f, 0.665f}}},    {224, 128, {5.7f, 0.63f}, {{4.1f, 0.69f}, {7.5f, 0.71f}}},
    {256, 128, {6.5f, 0.69f}, {{4.3f, 0.743f}, {9.f, 0.76f}}},
    {160, 256, {8.f, 0.8f}, {{4.85f, 0.872f}, {10.5f, 0.93f}}},   {192, 256, {9.f, 0.85f}, {{5.5f, 0.9f}, {13.f, 0.96f}}},
    {224, 256, {12.f, 0.93f}, {{6.1f, 1.f}, {16.5f, 1.07f}}},
    {256, 256, {15.f, 1.f}, {{6.7f, 1.1f}, {20.f, 1.19f}}},
};
// Tiles of 96 and 224 rows are for the runs of rows that leave the last round of the others' a quarter empty; up to K = 512, where a round is its start and its end, a
// twentieth at the most (256 blocks, 4096 columns, us by 96 x 128 / 128 x 128 tiles: K = 256 8.5 / 8.8, 512 9.9 / 10.2, 1024 12.6 / 13.4, 2048 21.5 / 23.9, 8192 63.3 / 72.9; by 192, 224
// and 256 x 256: K = 2048 46.6, 50.6, 55.1), so they begin past that.  2048 columns over 2048, 1102 rows 17.3 / 15.1, over 8192, 1379 rows 62.9 / 54.3; 10240 over 2048, 213 rows
// 21.8 / 18.8; 4544 over 5184, 615 rows 51.0 / 41.3; of 280 drawn ones 58 take them, at 0.90 of the time.
struct RowsChoice {
  RowsForm form;
  float us;
};
// `second`: the product has a second operand.
static RowsChoice rows_form(int rows, int M, int N, int K, bool second) {
  const int stages = (K + BK - 1) / BK;
  const RowsForm first = K < 8 * BK ? ROWS_64X64 : ROWS_32X32;   // (a short K does not fill the small tiles' many stages)
  RowsChoice best{first, 0.f};
  for (int form = first; form < ROWS_FORMS; ++form) {
    const RowsPrice& p = ROWS_PRICES[form];
    if (form > ROWS_128X128 && (M < p.bm || N < p.bn || (second && N % 8 != 0))) continue;
    if (stages <= 8 && (form == ROWS_96X128 || form == ROWS_224X128 || form == ROWS_224X256)) continue;
    const RoundPrice& of = stages > SHORT_STAGES ? p.long_k : p.short_k[second];
    const long tiles = (long)((rows + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
    const float us = (float)((tiles + 255) / 256) * (of.start + of.stage * stages);
    if (form == first || us < best.us) best = {(RowsForm)form, us};
  }
  return best;
}
template <bool TAIL>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, bf16_t* __restrict__ C,
                                                        int M, int N, int K, const int* __restrict__ valid, FormTable forms, QkvTail tail) {
  const FormOfRows chosen = form_of_rows(forms, valid, M);
  const int Mv = chosen.rows, patched = chosen.patched;
#define IRON_ROWS(FORM, MI, NT) \
  case FORM: \
    static_assert(ROWS_PRICES[FORM].bm == 32 * MI && ROWS_PRICES[FORM].bn == 32 * NT, "the tile that was priced"); \
    gemm_big_body<BigTile<2, 2, MI, NT>, false, false, false, TAIL>(A, B, C, M, N, K, Mv, (M + 32 * MI - 1) / (32 * MI), (N + 32 * NT - 1) / (32 * NT), \
                                                                    patched, GatedPair{}, tail); \
    break
  switch (chosen.form) {
    IRON_ROWS(ROWS_96X128, 3, 4);
    IRON_ROWS(ROWS_160X128, 5, 4);
    IRON_ROWS(ROWS_192X128, 6, 4);
    IRON_ROWS(ROWS_224X128, 7, 4);
    IRON_ROWS(ROWS_256X128, 8, 4);
    IRON_ROWS(ROWS_160X256, 5, 8);
    IRON_ROWS(ROWS_192X256, 6, 8);
    IRON_ROWS(ROWS_224X256, 7, 8);
    IRON_ROWS(ROWS_256X256, 8, 8);
    case ROWS_128X128:
      gemm_nt16_body<false>(A, B, C, M, N, K, Mv, (M + 127) / 128, (N + 127) / 128, patched, tail);
      break;
    case ROWS_128X64:
      gemm_nt64_body<5, false, 4>(A, B, C, M, N, K, Mv, (M + 127) / 128, (N + 63) / 64, patched, tail);
      break;
    case ROWS_64X64:
      gemm_nt64_body<8>(A, B, C, M, N, K, Mv, (M + 63) / 64, (N + 63) / 64, patched, tail);
      break;
    case ROWS_64X32:
      gemm_nt64_body<13, false, 1, 4>(A, B, C, M, N, K, Mv, (M + 63) / 64, (N + 31) / 32, patched, tail);
      break;
    default: {
      if (rows_by_long_stages(Mv, N, K, (int)gridDim.x)) gemm_long_body<LONG_PLAIN, 32, 7>(A, B, C, N, K, Mv, tail);
      else gemm_nt64_body<20, false, 1, 2, 1>(A, B, C, M, N, K, Mv, (M + 31) / 32, (N + 31) / 32, patched, tail);
    }
  }
#undef IRON_ROWS
}

// A launch whose blocks choose their form: the table that they choose by, and how many there are.
struct FormPlan {
  FormTable table;
  int blocks;
};
template <class Price, int FORMS, class Best>
static FormPlan form_plan(const Price (&prices)[FORMS], int M, int N, bool bounded, Best best) {
  int upto[FORMS] = {};   // each form's grid covers the rows it is chosen for
  FormPlan plan{form_table(M, bounded, best, upto), 1};
  for (int form = 0; form < FORMS; ++form) {
    // Tile rows rounded up to whole patches where that lets the XCD-aware order apply: the added
    // tiles lie past the bound any block of that tiling runs for, and leave at once.
    int tile_rows = (upto[form] + prices[form].bm - 1) / prices[form].bm;
    const int tile_cols = (N + prices[form].bn - 1) / prices[form].bn, whole = (tile_rows + 7) & ~7;
    if (tile_rows >= 8 && !patched_order(tile_rows, tile_cols) && patched_order(whole, tile_cols)) tile_rows = whole;
    plan.table.patched |= (tile_rows >= 8 && patched_order(tile_rows, tile_cols)) << form;
    if (tile_rows * tile_cols > plan.blocks) plan.blocks = tile_rows * tile_cols;
  }
  return plan;
}
// Under a bound the plan is a price for every form and run of rows, 1.5 us of the host's time at 2048 rows and 3 at 4096 (asked for again 0.02), and follows
// from the sizes alone: a thread keeps the last ones it made (a decoder layer has up to five).
constexpr int PLANS_HELD = 16;
struct HeldPlan {
  int M, N, K, variant;   // M 0: none
  FormPlan plan;
};
template <class Make>
static FormPlan held_plan(HeldPlan (&held)[PLANS_HELD], int M, int N, int K, int variant, Make make) {
  HeldPlan& h = held[((uint32_t)M * 31 + (uint32_t)N * 17 + (uint32_t)K / 8 * 7 + variant) % 251 % PLANS_HELD];
  if (h.M != M || h.N != N || h.K != K || h.variant != variant) h = HeldPlan{M, N, K, variant, make()};
  return h.plan;
}
static FormPlan rows_plan(int M, int N, int K, bool bounded, bool second) {
  auto make = [&] { return form_plan(ROWS_PRICES, M, N, bounded, [&](int rows) { return (int)rows_form(rows, M, N, K, second).form; }); };
  static thread_local HeldPlan held[PLANS_HELD];
  return bounded ? held_plan(held, M, N, K, second, make) : make();
}
// Fewer than 128 tiles of 128 x 128 are 64 x 64 ones on 64 KB of LDS, two blocks a CU and their whole register file of 256 each, which the forms above leave to one
// block: over a short K always (us, one a CU / two, with a second operand: 2048 x 528 x 256 6.6 / 5.5, 1024 x 1160 x 192 6.5 / 5.7, 2 rows of 256 x 4568 x 64 4.1 /
// 3.6, which is the table's trip); over a longer one, where few rows have smaller tiles, without a bound and while there are more than one a CU and little of B for each
// to wait for (2048 x 528 x 512 8.9 / 7.9, 2048 x 624 x 1024 11.7 / 11.0, 2048 x 960 x 1536 16.2 / 15.6; but 1024 x 1904 x 1024 13.0 / 13.9, 2048 x 960 x 4096
// 30.2 / 31.3).  Under a bound and K of 512 and more the forms above stay: at the bound's most rows they take 0.5 to 1 us longer than two a CU,
// at few rows 1 to 2 less (2048 x 568 x 960 under 119 rows 7.0 / 5.7).  Up to 64 rows, whose tiles are 64 x 64 whatever the bound, of more columns: over a short K as well
// (one a CU / two: 2 x 32000 x 168 6.3 / 5.2, 64 x 19760 x 128 with a second operand 6.9 / 6.0; over 328 drawn ones 1.09), and to K = 1024 where there are more than two a CU
// (19 drawn ones 1.13; up to two, K from 512 on, 70 of them 0.94).
static bool two_a_cu(int M, int N, int K, bool bounded) {
  const long tiles64 = (long)((M + 63) / 64) * ((N + 63) / 64);
  if (M <= 64 && (K < 8 * BK || (K < 16 * BK && tiles64 > 512))) return true;
  if ((long)((M + 127) / 128) * ((N + 127) / 128) >= 128) return false;
  return K < 8 * BK || (!bounded && tiles64 > 256 && tiles64 <= 512 && (long)N * K <= 3 << 19);
}

static int launch_gemm_rows(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, const int* valid, hipStream_t s,
                            const QkvTail& tail = QkvTail{}) {
  if (two_a_cu(M, N, K, valid != nullptr)) return launch_gemm_nt<false, false, 1>(A, B, C, M, N, K, valid, s, tail);
  const FormPlan plan = rows_plan(M, N, K, valid != nullptr, tail.residual != nullptr);
  constexpr size_t lds = Tile256Four::LDS_BYTES;
  static_assert(lds >= (size_t)NT_STAGES * 256 * BK * 2 && lds >= (size_t)long_lds(32, 8, 7), "the other bodies' stages fit too");
  static LdsOptIn opt_in[2];
  const auto kernel = tail.residual != nullptr ? &gemm_rows_kernel<true> : &gemm_rows_kernel<false>;
  if (hipError_t e = opt_in[tail.residual != nullptr].ensure(reinterpret_cast<const void*>(kernel), lds); e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(kernel, dim3(plan.blocks), dim3(256), lds, s, A, B, C, M, N, K, valid, plan.table, tail);
  IRON_LAUNCH_CHECK();
}

// A residual product of few rows over a long K, followed by the RMSNorm of its rows (a prompt chunk's
// down projection: 512 live rows x 2048 columns over K = 8192, then the next layer's input norm).
// 128 x 128 tiles would occupy a quarter of the CUs and the 64 x 64 ones that fill the chip fetch
// every operand row twice as often, so a tile's K is dealt over `splits` blocks -- chosen on the
// device by the row bound and K: 16 or 8 where that many a tile fit the chip in slices of eight stages or more, 4 where those would be too
// short, else as many as the chip has CUs for, 7 to 2, in slices that differ by a stage; past half the chip whole K, by tiles of 96 rows while
// those are one round -- each leaving its float32 sums in a workspace slice.  A second launch, a block a row,
// adds a row's slices in slice order (the same sums whatever ran first), rounds once, adds the
// residual, stores the row and norms it as rmsnorm_kernel does: that launch stands where the
// norm's own stood, so the slices' sum costs no launch of its own.
constexpr int kSplitKMax = 4;    // slices the second launch asks for at a time; K is whole stages of as many
__device__ __host__ inline int splitk_for(int tile_rows, int tiles_n, int K) {
  const int live_tiles = tile_rows * tiles_n;
  // Past four slices while the chip would idle and a slice keeps eight stages; ten where the slices of several tile rows pass half
  // the chip, whose sums cost the second launch more.  us with the norm, weights out of memory, N = 2048, fewer slices and more: K = 8192 29 rows
  // 26.0 / 16.3 (16), 128 28.5 / 19.8, 256 29.5 / 23.0 (8); K = 14336 41.3 / 21.6, 43.5 / 24.9, 43.8 / 31.1; K = 4096 29 rows 15.8 / 12.9 (8), but 256 20.6 / 21.8,
  // and 256 rows of N = 1024 over 8192 by 8 slices 20.1, by 16 21.6.
  auto keeps = [=](int splits) {
    const int stages = tile_rows > 1 && 2 * live_tiles * splits > 256 ? 10 : 8;
    return live_tiles * splits <= 256 && K % (splits * BK) == 0 && K >= splits * stages * BK;
  };
  if (keeps(16)) return 16;
  if (keeps(8)) return 8;
  // Between eight and two, as many as the chip has CUs for, though their stages do not come out even (us with the norm, weights out of memory, four slices and five: 2048 columns
  // over 8192, 300 rows 26.5 / 25.2, 384 30.9 / 28.2; two and three: 600 rows 44.0 / 35.0, 3072 over 8192, 384 48.1 / 38.2, 2560 over 9728, 512 55.9 / 44.3; four and six, 130 28.3 / 25.7).
  if (live_tiles * 8 > 256 && live_tiles * 2 <= 256) return 256 / live_tiles;
  return live_tiles * 4 <= 256 ? 4 : (live_tiles * 2 <= 256 ? 2 : 1);
}
// Rows a slice of the workspace holds when K is dealt `splits` ways: the most that split count runs for.
__device__ __host__ inline size_t splitk_slice_rows(int splits, int tiles_n) {
  return (size_t)((256 / splits) / tiles_n) * 128;
}

__global__ __launch_bounds__(256) void gemm_splitk_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                          bf16_t* __restrict__ C, int M, int N, int K,
                                                          const int* __restrict__ valid, Tiling whole, QkvTail tail,
                                                          float* __restrict__ partial) {
  const int Mv = bound_or(valid, M);
  const int tiles_n = whole.tiles_n, tile_rows = (Mv + 127) / 128, live_tiles = tile_rows * tiles_n;
  const int splits = splitk_for(tile_rows, tiles_n, K), id = blockIdx.x;
  if (splits == 1) {   // whole K a block, the residual in its epilogue: iron_gemm_residual_bf16's 128 x 128 launch, or tiles of 96 rows where they are one round
    const int tiles96 = (Mv + 95) / 96 * tiles_n;
    if (tiles96 <= min(256, (int)gridDim.x) && M >= 96 && N % 128 == 0)
      gemm_big_body<BigTile<2, 2, 3, 4>, false, false, false, true>(A, B, C, M, N, K, Mv, (M + 95) / 96, tiles_n, 0, GatedPair{}, tail);
    else if (id < whole.tiles_m * whole.tiles_n)
      gemm_nt16_body<false>(A, B, C, M, N, K, Mv, whole.tiles_m, whole.tiles_n, whole.patched, tail);
    return;
  }
  // The live (tile, slice) pairs are the first ids, so that they go out one a CU whatever the
  // launch's size; an XCD (id mod 8) serves one slice of K and a band of tile columns, whose
  // A and B pieces it then re-reads from its own L2.
  const int live = live_tiles * splits;
  if (id >= live) return;
  int tile, split;
  if (live % 8 == 0 && 8 % splits == 0) {
    const int xcd = id & 7, per = 8 / splits;
    split = xcd % splits;
    tile = (id >> 3) * per + xcd / splits;
  } else {
    split = id % splits;
    tile = id / splits;
  }
  tail.residual = nullptr;   // the second launch adds it
  const int stages = K / BK, first = split * stages / splits;
  tail.k_begin = first * BK;
  tail.k_len = ((split + 1) * stages / splits - first) * BK;
  tail.partial = partial + (size_t)split * splitk_slice_rows(splits, tiles_n) * N;
  tail.tile_plus1 = tile + 1;
  gemm_nt16_body<false>(A, B, C, M, N, K, Mv, (Mv + 127) / 128, tiles_n, 0, tail);
}

// The second launch: row `blockIdx.x` of C finished (from the slices, or as the first launch left
// it where K was not dealt) and normed into Y.  A thread holds CHUNKS 16-byte pieces of the row;
// every load of a piece goes out before any is used, through bounded buffers (a thread past the
// row's end reads zeros and takes no branch).  The norm's arithmetic is rmsnorm_kernel's, sum by
// sum, so Y is what iron_rmsnorm_bf16 makes of C bit for bit.
template <int CHUNKS>
__global__ __launch_bounds__(256) void gemm_finish_rows_kernel(const float* __restrict__ partial,
                                                               const bf16_t* residual, float scale, bf16_t* C,
                                                               const bf16_t* __restrict__ gain,
                                                               bf16_t* __restrict__ Y, int M, int N, float eps,
                                                               const int* __restrict__ valid, int tiles_n, int K) {
  const int row = blockIdx.x, nchunk = N >> 3;
  const __amdgpu_buffer_rsrc_t gain_bytes = bounded_bytes(gain, N * 2);
  uint4 gains[CHUNKS];
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) gains[i] = load_bounded(gain_bytes, 16 * (threadIdx.x + 256 * i));
  const int Mv = bound_or(valid, M);
  if (row >= Mv) return;
  const int splits = splitk_for((Mv + 127) / 128, tiles_n, K);
  uint4* c_row = reinterpret_cast<uint4*>(C + (size_t)row * N);
  uint4 held[CHUNKS];
  if (splits == 1) {
    const __amdgpu_buffer_rsrc_t row_bytes = bounded_bytes(c_row, N * 2);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) held[i] = load_bounded(row_bytes, 16 * (threadIdx.x + 256 * i));
  } else {
    const size_t slice = splitk_slice_rows(splits, tiles_n) * N;
    const __amdgpu_buffer_rsrc_t res_bytes = bounded_bytes(residual + (size_t)row * N, N * 2);
    uint4 added[CHUNKS], part[CHUNKS][kSplitKMax][2];
    // Slices first .. first + 3 of every piece, all requested before any is used.
    auto request = [&](int first) {
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i)
#pragma unroll
        for (int sl = 0; sl < kSplitKMax; ++sl) {
          // slices past the split count: an empty buffer, zeros
          const bool there = first + sl < splits;
          const __amdgpu_buffer_rsrc_t sums = bounded_bytes(partial + (there ? first + sl : 0) * slice + (size_t)row * N,
                                                            there ? N * 4 : 0);
          part[i][sl][0] = load_bounded(sums, 32 * (threadIdx.x + 256 * i));
          part[i][sl][1] = load_bounded(sums, 32 * (threadIdx.x + 256 * i) + 16);
        }
    };
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) added[i] = load_bounded(res_bytes, 16 * (threadIdx.x + 256 * i));
    request(0);
    f32x4 sum[CHUNKS][2];
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sum[i][h] = __builtin_bit_cast(f32x4, part[i][0][h]);
#pragma unroll
        for (int sl = 1; sl < kSplitKMax; ++sl)
          if (sl < splits) sum[i][h] += __builtin_bit_cast(f32x4, part[i][sl][h]);
      }
    for (int first = kSplitKMax; first < splits; first += kSplitKMax) {   // (slices past the last: zeros)
      request(first);
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int sl = 0; sl < kSplitKMax; ++sl) sum[i][h] += __builtin_bit_cast(f32x4, part[i][sl][h]);
    }
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      float x[8], rf[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = sum[i][e >> 2][e & 3];
      unpack8(added[i], rf);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = fmaf(scale, round_bf16(x[e]), rf[e]);
      held[i] = pack8(x);
      const int c = threadIdx.x + 256 * i;
      if (c < nchunk) c_row[c] = held[i];
    }
  }

  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) {
    float f[8];
    unpack8(held[i], f);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf(f[j], f[j], ss);
  }
  ss = wave_sum(ss);
  __shared__ float part_sums[4];
  if ((threadIdx.x & 63) == 0) part_sums[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float total = part_sums[0] + part_sums[1] + part_sums[2] + part_sums[3];
  const float inv = 1.0f / sqrtf(total / (float)N + eps);
  uint4* y_row = reinterpret_cast<uint4*>(Y + (size_t)row * N);
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) {
    const int c = threadIdx.x + 256 * i;
    float f[8], g[8];
    unpack8(held[i], f);
    unpack8(gains[i], g);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = round_bf16(f[j] * inv) * g[j];
    if (c < nchunk) y_row[c] = pack8(f);
  }
}

// A gated feed-forward's two first projections on one 128 x 128 tile position AT ONCE: a stage is the
// A tile and both weights' tiles (48 KB, three stages), an A fragment read out of LDS serves both
// products, and the gated epilogue has both accumulators in registers in the same layout, so the
// gate's product is stored (rounded, as the separate product stores it) and never read back.
// Against the same body run twice this fetches A once instead of twice (a quarter of the bytes a
// CU draws from L2 and a quarter of its LDS fragment reads).  Each product's MFMAs run in the order
// of the single-product body, so G and C are the separate launches' bit for bit.
// GROUPED: the caller has chosen the tile (tiles_m, tiles_n stand for its place), A's rows are those `a_rows` lists, and the
// gate's product is not stored.
template <bool GROUPED = false>
__device__ __forceinline__ void gemm_nt16_pair_body(const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bg,
                                                    const bf16_t* __restrict__ Bu, bf16_t* __restrict__ G,
                                                    bf16_t* __restrict__ C, int M, int N, int K,
                                                    int Mv, int tiles_m, int tiles_n,
                                                    int patched, int activation, const int* __restrict__ a_rows = nullptr) {
  constexpr int NT_BM = 128, NT_BN = 128;
  constexpr int PART = NT_BM * BK * 2;             // a 128 x 64 tile's 16 KB: A, then the gate's, then the up projection's
  constexpr int STAGE = 3 * PART, STAGES = PAIR_STAGES;
  constexpr int INST = NT_BM / 8 / 4;              // 1 KB loads of each part a wave issues per stage
  constexpr int LOADS = 3 * INST;
  static_assert(BK == 64 && INST == 4, "two 32-wide k-steps a stage, twelve loads a wave");
  extern __shared__ __align__(16) char smem_nt[];

  int tm = tiles_m, tn = tiles_n;
  if constexpr (!GROUPED) {
    if (!live_tile(blockIdx.x, tiles_m, tiles_n, patched, (Mv + NT_BM - 1) / NT_BM, tm, tn)) return;
  }
  const int m0 = tm * NT_BM;
  if (m0 >= Mv) return;
  const int n0 = tn * NT_BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int lrow = lane >> 3, pch = lane & 7;
  int a_voff[INST], b_voff[INST];
#pragma unroll
  for (int i = 0; i < INST; ++i) {
    const int r = (wave * INST + i) * 8 + lrow;
    const int lch = pch ^ ((r >> 1) & 7);
    if constexpr (GROUPED) a_voff[i] = (int)(((size_t)a_rows[m0 + r] * K + lch * 8) * 2);
    else a_voff[i] = m0 + r < Mv ? (r * K + lch * 8) * 2 : NOWHERE;
    b_voff[i] = (int)(((size_t)(min(n0 + r, N - 1) - n0) * K + lch * 8) * 2);
  }
  const bf16_t* a_tile = GROUPED ? A : A + (size_t)m0 * K;
  const bf16_t* g_tile = Bg + (size_t)n0 * K;
  const bf16_t* u_tile = Bu + (size_t)n0 * K;
  auto issue_one = [&](char* st, int kt, int idx) {   // idx: 0..3 A, 4..7 the gate's weights, 8..11 the up projection's
    const int k0 = kt * BK, part = idx / INST, piece = idx % INST;
    const bf16_t* from = part == 0 ? a_tile : (part == 1 ? g_tile : u_tile);
    const __amdgpu_buffer_rsrc_t rows = stage_rows(from + k0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, IRON_LDS_PTR(st + part * PART + (wave * INST + piece) * 1024), 16,
                                             (int)(part == 0 ? a_voff[piece] : b_voff[piece]), 0, 0, 0);
  };

  f32x4 accg[4][4], accu[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) accg[i][j][e] = accu[i][j][e] = 0.f;

  const int nk = K / BK;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
    for (int idx = 0; idx < LOADS; ++idx) issue_one(smem_nt + s * STAGE, min(s, nk - 1), idx);

  // Fragments: lane -> row fr of a 16-row tile, 16-byte chunk kq of the k-step's four.
  const int fr = lane & 15, kq = lane >> 4;
  const int swz = (fr >> 1) & 7;   // tile rows are multiples of 16 apart: one swizzle for all
  const int a_row = (wm * 64 + fr) * 128, b_row = (wn * 64 + fr) * 128;
  auto a_frag = [&](const char* st, int ks, int i) {
    return *reinterpret_cast<const bf16x8*>(st + a_row + i * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };
  auto b_frag = [&](const char* st, int part, int ks, int j) {
    return *reinterpret_cast<const bf16x8*>(st + part * PART + b_row + j * 16 * 128 + (((ks * 4 + kq) ^ swz) << 4));
  };

  wait_vmcnt<(STAGES - 2) * LOADS>();   // stage 0 has landed once only the younger one is out
  block_barrier();
  bf16x8 af[2][4], bg[2][4], bu[2][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) bg[0][i] = b_frag(smem_nt, 1, 0, i);
#pragma unroll
  for (int i = 0; i < 4; ++i) bu[0][i] = b_frag(smem_nt, 2, 0, i);
#pragma unroll
  for (int i = 0; i < 4; ++i) af[0][i] = a_frag(smem_nt, 0, i);
  // One stage of the loop, which is unrolled over the three stage buffers (stage_c = kt % STAGES): a
  // fragment's stage then rides in its read's offset field instead of a vector add a read.
  auto stage_step = [&](int kt, auto stage_c) {
    constexpr int S = decltype(stage_c)::value;
    // Prefetch goes into the buffer of stage kt-1.  Past the end the last stage is fetched again
    // (into buffers nobody reads any more) rather than branch: every iteration issues the same
    // loads, which keeps the wait counts exact and the scheduling region whole.
    const int kn = min(kt + STAGES - 1, nk - 1);
    char* nst = smem_nt + ((S + STAGES - 1) % STAGES) * STAGE;
    const char* st = smem_nt + S * STAGE;
    const char* st1 = smem_nt + ((S + 1) % STAGES) * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks == 1) {
        // The stage's one barrier, before its second k-step (whose fragments are in registers): of
        // the loads in flight the oldest LOADS are stage kt+1's, then the half of stage kt+2's
        // issued so far; after it nobody reads stage kt any more.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vmcnt<LOADS / 2>();
        block_barrier();
      }
      const char* from = ks == 0 ? st : st1;
      const int nks = ks ^ 1;
      // Source order is issue order (nothing crosses a sched_barrier): after an MFMA one fragment
      // read of the next k-step (the weights' first: its first MFMAs need all of them) or one load.
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j < 4) mfma_16x16x32_in_place(accg[i][j], bg[ks][j], af[ks][i]);
          else mfma_16x16x32_in_place(accu[i][j - 4], bu[ks][j - 4], af[ks][i]);
          __builtin_amdgcn_sched_barrier(0);
          const int slot = i * 8 + j;
          if (slot < 4) bg[nks][slot] = b_frag(from, 1, nks, slot);
          else if (slot < 8) bu[nks][slot - 4] = b_frag(from, 2, nks, slot - 4);
          else if (slot < 12) af[nks][slot - 8] = a_frag(from, nks, slot - 8);
          else if ((slot & 1) && slot < 12 + LOADS) issue_one(nst, kn, ks * (LOADS / 2) + (slot - 13) / 2);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  static_assert(STAGES == 3, "the loop below names the three stage buffers");
  for (int kt0 = 0; kt0 < nk; kt0 += STAGES) {
    stage_step(kt0, std::integral_constant<int, 0>{});
    if (kt0 + 1 < nk) stage_step(kt0 + 1, std::integral_constant<int, 1>{});
    if (kt0 + 2 < nk) stage_step(kt0 + 2, std::integral_constant<int, 2>{});
  }

  wait_vmcnt<0>();   // the idle fetches of the last iterations land ...
  block_barrier();   // ... in every wave, and every wave is done with the stages, before LDS is reused

  // Output through LDS, a product at a time: the wave lays its 64 x 64 out row-major (rows padded by
  // 16 bytes) and each lane then owns 8 consecutive columns of a row, so a row of the tile leaves as
  // one 128-byte segment.  First the gate's product as it is stored, where it is asked for; then, made in the accumulators'
  // own layout, bf16(bf16(act(bf16 g)) * bf16 u).
  constexpr int OROWB = 64 * 2 + 16;
  char* ot = smem_nt + wave * (64 * OROWB);
  const int out_row = lane >> 3, out_col = (lane & 7) * 8;
  const int out_n = n0 + wn * 64 + out_col;
  const bool whole = (N & 7) == 0 && out_n + 8 <= N;
  auto leave = [&](bf16_t* to) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int row = r * 8 + out_row, m = m0 + wm * 64 + row;
      const uint4 v = *reinterpret_cast<const uint4*>(ot + row * OROWB + out_col * 2);
      if (m >= Mv || out_n >= N) continue;
      bf16_t* p = to + (size_t)m * N + out_n;
      if (whole) *reinterpret_cast<uint4*>(p) = v;
      else store_ragged(p, v, N - out_n);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();   // the rows are read before the next product overwrites them
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if (!GROUPED && G != nullptr) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<uint2*>(ot + (i * 16 + fr) * OROWB + (j * 16 + 4 * kq) * 2) =
            make_uint2(pack_bf16(accg[i][j][0], accg[i][j][1]), pack_bf16(accg[i][j][2], accg[i][j][3]));
    leave(G);
  }
  auto gated = [&](auto kind) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float c[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          c[e] = round_bf16(gate_of(decltype(kind)::value, round_bf16(accg[i][j][e]))) * round_bf16(accu[i][j][e]);
        *reinterpret_cast<uint2*>(ot + (i * 16 + fr) * OROWB + (j * 16 + 4 * kq) * 2) =
            make_uint2(pack_bf16(c[0], c[1]), pack_bf16(c[2], c[3]));
      }
  };
  // The kind of gate is chosen once: asked an element, its branches kept the matrix results of one wave a
  // SIMD waiting for each other.
  if (activation == 1) gated(std::integral_constant<int, 1>{});
  else if (activation == 2) gated(std::integral_constant<int, 2>{});
  else gated(std::integral_constant<int, 3>{});
  leave(C);
}

// A gated feed-forward's two first projections over many rows as ONE launch, the tile chosen on the
// device by the row bound as in gemm_rows_kernel.  Tiles of BN / 2 columns of both weights: a wave's columns are half gate and half up projection, so
// the gated product is made in its registers (64 rows: on the 64 x 64 tile's loop, two waves a product; 29 x 8192 x 2048 29.7 -> 20.5 us; up to 32 rows by gemm_long_body, 15.8).
// Which tile: by rounds of blocks over the CUs, as big_form, at what a round was measured to take with weights out of memory.  8192 columns over
// K = 2048, us, by 64 x (32 + 32), 128 x (128 + 128) and 256 x (128 + 128) tiles alone and by these: 128 rows 27.9 / 25.9, 256 38.5 / 27.4, 384 39.6 /
// 33.2, 500 41.3 / 38.6, 640 58.5 / 45.7, 768 59.1 / 48.8, 1280 111 / 87, 1536 113 / 93, 1792 114 / 105.
// (96 and 224 rows as in RowsForm: 8192 columns over 2048, 119 rows 25.8 / 21.1, 394 34.7 / 31.8, 411 36.6 / 32.9, 133 to 187 23.2 / 22.3 to 23.6 / 23.9; 240 drawn ones, 69 of them, at 0.93.)
enum PairForm { PAIR_64X32, PAIR_EDGED, PAIR_96X64, PAIR_128X64, PAIR_160X64, PAIR_192X64, PAIR_224X64, PAIR_128X128, PAIR_160X128, PAIR_192X128, PAIR_224X128, PAIR_256X128, PAIR_FORMS };
struct PairPrice {
  int bm, bn;   // rows and columns of each product
  float start, stage;
};
constexpr PairPrice PAIR_PRICES[PAIR_FORMS] = {
    {64, 32, 3.f, 0.28f},    {128, 128, 7.f, 0.95f},    // (a product whose columns are no whole tiles: 128 rows at the edges' cost)
    {96, 64, 3.9f, 0.505f},  {128, 64, 4.f, 0.58f},   {160, 64, 4.5f, 0.64f},  {192, 64, 5.f, 0.73f},   {224, 64, 5.5f, 0.815f}, {128, 128, 6.f, 0.90f},
    {160, 128, 6.5f, 1.12f}, {192, 128, 7.5f, 1.2f},  {224, 128, 8.5f, 1.36f}, {256, 128, 9.5f, 1.5f},
};
// Whole tiles of 128 x (128 + 128) are made by the body that takes edges up to K = 2048 (us, by gemm_big_body and by that: 2048 x 2048 x 1920 33.5 / 29.6, x 960 20.9 / 19.3,
// 1024 x 4096 x 512 15.4 / 14.2; 430 drawn ones 0.90 to 0.95 with weights that the last-level cache holds, 0.98 to 1.02 out of memory), past it by gemm_big_body (0.91 and 1.03).
static PairForm pair_form(int rows, int M, int N, int K) {
  PairForm best = PAIR_64X32;
  float price = 0.f;
  const bool edged = K < 32 * BK && M >= 128 && N % 128 == 0;
  for (int form = PAIR_64X32; form < PAIR_FORMS; ++form) {
    if (edged && form == PAIR_128X128) continue;
    const PairPrice& p = PAIR_PRICES[edged && form == PAIR_EDGED ? PAIR_128X128 : form];
    if (form > PAIR_EDGED && (M < p.bm || N % p.bn != 0)) continue;
    if (K <= 8 * BK && (form == PAIR_96X64 || form == PAIR_224X64)) continue;   // (as in rows_form)
    const long tiles = (long)((rows + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
    const float us = (float)((tiles + 255) / 256) * (p.start + p.stage * (K / BK));
    if (form == PAIR_64X32 || us < price) best = (PairForm)form, price = us;
  }
  return best;
}
__global__ __launch_bounds__(256) void gemm_gated_pair_kernel(const bf16_t* __restrict__ A,
                                                              const bf16_t* __restrict__ Bg,
                                                              const bf16_t* __restrict__ Bu, bf16_t* __restrict__ G,
                                                              bf16_t* __restrict__ C, int M, int N, int K,
                                                              const int* __restrict__ valid, FormTable forms, int activation) {
  const FormOfRows chosen = form_of_rows(forms, valid, M);
  const int Mv = chosen.rows, patched = chosen.patched;
  const GatedPair pair{Bu, G, activation};
#define IRON_PAIR(FORM, MI, NT) \
  case FORM: \
    static_assert(PAIR_PRICES[FORM].bm == 32 * MI && PAIR_PRICES[FORM].bn == 16 * NT, "the tile that was priced"); \
    gemm_big_body<BigTile<2, 2, MI, NT>, false, false, true>(A, Bg, C, M, N, K, Mv, (M + 32 * MI - 1) / (32 * MI), N / (16 * NT), patched, pair); \
    break
  switch (chosen.form) {
    IRON_PAIR(PAIR_96X64, 3, 4);
    IRON_PAIR(PAIR_128X64, 4, 4);
    IRON_PAIR(PAIR_160X64, 5, 4);
    IRON_PAIR(PAIR_192X64, 6, 4);
    IRON_PAIR(PAIR_224X64, 7, 4);
    IRON_PAIR(PAIR_128X128, 4, 8);
    IRON_PAIR(PAIR_160X128, 5, 8);
    IRON_PAIR(PAIR_192X128, 6, 8);
    IRON_PAIR(PAIR_224X128, 7, 8);
    IRON_PAIR(PAIR_256X128, 8, 8);
    case PAIR_EDGED:
      gemm_nt16_pair_body(A, Bg, Bu, G, C, M, N, K, Mv, (M + 127) / 128, (N + 127) / 128, patched, activation);
      break;
    default: {
      QkvTail gate{};
      gate.gated = activation;
      if (pair_by_long_stages(Mv, N, K)) gemm_long_body<LONG_PAIR, 32, 3>(A, Bg, C, N, K, Mv, gate, Bu, G);
      else gemm_nt64_body<8, true>(A, Bg, C, M, N, K, Mv, (M + 63) / 64, (N + 31) / 32, patched, gate, Bu, G);
    }
  }
#undef IRON_PAIR
}

static FormPlan pair_plan(int M, int N, int K, bool bounded) {
  auto make = [&] { return form_plan(PAIR_PRICES, M, N, bounded, [&](int rows) { return (int)pair_form(rows, M, N, K); }); };
  static thread_local HeldPlan held[PLANS_HELD];
  return bounded ? held_plan(held, M, N, K, 0, make) : make();
}
static int launch_gemm_gated_pair(const bf16_t* A, const bf16_t* Bg, const bf16_t* Bu, bf16_t* G, bf16_t* C, int M,
                                  int N, int K, const int* valid, int activation, hipStream_t s) {
  const FormPlan plan = pair_plan(M, N, K, valid != nullptr);
  constexpr size_t lds = Tile256Four::LDS_BYTES;   // the largest tile's, more than the others'
  static_assert(lds >= (size_t)PAIR_STAGES * 3 * 128 * BK * 2 && lds >= (size_t)NT_STAGES * 256 * BK * 2 && lds >= (size_t)long_lds(32, 64, 3),
                "the other bodies' stages fit too");
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_gated_pair_kernel), lds); e != hipSuccess) {
    set_error("gemm_gated_pair: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(gemm_gated_pair_kernel, dim3(plan.blocks), dim3(256), lds, s, A, Bg, Bu, G, C, M, N, K, valid, plan.table, activation);
  IRON_LAUNCH_CHECK();
}

// Products of rows dealt to several weights of one shape, stacked: the rows lie (or are listed) weight by weight, each
// weight's padded to whole 128-row tiles, and GroupedTiles says which weight a row tile belongs to.  Blocks of an XCD share
// columns of tiles, and go down them weight by weight: a weight's tile crosses HBM once.
__device__ __forceinline__ bool grouped_tile(const GroupedTiles& g, int tiles_n, int& tm, int& tn, int& which) {
  if (tiles_n % 8 == 0) {
    const int loc = blockIdx.x >> 3;
    tm = loc % g.most;
    tn = (loc / g.most) * 8 + ((int)blockIdx.x & 7);
  } else {
    tm = (int)blockIdx.x % g.most;
    tn = (int)blockIdx.x / g.most;
  }
  if (tm >= *g.count) return false;
  which = g.which[tm];
  return true;
}
__global__ __launch_bounds__(256) void gemm_grouped_pair_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bg,
                                                                const bf16_t* __restrict__ Bu, bf16_t* __restrict__ C, int N, int K,
                                                                GroupedTiles g, const int* __restrict__ a_rows, int activation) {
  int tm, tn, e;
  if (!grouped_tile(g, (N + 127) / 128, tm, tn, e)) return;
  gemm_nt16_pair_body<true>(A, Bg + (size_t)e * N * K, Bu + (size_t)e * N * K, nullptr, C, g.most * 128, N, K, g.most * 128, tm, tn, 0, activation, a_rows);
}
__global__ __launch_bounds__(256) void gemm_grouped_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, bf16_t* __restrict__ C,
                                                           int N, int K, GroupedTiles g) {
  int tm, tn, e;
  const int tiles_n = (N + 127) / 128;
  if (!grouped_tile(g, tiles_n, tm, tn, e)) return;
  QkvTail tail{};
  tail.tile_plus1 = tm * tiles_n + tn + 1;
  gemm_nt16_body<false>(A, B + (size_t)e * N * K, C, g.most * 128, N, K, g.most * 128, g.most, tiles_n, 0, tail);
}

int launch_grouped_pair(const bf16_t* A, const bf16_t* Bg, const bf16_t* Bu, bf16_t* C, int N, int K, const GroupedTiles& g,
                        const int* a_rows, int activation, hipStream_t s) {
  constexpr size_t lds = (size_t)PAIR_STAGES * 3 * 128 * BK * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_grouped_pair_kernel), lds); e != hipSuccess) {
    set_error("gemm_grouped_pair: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(gemm_grouped_pair_kernel, dim3(g.most * ((N + 127) / 128)), dim3(256), lds, s, A, Bg, Bu, C, N, K, g, a_rows, activation);
  IRON_LAUNCH_CHECK();
}
int launch_grouped(const bf16_t* A, const bf16_t* B, bf16_t* C, int N, int K, const GroupedTiles& g, hipStream_t s) {
  constexpr size_t lds = (size_t)NT_STAGES * 256 * BK * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_grouped_kernel), lds); e != hipSuccess) {
    set_error("gemm_grouped: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL(gemm_grouped_kernel, dim3(g.most * ((N + 127) / 128)), dim3(256), lds, s, A, B, C, N, K, g);
  IRON_LAUNCH_CHECK();
}

// Products whose 128 x 128 tiles come out badly as rounds over the chip: the last `shared` tiles' K is dealt over
// `slices` blocks each, which leave float32 sums in a workspace; a second launch adds them up and
// rounds once.  A few tiles over a long K share all of them (one block's chain of stages is what the
// product takes: 383 x 1472 x 6520 36 tiles of 102 stages), tiles that just miss a whole number of rounds share the
// last, nearly empty round's.
struct TileShares {
  int whole, shared, slices;
};

template <bool B_KN, bool C_NM>
__global__ __launch_bounds__(256) void gemm_shared_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                          bf16_t* __restrict__ C, int M, int N, int K, int tiles_m,
                                                          int tiles_n, TileShares deal, float* __restrict__ sums) {
  QkvTail tail{};
  int tile = blockIdx.x;
  if (tile >= deal.whole) {
    const int at = tile - deal.whole, slice = at / deal.shared, nth = at - slice * deal.shared;
    const int stages = (K + k_pad(K)) / BK, from = slice * stages / deal.slices, to = (slice + 1) * stages / deal.slices;
    tile = deal.whole + nth;
    tail.k_begin = from * BK;
    tail.k_len = (to - from) * BK;
    tail.tile_sums = sums + (size_t)at * (128 * 128);
  }
  int tm, tn;
  tile_of_block(tile, tiles_m, tiles_n, 0, tm, tn);
  tail.tile_plus1 = tm * tiles_n + tn + 1;
  gemm_nt16_body<false, B_KN, C_NM, true>(A, B, C, M, N, K, M, tiles_m, tiles_n, 0, tail);
}

// The shared tiles' sums added up in the order of k, eight columns a thread, eight blocks a tile.
template <bool B_KN, bool C_NM>
__global__ __launch_bounds__(256) void gemm_shared_finish_kernel(const float* __restrict__ sums, bf16_t* __restrict__ C,
                                                                 int M, int N, int tiles_m, int tiles_n, TileShares deal) {
  const int nth = blockIdx.x >> 3, at = ((blockIdx.x & 7) * 256 + threadIdx.x) * 8;
  const float* from = sums + (size_t)nth * (128 * 128) + at;
  const size_t slice = (size_t)deal.shared * (128 * 128);
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll 4
  for (int p = 0; p < deal.slices; ++p) {
    lo += *reinterpret_cast<const f32x4*>(from + p * slice);
    hi += *reinterpret_cast<const f32x4*>(from + p * slice + 4);
  }
  int tm, tn;
  tile_of_block(deal.whole + nth, tiles_m, tiles_n, 0, tm, tn);
  const int m0 = tm * 128, n0 = B_KN ? max(min(tn * 128, N - 128), 0) : tn * 128;
  const int row = (C_NM ? n0 : m0) + (at >> 7), col = (C_NM ? m0 : n0) + (at & 127);
  const int rows = C_NM ? N : M, cols = C_NM ? M : N;
  if (row >= rows || col >= cols) return;
  bf16_t* to = C + (size_t)row * cols + col;
  const uint32_t w[4] = {pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
  store_ragged(to, make_uint4(w[0], w[1], w[2], w[3]), cols - col);
}

template <bool B_KN, bool C_NM>
static int launch_gemm_shared(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, const TileShares& deal,
                              float* sums, hipStream_t s) {
  const int tiles_m = (M + 127) / 128, tiles_n = (N + 127) / 128;
  constexpr size_t lds = (size_t)NT_STAGES * 256 * BK * 2;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_shared_kernel<B_KN, C_NM>), lds); e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL((gemm_shared_kernel<B_KN, C_NM>), dim3(deal.whole + deal.shared * deal.slices), dim3(256), lds, s, A, B,
                     C, M, N, K, tiles_m, tiles_n, deal, sums);
  hipLaunchKernelGGL((gemm_shared_finish_kernel<B_KN, C_NM>), dim3(deal.shared * 8), dim3(256), 0, s, sums, C, M, N, tiles_m,
                     tiles_n, deal);
  IRON_LAUNCH_CHECK();
}

template <class T, bool B_KN, bool STREAM_OUT>
static int launch_gemm_big_as(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, const int* valid, hipStream_t s) {
  const int tiles_m = (M + T::BM - 1) / T::BM, tiles_n = (N + T::BN - 1) / T::BN;
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_big_kernel<T, B_KN, STREAM_OUT>), T::LDS_BYTES);
      e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL((gemm_big_kernel<T, B_KN, STREAM_OUT>), dim3(tiles_m * tiles_n), dim3(T::WAVES * 64), T::LDS_BYTES, s,
                     A, B, C, M, N, K, valid, tiles_m, tiles_n, patched_order(tiles_m, tiles_n));
  IRON_LAUNCH_CHECK();
}

// The same without a bound: a product of up to 32 rows, B_ROWS rows of B a block.
template <int B_ROWS, int STAGES>
__global__ __launch_bounds__(256) void gemm_long_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, bf16_t* __restrict__ C, int M, int N, int K) {
  gemm_long_body<LONG_PLAIN, 32, STAGES, B_ROWS, true>(A, B, C, N, K, M, QkvTail{});
}
template <int B_ROWS, int STAGES>
static int launch_gemm_long(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, hipStream_t s) {
  constexpr size_t lds = long_lds(32, B_ROWS, STAGES);
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_long_kernel<B_ROWS, STAGES>), lds); e != hipSuccess) {
    set_error("gemm: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipLaunchKernelGGL((gemm_long_kernel<B_ROWS, STAGES>), dim3((N + B_ROWS - 1) / B_ROWS), dim3(256), lds, s, A, B, C, M, N, K);
  IRON_LAUNCH_CHECK();
}
static int long_columns(int N) { return N <= 8 * 256 ? 8 : (N <= 16 * 256 ? 16 : (N <= 32 * 256 ? 32 : 64)); }
static int launch_gemm_long(const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, hipStream_t s) {
  switch (long_columns(N)) {
    case 8: return launch_gemm_long<8, 8>(A, B, C, M, N, K, s);
    case 16: return launch_gemm_long<16, 6>(A, B, C, M, N, K, s);
    case 32: return launch_gemm_long<32, 5>(A, B, C, M, N, K, s);
    default: return launch_gemm_long<64, 3>(A, B, C, M, N, K, s);
  }
}

// Whole tiles larger than 128 x 128, by how the rounds they make over the chip's 256 CUs come out: a round of a tile was measured
// to take `start` us (its entry, first loads and stores) and `stage` for each 64 of K, `loose` where rows straddle cache lines; [0] with B (N,K), [1] (K,N).
// The stage grows with the tile's area, so what a product gains is the part of its rounds that is not filled (us, by 128 x 128 or 256 x 256 tiles
// alone and by the tile chosen here): 777 x 10240 x 2560 53 -> 37 (weights out of memory 63 -> 50), 2012 x 3008 x 1608 34.4 -> 24.4, 2856 x 2325 x 3176 77 -> 51, 1636 x 5256 x 6200 with
// B (K,N) 153 -> 119, 908 x 5328 x 344 with B (K,N) 14.8 -> 9.9, 3000 x 3000 x 3000 74 -> 54.
// Tiles of 96 x 128 by four waves and of 224 x 256 past K = 512 (up to there a round is its start and its end): 1903 x 1298 x 4440 44.3 -> 38.5, 137 x 8852 x 6136 58.4 ->
// 49.4, 1958 x 12862 x 1248 65.7 -> 60.8, 2592 x 10736 x 1848 with B (K,N) 96.6 -> 90.9; fifty drawn products that take them 0.927 of the time, the worst 1.06 (8100 x 296 x
// 3696).  160 x 128 and 224 x 128 by four waves take what 128 x 192 and 128 x 256 by eight do.
enum BigForm { BIG_NONE, BIG_256, BIG_192X256, BIG_160X256, BIG_128X256, BIG_128X192, BIG_224X256, BIG_96X128, BIG_FORMS };
struct BigPrice {
  int bm, bn;
  float start, stage[2], loose[2];
};
constexpr BigPrice BIG_PRICES[BIG_FORMS] = {
    {128, 128, 2.8f, {0.415f, 0.426f}, {0.615f, 0.49f}},   // (the 128 x 128 kernel)
    {256, 256, 7.5f, {1.36f, 1.42f}, {1.63f, 1.48f}},  {192, 256, 5.9f, {1.10f, 1.16f}, {1.38f, 1.22f}},
    {160, 256, 4.9f, {0.92f, 0.955f}, {1.08f, 1.00f}}, {128, 256, 4.4f, {0.76f, 0.80f}, {0.95f, 0.835f}},
    {128, 192, 3.2f, {0.595f, 0.f}, {0.76f, 0.f}},     // (a stage of (K,N) rows of 192 columns is no whole number of loads)
    {224, 256, 6.8f, {1.243f, 1.283f}, {1.505f, 1.35f}}, {96, 128, 2.f, {0.366f, 0.f}, {0.54f, 0.f}},
};
static float big_price(BigForm form, int M, int N, int K, bool b_nk) {
  const BigPrice& p = BIG_PRICES[form];
  const long tiles = (long)((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
  return (float)((tiles + 255) / 256) * (p.start + (K % BK == 0 ? p.stage : p.loose)[!b_nk] * ((K + BK - 1) / BK));
}
// The form before `end` for a product without a row bound, and what it and the 128 x 128 tiles are expected to take.
static BigForm big_form(int M, int N, int K, bool b_nk, float& price, float& price128, int end = BIG_FORMS) {
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  BigForm best = BIG_NONE;
  price = price128 = big_price(BIG_NONE, M, N, K, b_nk);
  if (!b_nk && (long)(K + BK) * N * 2 >= (1L << 31)) return best;   // (a (K,N) matrix is addressed with 32-bit byte offsets)
  for (int form = BIG_256; form < end; ++form) {
    if (M < BIG_PRICES[form].bm || N < BIG_PRICES[form].bn || (!b_nk && BIG_PRICES[form].bn != 256) || (form > BIG_128X192 && K <= 8 * BK)) continue;
    const float p = big_price((BigForm)form, M, N, K, b_nk);
    // (past four rounds of 256 x 256 tiles the smaller ones' traffic tells: 5540 x 12392 x 7728 1011 us by those, 1024 by 160 x 256, 881 by its price; with B (K,N) 128 x 128
    // tiles take more than theirs, a larger one's first rounds less: by them and by the larger 8192 x 1400 x 1608 53 / 42, 32000 x 1040 x 3904 359 / 275, 749 x 26520 x 4912
    // 282 / 193; over 869 drawn products, two thirds of them (K,N), the form taken is within 0.6 % of the best on average, 1.4 % at the line of B (N,K))
    const float line = best == BIG_NONE && !b_nk ? 1.1f : (best == BIG_256 && tiles256 > 3 * 256 ? 0.9f : 0.97f);
    if (p < line * price) best = (BigForm)form, price = p;
  }
  return best;
}
template <bool B_KN>
static int launch_gemm_big(BigForm form, const bf16_t* A, const bf16_t* B, bf16_t* C, int M, int N, int K, const int* valid, hipStream_t s) {
  // Over a long K the tiles leave by non-temporal stores (see the body's epilogue).
  if (form == BIG_256 && K >= 4096) return launch_gemm_big_as<Tile256, B_KN, true>(A, B, C, M, N, K, valid, s);
  if (form == BIG_256) return launch_gemm_big_as<Tile256, B_KN, false>(A, B, C, M, N, K, valid, s);
  if (form == BIG_224X256) return launch_gemm_big_as<Tile224x256, B_KN, false>(A, B, C, M, N, K, valid, s);
  if (form == BIG_192X256) return launch_gemm_big_as<Tile192x256, B_KN, false>(A, B, C, M, N, K, valid, s);
  if (form == BIG_160X256) return launch_gemm_big_as<Tile160x256, B_KN, false>(A, B, C, M, N, K, valid, s);
  if constexpr (!B_KN)
    if (form == BIG_128X192 || form == BIG_96X128)
      return form == BIG_96X128 ? launch_gemm_big_as<Tile96x128, false, false>(A, B, C, M, N, K, valid, s) : launch_gemm_big_as<Tile128x192, false, false>(A, B, C, M, N, K, valid, s);
  return launch_gemm_big_as<Tile128x256, B_KN, false>(A, B, C, M, N, K, valid, s);
}

}  // namespace iron

using namespace iron;

static int check_gemm(const uint16_t* A, const uint16_t* B, const uint16_t* C, int M, int N, int K, int b_col_maj) {
  IRON_REQUIRE(A && B && C, "gemm: null operand");
  IRON_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: M (%d), N (%d), K (%d) must be positive", M, N, K);
  IRON_REQUIRE(K % 8 == 0, "gemm: K (%d) must be a multiple of 8 (16-byte loads)", K);
  IRON_REQUIRE(K <= (1 << 22) && N <= (1 << 22),
               "gemm: K (%d) and N (%d) may be at most 2^22 (a tile's rows are addressed with 32-bit offsets)", K, N);
  IRON_REQUIRE((((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) == 0,
               "gemm: operands must be 16-byte aligned");
  IRON_REQUIRE(b_col_maj || N % 8 == 0,
               "gemm: N (%d) must be a multiple of 8 when B is (K,N) (16-byte loads along N)", N);
  return 0;
}

// Tiles of 32 columns (B (N,K)) by 32 or 64 rows (rows 0: neither), while they are one round over the chip: a CU then draws a half or three
// quarters of what it draws for a 64 x 64 tile (see gemm_nt64_body), which is what a product without a full round of those takes; and what they were
// measured to take (a twentieth off over 270 shapes). us, weights out of memory, by the kernels chosen before and by these: 97 x 711 x 1936 10.9 / 6.8,
// 250 x 232 x 2584 13.9 / 7.8, 163 x 2113 x 4088 26.1 / 16.4; against shared K 112 x 886 x 2704 18.7 / 9.1, 58 x 411 x 4416 19.5 / 10.4; out of the
// last-level cache 510 x 331 x 2232 9.3 / 7.1, 41 x 4827 x 3112 21.2 / 11.0. Two stages are too few for them to pay.
// With B (K,N) the columns are 64, a cache line of a row of B; 128 x 128 tiles and those: 521 x 416 x 1320 12.3 / 7.5, 50 x 6672 x 1880 21.6 / 13.1,
// 130 x 88 x 1008 8.9 / 5.8; a long K shared stays so, 135 x 440 x 8096 14.8 / 36.  C (N,M) of it likewise: 248 x 1472 x 1480 12.7 / 7.6, 883 x 160 x 1032
// 10.8 / 6.8, 110 x 176 x 248 6.2 / 3.9.
struct SmallTiles {
  int rows;
  float us;
};
// B (K,N) past 16 MB comes from memory, a line of a row at a time.
static bool kn_from_memory(int N, int K) { return (long)N * K > 8000000; }
static SmallTiles small_tiles(int M, int N, int K, bool b_nk) {
  const int columns = b_nk ? 32 : 64;
  const long low = (long)((M + 31) / 32) * ((N + columns - 1) / columns), high = (long)((M + 63) / 64) * ((N + columns - 1) / columns);
  const float stages = (float)((K + BK - 1) / BK);
  if (K < 3 * BK || high > 256) return {0, 0.f};
  const float from_memory = !b_nk && kn_from_memory(N, K) ? 0.08f : 0.f;
  if (!b_nk && low <= 256) return {32, 3.f + stages * (0.165f + 0.02f * low / 256 + from_memory)};
  if (!b_nk) return {64, 3.2f + stages * (0.19f + 0.02f * high / 256 + from_memory)};
  if (low <= 256) return {32, 3.05f + stages * (0.108f + (K % BK == 0 ? 0.02f : 0.034f) * low / 256)};
  return {64, 3.2f + stages * (0.14f + 0.035f * high / 256)};
}

// How a product's 128 x 128 tiles are shared (none: slices 0), M and N as the tiles see them, by what was
// measured, in us.  Unshared: 3 a launch; a stage of 64 k 0.5 a round of 128 x 128 tiles; on the 64 x 64 tiles
// that few tiles of B (N,K) take, 0.13 to 0.23 up to a block a CU, and 0.14 (a few blocks) to 0.34 where K is no multiple of 64.
// Shared: the second launch and 0.028 a slice of a tile (its 64 KB out and back) on top, which the slices
// are chosen against.  Both sides: 97 x 400 x 7392 with B (K,N) 48.8 -> 14.0, 383 x 1472 x 6520 50.7 -> 25.0, 86 x 1728 x
// 5560 with B (N,K) 26.6 -> 16.0, 5300 x 864 x 7744 (294 tiles) 92 -> 74; not 1024 x 1024 x 4096, 15.5 against 21.2.
static TileShares gemm_shares_of_tiles(int M, int N, int K, bool b_nk, float* price = nullptr) {
  const TileShares none{0, 0, 0};
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (K < BK || tiles > 3 * 256) return none;
  const int stages = (K + BK - 1) / BK, t = (int)tiles;
  const int shared = t <= 128 ? t : (t > 256 ? t % 256 : 0);   // all tiles, or those of the last round
  if (shared == 0 || shared > 128) return none;
  const int by_cost = (int)(4.2f * sqrtf((float)stages / shared) + 0.5f);
  int slices = 256 / shared < stages / 6 ? 256 / shared : stages / 6;
  if (slices > by_cost) slices = by_cost;
  if (slices < 2) return none;
  const float fill = (float)((long)((M + 63) / 64) * ((N + 63) / 64)) / 256.f;
  const float stage64 = K % BK == 0 ? 0.13f + 0.10f * fill : fminf(0.14f + 3.f * fill, 0.22f + 0.12f * fill);
  const float now = 3.f + stages * (b_nk && t <= 128 ? stage64 : 0.5f * ((t + 255) / 256));
  const float then = 7.f + 0.028f * slices * shared + 0.5f * ((stages + slices - 1) / slices + stages * ((t - shared) / 256));
  if (price != nullptr) *price = then;
  return then < 0.9f * now ? TileShares{t - shared, shared, slices} : none;
}

// Whether the few-row kernels take a product of B (N,K).  Their blocks read all of A each, so they grow with rows x K
// (2048 x 8192 16 / 33 / 63 rows 10.3 / 27.1 / 35.8 us, 5256 x 6192 27 / 44 / 64) where the tiles do not (17.3 and 27);
// the line lies where the two met over twenty shapes, short K to the few rows (63 x 1304 x 1032 6.4 against 7.8).  Up to sixteen rows
// of a matrix that the strips take a tile a block stay ahead of the tiles past that line (weights out of memory: 16 rows 2048 x 9216 13.3
// against 18.2, 2048 x 16384 18.0 against 23.4, 1000 x 16384 15.3 against 17.7, 304 x 14336 13.3 against 13.5; not
// 14 x 304 x 18944, 16.0 against 14.9).  Past the line the few rows stay where what they are measured to take, weights out of memory, is the less:
// 2.6 us and, a thousand of K, what the rows and the rounds of blocks make of it; the tiles 11 and the matrix at 5 TB/s where they are shared,
// else 3.3 and their chain of stages, dearer where rows straddle cache lines (few rows against tiles: 45 x 1928 x 3192 16.4 / 23.7, 48 x 3992 x 1424
// 8.5 / 12.4, 63 x 2048 x 6144 28.9 / 32.7, 16 x 4096 x 10192 24.2 / 31.6, but 40 x 2048 x 8192 28.9 / 17.6, 56 x 6000 x 3192 36.4 / 28.0).
// More than 32 rows give way to tiles of 32 columns that take a good deal less (few rows against those: 34 x 7452 x 2312 19.0 / 11.7, 40 x 3208 x 3744
// 17.2 / 12.1, 35 x 1828 x 2512 11.2 / 8.3; but 59 x 344 x 480 3.1 / 3.9).
static bool gemm_of_few_rows(int M, int N, int K) {
  if (M >= 64) return false;
  const float rows = M <= 16 ? 1.1f + 0.045f * M : 1.55f + 0.0435f * M;
  const float each = N < 8192 ? rows * ((N + 4095) / 4096) : (M <= 16 ? 3.5f : 4.15f + 0.028f * M);   // (N = 8192: 32 columns a block)
  const float few = 2.6f + 1e-3f * K * each;
  if (const SmallTiles small = small_tiles(M, N, K, true); M > 32 && small.rows > 0 && small.us < 0.72f * few) return false;
  if (M <= 16 && N <= 2048 && K <= 16384 && (long)N * K >= (1 << 21)) return true;
  if ((long)M * K < 140000 && (M < 48 || K < 1408)) return true;
  if (N > 8192 || K < BK) return false;
  const float stage = K % BK == 0 ? 0.17f + 0.0018f * M : 0.2f + 0.0048f * M;
  const float tiles = gemm_shares_of_tiles(M, N, K, true).slices > 0 ? 11.f + 4e-7f * N * K : 3.3f + stage * ((K + BK - 1) / BK);
  return 1.05f * few < tiles;
}

// Seventeen to thirty-two rows against B (N,K) while a round of blocks takes all of it: long stages (gemm_long_body) instead of strips, whose two tiles of rows come straight from memory
// a fragment at a time, of 64 x 32 tiles or of shared ones.  us with the same weights again and out of memory, those / this: 31 x 2048 x 4096 11.0 / 8.9 and 12.2 / 8.9, 21 x 4096 x
// 8192 20.6 / 16.2, 21.8 / 18.2, 26 x 16384 x 4096 40.4 / 25.2, 42.5 / 25.9, 27 x 10240 x 1024 8.8 / 6.7, 10.5 / 6.8, 22 x 1024 x 8192 14.3 / 13.3, 15.4 / 12.8; but where the
// last-level cache holds more weights than that, or rows straddle lines, 29 x 4857 x 5648 13.4 / 18.2, 28 x 10240 x 8192 26.3 / 33.6, 22 x 5808 x 1848 7.7 / 8.2 (11.6 / 8.4 out of memory), 19 x 1925 x 3552 7.5 / 8.1,
// over few columns 18 x 140 x 5920 9.0 / 10.0, over a short K 28 x 2048 x 512 5.6 / 6.0, and up to sixteen rows strips stay: 10 x 8192 x 4096 16.0 / 18.1, 13 x 422 x 5976 8.0 / 10.4.
static bool gemm_of_long_stages(int M, int N, int K) {
  return M > 16 && M <= 32 && (K > 1024 || (N > 32 * 256 && K >= LONG_K)) && N >= 256 && N <= 64 * 256 && (K % BK == 0 ? K <= (N <= 16 * 256 ? 8192 : 4096) : N <= 16 * 256 && K <= 2048);
}

// Whether the direct-to-LDS kernels take a product, B (N,K) with C (N,M) turned round before.  They take any K from one stage on (k_pad),
// any M, and any N of B (N,K); against the general kernel, which loads through registers: 2048 x 2048 x 2056 42.5 -> 26.0 us, 86 x 1728 x
// 5560 59 -> 26.5, (K,N) 2048 x 2048 x 2040 65 -> 22.0, 300 x 1000 x 1000 33.6 -> 9.8, 2048 x 2616 x 72 9.8 -> 6.9, 7137 x 6620 x 80 49.0 -> 30.8.
// (A K that is no multiple of 64 stays dearer than its neighbour that is, 26.0 us against 19.4: its rows' 128-byte
// pieces straddle two cache lines.)  The general kernel, of which a CU holds several blocks, keeps a short K where there is one row or column
// of tiles (general against direct: (K,N) 107 x 240 x 64 3.7 / 4.6, 100 x 8008 x 64 4.4 / 4.9, but 200 x 240 x 64 5.8 / 4.6;
// (N,M) of 3 x 3904 x 224 5.8 / 6.3; (N,K) 490 x 22 x 64 3.2 / 3.8, under a bound 63 x 424 x 64 3.2 / 3.8).
static bool gemm_direct_to_lds(int M, int N, int K, int b_col_maj, int c_col_maj, bool bounded) {
  if (K < BK || (c_col_maj && (b_col_maj || bounded))) return false;
  if (!b_col_maj) return (M >= 128 && N >= 128) || K > (c_col_maj && M < 8 ? 4 : 2) * BK;
  return (M >= 64 && N >= 64) || K > 2 * BK;
}

// What a product without a bound takes, B (N,K) with C (N,M) turned round before: one answer for the launch, for the workspace and for whoever asks.
// `deal`: how its tiles' K is shared where the caller brings a workspace.  Small tiles are the cheaper wherever they are one round, 128 tiles of 128 x 128
// with a dimension of at most 64 among them (us, weights out of memory, half-empty 128 x 128 tiles / shared / small: 64 x 16384 x 8192 with B (K,N) 70 / 58 / 54,
// 16384 x 64 71 / 87 / 59; 64 x 16320 x 200 6.0 unshared, 5.0 small).
enum class GemmForm { FEW_ROWS, LONG_STAGES, SMALL, BIG, TILES_64, TILES_128, GENERAL };
struct GemmPlan {
  GemmForm form;
  SmallTiles small;
  BigForm big;
  TileShares deal;
};
// `all`: false leaves out long stages and the tiles of 96 and 224 rows, for iron_gemm_shared_bf16.
static GemmPlan gemm_plan(int M, int N, int K, bool b_nk, bool c_nm, bool all = true) {
  GemmPlan plan{GemmForm::GENERAL, {0, 0.f}, BIG_NONE, {0, 0, 0}};
  if (all && b_nk && !c_nm && gemm_of_long_stages(M, N, K)) {
    plan.form = GemmForm::LONG_STAGES;
    return plan;
  }
  if (b_nk && !c_nm && gemm_of_few_rows(M, N, K)) {   // fewer rows than the smallest tile: bound by streaming B
    plan.form = GemmForm::FEW_ROWS;
    return plan;
  }
  if (!gemm_direct_to_lds(M, N, K, b_nk, c_nm, false)) return plan;
  const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
  float big = 0.f, price128 = 0.f, shared = 0.f;
  plan.small = small_tiles(M, N, K, b_nk);
  if (!c_nm && tiles128 >= 128) plan.big = big_form(M, N, K, b_nk, big, price128, all ? BIG_FORMS : BIG_224X256);
  // 128 x 128 tiles that would occupy under half the CUs give way to 64 x 64 ones, and so do tiles that up to 64 rows would half fill at
  // most (64 x 16384 x 8184: 93 -> 68 us).
  plan.form = plan.small.rows > 0 ? GemmForm::SMALL : (plan.big != BIG_NONE ? GemmForm::BIG : (b_nk && (tiles128 < 128 || M <= 64) ? GemmForm::TILES_64 : GemmForm::TILES_128));
  const TileShares deal = gemm_shares_of_tiles(M, N, K, b_nk, &shared);
  // (small tiles against shared ones, us out of memory and with the same weights again: with B (K,N) 59 x 6144 x 4712 28.0 / 21.3 and 18.6 / 19.8, 9 x 6144 x 3824
  // 21.5 / 18.8 and 14.1 / 17.9, but 10 x 12288 x 2736 18.7 / 21.9 and 14.5 / 19.6; rows of a smaller B (K,N) that straddle cache lines cost the small tiles more,
  // 30 x 2776 x 3248 shared 16.1, by those 21.0; whole tiles of another size where they take no more)
  const float line = !b_nk && kn_from_memory(N, K) ? 0.9f : (b_nk || N % BK == 0 ? 0.78f : 0.68f);
  const bool alone = plan.form == GemmForm::SMALL ? plan.small.us < line * shared : plan.form == GemmForm::BIG && big + 3.f <= shared;
  if (!alone) plan.deal = deal;
  return plan;
}

extern "C" int iron_gemm_bf16(const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K,
                              int b_col_maj, int c_col_maj, const int* valid, const int* valid_k,
                              void* stream) {
  if (const int rc = check_gemm(A, B, C, M, N, K, b_col_maj); rc != 0) return rc;
  hipStream_t s = (hipStream_t)stream;
  // The (N,M) output of A and B (N,K) is the (M,N) output of B and A: both are rows of K (2048^3 41.5 ->
  // 19.4 us against the general kernel's strided stores).
  if (b_col_maj && c_col_maj && valid == nullptr && valid_k == nullptr && M <= (1 << 22)) {
    const uint16_t* rows = A;
    A = B, B = rows;
    const int m = M;
    M = N, N = m;
    c_col_maj = 0;
  }
  if (valid == nullptr && valid_k == nullptr) {
    const GemmPlan plan = gemm_plan(M, N, K, b_col_maj, c_col_maj);
    const bool high = plan.small.rows == 64;
    switch (plan.form) {
      case GemmForm::FEW_ROWS:
        return iron_gemm_few_bf16(A, B, nullptr, C, M, N, K, 0, stream);
      case GemmForm::LONG_STAGES:
        return launch_gemm_long(A, B, C, M, N, K, s);
      case GemmForm::SMALL:
        if (b_col_maj) return high ? launch_gemm_small<13, 1, 4, 2>(A, B, C, M, N, K, s) : launch_gemm_small<20, 1, 2, 1>(A, B, C, M, N, K, s);
        if (c_col_maj) return high ? launch_gemm_small<10, 2, 2, 2, true, true>(A, B, C, M, N, K, s) : launch_gemm_small<13, 1, 2, 2, true, true>(A, B, C, M, N, K, s);
        return high ? launch_gemm_small<10, 2, 2, 2, true>(A, B, C, M, N, K, s) : launch_gemm_small<13, 1, 2, 2, true>(A, B, C, M, N, K, s);
      case GemmForm::BIG:
        return b_col_maj ? launch_gemm_big<false>(plan.big, A, B, C, M, N, K, nullptr, s) : launch_gemm_big<true>(plan.big, A, B, C, M, N, K, nullptr, s);
      case GemmForm::TILES_64:
        return launch_gemm_nt<false, false, 1>(A, B, C, M, N, K, nullptr, s);
      case GemmForm::TILES_128:
        if (b_col_maj) return launch_gemm_nt<false>(A, B, C, M, N, K, nullptr, s);
        return c_col_maj ? launch_gemm_nt<true, false, 2, 4, true>(A, B, C, M, N, K, nullptr, s) : launch_gemm_nt<true>(A, B, C, M, N, K, nullptr, s);
      case GemmForm::GENERAL:
        break;
    }
  } else if (valid_k == nullptr && gemm_direct_to_lds(M, N, K, b_col_maj, c_col_maj, true)) {
    return b_col_maj ? launch_gemm_rows(A, B, C, M, N, K, valid, s) : launch_gemm_nt<true>(A, B, C, M, N, K, valid, s);
  }
  // 128x128 tiles fill the 256 CUs once at 2048x2048; narrower problems take 64-wide tiles.
  const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (tiles128 >= 128 || (M >= 128 && N >= 128))
    return launch_gemm<128, 128, 2, 2>(A, B, C, M, N, K, b_col_maj, c_col_maj, valid, valid_k, s);
  return launch_gemm<64, 64, 2, 2>(A, B, C, M, N, K, b_col_maj, c_col_maj, valid, valid_k, s);
}

extern "C" int64_t iron_gemm_workspace_bytes(int M, int N, int K, int b_col_maj, int c_col_maj) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 != 0) return 0;
  const bool turned = b_col_maj && c_col_maj;
  const TileShares deal = gemm_plan(turned ? N : M, turned ? M : N, K, b_col_maj, c_col_maj && !turned).deal;
  return (int64_t)deal.slices * deal.shared * 128 * 128 * sizeof(float);
}

extern "C" int iron_gemm_shared_bf16(const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K,
                                     int b_col_maj, int c_col_maj, void* workspace, void* stream) {
  if (const int rc = check_gemm(A, B, C, M, N, K, b_col_maj); rc != 0) return rc;
  IRON_REQUIRE(workspace != nullptr && ((uintptr_t)workspace & 15) == 0, "gemm_shared: a workspace, 16-byte aligned");
  IRON_REQUIRE(M <= (1 << 22), "gemm_shared: M (%d) may be at most 2^22", M);
  if (b_col_maj && c_col_maj) {   // (as iron_gemm_bf16)
    const uint16_t* rows = A;
    A = B, B = rows;
    const int m = M;
    M = N, N = m;
    c_col_maj = 0;
  }
  const TileShares deal = gemm_plan(M, N, K, b_col_maj, c_col_maj).deal;
  // (Products that tiles of 96 and 224 rows or long stages made cheaper than shared ones are taken all the same, by those: whoever brings a workspace of their own
  // size for them need not ask first.)
  if (deal.slices == 0 && gemm_plan(M, N, K, b_col_maj, c_col_maj, false).deal.slices > 0) return iron_gemm_bf16(A, B, C, M, N, K, b_col_maj, c_col_maj, nullptr, nullptr, stream);
  IRON_REQUIRE(deal.slices > 0, "gemm_shared: a product of %d x %d over %d shares no tiles (iron_gemm_workspace_bytes is 0)", M, N, K);
  hipStream_t s = (hipStream_t)stream;
  float* sums = (float*)workspace;
  if (b_col_maj) return launch_gemm_shared<false, false>(A, B, C, M, N, K, deal, sums, s);
  if (c_col_maj) return launch_gemm_shared<true, true>(A, B, C, M, N, K, deal, sums, s);
  return launch_gemm_shared<true, false>(A, B, C, M, N, K, deal, sums, s);
}

// What the launches above and below decide on the host, for whoever asks without a launch.
extern "C" int iron_gemm_tile(int kind, int M, int N, int K, int b_col_maj, int c_col_maj, int rows) {
  if (kind < 0 || kind > 3 || M <= 0 || N <= 0 || K <= 0 || K % 8 != 0 || K > (1 << 22) || N > (1 << 22)) return 0;
  auto tile = [](int bm, int bn) { return bm << 16 | bn; };
  auto by_long_stages = [=](int columns) { return tile(32, 1 << 15 | columns); };
  if (kind > 0) {
    if (kind < 3 && two_a_cu(M, N, K, rows > 0)) return tile(64, 64);
    const FormPlan plan = kind == 3 ? pair_plan(M, N, K, true) : rows_plan(M, N, K, true, kind == 2);
    const int live = rows > 0 && rows < M ? rows : M, form = form_of_rows(plan.table, live);
    if (kind == 3 && form == PAIR_64X32 && pair_by_long_stages(live, N, K)) return by_long_stages(long_b_rows(LONG_PAIR) / 2);
    if (kind < 3 && form == ROWS_32X32 && rows_by_long_stages(live, N, K, plan.blocks)) return by_long_stages(long_b_rows(LONG_PLAIN));
    return kind == 3 ? tile(PAIR_PRICES[form].bm, PAIR_PRICES[form].bn) : tile(ROWS_PRICES[form].bm, ROWS_PRICES[form].bn);
  }
  const bool turned = b_col_maj && c_col_maj;
  const GemmPlan plan = gemm_plan(turned ? N : M, turned ? M : N, K, b_col_maj, c_col_maj && !turned);
  switch (plan.form) {
    case GemmForm::LONG_STAGES: return by_long_stages(long_columns(turned ? M : N));
    case GemmForm::SMALL: return tile(plan.small.rows, b_col_maj ? 32 : 64);
    case GemmForm::BIG: return tile(BIG_PRICES[plan.big].bm, BIG_PRICES[plan.big].bn);
    case GemmForm::TILES_64: return tile(64, 64);
    case GemmForm::TILES_128: return tile(128, 128);
    default: return 0;
  }
}

// A product over many rows whose epilogue reads a second (M, N) operand: the residual sum or the gate.
static int gemm_with_tail(const char* what, const uint16_t* A, const uint16_t* B, const uint16_t* R, uint16_t* C,
                          int M, int N, int K, const QkvTail& tail, const int* valid, void* stream) {
  IRON_REQUIRE(A && B && R && C, "%s: null operand", what);
  IRON_REQUIRE(K <= (1 << 22) && N <= (1 << 22),
               "%s: K (%d) and N (%d) may be at most 2^22 (a tile's rows are addressed with 32-bit offsets)", what, K, N);
  IRON_REQUIRE(M >= 64 && N >= 64 && K > 0 && K % BK == 0,
               "%s: M (%d) and N (%d) at least 64, K (%d) a positive multiple of %d", what, M, N, K, BK);
  IRON_REQUIRE((((uintptr_t)A | (uintptr_t)B | (uintptr_t)R | (uintptr_t)C) & 15) == 0,
               "%s: operands must be 16-byte aligned", what);
  hipStream_t s = (hipStream_t)stream;
  return launch_gemm_rows(A, B, C, M, N, K, valid, s, tail);
}

extern "C" int iron_gemm_residual_bf16(const uint16_t* A, const uint16_t* B, const uint16_t* R, uint16_t* C, int M,
                                       int N, int K, float residual_scale, const int* valid, void* stream) {
  QkvTail tail{};
  tail.residual = R;
  tail.residual_scale = residual_scale;
  return gemm_with_tail("gemm_residual", A, B, R, C, M, N, K, tail, valid, stream);
}

// Whether (and with how much workspace) a residual product followed by its rows' norm is worth
// dealing its K over several blocks: whole 128-column tiles too few to fill the chip at some row
// count, a K long enough to cut, rows a block of the second launch can hold.
extern "C" int64_t iron_gemm_residual_norm_workspace_bytes(int M, int N, int K) {
  if (M < 128 || N < 128 || N % 128 != 0 || N > 8192 || K < 4096 || K % (BK * kSplitKMax) != 0) return 0;
  const int tiles_n = N / 128;
  // 256 tiles' worth of rows are room for every split count: splits * ((256 / splits) / tiles_n) <= 256 / tiles_n.
  return (int64_t)(256 / tiles_n) * 128 * N * (int64_t)sizeof(float);
}

extern "C" int iron_gemm_residual_norm_bf16(const uint16_t* A, const uint16_t* B, const uint16_t* R,
                                            const uint16_t* gain, uint16_t* C, uint16_t* Y, int M, int N, int K,
                                            float residual_scale, float eps, const int* valid, void* workspace,
                                            void* stream) {
  IRON_REQUIRE(A && B && R && gain && C && Y && workspace, "gemm_residual_norm: null operand");
  IRON_REQUIRE(iron_gemm_residual_norm_workspace_bytes(M, N, K) > 0,
               "gemm_residual_norm: M (%d) at least 128, N (%d) a multiple of 128 up to 8192, K (%d) a multiple of %d "
               "from 4096 on (other shapes: iron_gemm_residual_bf16, then iron_rmsnorm_bf16)", M, N, K, BK * kSplitKMax);
  IRON_REQUIRE(K <= (1 << 22), "gemm_residual_norm: K (%d) may be at most 2^22 (a tile's rows are addressed with 32-bit offsets)", K);
  IRON_REQUIRE((((uintptr_t)A | (uintptr_t)B | (uintptr_t)R | (uintptr_t)gain | (uintptr_t)C | (uintptr_t)Y |
                 (uintptr_t)workspace) & 15) == 0,
               "gemm_residual_norm: operands must be 16-byte aligned");
  IRON_REQUIRE(Y != C && Y != R, "gemm_residual_norm: the normed rows need a buffer of their own");
  hipStream_t s = (hipStream_t)stream;
  int tiles_m = (M + 127) / 128;
  const int tiles_n = N / 128;
  // Whole-K tiles in the XCD-aware order where whole patches allow it (the added tile rows lie past M).
  if (tiles_m >= 8 && !patched_order(tiles_m, tiles_n) && patched_order((tiles_m + 7) & ~7, tiles_n))
    tiles_m = (tiles_m + 7) & ~7;
  const Tiling whole{tiles_m, tiles_n, patched_order(tiles_m, tiles_n)};
  QkvTail tail{};
  tail.residual = R;
  tail.residual_scale = residual_scale;
  constexpr size_t lds = (size_t)NT_STAGES * 256 * BK * 2;
  static_assert(lds >= BigTile<2, 2, 3, 4>::LDS_BYTES, "the tiles of 96 rows fit too");
  static LdsOptIn opt_in;
  if (hipError_t e = opt_in.ensure(reinterpret_cast<const void*>(&gemm_splitk_kernel), lds); e != hipSuccess) {
    set_error("gemm_residual_norm: %s", hipGetErrorString(e));
    return (int)e;
  }
  const int blocks = whole.tiles_m * whole.tiles_n > 256 ? whole.tiles_m * whole.tiles_n : 256;
  hipLaunchKernelGGL(gemm_splitk_kernel, dim3(blocks), dim3(256), lds, s, A, B, C, M, N, K, valid, whole, tail,
                     (float*)workspace);
  const int chunks = (N / 8 + 255) / 256;
#define IRON_FINISH(CH)                                                                                          \
  hipLaunchKernelGGL((gemm_finish_rows_kernel<CH>), dim3(M), dim3(256), 0, s, (const float*)workspace, R,        \
                     residual_scale, C, gain, Y, M, N, eps, valid, tiles_n, K)
  if (chunks <= 1) IRON_FINISH(1);
  else if (chunks == 2) IRON_FINISH(2);
  else IRON_FINISH(4);
#undef IRON_FINISH
  IRON_LAUNCH_CHECK();
}

extern "C" int iron_gemm_gated_bf16(const uint16_t* A, const uint16_t* B, const uint16_t* G, uint16_t* C, int M,
                                    int N, int K, int activation, const int* valid, void* stream) {
  IRON_REQUIRE(activation >= 1 && activation <= 3, "gemm_gated: activation (%d) is 1 (SiLU), 2 (GELU, tanh form) or 3 (ReLU)",
               activation);
  QkvTail tail{};
  tail.residual = G;
  tail.gated = activation;
  return gemm_with_tail("gemm_gated", A, B, G, C, M, N, K, tail, valid, stream);
}

// G may be null: the gate's product is then stored nowhere.  It is as many bytes as the output, behind each tile's last product, where nothing is left to
// hide them under (weights out of memory, us with and without: 2048 x 8192 x 2048 111 / 107, 857 rows 52 / 50, 4096 x 14336 x 4096 699 / 677, 1024 x 4096 x 1024
// 23.4 / 21.5, 200 rows of 2048 x 512 8.0 / 7.65).
static int gemm_gated_pair(const char* what, const uint16_t* A, const uint16_t* Bg, const uint16_t* Bu, uint16_t* G, uint16_t* C, int M, int N, int K,
                           int activation, const int* valid, void* stream) {
  IRON_REQUIRE(A && Bg && Bu && C, "%s: null operand", what);
  IRON_REQUIRE(activation >= 1 && activation <= 3, "%s: activation (%d) is 1 (SiLU), 2 (GELU, tanh form) or 3 (ReLU)", what,
               activation);
  if (M < 64 && valid == nullptr) return iron_gemm_few_bf16(A, Bg, Bu, C, M, N, K, activation, stream);
  IRON_REQUIRE(G != C, "%s: the gate's product and the output are different buffers", what);
  IRON_REQUIRE(K <= (1 << 22) && N <= (1 << 22),
               "%s: K (%d) and N (%d) may be at most 2^22 (a tile's rows are addressed with 32-bit offsets)", what, K, N);
  IRON_REQUIRE(M >= 64 && N >= 64 && K > 0 && K % BK == 0,
               "%s: M (%d) and N (%d) at least 64, K (%d) a positive multiple of %d", what, M, N, K, BK);
  IRON_REQUIRE((((uintptr_t)A | (uintptr_t)Bg | (uintptr_t)Bu | (uintptr_t)G | (uintptr_t)C) & 15) == 0,
               "%s: operands must be 16-byte aligned", what);
  return launch_gemm_gated_pair(A, Bg, Bu, G, C, M, N, K, valid, activation, (hipStream_t)stream);
}

extern "C" int iron_gemm_gated_pair_bf16(const uint16_t* A, const uint16_t* Bg, const uint16_t* Bu, uint16_t* G,
                                         uint16_t* C, int M, int N, int K, int activation, const int* valid,
                                         void* stream) {
  IRON_REQUIRE(G || M < 64, "gemm_gated_pair: null operand");
  return gemm_gated_pair("gemm_gated_pair", A, Bg, Bu, G, C, M, N, K, activation, valid, stream);
}

extern "C" int iron_gemm_gated_product_bf16(const uint16_t* A, const uint16_t* Bg, const uint16_t* Bu, uint16_t* C, int M, int N, int K, int activation,
                                            const int* valid, void* stream) {
  return gemm_gated_pair("gemm_gated_product", A, Bg, Bu, nullptr, C, M, N, K, activation, valid, stream);
}

static int prefill_qkv(const uint16_t* x, const uint16_t* Wq, const uint16_t* Wk, const uint16_t* Wv,
                       const uint16_t* angles, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out, int rows,
                       int hidden, int heads, int kv_heads, int d, const int* valid, const int* kv_row0,
                       int kv_rows, void* stream) {
  IRON_REQUIRE(x && Wq && Wk && Wv && angles && q_out && k_out && v_out, "prefill_qkv: null operand");
  IRON_REQUIRE(d == 64, "prefill_qkv: d (%d) must be 64 (a wave's 64 output columns are one head)", d);
  IRON_REQUIRE(rows >= 64 && heads > 0 && kv_heads > 0 && heads % 2 == 0 && kv_heads % 2 == 0,
               "prefill_qkv: rows (%d) at least 64; heads (%d) and kv_heads (%d) positive and even "
               "(whole 128-column tiles)", rows, heads, kv_heads);
  IRON_REQUIRE(hidden > 0 && hidden % BK == 0, "prefill_qkv: hidden (%d) must be a positive multiple of %d", hidden, BK);
  IRON_REQUIRE(hidden <= (1 << 22), "prefill_qkv: hidden (%d) may be at most 2^22 (a tile's rows are addressed with 32-bit offsets)", hidden);
  IRON_REQUIRE((((uintptr_t)x | (uintptr_t)Wq | (uintptr_t)Wk | (uintptr_t)Wv | (uintptr_t)angles |
                 (uintptr_t)q_out | (uintptr_t)k_out | (uintptr_t)v_out) & 15) == 0,
               "prefill_qkv: operands must be 16-byte aligned");
  QkvTail tail{Wk, Wv, k_out, v_out, angles, kv_heads * d};
  tail.kv_row0 = kv_row0;
  tail.kv_rows = kv_rows;
  hipStream_t s = (hipStream_t)stream;
  // 192-wide tiles (three heads) when they make fewer rounds over the chip than 128-wide ones: in
  // units of a 128 x 128 tile's work a launch costs rounds x tile width.  The row bound is read on
  // the device, so with one the blocks of one launch choose the tiling by it.
  const int total = heads + 2 * kv_heads, cus = 256;
  auto cost = [&](int live_rows, int tile_n, int n_tiles) {
    const int tiles = ((live_rows + 127) / 128) * n_tiles;
    return (double)((tiles + cus - 1) / cus) * tile_n;
  };
  const bool wide_ok = total % 3 == 0;
  auto wide_wins = [&](int live_rows) {
    return wide_ok && cost(live_rows, 192, total / 3) < cost(live_rows, 128, total / 2);
  };
  // One-head tiles while they fit one round over the chip and beat both of the others' cost.
  auto thin_wins = [&](int live_rows) {
    const double c = cost(live_rows, 64, total);
    return ((live_rows + 127) / 128) * total <= cus && c < cost(live_rows, 128, total / 2) &&
           (!wide_ok || c < cost(live_rows, 192, total / 3));
  };
  int thin_upto = 0;
  for (int live = 128; live <= ((rows + 127) / 128) * 128; live += 128)
    if (thin_wins(live)) thin_upto = live;
  if (thin_upto >= rows && (valid == nullptr ? rows : 1) > few_qkv_rows(total, hidden, 64)) return launch_qkv64(x, Wq, q_out, rows, heads, kv_heads, hidden, valid, s, tail);
  // The bound above which the winner at `rows` wins, if the two ever change places below `rows`.
  int above = -1;
  if (valid != nullptr)
    for (int live = 128; live <= rows; live += 128)
      if (wide_wins(live) != wide_wins(rows)) above = live;
  if (valid == nullptr && rows > few_qkv_rows(total, hidden, 64)) thin_upto = 0;
  if (above < 0 && thin_upto == 0) {
    if (wide_wins(rows)) return launch_qkv192(x, Wq, q_out, rows, heads, kv_heads, hidden, valid, s, tail);
    return launch_gemm_nt<false, true>(x, Wq, q_out, rows, heads * d, hidden, valid, s, tail);
  }
  return launch_qkv_either(x, Wq, q_out, rows, heads, kv_heads, hidden, valid, s, tail, above, wide_wins(rows), wide_ok,
                           thin_upto);
}

extern "C" int iron_prefill_qkv_bf16(const uint16_t* x, const uint16_t* Wq, const uint16_t* Wk,
                                     const uint16_t* Wv, const uint16_t* angles, uint16_t* q_out,
                                     uint16_t* k_out, uint16_t* v_out, int rows, int hidden, int heads,
                                     int kv_heads, int d, const int* valid, void* stream) {
  return prefill_qkv(x, Wq, Wk, Wv, angles, q_out, k_out, v_out, rows, hidden, heads, kv_heads, d, valid, nullptr, 0,
                     stream);
}

extern "C" int iron_prefill_qkv_cache_bf16(const uint16_t* x, const uint16_t* Wq, const uint16_t* Wk,
                                           const uint16_t* Wv, const uint16_t* angles, uint16_t* q_out,
                                           uint16_t* keys, uint16_t* values, int rows, int hidden, int heads,
                                           int kv_heads, int d, int cache_rows, const int* start,
                                           const int* valid, void* stream) {
  IRON_REQUIRE(start != nullptr, "prefill_qkv_cache: null start");
  IRON_REQUIRE(cache_rows > 0, "prefill_qkv_cache: cache_rows (%d) must be positive", cache_rows);
  // Whatever the bound word holds it is at most `rows`: the rows under it then fit the cache from some row on.
  IRON_REQUIRE(rows <= cache_rows, "prefill_qkv_cache: the chunk's %d rows must fit the cache's %d", rows, cache_rows);
  return prefill_qkv(x, Wq, Wk, Wv, angles, q_out, keys, values, rows, hidden, heads, kv_heads, d, valid, start,
                     cache_rows, stream);
}
