// Decode projections y = x @ W^T as one weight stream per compute unit: partials at
// 17..64 rows of x, gate/up from 9 and the LM head from 5 (skinny_gemm.hip
// says which calls; engine/kernels/skinny_gemm.py:28-121 is the reference).
//
// What bounds it: HBM, the weight read once; at these row counts x (up to 64 x
// K) comes from L2 for every column block and weighs as much as the weights
// do in the CU's own traffic.  So one 8-wave workgroup per CU takes an equal
// share of the output columns (the fewest, widest column blocks that fill the
// chip, so x is re-read the least), and everything moves by
// global_load_lds_dwordx4 straight into an LDS ring of three stages, 128 k wide
// for blocks of up to 8 tiles and 64 beyond: no registers hold loads in
// flight, and up to two stages (96 KB) per CU are, whatever the waves are
// doing.  One barrier per stage; a stage's loads are waited for by count
// (vmcnt, S - 2 stages stay in flight over the wait).  A workgroup whose
// columns need several blocks runs them through one continuous ring.  K ranges
// of a few stages do not fill it (64-row qkv and o_proj, four stages: 42 reads
// in flight per CU where the LM head holds 95).
//
//   A operand = 16 rows of W (one n-tile), B operand = 16 rows of x (one
//   m-tile), 32 k per v_mfma_f32_16x16x32_bf16; lane l's result is
//   D[4*(l/16) + i][l % 16] = y[m0 + l%16][n0 + 4*(l/16) + i].
//   Waves: MG groups of two m-tiles times 8 / MG groups of n-tiles
//   (tile t to group t % (8 / MG)); every output has one wave and one chain
//   of additions, so no reduction between waves is needed.
//
// A ring tile is 16 rows of 256 or 128 bytes; 16-byte piece p of row r sits at
// piece p ^ swizzle(r), so the 16 lanes of a fragment read touch all 64 banks
// once.  The DMA writes linearly, so the lanes fetch permuted pieces of a
// row's own bytes.
//
// Every call's order of additions is a function of K and its split count
// (launch_stream), not of the columns or of the rows beside a row.
//
// Gate/up tiles hold 8 gate rows over the matching 8 up rows: the SiLU
// epilogue is local to the wave.
#include "qf_skinny.h"
#include "qf_silu.h"

namespace qf {
namespace {

constexpr int kStreamWaves = 8;
constexpr int kStreamBlock = kStreamWaves * kWave;
constexpr int kLdsBytes = 160 << 10;
constexpr int kLoadBytes = 16 * kWave;             // one load instruction of a wave
constexpr int kMaxStages = 3;

// Slot of 16-byte piece p in row r of a ring tile is p ^ swizzle(r): the 16
// rows' slots of one piece then cover all 64 banks once.
template <int KW>
__device__ __forceinline__ int swizzle(int r) { return KW == 128 ? r : (r >> 1) & 7; }

struct StreamArgs {
  const uint16_t* x;
  const uint16_t* w;
  float* partials;
  uint16_t* out;
  int64_t k;
  int32_t m, n;
  int32_t chunks;        // 64-wide k chunks per split
  int32_t tiles;         // n-tiles (gate/up: of 8 output columns) of the whole output
  int32_t groups;        // column groups: one workgroup each per split
  int32_t block_tiles;   // tiles of a column block, at most
  int32_t splits;
  int32_t splits_major;  // 1: consecutive workgroups take the splits of one column group
};

// One 1 KB load: lane l's 16 bytes go to LDS byte dst + 16 l.  Inline assembly
// so that the compiler does not order later LDS reads after it; the ring's
// waits are explicit.  NT: streamed once.
template <bool NT>
__device__ __forceinline__ void dma16(const uint16_t* src, uint32_t dst) {
  uint32_t saved;
  if constexpr (NT)
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
        "global_load_lds_dwordx4 %2, off nt\n\ts_mov_b32 m0, %0"
        : "=&s"(saved) : "s"(dst), "v"(src) : "memory");
  else
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
        "global_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
        : "=&s"(saved) : "s"(dst), "v"(src) : "memory");
}

// All of the wave's LDS reads done, and all but the newest N of its loads.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
// All but the newest `stages` (at most MAX) stages of `per` (at most PER) loads each.
template <int PER, int MAX>
__device__ __forceinline__ void wait_stages(int per, int stages) {
  if constexpr (MAX == 0 || PER == 0) {
    wait_loads<0>();
  } else {
    if (stages < MAX) wait_stages<PER, MAX - 1>(per, stages);
    else if (per < PER) wait_stages<PER - 1, MAX>(per, stages);
    else wait_loads<MAX * PER>();
  }
}

// KW: k per ring stage; PHASED: K in quarters, from a start of the group's own.
template <int MT, int NT, int KW, int EPI, bool PHASED>
__global__ __launch_bounds__(kStreamBlock, 2) void stream_kernel(StreamArgs a) {
  constexpr bool PAIRS = EPI == kEpiSiluMul;
  constexpr int MG = MT > 2 ? 2 : 1;               // wave groups over m
  constexpr int MTW = MT > 1 ? 2 : 1;              // m-tiles per wave
  constexpr int NG = kStreamWaves / MG;            // wave groups over n
  constexpr int NTW = (NT + NG - 1) / NG;          // n-tiles per wave, at most
  constexpr int kTiles = NT + MT;
  constexpr int kRowBytes = KW * 2;
  constexpr int kTileBytes = kTile * kRowBytes;
  constexpr int kSteps = KW / kStep;
  constexpr int kPieces = KW / 8;                  // 16-byte pieces per row
  constexpr int kLoadRows = kWave / kPieces;       // rows per load
  constexpr int kTileLoads = kTile / kLoadRows;    // loads per tile
  constexpr int TG = kStreamWaves / kTileLoads;    // tile groups of loading waves
  constexpr int kStageBytes = kTiles * kTileBytes;
  constexpr int kFit = kLdsBytes / kStageBytes;
  constexpr int S = kFit < kMaxStages ? kFit : kMaxStages;
  static_assert(S >= 2, "ring");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[S * kStageBytes];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane % kTile, g = lane / kTile;
  const int wn = wave % NG, wm = wave / NG;
  const int split = a.splits_major ? blockIdx.x % a.splits : blockIdx.x / a.groups;
  const int group = a.splits_major ? blockIdx.x / a.splits : blockIdx.x % a.groups;
  const int t_lo = (int)((int64_t)group * a.tiles / a.groups);
  const int t_hi = (int)((int64_t)(group + 1) * a.tiles / a.groups);
  const int64_t kbase = (int64_t)split * a.chunks * kChunk;
  const int stages = (a.chunks * kChunk + KW - 1) / KW;
  const bool ragged = !PHASED && KW > kChunk && (a.chunks & 1);  // last stage half filled
  const int width = a.block_tiles;                 // <= NT: no loads for the rest
  const int blocks = (t_hi - t_lo + width - 1) / width;
  const int total = blocks * stages;

  // Loads: tile i of a stage (NT of W, then MT of x) is loaded by the waves
  // of tile group i % TG, load q of it rows q * kLoadRows ...; lane l fetches
  // row l / kPieces of the load, the piece that belongs at slot l % kPieces.
  const int tg = wave / kTileLoads, q = wave % kTileLoads;
  const int lrow = q * kLoadRows + lane / kPieces;
  const int piece = (lane % kPieces) ^ swizzle<KW>(lrow);
  const int64_t wlane = (int64_t)(lane / kPieces) * a.k;
  // x tiles x0, x0 + TG, ...: tile NT + mt of the stage is of group (NT + mt) % TG
  constexpr int kXLoads = (MT + TG - 1) / TG;
  const int x0 = (tg + kTiles * TG - NT) % TG;
  const uint16_t* xrow[kXLoads];
#pragma unroll
  for (int c = 0; c < kXLoads; ++c) {
    const int row = kTile * (x0 + TG * c) + lrow;
    xrow[c] = a.x + (int64_t)(row < a.m ? row : a.m - 1) * a.k + kbase;
  }
  const uint32_t ring0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)ring +
                         kLoadBytes * q;
  // PHASED: part v of a group's pass over K is quarter v ^ phase, and the
  // quarters are added as (q0 + q1) + (q2 + q3).  Whatever the phase, the same
  // sums are formed (with their two sides in either order, which rounds the
  // same), so a weight row's result does not depend on its group, on N or on
  // how the columns are sharded.  The phase is hashed so that it does not run
  // with the group's address bits (16,384-column gate/up at K = 4096, 64 rows:
  // 77 us with a start that follows the group number, 45 hashed).
  constexpr int kParts = PHASED ? 4 : 1;
  const int per_part = stages / kParts;            // PHASED: K is a multiple of 1,024
  const int phase = PHASED ? (int)(((uint32_t)group * 0x9E3779B1u) >> 30) : 0;
  // Loads of this wave per stage: its tiles of the block's W, and of x.
  const int per_stage = (width > tg ? (width - tg + TG - 1) / TG : 0) +
                        (MT > x0 ? (MT - x0 + TG - 1) / TG : 0);
  // Next stage to issue: stage is_in of part is_part of the block at is_tile.
  int is_tile = t_lo, is_part = 0, is_in = 0, is_stage = phase * per_part;
  auto issue = [&](int slot) {
    // Past the split's range in a half-filled last stage: re-read its first
    // half (those LDS pieces are not used).
    const bool cut = ragged && is_stage == stages - 1;
    const int64_t off = (int64_t)is_stage * KW + 8 * (cut ? piece & 7 : piece);
    const uint32_t dst = ring0 + slot * kStageBytes;
#pragma unroll
    for (int c = 0; c < (NT + TG - 1) / TG; ++c) {
      const int i = tg + TG * c;
      if (i < width) {
        int t = is_tile + i;
        if (t >= t_hi) t = is_tile;                // the last block's missing tiles: its first again
        const int64_t row = PAIRS ? (q < kTileLoads / 2 ? 0 : (int64_t)a.n - 8) + 8 * (int64_t)t +
                                        q * kLoadRows
                                  : (int64_t)kTile * t + q * kLoadRows;
        dma16<true>(a.w + row * a.k + kbase + wlane + off, dst + i * kTileBytes);
      }
    }
#pragma unroll
    for (int c = 0; c < kXLoads; ++c) {
      const int mt = x0 + TG * c;
      if (mt < MT) dma16<false>(xrow[c] + off, dst + (NT + mt) * kTileBytes);
    }
    ++is_stage;
    if (++is_in == per_part) {
      is_in = 0;
      if (++is_part == kParts) {
        is_part = 0;
        is_tile += width;
      }
      is_stage = (is_part ^ phase) * per_part;
    }
  };

  f32x4 acc[NTW][MTW];
  // PHASED: the quarter, and the half, that wait for the other side of their sum.
  f32x4 quarter[PHASED ? NTW : 1][PHASED ? MTW : 1], half[PHASED ? NTW : 1][PHASED ? MTW : 1];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int j = 0; j < MTW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  int rd[kSteps];                                  // fragment of k step s: row r, piece 4 s + g
#pragma unroll
  for (int s = 0; s < kSteps; ++s) rd[s] = r * kRowBytes + 16 * ((4 * s + g) ^ swizzle<KW>(r));
  auto products = [&](const uint8_t* buf, auto nt_tag, auto steps_tag) {
    constexpr int N = decltype(nt_tag)::value, STEPS = decltype(steps_tag)::value;
    uint4 fw[STEPS][N > 0 ? N : 1], fx[STEPS][MTW];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
#pragma unroll
      for (int j = 0; j < MTW; ++j) {
        int mt = wm * MTW + j;
        if (MT % MTW != 0 && mt >= MT) mt = MT - 1;  // rows past the last tile: never stored
        fx[s][j] = *reinterpret_cast<const uint4*>(buf + (NT + mt) * kTileBytes + rd[s]);
      }
#pragma unroll
      for (int i = 0; i < N; ++i)
        fw[s][i] = *reinterpret_cast<const uint4*>(buf + (wn + NG * i) * kTileBytes + rd[s]);
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < MTW; ++j) acc[i][j] = mfma(fw[s][i], fx[s][j], acc[i][j]);
  };
  auto stage_products = [&](const uint8_t* buf, auto steps_tag) {
    // Groups past the last full round of n-tiles have one tile fewer.
    if (NT % NG == 0 || wn < NT % NG) products(buf, std::integral_constant<int, NTW>{}, steps_tag);
    else products(buf, std::integral_constant<int, NTW - 1>{}, steps_tag);
  };

  float best[MTW];                                 // argmax form only
  int besti[MTW];
#pragma unroll
  for (int j = 0; j < MTW; ++j) {
    best[j] = -__builtin_inff();
    besti[j] = INT32_MAX;
  }
  auto store = [&](int tile0) {
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      const int t = tile0 + wn + NG * i;
      const bool live = wn + NG * i < width && t < t_hi;
#pragma unroll
      for (int j = 0; j < MTW; ++j) {
        const int m = kTile * (wm * MTW + j) + r;
        const f32x4 v = acc[i][j];
        if constexpr (EPI == kEpiPartials) {
          if (live && m < a.m)
            *reinterpret_cast<f32x4*>(a.partials + ((int64_t)split * a.m + m) * a.n + kTile * t +
                                      4 * g) = v;
        } else if constexpr (EPI == kEpiSiluMul) {
          // Lanes g = 0, 1 hold gate columns 8 t + 4 g .. + 3, g = 2, 3 the
          // matching up columns; each projection and the SiLU round to bf16.
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = __shfl_xor(v[e], 32);
          if (live && g < 2 && m < a.m) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              y[e] = from_bf16(to_bf16(silu_f32(from_bf16(to_bf16(v[e]))))) *
                     from_bf16(to_bf16(y[e]));
            *reinterpret_cast<uint2*>(a.out + (int64_t)m * a.n + 8 * t + 4 * g) =
                make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
          }
        } else {
          // bf16 logits; per lane and row the largest so far, lowest column on
          // ties (NaN largest).
          if (live && m < a.m) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              y[e] = from_bf16(to_bf16(v[e]));
              const int col = kTile * t + 4 * g + e;
              if (better(y[e], col, best[j], besti[j])) {
                best[j] = y[e];
                besti[j] = col;
              }
            }
            if (a.out)
              *reinterpret_cast<uint2*>(a.out + (int64_t)m * a.n + kTile * t + 4 * g) =
                  make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
          }
        }
      }
    }
  };

#pragma unroll
  for (int d = 0; d < S - 1; ++d)
    if (d < total) issue(d);
  int slot = 0, next = S - 1;
  constexpr int kMostLoads = (NT + TG - 1) / TG + kXLoads;
  // Stage `it` of the sequence; `last`: the last one of its block.
  auto step = [&](int it, bool last) {
    wait_stages<kMostLoads, S - 2>(per_stage, total - 1 - it);  // of the stages after this one
    __builtin_amdgcn_s_barrier();                  // stage `it` is whole; stage `it - 1` is read
    asm volatile("" ::: "memory");
    if (it + S - 1 < total) issue(next);
    const uint8_t* buf = ring + slot * kStageBytes;
    if (ragged && last) stage_products(buf, std::integral_constant<int, kChunk / kStep>{});
    else stage_products(buf, std::integral_constant<int, kSteps>{});
    slot = slot + 1 == S ? 0 : slot + 1;
    next = next + 1 == S ? 0 : next + 1;
  };
  clear();
  int tile0 = t_lo;
  if constexpr (PHASED) {
    for (int it = 0; it < total; tile0 += width) {
#pragma unroll
      for (int part = 0; part < kParts; ++part) {
        for (int at = 0; at < per_part; ++at, ++it) step(it, false);
#pragma unroll
        for (int i = 0; i < NTW; ++i)
#pragma unroll
          for (int j = 0; j < MTW; ++j) {
            if (part % 2 == 1) acc[i][j] += quarter[i][j];
            if (part == 3) acc[i][j] += half[i][j];
            if (part % 2 == 0) quarter[i][j] = acc[i][j];
            if (part == 1) half[i][j] = acc[i][j];
          }
        if (part == 3) store(tile0);
        clear();
      }
    }
  } else {
    int at = 0;
    for (int it = 0; it < total; ++it) {
      step(it, at == stages - 1);
      if (++at == stages) {
        store(tile0);
        clear();
        at = 0;
        tile0 += width;
      }
    }
  }

  if constexpr (EPI == kEpiArgmax) {
    // One candidate per row and workgroup: over the four lanes of a row, then,
    // through the drained ring, over the waves of its m-tile.  (One per 16
    // columns gave the last kernel 9,496 a row to read, and as many 8-byte
    // stores: the Qwen3-4B head with logits at 64 rows 147.4 -> 144.9 us.)
    uint2* cand = reinterpret_cast<uint2*>(ring);  // [NG][MG * MTW * 16 rows]
    constexpr int kRows = MG * MTW * kTile;
    __syncthreads();                               // the last stage is read
#pragma unroll
    for (int j = 0; j < MTW; ++j) {
#pragma unroll
      for (int mask = 16; mask <= 32; mask *= 2) {
        const float ov = __shfl_xor(best[j], mask);
        const int oi = __shfl_xor(besti[j], mask);
        if (better(ov, oi, best[j], besti[j])) {
          best[j] = ov;
          besti[j] = oi;
        }
      }
      if (g == 0)
        cand[wn * kRows + kTile * (wm * MTW + j) + r] =
            make_uint2(__float_as_uint(best[j]), (uint32_t)besti[j]);
    }
    __syncthreads();
    const int m = threadIdx.x;
    if (m < a.m) {                                 // a.m <= kRows
      uint2 top = cand[m];
#pragma unroll
      for (int w = 1; w < NG; ++w) {
        const uint2 c = cand[w * kRows + m];
        if (better(__uint_as_float(c.x), (int)c.y, __uint_as_float(top.x), (int)top.y)) top = c;
      }
      reinterpret_cast<uint2*>(a.partials)[(int64_t)m * a.groups + group] = top;
    }
  }
}

// Column groups (stream_groups): each an equal run of n-tiles; a block of it is as wide as the
// ring takes (x is re-read once per block), evenly cut.
// PHASED beyond 32 rows: 16, where the two held sums still fit the registers
// (19 spill: the 151,936-column head at K = 2048, 64 rows 159 us, 16 132).
template <int MT, bool PHASED>
constexpr int kMaxBlockTiles = PHASED && MT > 2 ? 16 : 19;

template <int MT, int EPI, bool PHASED>
int launch_stream_as(const SkinnyArgs& s, int splits, hipStream_t stream) {
  StreamArgs a;
  a.x = s.x;
  a.w = s.w;
  a.partials = s.partials;
  a.out = s.out;
  a.k = s.k;
  a.m = s.m;
  a.n = s.n;
  a.chunks = s.chunks;
  a.splits = splits;
  a.tiles = s.n / (EPI == kEpiSiluMul ? kTile / 2 : kTile);
  a.groups = stream_groups(a.tiles, splits);
  const int most = (a.tiles + a.groups - 1) / a.groups;          // tiles of a group
  constexpr int kMost = kMaxBlockTiles<MT, PHASED>;
  const int blocks = (most + kMost - 1) / kMost;
  const int need = (most + blocks - 1) / blocks;                 // tiles of a block
  a.block_tiles = need;
  a.splits_major = splits > 1 && s.k >= s.n ? 1 : 0;
  const dim3 grid((unsigned)((int64_t)a.groups * splits));
#define QF_STREAM(NT, KW)                                                              \
  if constexpr (NT <= kMost)                                                           \
  if (need <= NT) {                                                                    \
    hipLaunchKernelGGL((stream_kernel<MT, NT, KW, EPI, PHASED>), grid,                 \
                       dim3(kStreamBlock), 0, stream, a);                              \
    return launch_status();                                                            \
  }
  // A block loads the tiles it has, not its kernel's NT (a ladder, not every
  // count): 89,344-column head at K = 2560, 22 tiles a workgroup as 2 x 11 on the
  // 13-tile kernel, 64 rows 101 -> 95.8 us, 5 rows 79.2 -> 73.9.
  // Up to 8 tiles 128 k per stage (256-byte runs of each weight row), wider
  // blocks 64 k, so that three stages fit the LDS (Qwen3-4B qkv, 8 tiles, at
  // 32 and 64 rows 9.2 -> 8.7 and 10.9 -> 10.2 us with 128; gate/up, 5 tiles, at
  // 64 rows 27.5 -> 23.9; down and LM head, 13 and 19 tiles, 16.0 -> 13.9 and
  // 154 -> 140 with 64 and the wider blocks it allows).  More than three stages
  // in flight measured slower or even.
  QF_STREAM(1, 128)
  QF_STREAM(2, 128)
  QF_STREAM(3, 128)
  QF_STREAM(4, 128)
  QF_STREAM(5, 128)
  QF_STREAM(6, 128)
  QF_STREAM(8, 128)
  QF_STREAM(10, 64)
  QF_STREAM(13, 64)
  QF_STREAM(16, 64)
  QF_STREAM(19, 64)
#undef QF_STREAM
  return QF_E_SHAPE;  // not reached: need <= kMaxBlockTiles
}

// All workgroups in step read the same columns of rows a constant stride apart,
// and strides of 2, 4 or 8 KB send those to few memory channels.  So at K a
// multiple of 1,024 in one range, a quarter of the workgroups starts in each
// quarter of K (64 rows, in order -> PHASED: 151,936-column head at K = 2048
// 155 -> 132 us; at K = 1024 73 -> 76, but 130,304 columns 71 -> 62; 12,288-column
// gate/up at K = 4096 41.8 -> 36.6, at K = 2048 24.0 -> 21.1).  Other strides
// measured even (K = 2560) and split ranges start apart by themselves: there K
// goes in order.
template <int MT, int EPI>
int launch_stream(const SkinnyArgs& a, int splits, hipStream_t s) {
  if constexpr (EPI != kEpiPartials)
    if (a.k % 1024 == 0) return launch_stream_as<MT, EPI, true>(a, splits, s);
  return launch_stream_as<MT, EPI, false>(a, splits, s);
}

template <int EPI>
int dispatch_stream(const SkinnyArgs& a, int splits, hipStream_t s) {
  switch ((a.m + kTile - 1) / kTile) {
    case 1:
      if constexpr (EPI != kEpiPartials) return launch_stream<1, EPI>(a, splits, s);
      else return QF_E_SHAPE;  // up to 16 rows: skinny_gemm.hip
    case 2: return launch_stream<2, EPI>(a, splits, s);
    case 3: return launch_stream<3, EPI>(a, splits, s);
    default: return launch_stream<4, EPI>(a, splits, s);
  }
}

}  // namespace

int stream_partials(const SkinnyArgs& a, int splits, hipStream_t s) {
  return dispatch_stream<kEpiPartials>(a, splits, s);
}
int stream_silu(const SkinnyArgs& a, hipStream_t s) { return dispatch_stream<kEpiSiluMul>(a, 1, s); }
int stream_argmax(const SkinnyArgs& a, hipStream_t s) { return dispatch_stream<kEpiArgmax>(a, 1, s); }

}  // namespace qf
