// What the decode projections share (skinny_gemm.hip, stream_gemm.hip): tile
// sizes, the matrix-core step, the argmax order and the arguments of a launch.
#pragma once

#include "qf_device.h"

namespace qf {

constexpr int kTile = 16;    // rows of W (output columns) per n-tile; rows of x per m-tile
constexpr int kStep = 32;    // k per MFMA
constexpr int kChunk = 64;   // the shape rule's k granularity
constexpr int kMaxRows = 64;

// Epilogues.
constexpr int kEpiPartials = 0;  // f32 split-K partials [S, M, N]
constexpr int kEpiSiluMul = 1;   // packed gate/up -> bf16 silu(gate) * up [M, N]
constexpr int kEpiArgmax = 2;    // bf16 logits (optional) + argmax candidates per workgroup

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(const uint4& a, const uint4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                  __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Is (v, i) ahead of (bv, bi) in argmax order: larger value, NaN above
// everything, the lower index on equal values (torch.argmax's first maximum)?
__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
  const bool vn = v != v, bn = bv != bv;
  if (vn || bn) return vn && (!bn || i < bi);
  return v > bv || (v == bv && i < bi);
}

struct SkinnyArgs {
  const uint16_t* x;   // [m, k]
  const uint16_t* w;   // [n, k], or [2n, k] gate rows then up rows
  float* partials;     // [splits, m, n]; argmax: (value, index) pairs [m, workgroups]
  uint16_t* out;       // [m, n] (argmax: optional bf16 logits, may be null)
  int64_t k;
  int32_t m;
  int32_t n;           // output columns
  int32_t chunks;      // 64-wide k chunks per split
  int32_t splits_major; // 1: blockIdx.x is the split and blockIdx.y the column block
  // kXMerged only: x row m, columns [128 h, 128 h + 128), is the merge of the
  // attention segments of virtual head m * seg_kv_heads + h / seg_groups,
  // query group h % seg_groups (partials [V, S, G, 128], stats [V, S, 2, G]).
  const float* seg_partials;
  const float* seg_stats;
  int32_t seg_splits;
  int32_t seg_groups;
  int32_t seg_kv_heads;
  // kXNormed only: x (the residual stream `total`, bf16 [m, k]) enters as
  //   inv = 1 / sqrt(f32(sum_g sq[m][g]) / k + eps),  bf16(bf16(x * inv) * gain)
  // with sq f64 [m, QF_ROW_GROUPS] (per-workgroup sums of squares from
  // qf_linear_residual) and gain bf16 [k].
  const double* sq;
  const uint16_t* gain;
  float eps;
};

// Column groups of a weight stream: one workgroup per CU over all splits
// (fewer for small outputs).
inline int32_t stream_groups(int32_t tiles, int splits) {
  const int fill = kCUs / splits < 1 ? 1 : kCUs / splits;
  return fill < tiles ? fill : tiles;
}

// The weight streams (stream_gemm.hip; partials at 17..64 rows, the others at
// any): x, w, partials / out, k, m, n and chunks set, checked by the caller.
int stream_partials(const SkinnyArgs& a, int splits, hipStream_t s);
int stream_silu(const SkinnyArgs& a, hipStream_t s);
int stream_argmax(const SkinnyArgs& a, hipStream_t s);

}  // namespace qf
