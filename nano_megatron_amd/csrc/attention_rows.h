// Attention one row at a time: a wavefront per query row (dK/dV: per key), lane
// l holding head-dim elements l and l + 64 (head_dim <= 128).
//
// A hidden key or query is not read here at all.  The matrix products of the
// tiled kernels take every row of a tile, hidden ones with weight zero, and
// 0 x NaN (or infinity) is NaN: a tiled kernel whose result for a row is NaN
// runs that row again through these functions before it stores it, so padded
// keys and queries may hold anything under any mask.  Finite data never gets
// here, and costs the tiled kernels one comparison per result.
#pragma once

#include "attention_common.h"
#include "dropout_math.h"

namespace nmb {
namespace {

struct MaskRef {
  const void* p;
  int64_t sb, sh, sq, sk;  // element strides of [batch, q_heads, seq_q, seq_k] (0: broadcast)
};

// What a row's attention takes besides its tensors: the first element of the
// mask's (batch, head), and the element of (batch, head, query 0, key 0) in
// the dropout stream.
struct RowMask {
  MaskRef mr;
  int64_t base;
  uint64_t drop0;
  DropoutParams dp;
};

__device__ __forceinline__ RowMask row_mask(const AttnShape& p, const MaskRef& mr, const DropoutParams& dp, int b,
                                            int h) {
  return RowMask{mr, b * mr.sb + h * mr.sh, (static_cast<uint64_t>(b) * p.Hq + h) * p.Sq * p.Sk, dp};
}

// MK 0: no mask, 1: boolean, 2: additive (-inf drops the key)
template <typename T, int MK>
__device__ __forceinline__ bool row_visible(const RowMask& rm, int i, int j, float& add) {
  add = 0.f;
  if constexpr (MK == 0) return true;
  const int64_t off = rm.base + i * rm.mr.sq + j * rm.mr.sk;
  if constexpr (MK == 1) {
    return static_cast<const uint8_t*>(rm.mr.p)[off] != 0;
  } else {
    add = to_f32(static_cast<const T*>(rm.mr.p)[off]);
    return add != -__builtin_inff();
  }
}

template <bool DROP>
__device__ __forceinline__ float row_keep(const RowMask& rm, const AttnShape& p, int i, int j) {
  if constexpr (!DROP) return 1.f;
  return drop_factor(rm.dp, rm.drop0 + static_cast<uint64_t>(i) * p.Sk + j);
}

template <typename T>
__device__ __forceinline__ float row_dot(const T* a, const T* b, int D, int lane) {
  float s = 0.f;
  for (int d = lane; d < D; d += 64) s += to_f32(a[d]) * to_f32(b[d]);
  return wave_sum(s);
}

// Query row i (at qr) over one K/V block whose rows start at kb, vb: the
// running maximum, sum and outputs.
template <typename T, int MK, bool DROP>
__device__ void row_fwd(const T* qr, const T* kb, const T* vb, int64_t koff, int i, const AttnShape& p, int D,
                        const RowMask& rm, int lane, float& m, float& l, float (&acc)[2]) {
  for (int j = 0; j < p.Sk; ++j) {
    if (p.causal && koff + j > p.q_offset + i) break;
    float add;
    if (!row_visible<T, MK>(rm, i, j, add)) continue;
    const T* vr = vb + static_cast<int64_t>(j) * p.kv_ss;
    const float s = row_dot(qr, kb + static_cast<int64_t>(j) * p.kv_ss, D, lane) * p.scale + add;
    const float mn = fmaxf(m, s);
    const float alpha = expf(m - mn), pv = expf(s - mn);
    m = mn;
    l = l * alpha + pv;
    const float pz = pv * row_keep<DROP>(rm, p, i, j);  // dropout acts after the normalisation
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int d = lane + 64 * c;
      if (d < D) acc[c] = acc[c] * alpha + pz * to_f32(vr[d]);
    }
    if (l != l) break;  // NaN: sum and outputs stay so
  }
}

// 1 / sum of a row's probabilities (0 for a row without any)
__device__ __forceinline__ float inverse_sum(float s) { return s > 0.f ? 1.f / s : (s == 0.f ? 0.f : s); }

// dQ of query row i (before the scale), from its lse and delta; psum: the sum
// of its probabilities.
template <typename T, int MK, bool DROP>
__device__ void row_dq(const T* qr, const T* dr, const T* kb, const T* vb, int64_t koff, int i, float lse, float delta,
                       const AttnShape& p, int D, const RowMask& rm, int lane, float (&acc)[2], float& psum) {
  if (lse == -__builtin_inff()) return;
  for (int j = 0; j < p.Sk; ++j) {
    if (p.causal && koff + j > p.q_offset + i) break;
    float add;
    if (!row_visible<T, MK>(rm, i, j, add)) continue;
    const T* kr = kb + static_cast<int64_t>(j) * p.kv_ss;
    const T* vr = vb + static_cast<int64_t>(j) * p.kv_ss;
    const float pv = expf(row_dot(qr, kr, D, lane) * p.scale + add - lse);
    psum += pv;
    const float ds = pv * (row_keep<DROP>(rm, p, i, j) * row_dot(dr, vr, D, lane) - delta);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int d = lane + 64 * c;
      if (d < D) acc[c] += ds * to_f32(kr[d]);
    }
  }
}

// dK (before the scale) and dV of key j (rows kr, vr) from the queries of one
// head (rows from qb, db; lse, delta and, if given, norm of the head).
template <typename T, int MK, bool DROP>
__device__ void row_dkdv(const T* kr, const T* vr, const T* qb, const T* db, const float* lse, const float* delta,
                         const float* norm, int64_t koff, int j, const AttnShape& p, int D, const RowMask& rm, int lane,
                         float (&dk)[2], float (&dv)[2]) {
  for (int i = 0; i < p.Sq; ++i) {
    const float ls = lse[i];
    float add;
    if ((p.causal && koff + j > p.q_offset + i) || ls == -__builtin_inff() || !row_visible<T, MK>(rm, i, j, add))
      continue;
    const T* qr = qb + static_cast<int64_t>(i) * p.q_ss;
    const T* dr = db + static_cast<int64_t>(i) * p.o_ss;
    float pv = expf(row_dot(qr, kr, D, lane) * p.scale + add - ls);
    if (norm != nullptr) pv *= norm[i];
    const float z = row_keep<DROP>(rm, p, i, j);
    const float ds = pv * (z * row_dot(dr, vr, D, lane) - delta[i]);
    const float pz = pv * z;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int d = lane + 64 * c;
      if (d < D) {
        dv[c] += pz * to_f32(dr[d]);
        dk[c] += ds * to_f32(qr[d]);
      }
    }
  }
}

template <typename T>
__device__ __forceinline__ void row_store(T* row, const float (&v)[2], float f, int D, int lane) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int d = lane + 64 * c;
    if (d < D) row[d] = from_f32<T>(v[c] * f);
  }
}

// the rows (bit 0 .. 15) that a lane of any of the wave's four 16-lane groups names
__device__ __forceinline__ uint32_t rows_of(uint64_t lanes) {
  const uint32_t x = static_cast<uint32_t>(lanes) | static_cast<uint32_t>(lanes >> 32);
  return (x | x >> 16) & 0xffffu;
}

}  // namespace
}  // namespace nmb
