// Attention for any head dim <= 128, any strides, fp32 or bf16 storage.
#pragma once

#include "attention_common.h"
#include "dropout_math.h"

namespace nmb {
namespace {

// ---------------------------------------------------------------- delta (fp32 path)
// delta[b, h, i] = sum_d dO[b, i, h, d] * O[b, i, h, d] (fp32).
template <typename T>
__global__ __launch_bounds__(256) void attn_delta_kernel(const T* __restrict__ o,
                                                         const T* __restrict__ dout,
                                                         float* __restrict__ delta, AttnShape p,
                                                         int D) {
  const int64_t rows = static_cast<int64_t>(p.B) * p.Sq * p.Hq;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; r < rows;
       r += static_cast<int64_t>(gridDim.x) * 256) {
    const int h = static_cast<int>(r % p.Hq);
    const int64_t bi = r / p.Hq;
    const int i = static_cast<int>(bi % p.Sq);
    const int b = static_cast<int>(bi / p.Sq);
    const int64_t off = b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh;
    float s = 0.f;
    for (int d = 0; d < D; ++d) s += to_f32(o[off + d]) * to_f32(dout[off + d]);
    delta[(static_cast<int64_t>(b) * p.Hq + h) * p.Sq + i] = s;
  }
}

// ---------------------------------------------------------------- generic path
// One wavefront per query row; lane owns head_dim elements lane and lane + 64
// (head_dim <= 128).  The fp32 configuration's attention, and attention with
// an explicit mask where attention_masked.hip's MFMA kernels do not apply (the reference passes attention_mask
// to SDPA, nn/kernels/torch_backend.py:60-76): MK 0 no mask, 1 a boolean mask
// (one byte per entry, nonzero = attend), 2 an additive mask in the attention
// dtype (added to the scaled scores; -inf drops the key).  A query row with no
// visible key gives zeros and lse = -inf, as the safe softmax of the
// reference's SDPA does.  Attention dropout (SDPA's dropout_p, applied to the
// normalised probabilities): probability (b, h, i, j) is multiplied by the
// dropout_math.h factor of index ((b * Hq + h) * Sq + i) * Sk + j; l and the
// lse stay those of the undropped softmax.
struct MaskRef {
  const void* p;
  int64_t sb, sh, sq, sk;  // element strides of [batch, q_heads, seq_q, seq_k] (0: broadcast)
};

template <typename T, int MK>
__device__ __forceinline__ bool visible(const MaskRef& mr, int b, int h, int64_t i, int64_t j, float& add) {
  if constexpr (MK == 0) {
    return true;
  } else {
    const int64_t off = b * mr.sb + h * mr.sh + i * mr.sq + j * mr.sk;
    if constexpr (MK == 1) {
      return static_cast<const uint8_t*>(mr.p)[off] != 0;
    } else {
      add = to_f32(static_cast<const T*>(mr.p)[off]);
      return add != -__builtin_inff();
    }
  }
}

template <typename T>
__device__ __forceinline__ float dot_row(const T* a, const T* b, int D, int lane) {
  float s = 0.f;
  for (int d = lane; d < D; d += 64) s += to_f32(a[d]) * to_f32(b[d]);
  return wave_sum(s);
}

template <typename T, int MK>
__global__ __launch_bounds__(64) void attn_fwd_generic_kernel(const T* __restrict__ q, KVBlocks kv,
                                                              T* __restrict__ o, float* __restrict__ lse,
                                                              AttnShape p, int D, MaskRef mr,
                                                              DropoutParams dp) {
  const int lane = threadIdx.x;
  const int i = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int hk = h / (p.Hq / p.Hkv);
  const T* qr = q + b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh;
  const int64_t qa = p.q_offset + i;
  const uint64_t prow = ((static_cast<uint64_t>(b) * p.Hq + h) * p.Sq + i) * p.Sk;  // dropout index base
  float m = -__builtin_inff(), l = 0.f;
  float acc[2] = {0.f, 0.f};
  for (int blk = 0; blk < p.nblk; ++blk) {
    const T* kb = static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const T* vb = static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const int64_t koff = kv.koff[blk];
    for (int j = 0; j < p.Sk; ++j) {
      if (p.causal && koff + j > qa) break;
      float add = 0.f;
      if (!visible<T, MK>(mr, b, h, i, j, add)) continue;
      const T* kr = kb + static_cast<int64_t>(j) * p.kv_ss;
      const T* vr = vb + static_cast<int64_t>(j) * p.kv_ss;
      const float sc = dot_row(qr, kr, D, lane) * p.scale + add;
      const float mnew = fmaxf(m, sc);
      const float alpha = expf(m - mnew);
      const float pv = expf(sc - mnew);
      l = l * alpha + pv;
      const float pz = pv * drop_factor(dp, prow + j);  // dropout acts after the normalisation
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int d = lane + 64 * c;
        if (d < D) acc[c] = acc[c] * alpha + pz * to_f32(vr[d]);
      }
      m = mnew;
    }
  }
  T* orow = o + b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh;
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int d = lane + 64 * c;
    if (d < D) orow[d] = from_f32<T>(acc[c] * inv);
  }
  if (lane == 0)
    lse[(static_cast<int64_t>(b) * p.Hq + h) * p.Sq + i] = l > 0.f ? m + logf(l) : -__builtin_inff();
}

template <typename T, int MK>
__global__ __launch_bounds__(64) void attn_bwd_dq_generic_kernel(
    const T* __restrict__ q, KVBlocks kv, const T* __restrict__ dout,
    const float* __restrict__ lse, const float* __restrict__ delta, T* __restrict__ dq,
    AttnShape p, int D, MaskRef mr, DropoutParams dp) {
  const int lane = threadIdx.x;
  const int i = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int hk = h / (p.Hq / p.Hkv);
  const T* qr = q + b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh;
  const T* dr = dout + b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh;
  const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq + i;
  const uint64_t prow = static_cast<uint64_t>(row) * p.Sk;
  const float ls = lse[row], dl = delta[row];
  const int64_t qa = p.q_offset + i;
  float acc[2] = {0.f, 0.f};
  if (ls != -__builtin_inff()) {
    for (int blk = 0; blk < p.nblk; ++blk) {
      const T* kb = static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh;
      const T* vb = static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh;
      const int64_t koff = kv.koff[blk];
      for (int j = 0; j < p.Sk; ++j) {
        if (p.causal && koff + j > qa) break;
        float add = 0.f;
        if (!visible<T, MK>(mr, b, h, i, j, add)) continue;
        const T* kr = kb + static_cast<int64_t>(j) * p.kv_ss;
        const T* vr = vb + static_cast<int64_t>(j) * p.kv_ss;
        const float pv = expf(dot_row(qr, kr, D, lane) * p.scale + add - ls);
        // dropout: dP = Z (dO . V) with Z = keep / (1 - p); delta = rowsum(dO o O) still
        // equals sum_j P Z (dO . V), so dS = P (dP - delta)
        const float ds = pv * (drop_factor(dp, prow + j) * dot_row(dr, vr, D, lane) - dl);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int d = lane + 64 * c;
          if (d < D) acc[c] += ds * to_f32(kr[d]);
        }
      }
    }
  }
  T* out = dq + b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int d = lane + 64 * c;
    if (d < D) out[d] = from_f32<T>(acc[c] * p.scale);
  }
}

template <typename T, int MK>
__global__ __launch_bounds__(64) void attn_bwd_dkdv_generic_kernel(
    const T* __restrict__ q, KVBlocks kv, const T* __restrict__ dout,
    const float* __restrict__ lse, const float* __restrict__ delta, AttnShape p, int D, MaskRef mr,
    DropoutParams dp) {
  const int lane = threadIdx.x;
  const int j = blockIdx.x, hk = blockIdx.y;
  const int blk = static_cast<int>(blockIdx.z) % p.nblk;
  const int b = static_cast<int>(blockIdx.z) / p.nblk;
  const int group = p.Hq / p.Hkv;
  const int64_t koff = kv.koff[blk];
  const int64_t kvo = b * p.kv_sb + static_cast<int64_t>(j) * p.kv_ss + hk * p.kv_sh;
  const T* kr = static_cast<const T*>(kv.k[blk]) + kvo;
  const T* vr = static_cast<const T*>(kv.v[blk]) + kvo;
  float dk[2] = {0.f, 0.f}, dv[2] = {0.f, 0.f};
  int i0 = 0;
  if (p.causal) {
    const int64_t fq = koff + j - p.q_offset;
    i0 = fq <= 0 ? 0 : (fq >= p.Sq ? p.Sq : static_cast<int>(fq));
  }
  for (int hi = 0; hi < group; ++hi) {
    const int h = hk * group + hi;
    for (int i = i0; i < p.Sq; ++i) {
      const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq + i;
      const float ls = lse[row];
      if (ls == -__builtin_inff()) continue;
      float add = 0.f;
      if (!visible<T, MK>(mr, b, h, i, j, add)) continue;
      const T* qr = q + b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh;
      const T* dr = dout + b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh;
      const float pv = expf(dot_row(qr, kr, D, lane) * p.scale + add - ls);
      const float z = drop_factor(dp, static_cast<uint64_t>(row) * p.Sk + j);
      const float ds = pv * (z * dot_row(dr, vr, D, lane) - delta[row]);
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
  T* dkr = static_cast<T*>(kv.dk[blk]) + kvo;
  T* dvr = static_cast<T*>(kv.dv[blk]) + kvo;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int d = lane + 64 * c;
    if (d < D) {
      dkr[d] = from_f32<T>(dk[c] * p.scale);
      dvr[d] = from_f32<T>(dv[c]);
    }
  }
}

}  // namespace
}  // namespace nmb
