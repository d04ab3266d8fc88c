// Attention on the fp32 matrix core (v_mfma_f32_16x16x4_f32) for any head dim
// <= 128, any strides, fp32 or bf16 storage, up to 8 K/V blocks, an optional
// mask and dropout: the fp32 configuration's attention, and masked attention
// where attention_masked.hip's bf16 kernels do not apply.
//
// Masks (the reference passes attention_mask to SDPA,
// nn/kernels/torch_backend.py:60-76): MK 0 no mask, 1 a boolean mask (one byte
// per entry, nonzero = attend), 2 an additive mask in the attention dtype
// (added to the scaled scores; -inf drops the key).  A query row with no
// visible key gives zeros and lse = -inf, as the safe softmax of the
// reference's SDPA does.  Attention dropout (SDPA's dropout_p, applied to the
// normalised probabilities): probability (b, h, i, j) is multiplied by the
// dropout_math.h factor of index ((b * Hq + h) * Sq + i) * Sk + j; l and the
// lse stay those of the undropped softmax.
//
// A workgroup owns 16 queries (dK/dV: 16 keys) of one head, and its four
// wavefronts take the 16-row tiles of the other side in turn, each with
// accumulators of its own that are merged through LDS in wave order at the
// end: the smoke configuration's 128-token sequences are latency-bound, and
// this gives 128 workgroups of four short chains instead of one wavefront
// walking every key.  S^T = K Q^T puts the scores of one query and four
// consecutive keys (4 g + e) in a lane, which are the B operand of the e-th
// MFMA of the next product as they are.  Operands come straight from global
// memory (each is used by one wave), the next tile's in flight during the
// current one's MFMAs: rows as four consecutive head-dim elements per lane (16
// j + 4 g + e, summed over e in separate accumulators so that the chains stay
// short), columns as one element per row.  Measured at 4 x 4 heads x 128
// tokens, D 64 (fp32): forward 9.8 us, dQ 11.6 us, dK/dV 11.9 us; one
// wavefront per row took 97, 123 (and 18 for delta) and 84 us.
#pragma once

#include "attention_rows.h"

namespace nmb {
namespace {

__device__ __forceinline__ f32x4 mfma_f32x4(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Row operand: elements 16 j + 4 g + e of a row of D (zeros past D, or
// everywhere when !ok, in which case p must still be readable); vec: 16-byte
// loads (fp32, D a multiple of 4).
template <typename T, int DM>
__device__ __forceinline__ void load_row(const T* p, bool ok, int D, int g, bool vec, f32x4 (&v)[DM / 16]) {
#pragma unroll
  for (int j = 0; j < DM / 16; ++j) {
    const int d = 16 * j + 4 * g;
    f32x4 t = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (sizeof(T) == 4) {
      if (vec) {
        if (d < D) t = *reinterpret_cast<const f32x4*>(p + d);
        v[j] = t;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < D) t[e] = p[d + e];
        v[j] = t;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < D) t[e] = to_f32(p[d + e]);
      v[j] = t;
    }
    if (!ok) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// Column operand: element d = 16 dt + l16 of rows r0 + 4 g + e of a matrix of
// n rows (zeros past n and past D).
template <typename T, int DM>
__device__ __forceinline__ void load_cols(const T* base, int64_t stride, int r0, int n, int D, int l16, int g,
                                          float (&v)[4][DM / 16]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = r0 + 4 * g + e;
    const T* p = base + static_cast<int64_t>(min(r, n - 1)) * stride;
#pragma unroll
    for (int dt = 0; dt < DM / 16; ++dt) {
      const int d = 16 * dt + l16;
      const float x = d < D ? to_f32(p[d]) : 0.f;
      v[e][dt] = r < n ? x : 0.f;
    }
  }
}

// 16 x 16 scores: sum over the head dim of a[row] b[col] (a, b row operands)
template <int DM>
__device__ __forceinline__ f32x4 row_product(const f32x4 (&a)[DM / 16], const f32x4 (&b)[DM / 16]) {
  f32x4 s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < DM / 16; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = mfma_f32x4(a[j][e], b[j][e], s[e]);
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (s[0][e] + s[1][e]) + (s[2][e] + s[3][e]);
  return r;
}

// scale * s plus the mask entry at element offset off, or -inf if masked
template <typename T, int MK>
__device__ __forceinline__ float score(float s, float scale, const MaskRef& mr, int64_t off, bool hidden) {
  if constexpr (MK == 0) {
    return hidden ? -__builtin_inff() : s * scale;
  } else if constexpr (MK == 1) {
    return hidden || static_cast<const uint8_t*>(mr.p)[off] == 0 ? -__builtin_inff() : s * scale;
  } else {
    const float add = to_f32(static_cast<const T*>(mr.p)[off]);
    return hidden || add == -__builtin_inff() ? -__builtin_inff() : fmaf(s, scale, add);
  }
}

// A row (of 4 g + e) hidden from all 16 columns may hold anything: its column
// operand becomes zeros, so that the padding of a batch does not bring 0 x NaN
// to the sums (rows hidden from some of the columns may: attention_rows.h).
template <int DM>
__device__ __forceinline__ void drop_hidden(const bool (&hidden)[4], int g, float (&v)[4][DM / 16]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint64_t m = __ballot(hidden[e]);
    if (((m >> (16 * g)) & 0xffff) == 0xffff)
#pragma unroll
      for (int dt = 0; dt < DM / 16; ++dt) v[e][dt] = 0.f;
  }
}

// 16-key tiles of a block that a query up to absolute position q_last can see
__device__ __forceinline__ int visible_tiles16(const AttnShape& p, int64_t koff, int64_t q_last) {
  int n = (p.Sk + 15) >> 4;
  if (p.causal) {
    const int64_t lim = q_last - koff;
    if (lim < 0) return 0;
    const int64_t t = (lim >> 4) + 1;
    if (t < n) n = static_cast<int>(t);
  }
  return n;
}

// acc[dt] (X^T[d = 16 dt + 4 g + e][row l16]) of the four waves, into LDS rows
// [wave][row][d]; a barrier follows.
template <int DM>
struct WaveSums {
  static constexpr int kLd = DM + 4;
  float v[4][16][kLd];
  __device__ __forceinline__ void put(int wave, int l16, int g, const f32x4 (&acc)[DM / 16]) {
#pragma unroll
    for (int dt = 0; dt < DM / 16; ++dt) *reinterpret_cast<f32x4*>(&v[wave][l16][16 * dt + 4 * g]) = acc[dt];
  }
};

template <typename T, int DM, int MK, bool DROP>
__global__ __launch_bounds__(256) void attn_f32_fwd_kernel(const T* __restrict__ q, KVBlocks kv, T* __restrict__ o,
                                                           float* __restrict__ lse, AttnShape p, int D, int vec,
                                                           MaskRef mr, DropoutParams dp) {
  constexpr int DT = DM / 16;
  __shared__ __attribute__((aligned(16))) WaveSums<DM> sums;
  __shared__ float sM[4][16], sL[4][16];
  __shared__ uint32_t sBad;  // rows with a NaN
  if (threadIdx.x == 0) sBad = 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int q0 = 16 * (static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x));  // heavy tiles first
  const int h = blockIdx.y, b = blockIdx.z;
  const int hk = h / (p.Hq / p.Hkv);
  const int qi = q0 + l16, qr = min(qi, p.Sq - 1);
  const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq;
  const int64_t mask_row = b * mr.sb + h * mr.sh + qr * mr.sq;
  f32x4 qf[DT];
  load_row<T, DM>(q + b * p.q_sb + static_cast<int64_t>(qr) * p.q_ss + h * p.q_sh, true, D, g, vec, qf);
  float m = -__builtin_inff(), l = 0.f;
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t q_last = p.q_offset + min(q0 + 15, p.Sq - 1);
  int seen = 0;  // tiles of the blocks before
  for (int blk = 0; blk < p.nblk; ++blk) {
    const T* kb = static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const T* vb = static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const int nt = visible_tiles16(p, kv.koff[blk], q_last);
    f32x4 kf[DT];
    float vf[4][DT];
    auto load = [&](int t) {
      const int key = 16 * t + l16;
      load_row<T, DM>(kb + static_cast<int64_t>(min(key, p.Sk - 1)) * p.kv_ss, key < p.Sk, D, g, vec, kf);
      load_cols<T, DM>(vb, p.kv_ss, 16 * t, p.Sk, D, l16, g, vf);
    };
    int t = (wave - seen) & 3;
    seen += nt;
    if (t < nt) load(t);
    for (; t < nt; t += 4) {
      const int k0 = 16 * t;
      f32x4 kc[DT];
      float vc[4][DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        kc[dt] = kf[dt];
#pragma unroll
        for (int e = 0; e < 4; ++e) vc[e][dt] = vf[e][dt];
      }
      if (t + 4 < nt) load(t + 4);
      const f32x4 s = row_product<DM>(kc, qf);
      const int lim = mask_limit(p, kv.koff[blk], k0, p.q_offset + qi);
      float x[4], tmax = -__builtin_inff();
      bool hidden[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * g + e;
        x[e] = score<T, MK>(s[e], p.scale, mr, mask_row + min(k0 + j, p.Sk - 1) * mr.sk, j > lim);
        hidden[e] = x[e] == -__builtin_inff();
        tmax = fmaxf(tmax, x[e]);
      }
      if constexpr (MK != 0) drop_hidden<DM>(hidden, g, vc);
      tmax = xor32_max(xor16_max(tmax));
      if (__any(tmax > m)) {
        const float mn = fmaxf(m, tmax);
        const float alpha = m == -__builtin_inff() ? 0.f : expf(m - mn);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
      }
      const float mc = m == -__builtin_inff() ? 0.f : m;
      bool keep[4] = {true, true, true, true};
      if constexpr (DROP)
        keep4(dp, static_cast<uint64_t>(row + qr) * p.Sk + k0 + 4 * g, (p.Sk & 1) == 0, keep);
      float pv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pv[e] = expf(x[e] - mc);
        l += pv[e];
        if constexpr (DROP) pv[e] = keep[e] ? pv[e] * dp.scale : 0.f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = mfma_f32x4(vc[e][dt], pv[e], acc[dt]);
    }
  }
  l = xor32_sum(xor16_sum(l));
  sums.put(wave, l16, g, acc);
  if (g == 0) {
    sM[wave][l16] = m;
    sL[wave][l16] = l;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * DM; i += 256) {
    const int r = i / DM, d = i % DM;
    if (q0 + r >= p.Sq) continue;
    const float mx = fmaxf(fmaxf(sM[0][r], sM[1][r]), fmaxf(sM[2][r], sM[3][r]));
    float lt = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = sM[w][r] == -__builtin_inff() ? 0.f : expf(sM[w][r] - mx);
      lt += f * sL[w][r];
      v += f * sums.v[w][r][d];
    }
    if (v != v) atomicOr(&sBad, 1u << r);
    if (d < D)
      o[b * p.o_sb + static_cast<int64_t>(q0 + r) * p.o_ss + h * p.o_sh + d] =
          from_f32<T>(v * (lt > 0.f ? 1.f / lt : 0.f));
    if (d == 0) lse[row + q0 + r] = lt > 0.f ? mx + logf(lt) : -__builtin_inff();
  }
  __syncthreads();
  for (uint32_t bad = sBad; bad != 0; bad &= bad - 1) {  // NaN: see attention_rows.h
    const int i = q0 + __ffs(bad) - 1;
    if ((i & 3) != wave) continue;
    const RowMask rm = row_mask(p, mr, dp, b, h);
    float rmax = -__builtin_inff(), rl = 0.f, ra[2] = {0.f, 0.f};
    for (int blk = 0; blk < p.nblk; ++blk)
      row_fwd<T, MK, DROP>(q + b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh,
                           static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh,
                           static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh, kv.koff[blk], i, p, D, rm,
                           lane, rmax, rl, ra);
    row_store(o + b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh, ra, rl > 0.f ? 1.f / rl : 0.f, D, lane);
    if (lane == 0) lse[row + i] = rl > 0.f ? rmax + logf(rl) : -__builtin_inff();
  }
}

// dQ, and delta = rowsum(dO o O) for the dK/dV kernel (which equals
// sum_j P Z (dO . V) under dropout factors Z, so dS = P (Z dO . V - delta)).
// MK 2: the probabilities are normalised by their sum over the row, whose
// inverse goes to norm (if given) for the dK/dV kernel: beside a mask of the
// type's lowest value, lse = m + log(l) has no room for log(l), and exp(x -
// lse) of a row masked throughout by it is 1 for every key.
template <typename T, int DM, int MK, bool DROP>
__global__ __launch_bounds__(256) void attn_f32_dq_kernel(const T* __restrict__ q, KVBlocks kv,
                                                          const T* __restrict__ o, const T* __restrict__ dout,
                                                          const float* __restrict__ lse, float* __restrict__ delta,
                                                          float* __restrict__ norm, T* __restrict__ dq,
                                                          AttnShape p, int D, int vec, MaskRef mr,
                                                          DropoutParams dp) {
  constexpr int DT = DM / 16;
  __shared__ __attribute__((aligned(16))) WaveSums<DM> sums;
  __shared__ uint32_t sBad;  // rows with a NaN
  __shared__ float sN[4][16];
  if (threadIdx.x == 0) sBad = 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int q0 = 16 * (static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x));
  const int h = blockIdx.y, b = blockIdx.z;
  const int hk = h / (p.Hq / p.Hkv);
  const int qi = q0 + l16, qr = min(qi, p.Sq - 1);
  const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq;
  const int64_t mask_row = b * mr.sb + h * mr.sh + qr * mr.sq;
  const int64_t o_row = b * p.o_sb + static_cast<int64_t>(qr) * p.o_ss + h * p.o_sh;
  f32x4 qf[DT], df[DT];
  load_row<T, DM>(q + b * p.q_sb + static_cast<int64_t>(qr) * p.q_ss + h * p.q_sh, true, D, g, vec, qf);
  load_row<T, DM>(dout + o_row, true, D, g, vec, df);
  float dl = 0.f;
  {
    f32x4 of[DT];
    load_row<T, DM>(o + o_row, true, D, g, vec, of);
#pragma unroll
    for (int j = 0; j < DT; ++j)
      dl += (of[j][0] * df[j][0] + of[j][1] * df[j][1]) + (of[j][2] * df[j][2] + of[j][3] * df[j][3]);
  }
  dl = xor32_sum(xor16_sum(dl));
  if (wave == 0 && g == 0 && qi < p.Sq) delta[row + qi] = dl;
  const float ls = lse[row + qr];
  float psum = 0.f;
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t q_last = p.q_offset + min(q0 + 15, p.Sq - 1);
  int seen = 0;
  for (int blk = 0; blk < p.nblk; ++blk) {
    const T* kb = static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const T* vb = static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh;
    const int nt = visible_tiles16(p, kv.koff[blk], q_last);
    f32x4 kf[DT], vf[DT];
    float kcol[4][DT];
    auto load = [&](int t) {
      const int key = 16 * t + l16;
      const int64_t off = static_cast<int64_t>(min(key, p.Sk - 1)) * p.kv_ss;
      load_row<T, DM>(kb + off, key < p.Sk, D, g, vec, kf);
      load_row<T, DM>(vb + off, key < p.Sk, D, g, vec, vf);
      load_cols<T, DM>(kb, p.kv_ss, 16 * t, p.Sk, D, l16, g, kcol);
    };
    int t = (wave - seen) & 3;
    seen += nt;
    if (t < nt) load(t);
    for (; t < nt; t += 4) {
      const int k0 = 16 * t;
      const f32x4 s = row_product<DM>(kf, qf);
      const f32x4 dv = row_product<DM>(vf, df);
      float kc[4][DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 4; ++e) kc[e][dt] = kcol[e][dt];
      if (t + 4 < nt) load(t + 4);
      const int lim = mask_limit(p, kv.koff[blk], k0, p.q_offset + qi);
      bool keep[4] = {true, true, true, true}, hidden[4];
      if constexpr (DROP)
        keep4(dp, static_cast<uint64_t>(row + qr) * p.Sk + k0 + 4 * g, (p.Sk & 1) == 0, keep);
      float ds[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * g + e;
        const float x = score<T, MK>(s[e], p.scale, mr, mask_row + min(k0 + j, p.Sk - 1) * mr.sk, j > lim);
        hidden[e] = x == -__builtin_inff() || ls == -__builtin_inff();
        float dz = dv[e];
        if constexpr (DROP) dz = keep[e] ? dz * dp.scale : 0.f;
        const float pv = hidden[e] ? 0.f : expf(x - ls);
        if constexpr (MK == 2) psum += pv;
        ds[e] = hidden[e] ? 0.f : pv * (dz - dl);
      }
      if constexpr (MK != 0) drop_hidden<DM>(hidden, g, kc);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = mfma_f32x4(kc[e][dt], ds[e], acc[dt]);
    }
  }
  sums.put(wave, l16, g, acc);
  if constexpr (MK == 2) {
    psum = xor32_sum(xor16_sum(psum));
    if (g == 0) sN[wave][l16] = psum;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * DM; i += 256) {
    const int r = i / DM, d = i % DM;
    if (q0 + r >= p.Sq || d >= D) continue;
    float v = (sums.v[0][r][d] + sums.v[1][r][d]) + (sums.v[2][r][d] + sums.v[3][r][d]);
    if constexpr (MK == 2) {
      const float inv = inverse_sum((sN[0][r] + sN[1][r]) + (sN[2][r] + sN[3][r]));
      if (d == 0 && norm != nullptr) norm[row + q0 + r] = inv;
      v *= inv;
    }
    if (v != v) atomicOr(&sBad, 1u << r);
    dq[b * p.q_sb + static_cast<int64_t>(q0 + r) * p.q_ss + h * p.q_sh + d] = from_f32<T>(v * p.scale);
  }
  __syncthreads();
  for (uint32_t bad = sBad; bad != 0; bad &= bad - 1) {  // NaN: see attention_rows.h
    const int r = __ffs(bad) - 1, i = q0 + r;
    if ((i & 3) != wave) continue;
    const RowMask rm = row_mask(p, mr, dp, b, h);
    const int64_t q_off = b * p.q_sb + static_cast<int64_t>(i) * p.q_ss + h * p.q_sh;
    const float row_delta = __shfl(dl, r, 64);
    float ra[2] = {0.f, 0.f}, rsum = 0.f;
    for (int blk = 0; blk < p.nblk; ++blk)
      row_dq<T, MK, DROP>(q + q_off, dout + b * p.o_sb + static_cast<int64_t>(i) * p.o_ss + h * p.o_sh,
                          static_cast<const T*>(kv.k[blk]) + b * p.kv_sb + hk * p.kv_sh,
                          static_cast<const T*>(kv.v[blk]) + b * p.kv_sb + hk * p.kv_sh, kv.koff[blk], i,
                          lse[row + i], row_delta, p, D, rm, lane, ra, rsum);
    const float inv = MK == 2 ? inverse_sum(rsum) : 1.f;
    if (MK == 2 && lane == 0 && norm != nullptr) norm[row + i] = inv;
    row_store(dq + q_off, ra, p.scale * inv, D, lane);
  }
}

// dK, dV of 16 keys; the waves take the (query head, 16-query tile) pairs in
// turn.
template <typename T, int DM, int MK, bool DROP>
__global__ __launch_bounds__(256) void attn_f32_dkdv_kernel(const T* __restrict__ q, KVBlocks kv,
                                                            const T* __restrict__ dout,
                                                            const float* __restrict__ lse,
                                                            const float* __restrict__ delta,
                                                            const float* __restrict__ norm, AttnShape p, int D,
                                                            int vec, MaskRef mr, DropoutParams dp) {
  constexpr int DT = DM / 16;
  __shared__ __attribute__((aligned(16))) WaveSums<DM> sums;
  __shared__ uint32_t sBad;  // keys with a NaN
  if (threadIdx.x == 0) sBad = 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int j0 = 16 * static_cast<int>(blockIdx.x), hk = blockIdx.y;
  const int blk = static_cast<int>(blockIdx.z) % p.nblk;
  const int b = static_cast<int>(blockIdx.z) / p.nblk;
  const int group = p.Hq / p.Hkv;
  const int64_t koff = kv.koff[blk];
  const int64_t kv_off = b * p.kv_sb + hk * p.kv_sh;
  const int key = j0 + l16, kc = min(key, p.Sk - 1);
  const int64_t kr = kv_off + static_cast<int64_t>(kc) * p.kv_ss;
  f32x4 kf[DT], vf[DT];
  load_row<T, DM>(static_cast<const T*>(kv.k[blk]) + kr, true, D, g, vec, kf);
  load_row<T, DM>(static_cast<const T*>(kv.v[blk]) + kr, true, D, g, vec, vf);
  f32x4 dka[DT], dva[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dka[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    dva[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int n_qt = (p.Sq + 15) / 16;
  int qt0 = 0;
  if (p.causal) {
    const int64_t fq = koff + j0 - p.q_offset;
    qt0 = fq <= 0 ? 0 : (fq >= p.Sq ? n_qt : static_cast<int>(fq) / 16);
  }
  const int per_head = n_qt - qt0;
  f32x4 qf[DT], df[DT];
  float qcol[4][DT], dcol[4][DT];
  float ls[4], dl[4], nm[4];
  int h = hk * group, i0 = 0;  // of the tile loaded last
  auto load = [&](int t) {
    h = hk * group + t / per_head;
    i0 = 16 * (qt0 + t % per_head);
    const int qi = i0 + l16;
    const T* qb = q + b * p.q_sb + h * p.q_sh;
    const T* db = dout + b * p.o_sb + h * p.o_sh;
    load_row<T, DM>(qb + static_cast<int64_t>(min(qi, p.Sq - 1)) * p.q_ss, qi < p.Sq, D, g, vec, qf);
    load_row<T, DM>(db + static_cast<int64_t>(min(qi, p.Sq - 1)) * p.o_ss, qi < p.Sq, D, g, vec, df);
    load_cols<T, DM>(qb, p.q_ss, i0, p.Sq, D, l16, g, qcol);
    load_cols<T, DM>(db, p.o_ss, i0, p.Sq, D, l16, g, dcol);
    const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = min(i0 + 4 * g + e, p.Sq - 1);
      ls[e] = lse[row + r];
      dl[e] = delta[row + r];
      nm[e] = MK == 2 && norm != nullptr ? norm[row + r] : 1.f;
    }
  };
  const int total = group * per_head;
  int t = wave;
  if (t < total) load(t);
  for (; t < total; t += 4) {
    const int ch = h, ci = i0;
    const f32x4 s = row_product<DM>(qf, kf);
    const f32x4 dpv = row_product<DM>(df, vf);
    float qc[4][DT], dc[4][DT], lc[4], dlc[4], nmc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lc[e] = ls[e];
      nmc[e] = nm[e];
      dlc[e] = dl[e];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        qc[e][dt] = qcol[e][dt];
        dc[e][dt] = dcol[e][dt];
      }
    }
    if (t + 4 < total) load(t + 4);
    const int64_t row = (static_cast<int64_t>(b) * p.Hq + ch) * p.Sq;
    const int64_t mask_col = b * mr.sb + ch * mr.sh + kc * mr.sk;
    float pv[4], ds[4];
    bool hidden[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = ci + 4 * g + e, ic = min(i, p.Sq - 1);
      const bool off = i >= p.Sq || (p.causal && koff + key > p.q_offset + i) || lc[e] == -__builtin_inff();
      const float x = score<T, MK>(s[e], p.scale, mr, mask_col + ic * mr.sq, off);
      hidden[e] = x == -__builtin_inff();
      float pr = hidden[e] ? 0.f : expf(x - lc[e]);
      if constexpr (MK == 2) pr *= nmc[e];
      float z = 1.f;
      if constexpr (DROP) z = drop_factor(dp, static_cast<uint64_t>(row + ic) * p.Sk + key);
      pv[e] = pr * z;
      ds[e] = hidden[e] ? 0.f : pr * (z * dpv[e] - dlc[e]);
    }
    if constexpr (MK != 0) {
      drop_hidden<DM>(hidden, g, qc);
      drop_hidden<DM>(hidden, g, dc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        dva[dt] = mfma_f32x4(dc[e][dt], pv[e], dva[dt]);
        dka[dt] = mfma_f32x4(qc[e][dt], ds[e], dka[dt]);
      }
  }
  // dK, then dV through the same LDS rows
  T* outs[2] = {static_cast<T*>(kv.dk[blk]) + kv_off, static_cast<T*>(kv.dv[blk]) + kv_off};
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    sums.put(wave, l16, g, w == 0 ? dka : dva);
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * DM; i += 256) {
      const int r = i / DM, d = i % DM;
      if (j0 + r >= p.Sk || d >= D) continue;
      const float v = (sums.v[0][r][d] + sums.v[1][r][d]) + (sums.v[2][r][d] + sums.v[3][r][d]);
      if (v != v) atomicOr(&sBad, 1u << r);
      outs[w][static_cast<int64_t>(j0 + r) * p.kv_ss + d] = from_f32<T>(w == 0 ? v * p.scale : v);
    }
    __syncthreads();
  }
  for (uint32_t bad = sBad; bad != 0; bad &= bad - 1) {  // NaN: see attention_rows.h
    const int j = j0 + __ffs(bad) - 1;
    if ((j & 3) != wave) continue;
    const int64_t off = static_cast<int64_t>(j) * p.kv_ss;
    float rk[2] = {0.f, 0.f}, rv[2] = {0.f, 0.f};
    for (int h = hk * group; h < (hk + 1) * group; ++h) {
      const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq;
      row_dkdv<T, MK, DROP>(static_cast<const T*>(kv.k[blk]) + kv_off + off,
                            static_cast<const T*>(kv.v[blk]) + kv_off + off, q + b * p.q_sb + h * p.q_sh,
                            dout + b * p.o_sb + h * p.o_sh, lse + row, delta + row,
                            norm != nullptr ? norm + row : nullptr, koff, j, p, D, row_mask(p, mr, dp, b, h), lane, rk,
                            rv);
    }
    row_store(outs[0] + off, rk, p.scale, D, lane);
    row_store(outs[1] + off, rv, 1.f, D, lane);
  }
}

// ---------------------------------------------------------------- launches
// 16-byte row loads: fp32 rows of a multiple of 4 elements, all 16-byte aligned
template <typename T>
bool rows_vec4(const AttnShape& p, const KVBlocks& kv, int D, const void* q, const void* o, const void* dout) {
  if (sizeof(T) != 4 || D % 4 != 0) return false;
  const int64_t strides[] = {p.q_sb, p.q_ss, p.q_sh, p.kv_sb, p.kv_ss, p.kv_sh, p.o_sb, p.o_ss, p.o_sh};
  for (int64_t s : strides)
    if (s % 4 != 0) return false;
  if (!aligned16(q) || !aligned16(o) || !aligned16(dout)) return false;
  for (int i = 0; i < p.nblk; ++i)
    if (!aligned16(kv.k[i]) || !aligned16(kv.v[i])) return false;
  return true;
}

// launch(DM, MK, DROP) as compile-time values
template <class F>
void f32_select(int D, int mk, bool drop, F&& launch) {
  auto by_mask = [&](auto dm) {
    auto by_drop = [&](auto m) {
      if (drop) launch(dm, m, std::true_type{});
      else launch(dm, m, std::false_type{});
    };
    if (mk == 0) by_drop(std::integral_constant<int, 0>{});
    else if (mk == 1) by_drop(std::integral_constant<int, 1>{});
    else by_drop(std::integral_constant<int, 2>{});
  };
  if (D <= 64) by_mask(std::integral_constant<int, 64>{});
  else by_mask(std::integral_constant<int, 128>{});
}

template <typename T>
void f32_fwd_launch(const AttnShape& p, const KVBlocks& kv, const MaskRef& mr, const DropoutParams& dp, int kind,
                    bool drop, const void* q, void* o, float* lse, int D, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((p.Sq + 15) / 16), static_cast<unsigned>(p.Hq), static_cast<unsigned>(p.B));
  const int vec = rows_vec4<T>(p, kv, D, q, nullptr, nullptr);
  f32_select(D, kind, drop, [&](auto dm, auto mk, auto dr) {
    hipLaunchKernelGGL((attn_f32_fwd_kernel<T, dm.value, mk.value, dr.value>), grid, dim3(256), 0, stream,
                       static_cast<const T*>(q), kv, static_cast<T*>(o), lse, p, D, vec, mr, dp);
  });
}

template <typename T>
void f32_bwd_launch(const AttnShape& p, const KVBlocks& kv, const MaskRef& mr, const DropoutParams& dp, int kind,
                    bool drop, const void* q, const void* o, const void* dout, const float* lse, float* delta,
                    float* norm, void* dq, int D, hipStream_t stream) {
  const int vec = rows_vec4<T>(p, kv, D, q, o, dout);
  if (p.Sq > 0) {
    const dim3 grid(static_cast<unsigned>((p.Sq + 15) / 16), static_cast<unsigned>(p.Hq),
                    static_cast<unsigned>(p.B));
    f32_select(D, kind, drop, [&](auto dm, auto mk, auto dr) {
      hipLaunchKernelGGL((attn_f32_dq_kernel<T, dm.value, mk.value, dr.value>), grid, dim3(256), 0, stream,
                         static_cast<const T*>(q), kv, static_cast<const T*>(o), static_cast<const T*>(dout), lse,
                         delta, norm, static_cast<T*>(dq), p, D, vec, mr, dp);
    });
  }
  if (p.Sk > 0) {
    const dim3 grid(static_cast<unsigned>((p.Sk + 15) / 16), static_cast<unsigned>(p.Hkv),
                    static_cast<unsigned>(p.B * p.nblk));
    f32_select(D, kind, drop, [&](auto dm, auto mk, auto dr) {
      hipLaunchKernelGGL((attn_f32_dkdv_kernel<T, dm.value, mk.value, dr.value>), grid, dim3(256), 0, stream,
                         static_cast<const T*>(q), kv, static_cast<const T*>(dout), lse, delta, norm, p, D, vec, mr, dp);
    });
  }
}

}  // namespace
}  // namespace nmb
