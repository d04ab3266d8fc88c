// Attention with an explicit mask and / or attention dropout for gfx950:
// the reference passes attention_mask and dropout_p to SDPA
// (nn/kernels/torch_backend.py:60-76).  Semantics as attention_f32.h: a
// query row with no visible key gives zeros and lse = -inf, dropout multiplies
// the normalised probabilities by the dropout_math.h factor of element
// ((b Hq + h) Sq + i) Sk + j, and l and the lse stay those of the undropped
// softmax.
//
// bf16 at head_dim 64 and 128 runs on v_mfma_f32_16x16x32_bf16 with the tile
// layouts of the unmasked kernels (attention.hip): S^T = K Q^T per wave of 16
// queries (forward, dQ) or S = Q K^T per wave of 16 keys (dK/dV), 64 rows of
// the other side per step, streamed into LDS by direct loads.  Everything the
// one-row-per-wavefront kernels held in fp32 stays so: the scores, the row sum
// and the probabilities; a probability (and a dS) enters its product as the
// sum of three bf16 values that hold its fp32 bits, so those products run
// three times.  What bounds them: at B 8, Hq 16, S 512, D 64 (one pass, forward
// and backward, 15 GFLOP counted once, 67 MB) the exponentials, mask selects
// and splits on the VALU and the latency of each 64-row step, not the matrix
// cores; 64 queries (keys) per workgroup give 1,024 workgroups there and three
// per CU.  Measured there with a padding mask: forward 35 us, dQ 39 us, dK/dV
// 54 us (one wavefront per row: 1,939, 2,279 and 2,506 us); with dropout 0.1 at
// Hq 12 36, 40 and 63 us (1,823, 2,124 and 2,423 us).  With two bf16 terms (up
// to 2^-17 of a probability left out) they took 31, 35 and 46 us, and the
// errors of O and dV against 64 bits grew by 5e-7 and 1e-6 of themselves (the
// outputs' own rounding is 1.7e-3); with three they are within 1e-8 of the
// fp32 kernels' over 30 shapes.
//
// Boolean masks that are the same for every query (a padding mask) are read
// once per workgroup into one bit per key in LDS: key tiles without a visible
// key are skipped, and masked keys' rows are loaded as zeros.  Other masks are
// read from global memory per score, four at a time where their layout
// allows.  A row whose result is NaN, as hidden keys that hold NaN or infinity
// make it, is run again by attention_rows.h.
#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "attention_common.h"
#include "attention_f32.h"

namespace nmb {
namespace {

// mask kinds of the kernels below
constexpr int kNoMask = 0, kKeyMask = 1, kBoolMask = 2, kAddMask = 3;
constexpr int kMaxMaskKeys = 16384;  // keys of a kKeyMask: 2 KB of bits in LDS

// mask reads: four consecutive ones (along keys) as one load
struct MaskRead {
  MaskRef r;
  int vec4;
};

// p as three bf16 terms, to its fp32 bits (each rounding leaves a rest of fewer
// bits, the last at most 2^-25 |p|)
constexpr int kTerms = 3;
__device__ __forceinline__ void split(float p, bf16x8 (&t)[kTerms], int i) {
#pragma unroll
  for (int k = 0; k < kTerms; ++k) {
    t[k][i] = static_cast<bf16>(p);
    p -= static_cast<float>(t[k][i]);
  }
}

// Bit key % 64 of word key / 64: key is visible in the boolean mask row at
// mask (stride sk).  256 threads; ends with a barrier.
__device__ __forceinline__ void load_key_bits(uint64_t* bits, const uint8_t* mask, int64_t sk, int n_keys) {
  const int lane = threadIdx.x & 63;
  for (int k0 = 0; k0 < n_keys; k0 += 256) {
    const int key = k0 + static_cast<int>(threadIdx.x);
    const bool on = key < n_keys && mask[key * sk] != 0;
    const uint64_t w = __ballot(on);
    if (lane == 0) bits[key >> 6] = w;
  }
  __syncthreads();
}

// The mask values of 16 scores of one query (keys k0 + 16 mk + 4 g + e):
// visible, and for additive masks the value.  Keys at and past Sk read a
// valid entry (the caller masks them).
template <int MK>
struct QueryMask {
  float add[4][4];  // kAddMask
  uint32_t on[4];   // kBoolMask: bit e

  __device__ __forceinline__ void load(const MaskRead& m, int64_t row, int k0, int g, int Sk) {
#pragma unroll
    for (int mk = 0; mk < 4; ++mk) {
      const int key = k0 + 16 * mk + 4 * g;
      if constexpr (MK == kBoolMask) {
        const uint8_t* p = static_cast<const uint8_t*>(m.r.p) + row;
        on[mk] = 0;
        if (m.vec4) {
          const uint32_t w = *reinterpret_cast<const uint32_t*>(p + min(key, Sk - 4));
#pragma unroll
          for (int e = 0; e < 4; ++e) on[mk] |= ((w >> (8 * e)) & 0xff) != 0 ? 1u << e : 0u;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) on[mk] |= p[min(key + e, Sk - 1) * m.r.sk] != 0 ? 1u << e : 0u;
        }
      } else if constexpr (MK == kAddMask) {
        const bf16* p = static_cast<const bf16*>(m.r.p) + row;
        if (m.vec4) {
          const bf16x4 w = *reinterpret_cast<const bf16x4*>(p + min(key, Sk - 4));
#pragma unroll
          for (int e = 0; e < 4; ++e) add[mk][e] = static_cast<float>(w[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) add[mk][e] = static_cast<float>(p[min(key + e, Sk - 1) * m.r.sk]);
        }
      }
    }
  }
};

// scale * s (+ the additive mask), or -inf where the score is masked.  The
// mask is added in the natural domain: a mask of the type's lowest value must
// stay finite, so that a row masked throughout by it averages over all keys.
template <int MK>
__device__ __forceinline__ float masked_score(float s, float scale, const QueryMask<MK>& qm, uint64_t key_bits,
                                              int mk, int e, int idx, int lim) {
  float x;
  bool off = idx > lim;
  if constexpr (MK == kAddMask) {
    x = fmaf(s, scale, qm.add[mk][e]);
    off = off || qm.add[mk][e] == -__builtin_inff();
  } else {
    x = s * scale;
    if constexpr (MK == kBoolMask) off = off || !((qm.on[mk] >> e) & 1);
    if constexpr (MK == kKeyMask) off = off || !((key_bits >> (16 * mk + e)) & 1);
  }
  return off ? -__builtin_inff() : x;
}

// The K/V tiles (64 keys) a workgroup's queries see, in order: those below
// `end` with a visible key.
template <int MK>
struct KeyTiles {
  const uint64_t* bits;
  int end;
  __device__ __forceinline__ int from(int kt) const {
    if constexpr (MK == kKeyMask)
      while (kt < end && __builtin_amdgcn_readfirstlane(static_cast<int>(bits[kt] != 0)) == 0) ++kt;
    return kt;
  }
};

// K and V tiles kt of one (batch, KV head) into an LDS stage; rows past Sk
// and masked keys' rows read as zeros.  The descriptor starts at the tile, so
// the offsets stay below 64 rows.
template <int D, int MK>
__device__ __forceinline__ void issue_kv(const TileStream<D, 4>& ld, const bf16* kb, const bf16* vb, bf16* dk,
                                         bf16* dv, const AttnShape& p, int kt, const uint64_t* bits, int wave) {
  using TS = TileStream<D, 4>;
  const int r0 = kt * 64, rows = min(64, p.Sk - r0);
  const uint32_t bytes = static_cast<uint32_t>(((rows - 1) * p.kv_ss + D) * 2);
  const i32x4 rk = make_rsrc(kb + static_cast<int64_t>(r0) * p.kv_ss, bytes);
  const i32x4 rv = make_rsrc(vb + static_cast<int64_t>(r0) * p.kv_ss, bytes);
  uint64_t w = ~0ull;
  if constexpr (MK == kKeyMask) w = bits[kt];
  uint32_t off[TS::P];
#pragma unroll
  for (int j = 0; j < TS::P; ++j)
    off[j] = ld.row[j] < rows && ((w >> ld.row[j]) & 1) ? ld.off[j] : kOOB;
#pragma unroll
  for (int j = 0; j < TS::P; ++j) load_lds16(rk, dk + 512 * (wave * TS::P + j), off[j]);
#pragma unroll
  for (int j = 0; j < TS::P; ++j) load_lds16(rv, dv + 512 * (wave * TS::P + j), off[j]);
}

// zeros into the stage (keeps the number of loads per step constant)
template <int D>
__device__ __forceinline__ void issue_none(const void* any, bf16* a, bf16* b, int wave) {
  using TS = TileStream<D, 4>;
  const i32x4 rz = make_rsrc(any, 0);
#pragma unroll
  for (int j = 0; j < TS::P; ++j) load_lds16(rz, a + 512 * (wave * TS::P + j), kOOB);
#pragma unroll
  for (int j = 0; j < TS::P; ++j) load_lds16(rz, b + 512 * (wave * TS::P + j), kOOB);
}

// attention_rows.h's kind of a mask kind
template <int MK>
constexpr int row_kind = MK == kNoMask ? 0 : (MK == kAddMask ? 2 : 1);

// The wave's rows l16 with a NaN among their accumulators (lanes with `in`),
// which attention_rows.h runs again.
template <int DT>
__device__ __forceinline__ uint32_t nan_rows(const f32x4 (&acc)[DT], bool in) {
  bool nan = false;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 4; ++e) nan = nan || acc[dt][e] != acc[dt][e];
  return rows_of(__ballot(nan && in));
}

// three stages (48 KB, three workgroups per CU) at D 64, two (64 KB, two per
// CU) at D 128
template <int D>
constexpr int masked_stages() { return D == 64 ? 3 : 2; }

// ---------------------------------------------------------------- forward
template <int D, int MK, bool DROP>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_masked_fwd_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v, bf16* __restrict__ o,
    float* __restrict__ lse, AttnShape p, MaskRead mr, DropoutParams dp, int n_qt, int items, int per_xcd) {
  constexpr int BQ = 64, KS = D / 32, DT = D / 16, S = masked_stages<D>();
  using Tile = Tile64<D>;
  constexpr int kLoads = 2 * TileStream<D, 4>::P;
  __shared__ __attribute__((aligned(1024))) bf16 sK[S][Tile::kElems];
  __shared__ __attribute__((aligned(1024))) bf16 sV[S][Tile::kElems];
  __shared__ uint64_t sBits[MK == kKeyMask ? kMaxMaskKeys / 64 : 1];

  const int w = xcd_item(items, per_xcd);
  if (w < 0) return;
  const int bh = w / n_qt;
  const int qt = n_qt - 1 - (w % n_qt);  // heavy causal tiles first within a head
  const int b = bh / p.Hq, h = bh % p.Hq;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l16 = lane & 15, g = lane >> 4;
  const int hk = h / (p.Hq / p.Hkv);
  const int qi = qt * BQ + 16 * wave + l16;
  const int qr = min(qi, p.Sq - 1);
  const int64_t mask_row = b * mr.r.sb + h * mr.r.sh + qr * mr.r.sq;
  const uint64_t prow = (static_cast<uint64_t>(bh) * p.Sq + qr) * p.Sk;
  if constexpr (MK == kKeyMask)
    load_key_bits(sBits, static_cast<const uint8_t*>(mr.r.p) + b * mr.r.sb + h * mr.r.sh, mr.r.sk, p.Sk);

  const bf16* qb = q + b * p.q_sb + h * p.q_sh + static_cast<int64_t>(qr) * p.q_ss;
  const bf16* kb = k + b * p.kv_sb + hk * p.kv_sh;
  const bf16* vb = v + b * p.kv_sb + hk * p.kv_sh;
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = ld8(qb + ks * 32 + g * 8);
  wait_vmcnt<0>();
  TileStream<D, 4> ld;
  ld.init(p.kv_ss, wave, lane);
  KeyTiles<MK> tiles{sBits, visible_key_tiles(p, 0, p.q_offset + min(qt * BQ + BQ - 1, p.Sq - 1))};
  int kt = tiles.from(0), lt = kt;
  auto issue = [&](int st) {
    if (lt < tiles.end) {
      issue_kv<D, MK>(ld, kb, vb, sK[st], sV[st], p, lt, sBits, wave);
      lt = tiles.from(lt + 1);
    } else {
      issue_none<D>(k, sK[st], sV[st], wave);
    }
  };
#pragma unroll
  for (int st = 0; st < S - 1; ++st) issue(st);

  float m = -__builtin_inff(), l = 0.f;  // l: this lane's 16 keys of every tile
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; kt < tiles.end; ++it) {
    wait_vmcnt<(S - 2) * kLoads>();
    lds_barrier();
    const int k0 = kt * 64;
    QueryMask<MK> qm;
    qm.load(mr, mask_row, k0, g, p.Sk);
    issue((it + S - 1) % S);
    const bf16* tk = sK[it % S];
    const bf16* tv = sV[it % S];
    uint64_t bits = 0;
    if constexpr (MK == kKeyMask) bits = sBits[kt] >> (4 * g);
    kt = tiles.from(kt + 1);

    f32x4 s[4];
#pragma unroll
    for (int mk = 0; mk < 4; ++mk) s[mk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mk = 0; mk < 4; ++mk)
        s[mk] = mfma16(Tile::row8(tk, mk * 16 + l16, ks * 32 + g * 8), qf[ks], s[mk]);
    const int lim = mask_limit(p, 0, k0, p.q_offset + qi);
    float tmax = -__builtin_inff();
#pragma unroll
    for (int mk = 0; mk < 4; ++mk)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[mk][e] = masked_score<MK>(s[mk][e], p.scale, qm, bits, mk, e, mk * 16 + g * 4 + e, lim);
        tmax = fmaxf(tmax, s[mk][e]);
      }
    tmax = xor32_max(xor16_max(tmax));
    if (__any(tmax > m)) {  // wave-uniform
      const float mn = fmaxf(m, tmax);
      const float alpha = m == -__builtin_inff() ? 0.f : fast_exp2((m - mn) * kLog2e);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
    }
    const float mc = m == -__builtin_inff() ? 0.f : m;  // no visible key yet: P = 0
    bf16x8 pt[2][kTerms];
#pragma unroll
    for (int mk = 0; mk < 4; ++mk) {
      bool keep[4] = {true, true, true, true};
      if constexpr (DROP) keep4(dp, prow + k0 + 16 * mk + 4 * g, (p.Sk & 1) == 0, keep);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float pv = fast_exp2((s[mk][e] - mc) * kLog2e);
        l += pv;
        if constexpr (DROP) pv = keep[e] ? pv : 0.f;  // the factor 1 / (1 - p) at the end
        split(pv, pt[mk >> 1], 4 * (mk & 1) + e);
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const bf16x8 vv = Tile::col8(tv, 32 * s2, dt * 16, l16, g);
#pragma unroll
        for (int t = kTerms - 1; t >= 0; --t) acc[dt] = mfma16(vv, pt[s2][t], acc[dt]);
      }
  }
  wait_vmcnt<0>();  // no load may still write this workgroup's LDS when it ends
  l = xor32_sum(xor16_sum(l));
  uint32_t bad = nan_rows<DT>(acc, qi < p.Sq);
  if (qi < p.Sq && !(bad >> l16 & 1)) {
    const float inv = (l > 0.f ? 1.f / l : 0.f) * (DROP ? dp.scale : 1.f);
    bf16* orow = o + b * p.o_sb + h * p.o_sh + static_cast<int64_t>(qi) * p.o_ss;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      bf16x4 wv;
#pragma unroll
      for (int e = 0; e < 4; ++e) wv[e] = static_cast<bf16>(acc[dt][e] * inv);
      *reinterpret_cast<bf16x4*>(orow + dt * 16 + g * 4) = wv;
    }
    if (g == 0) lse[static_cast<int64_t>(bh) * p.Sq + qi] = l > 0.f ? m + logf(l) : -__builtin_inff();
  }
  for (; bad != 0; bad &= bad - 1) {
    const int i = qt * BQ + 16 * wave + __ffs(bad) - 1;
    float rmax = -__builtin_inff(), rl = 0.f, ra[2] = {0.f, 0.f};
    row_fwd<bf16, row_kind<MK>, DROP>(q + b * p.q_sb + h * p.q_sh + static_cast<int64_t>(i) * p.q_ss, kb, vb, 0, i, p,
                                      D, row_mask(p, mr.r, dp, b, h), lane, rmax, rl, ra);
    row_store(o + b * p.o_sb + h * p.o_sh + static_cast<int64_t>(i) * p.o_ss, ra, rl > 0.f ? 1.f / rl : 0.f, D, lane);
    if (lane == 0) lse[static_cast<int64_t>(bh) * p.Sq + i] = rl > 0.f ? rmax + logf(rl) : -__builtin_inff();
  }
}

// ---------------------------------------------------------------- dQ
// As the forward; also writes delta = rowsum(dO o O) (which equals
// sum_j P Z (dO . V) under dropout factors Z) for the dK/dV kernel, and with
// an additive mask the inverse of the row's sum of probabilities (norm;
// attention_f32.h says why).
template <int D, int MK, bool DROP>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_masked_dq_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ o, const bf16* __restrict__ dout, const float* __restrict__ lse,
    float* __restrict__ delta, float* __restrict__ norm, bf16* __restrict__ dq, AttnShape p, MaskRead mr,
    DropoutParams dp, int n_qt, int items, int per_xcd) {
  constexpr int BQ = 64, KS = D / 32, DT = D / 16, S = masked_stages<D>();
  using Tile = Tile64<D>;
  constexpr int kLoads = 2 * TileStream<D, 4>::P;
  __shared__ __attribute__((aligned(1024))) bf16 sK[S][Tile::kElems];
  __shared__ __attribute__((aligned(1024))) bf16 sV[S][Tile::kElems];
  __shared__ uint64_t sBits[MK == kKeyMask ? kMaxMaskKeys / 64 : 1];

  const int w = xcd_item(items, per_xcd);
  if (w < 0) return;
  const int bh = w / n_qt;
  const int qt = n_qt - 1 - (w % n_qt);
  const int b = bh / p.Hq, h = bh % p.Hq;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l16 = lane & 15, g = lane >> 4;
  const int hk = h / (p.Hq / p.Hkv);
  const int qi = qt * BQ + 16 * wave + l16;
  const int qr = min(qi, p.Sq - 1);
  const int64_t mask_row = b * mr.r.sb + h * mr.r.sh + qr * mr.r.sq;
  const uint64_t prow = (static_cast<uint64_t>(bh) * p.Sq + qr) * p.Sk;
  if constexpr (MK == kKeyMask)
    load_key_bits(sBits, static_cast<const uint8_t*>(mr.r.p) + b * mr.r.sb + h * mr.r.sh, mr.r.sk, p.Sk);

  const int64_t q_row = b * p.q_sb + h * p.q_sh + static_cast<int64_t>(qr) * p.q_ss;
  const int64_t o_row = b * p.o_sb + h * p.o_sh + static_cast<int64_t>(qr) * p.o_ss;
  const bf16* kb = k + b * p.kv_sb + hk * p.kv_sh;
  const bf16* vb = v + b * p.kv_sb + hk * p.kv_sh;
  bf16x8 qf[KS], df[KS];
  float dl = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = ld8(q + q_row + ks * 32 + g * 8);
    df[ks] = ld8(dout + o_row + ks * 32 + g * 8);
    const bf16x8 of = ld8(o + o_row + ks * 32 + g * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) dl += static_cast<float>(df[ks][e]) * static_cast<float>(of[e]);
  }
  dl = xor32_sum(xor16_sum(dl));
  const int64_t row = static_cast<int64_t>(bh) * p.Sq + qr;
  float ls = lse[row];
  ls = ls == -__builtin_inff() ? __builtin_inff() : ls;  // no visible key: P = 0
  if (qi < p.Sq && g == 0) delta[row] = dl;
  wait_vmcnt<0>();
  TileStream<D, 4> ld;
  ld.init(p.kv_ss, wave, lane);
  KeyTiles<MK> tiles{sBits, visible_key_tiles(p, 0, p.q_offset + min(qt * BQ + BQ - 1, p.Sq - 1))};
  int kt = tiles.from(0), lt = kt;
  auto issue = [&](int st) {
    if (lt < tiles.end) {
      issue_kv<D, MK>(ld, kb, vb, sK[st], sV[st], p, lt, sBits, wave);
      lt = tiles.from(lt + 1);
    } else {
      issue_none<D>(k, sK[st], sV[st], wave);
    }
  };
#pragma unroll
  for (int st = 0; st < S - 1; ++st) issue(st);

  float psum = 0.f;  // this lane's 16 keys of every tile
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; kt < tiles.end; ++it) {
    wait_vmcnt<(S - 2) * kLoads>();
    lds_barrier();
    const int k0 = kt * 64;
    QueryMask<MK> qm;
    qm.load(mr, mask_row, k0, g, p.Sk);
    issue((it + S - 1) % S);
    const bf16* tk = sK[it % S];
    const bf16* tv = sV[it % S];
    uint64_t bits = 0;
    if constexpr (MK == kKeyMask) bits = sBits[kt] >> (4 * g);
    kt = tiles.from(kt + 1);
    const int lim = mask_limit(p, 0, k0, p.q_offset + qi);
    bf16x8 st[2][kTerms];
#pragma unroll
    for (int mk = 0; mk < 4; ++mk) {
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, t = s;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = mfma16(Tile::row8(tk, mk * 16 + l16, ks * 32 + g * 8), qf[ks], s);
        t = mfma16(Tile::row8(tv, mk * 16 + l16, ks * 32 + g * 8), df[ks], t);
      }
      bool keep[4] = {true, true, true, true};
      if constexpr (DROP) keep4(dp, prow + k0 + 16 * mk + 4 * g, (p.Sk & 1) == 0, keep);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = masked_score<MK>(s[e], p.scale, qm, bits, mk, e, mk * 16 + g * 4 + e, lim);
        const float pv = fast_exp2((x - ls) * kLog2e);
        if constexpr (MK == kAddMask) psum += pv;
        float dz = t[e];
        if constexpr (DROP) dz = keep[e] ? dz * dp.scale : 0.f;
        const float ds = x == -__builtin_inff() ? 0.f : pv * (dz - dl);
        split(ds, st[mk >> 1], 4 * (mk & 1) + e);
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const bf16x8 kk = Tile::col8(tk, 32 * s2, dt * 16, l16, g);
#pragma unroll
        for (int t = kTerms - 1; t >= 0; --t) acc[dt] = mfma16(kk, st[s2][t], acc[dt]);
      }
  }
  wait_vmcnt<0>();  // no load may still write this workgroup's LDS when it ends
  if constexpr (MK == kAddMask) psum = xor32_sum(xor16_sum(psum));
  uint32_t bad = nan_rows<DT>(acc, qi < p.Sq);
  if (qi < p.Sq && !(bad >> l16 & 1)) {
    float f = p.scale;
    if constexpr (MK == kAddMask) {
      const float inv = inverse_sum(psum);
      if (g == 0 && norm != nullptr) norm[row] = inv;
      f *= inv;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      bf16x4 wv;
#pragma unroll
      for (int e = 0; e < 4; ++e) wv[e] = static_cast<bf16>(acc[dt][e] * f);
      *reinterpret_cast<bf16x4*>(dq + q_row + dt * 16 + g * 4) = wv;
    }
  }
  for (; bad != 0; bad &= bad - 1) {
    const int r = __ffs(bad) - 1, i = qt * BQ + 16 * wave + r;
    const float row_delta = __shfl(dl, r, 64);
    const int64_t q_off = b * p.q_sb + h * p.q_sh + static_cast<int64_t>(i) * p.q_ss;
    float ra[2] = {0.f, 0.f}, rsum = 0.f;
    row_dq<bf16, row_kind<MK>, DROP>(q + q_off, dout + b * p.o_sb + h * p.o_sh + static_cast<int64_t>(i) * p.o_ss, kb,
                                     vb, 0, i, lse[static_cast<int64_t>(bh) * p.Sq + i], row_delta, p, D,
                                     row_mask(p, mr.r, dp, b, h), lane, ra, rsum);
    const float inv = MK == kAddMask ? inverse_sum(rsum) : 1.f;
    if (MK == kAddMask && lane == 0 && norm != nullptr) norm[static_cast<int64_t>(bh) * p.Sq + i] = inv;
    row_store(dq + q_off, ra, p.scale * inv, D, lane);
  }
}

// ---------------------------------------------------------------- dK, dV
// Workgroup = 64 keys of one (batch, KV head), 16 per wave; loops over the
// query heads of the group and the 64-query tiles that can see the keys.
template <int D, int MK, bool DROP>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_masked_dkdv_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const bf16* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    const float* __restrict__ norm, bf16* __restrict__ dk, bf16* __restrict__ dv, AttnShape p, MaskRead mr, DropoutParams dp, int n_kt,
    int items, int per_xcd) {
  constexpr int BQ = 64, KS = D / 32, DT = D / 16, S = masked_stages<D>();
  using Tile = Tile64<D>;
  // Q, dO and one row statistic (waves 0 and 2 the lse, 1 and 3 delta; with an
  // additive mask wave 2 the rows' normalisers)
  using TS = TileStream<D, 4>;
  constexpr int kLoads = 2 * TS::P + 1;
  __shared__ __attribute__((aligned(1024))) bf16 sQ[S][Tile::kElems];
  __shared__ __attribute__((aligned(1024))) bf16 sD[S][Tile::kElems];
  __shared__ __attribute__((aligned(256))) float sStat[S][4][BQ];

  const int w = xcd_item(items, per_xcd);
  if (w < 0) return;
  const int kt = w % n_kt, bk = w / n_kt;
  const int b = bk / p.Hkv, hk = bk % p.Hkv;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l16 = lane & 15, g = lane >> 4;
  const int group = p.Hq / p.Hkv;
  const int kbase = kt * 64 + 16 * wave;
  const int key = kbase + l16, kc = min(key, p.Sk - 1);
  const int n_qt = (p.Sq + BQ - 1) / BQ;
  int qt0 = 0;  // first query tile that sees a key of the workgroup
  if (p.causal) {
    const int64_t fq = static_cast<int64_t>(kt) * 64 - p.q_offset;
    qt0 = fq <= 0 ? 0 : (fq >= p.Sq ? n_qt : static_cast<int>(fq) / BQ);
  }
  // a boolean mask that is the same for every query and head of the group
  // hides this lane's key from all of them
  bool visible_key = key < p.Sk;
  if constexpr (MK == kKeyMask) {
    if (mr.r.sh == 0)
      visible_key = visible_key && static_cast<const uint8_t*>(mr.r.p)[b * mr.r.sb + kc * mr.r.sk] != 0;
  }
  const int total = __syncthreads_or(visible_key) ? group * (n_qt - qt0) : 0;

  const int64_t kv_row = b * p.kv_sb + hk * p.kv_sh + static_cast<int64_t>(kc) * p.kv_ss;
  bf16x8 kf[KS], vf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    kf[ks] = visible_key ? ld8(k + kv_row + ks * 32 + g * 8) : zero8();
    vf[ks] = visible_key ? ld8(v + kv_row + ks * 32 + g * 8) : zero8();
  }
  f32x4 dka[DT], dva[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dka[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    dva[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  wait_vmcnt<0>();
  TS lq, ldo;
  lq.init(p.q_ss, wave, lane);
  ldo.init(p.o_ss, wave, lane);
  int l_ih = 0, l_qt = qt0;  // the next tile to load
  auto issue = [&](int it, int st) {
    if (it < total) {
      const int h = hk * group + l_ih, r0 = l_qt * BQ, rows = min(BQ, p.Sq - r0);
      if (++l_qt == n_qt) {
        l_qt = qt0;
        ++l_ih;
      }
      const i32x4 rq = make_rsrc(q + b * p.q_sb + h * p.q_sh + static_cast<int64_t>(r0) * p.q_ss,
                                 static_cast<uint32_t>(((rows - 1) * p.q_ss + D) * 2));
      const i32x4 rd = make_rsrc(dout + b * p.o_sb + h * p.o_sh + static_cast<int64_t>(r0) * p.o_ss,
                                 static_cast<uint32_t>(((rows - 1) * p.o_ss + D) * 2));
      lq.issue(rq, sQ[st], 0, rows, 0u, wave);
      ldo.issue(rd, sD[st], 0, rows, 0u, wave);
      const float* stats = wave & 1 ? delta : lse;
      if constexpr (MK == kAddMask)
        if (wave == 2 && norm != nullptr) stats = norm;
      const float* stat = stats + (static_cast<int64_t>(b) * p.Hq + h) * p.Sq + r0;
      load_lds4(make_rsrc(stat, static_cast<uint32_t>(rows * 4)), &sStat[st][wave][0],
                lane < rows ? static_cast<uint32_t>(4 * lane) : kOOB);
    } else {
      issue_none<D>(q, sQ[st], sD[st], wave);
      load_lds4(make_rsrc(q, 0), &sStat[st][wave][0], kOOB);
    }
  };
#pragma unroll
  for (int st = 0; st < S - 1; ++st) issue(st, st);
  int c_ih = 0, c_qt = qt0;
  for (int it = 0; it < total; ++it) {
    wait_vmcnt<(S - 2) * kLoads>();
    lds_barrier();
    const int h = hk * group + c_ih, q0 = c_qt * BQ;
    if (++c_qt == n_qt) {
      c_qt = qt0;
      ++c_ih;
    }
    // mask entries of (query q0 + 16 mq + 4 g + e, this lane's key); rows past
    // Sq read a valid one
    bool on[4][4];
    float add[4][4];
    if constexpr (MK == kBoolMask || MK == kAddMask) {
      const int64_t base = b * mr.r.sb + h * mr.r.sh + kc * mr.r.sk;
#pragma unroll
      for (int mq = 0; mq < 4; ++mq)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t off = base + min(q0 + 16 * mq + 4 * g + e, p.Sq - 1) * mr.r.sq;
          if constexpr (MK == kBoolMask) on[mq][e] = static_cast<const uint8_t*>(mr.r.p)[off] != 0;
          else add[mq][e] = static_cast<float>(static_cast<const bf16*>(mr.r.p)[off]);
        }
    }
    bool vis = visible_key;
    if constexpr (MK == kKeyMask) {
      if (mr.r.sh != 0)
        vis = vis && static_cast<const uint8_t*>(mr.r.p)[b * mr.r.sb + h * mr.r.sh + kc * mr.r.sk] != 0;
    }
    issue(it + S - 1, (it + S - 1) % S);
    const bf16* tq = sQ[it % S];
    const bf16* td = sD[it % S];
    const float* sL = sStat[it % S][0];
    const float* sDl = sStat[it % S][1];
    // tile-relative queries [qmin, qend) see this lane's key
    const int qend = min(BQ, p.Sq - q0);
    int qmin = 0;
    if (p.causal) {
      const int64_t f = static_cast<int64_t>(key) - p.q_offset - q0;
      qmin = f < 0 ? 0 : (f > BQ ? BQ : static_cast<int>(f));
    }
    if (!vis) qmin = BQ;
    const uint64_t pbase = (static_cast<uint64_t>(b) * p.Hq + h) * p.Sq + q0;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      bf16x8 pt[kTerms], st[kTerms];
#pragma unroll
      for (int m2 = 0; m2 < 2; ++m2) {
        const int mq = 2 * s2 + m2;
        f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, t = s;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          s = mfma16(Tile::row8(tq, mq * 16 + l16, ks * 32 + g * 8), kf[ks], s);
          t = mfma16(Tile::row8(td, mq * 16 + l16, ks * 32 + g * 8), vf[ks], t);
        }
        bool keep[4] = {true, true, true, true};
        if constexpr (DROP) {
          const uint64_t i0 = (pbase + mq * 16 + g * 4) * p.Sk + key;
          if ((p.Sk & 1) == 0) {
            // lanes 2j and 2j + 1 (keys of one pair) share every output: the
            // even lane forms those of queries 0 and 1, the odd lane those of
            // 2 and 3, and each passes on the other's halves
            const bool odd = lane & 1;
            const uint64_t z0 = splitmix64(dp.seed, (i0 + (odd ? 2u : 0u) * static_cast<uint64_t>(p.Sk)) >> 1);
            const uint64_t z1 = splitmix64(dp.seed, (i0 + (odd ? 3u : 1u) * static_cast<uint64_t>(p.Sk)) >> 1);
            const uint32_t a0 = static_cast<uint32_t>(z0), a1 = static_cast<uint32_t>(z1);
            const uint32_t b0 = static_cast<uint32_t>(z0 >> 32), b1 = static_cast<uint32_t>(z1 >> 32);
            const uint32_t r0 = __builtin_bit_cast(uint32_t, dpp<0xB1>(__builtin_bit_cast(float, odd ? a0 : b0)));
            const uint32_t r1 = __builtin_bit_cast(uint32_t, dpp<0xB1>(__builtin_bit_cast(float, odd ? a1 : b1)));
            keep[0] = (odd ? r0 : a0) >= dp.threshold;
            keep[1] = (odd ? r1 : a1) >= dp.threshold;
            keep[2] = (odd ? b0 : r0) >= dp.threshold;
            keep[3] = (odd ? b1 : r1) >= dp.threshold;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              keep[e] = keep_bits(dp.seed, i0 + static_cast<uint64_t>(e) * p.Sk) >= dp.threshold;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int ql = mq * 16 + g * 4 + e;
          float ls = sL[ql];
          ls = ls == -__builtin_inff() ? __builtin_inff() : ls;
          float x;
          bool off = ql < qmin || ql >= qend;
          if constexpr (MK == kAddMask) {
            x = fmaf(s[e], p.scale, add[mq][e]);
            off = off || add[mq][e] == -__builtin_inff();
          } else {
            x = s[e] * p.scale;
          }
          if constexpr (MK == kBoolMask) off = off || !on[mq][e];
          float pv = fast_exp2((x - ls) * kLog2e);
          if constexpr (MK == kAddMask) pv *= norm != nullptr ? sStat[it % S][2][ql] : 1.f;
          float dz = t[e];
          if constexpr (DROP) dz = keep[e] ? dz * dp.scale : 0.f;
          const float ds = off ? 0.f : pv * (dz - sDl[ql]);
          if constexpr (DROP) pv = keep[e] ? pv * dp.scale : 0.f;
          pv = off ? 0.f : pv;
          split(pv, pt, 4 * m2 + e);
          split(ds, st, 4 * m2 + e);
        }
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const bf16x8 bd = Tile::col8(td, 32 * s2, dt * 16, l16, g);
        const bf16x8 bq = Tile::col8(tq, 32 * s2, dt * 16, l16, g);
#pragma unroll
        for (int t = kTerms - 1; t >= 0; --t) {
          dva[dt] = mfma16(pt[t], bd, dva[dt]);
          dka[dt] = mfma16(st[t], bq, dka[dt]);
        }
      }
    }
  }
  wait_vmcnt<0>();  // no load may still write this workgroup's LDS when it ends
  // lane holds dK[key = kbase + 4 g + e][d = 16 dt + l16]
  uint32_t bad = 0;  // keys with a NaN
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    bool nan = false;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) nan = nan || dka[dt][e] != dka[dt][e] || dva[dt][e] != dva[dt][e];
    const uint64_t lanes = __ballot(nan);
#pragma unroll
    for (int gg = 0; gg < 4; ++gg)
      if ((lanes >> (16 * gg)) & 0xffff) bad |= 1u << (4 * gg + e);
  }
  const int64_t kv_off = b * p.kv_sb + hk * p.kv_sh;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int kr = kbase + 4 * g + e;
    if (kr >= p.Sk || (bad >> (4 * g + e) & 1)) continue;
    const int64_t r = kv_off + static_cast<int64_t>(kr) * p.kv_ss;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      dk[r + dt * 16 + l16] = static_cast<bf16>(dka[dt][e] * p.scale);
      dv[r + dt * 16 + l16] = static_cast<bf16>(dva[dt][e]);
    }
  }
  for (; bad != 0; bad &= bad - 1) {
    const int j = kbase + __ffs(bad) - 1;
    if (j >= p.Sk) break;
    const int64_t r = kv_off + static_cast<int64_t>(j) * p.kv_ss;
    float rk[2] = {0.f, 0.f}, rv[2] = {0.f, 0.f};
    for (int h = hk * group; h < (hk + 1) * group; ++h) {
      const int64_t row = (static_cast<int64_t>(b) * p.Hq + h) * p.Sq;
      row_dkdv<bf16, row_kind<MK>, DROP>(k + r, v + r, q + b * p.q_sb + h * p.q_sh, dout + b * p.o_sb + h * p.o_sh,
                                         lse + row, delta + row,
                                         MK == kAddMask && norm != nullptr ? norm + row : nullptr, 0, j, p, D,
                                         row_mask(p, mr.r, dp, b, h), lane, rk, rv);
    }
    row_store(dk + r, rk, p.scale, D, lane);
    row_store(dv + r, rv, 1.f, D, lane);
  }
}

// ---------------------------------------------------------------- dispatch
// The MFMA kernels take bf16 heads of 64 and 128 whose rows are 16-byte
// aligned with 64 rows inside one 2 GiB descriptor, and work items that fit
// one launch; every other call runs the fp32 matrix-core kernels of
// attention_f32.h.
bool mfma_shape(const AttnShape& p, int64_t D, int dtype, std::initializer_list<const void*> rows16) {
  if (dtype != NMB_BF16 || (D != 64 && D != 128) || p.Sk == 0) return false;
  for (const void* r : rows16)
    if (!aligned16(r)) return false;
  const int64_t strides[] = {p.q_sb, p.q_ss, p.q_sh, p.kv_sb, p.kv_ss, p.kv_sh, p.o_sb, p.o_ss, p.o_sh};
  for (int64_t s : strides)
    if (s % 8 != 0 || s < 0) return false;
  if (64 * std::max(p.q_ss, std::max(p.kv_ss, p.o_ss)) >= (int64_t{1} << 29)) return false;
  const int64_t tiles = std::max((p.Sq + 63) / 64, (p.Sk + 63) / 64);
  return static_cast<int64_t>(p.B) * p.Hq * tiles < (int64_t{1} << 30);
}

// mask_kind of the entry points -> kind of the kernels
int kernel_mask(const AttnShape& p, const MaskRef& m, int mask_kind, MaskRead* out) {
  *out = MaskRead{m, 0};
  if (mask_kind == 0) return kNoMask;
  if (mask_kind == 1 && m.sq == 0 && p.Sk <= kMaxMaskKeys) return kKeyMask;
  const int64_t group_bytes = mask_kind == 1 ? 4 : 8;
  out->vec4 = m.sk == 1 && p.Sk % 4 == 0 && m.sb % 4 == 0 && m.sh % 4 == 0 && m.sq % 4 == 0 &&
              reinterpret_cast<uintptr_t>(m.p) % group_bytes == 0;
  return mask_kind == 1 ? kBoolMask : kAddMask;
}

// f<D, MK, DROP> for the runtime values
#define NMB_MASKED_CASE(D, MK)                                    \
  if (D_ == D && kind == MK) {                                    \
    if (drop) launch(std::integral_constant<int, D>{}, std::integral_constant<int, MK>{}, std::true_type{}); \
    else launch(std::integral_constant<int, D>{}, std::integral_constant<int, MK>{}, std::false_type{});     \
    return;                                                       \
  }
template <class F>
void masked_select(int D_, int kind, bool drop, F&& launch) {
  NMB_MASKED_CASE(64, kNoMask)
  NMB_MASKED_CASE(64, kKeyMask)
  NMB_MASKED_CASE(64, kBoolMask)
  NMB_MASKED_CASE(64, kAddMask)
  NMB_MASKED_CASE(128, kNoMask)
  NMB_MASKED_CASE(128, kKeyMask)
  NMB_MASKED_CASE(128, kBoolMask)
  NMB_MASKED_CASE(128, kAddMask)
}
#undef NMB_MASKED_CASE

void mfma_fwd_launch(const AttnShape& p, const MaskRef& mref, const DropoutParams& dp, int mask_kind, bool drop,
                     int D, const void* q, const void* k, const void* v, void* o, float* lse, hipStream_t stream) {
  MaskRead mr;
  const int kind = kernel_mask(p, mref, mask_kind, &mr);
  const int n_qt = (p.Sq + 63) / 64;
  const int items = p.B * p.Hq * n_qt;
  int per;
  unsigned blocks;
  xcd_grid(items, &per, &blocks);
  masked_select(D, kind, drop, [&](auto dd, auto mk, auto dr) {
    hipLaunchKernelGGL((attn_masked_fwd_kernel<dd.value, mk.value, dr.value>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                       static_cast<bf16*>(o), lse, p, mr, dp, n_qt, items, per);
  });
}

void mfma_bwd_launch(const AttnShape& p, const MaskRef& mref, const DropoutParams& dp, int mask_kind, bool drop,
                     int D, const void* q, const void* k, const void* v, const void* o, const void* dout,
                     const float* lse, float* delta, float* norm, void* dq, void* dk, void* dv,
                     hipStream_t stream) {
  MaskRead mr;
  const int kind = kernel_mask(p, mref, mask_kind, &mr);
  const int n_qt = (p.Sq + 63) / 64, n_kt = (p.Sk + 63) / 64;
  int per;
  unsigned blocks;
  if (p.Sq > 0) {
    const int items = p.B * p.Hq * n_qt;
    xcd_grid(items, &per, &blocks);
    masked_select(D, kind, drop, [&](auto dd, auto mk, auto dr) {
      hipLaunchKernelGGL((attn_masked_dq_kernel<dd.value, mk.value, dr.value>), dim3(blocks), dim3(256), 0, stream,
                         static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                         static_cast<const bf16*>(o), static_cast<const bf16*>(dout), lse, delta,
                         norm, static_cast<bf16*>(dq), p, mr, dp, n_qt, items, per);
    });
  }
  const int items = p.B * p.Hkv * n_kt;
  xcd_grid(items, &per, &blocks);
  masked_select(D, kind, drop, [&](auto dd, auto mk, auto dr) {
    hipLaunchKernelGGL((attn_masked_dkdv_kernel<dd.value, mk.value, dr.value>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                       static_cast<const bf16*>(dout), lse, delta, norm, static_cast<bf16*>(dk),
                       static_cast<bf16*>(dv), p, mr, dp, n_kt, items, per);
  });
}

}  // namespace
}  // namespace nmb

using nmb::AttnShape;
using nmb::KVBlocks;

namespace nmb {
namespace {

// Shape, mask and dropout of the masked entry points: one K/V block at key
// offset 0; any head_dim <= 128 and any strides (of bf16 or fp32 data) are
// accepted.  mask_kind 0
// (no mask) serves attention with dropout alone.
int masked_setup(AttnShape* p, KVBlocks* kv, MaskRef* mr, DropoutParams* dp, const void* q, const void* k,
                 const void* v, int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                 int64_t seq_k, int64_t head_dim, const int64_t* qs, const int64_t* kvs, const int64_t* os,
                 const void* mask, int mask_kind, const int64_t* ms, int causal, int64_t q_offset,
                 float scale, float dropout_p, uint64_t seed, int dtype) {
  NMB_REQUIRE_SUPPORTED(dtype == NMB_BF16 || dtype == NMB_F32, "attention (masked): unsupported dtype code %d",
                        dtype);
  NMB_REQUIRE(mask_kind == 0 || mask_kind == 1 || mask_kind == 2,
              "attention (masked): mask_kind must be 0 (none), 1 (boolean) or 2 (additive), got %d",
              mask_kind);
  NMB_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "attention (masked): dropout_p must be in [0, 1), got %g",
              static_cast<double>(dropout_p));
  if (mask_kind != 0) {
    NMB_REQUIRE(mask != nullptr && ms != nullptr, "attention (masked): null mask");
    NMB_REQUIRE(ms[0] >= 0 && ms[1] >= 0 && ms[2] >= 0 && ms[3] >= 0,
                "attention (masked): mask strides must be non-negative");
  }
  const void* kb[1] = {k};
  const void* vb[1] = {v};
  const int64_t koff[1] = {0};
  const int st = fill_shape(p, kv, q, kb, vb, koff, 1, batch, q_heads, kv_heads, seq_q, seq_k, head_dim,
                            qs, kvs, os, causal, q_offset, scale, NMB_F32);
  if (st != NMB_OK) return st;
  *mr = mask_kind != 0 ? MaskRef{mask, ms[0], ms[1], ms[2], ms[3]} : MaskRef{};
  *dp = make_dropout(static_cast<double>(dropout_p), seed);
  return NMB_OK;
}

}  // namespace
}  // namespace nmb

extern "C" int nmb_attn_masked_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                                   int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                                   int64_t seq_k, int64_t head_dim, const int64_t* q_strides,
                                   const int64_t* kv_strides, const int64_t* o_strides, const void* mask,
                                   int mask_kind, const int64_t* mask_strides, int causal,
                                   int64_t q_offset, float scale, float dropout_p, uint64_t seed, int dtype,
                                   hipStream_t stream) {
  AttnShape p;
  KVBlocks kv;
  nmb::MaskRef mr;
  nmb::DropoutParams dp;
  const int st = nmb::masked_setup(&p, &kv, &mr, &dp, q, k, v, batch, q_heads, kv_heads, seq_q, seq_k,
                                   head_dim, q_strides, kv_strides, o_strides, mask, mask_kind, mask_strides,
                                   causal, q_offset, scale, dropout_p, seed, dtype);
  if (st != NMB_OK) return st;
  NMB_REQUIRE(o != nullptr && lse != nullptr, "attn_masked_fwd: null output");
  if (batch == 0 || seq_q == 0) return NMB_OK;
  if (nmb::mfma_shape(p, head_dim, dtype, {q, k, v, o}))
    nmb::mfma_fwd_launch(p, mr, dp, mask_kind, dropout_p > 0.f, static_cast<int>(head_dim), q, k, v, o, lse, stream);
  else if (dtype == NMB_BF16)
    nmb::f32_fwd_launch<nmb::bf16>(p, kv, mr, dp, mask_kind, dropout_p > 0.f, q, o, lse, static_cast<int>(head_dim),
                                   stream);
  else
    nmb::f32_fwd_launch<float>(p, kv, mr, dp, mask_kind, dropout_p > 0.f, q, o, lse, static_cast<int>(head_dim),
                               stream);
  NMB_CHECK_LAUNCH("attn_masked_fwd");
  return NMB_OK;
}

extern "C" int nmb_attn_masked_bwd(const void* q, const void* k, const void* v, const void* o,
                                   const void* dout, const float* lse, void* dq, void* dk, void* dv,
                                   void* workspace, size_t workspace_bytes, int64_t batch,
                                   int64_t q_heads, int64_t kv_heads, int64_t seq_q, int64_t seq_k,
                                   int64_t head_dim, const int64_t* q_strides, const int64_t* kv_strides,
                                   const int64_t* o_strides, const void* mask, int mask_kind,
                                   const int64_t* mask_strides, int causal, int64_t q_offset, float scale,
                                   float dropout_p, uint64_t seed, int dtype, hipStream_t stream) {
  AttnShape p;
  KVBlocks kv;
  nmb::MaskRef mr;
  nmb::DropoutParams dp;
  const int st = nmb::masked_setup(&p, &kv, &mr, &dp, q, k, v, batch, q_heads, kv_heads, seq_q, seq_k,
                                   head_dim, q_strides, kv_strides, o_strides, mask, mask_kind, mask_strides,
                                   causal, q_offset, scale, dropout_p, seed, dtype);
  if (st != NMB_OK) return st;
  NMB_REQUIRE(o != nullptr && dout != nullptr && lse != nullptr && dq != nullptr && dk != nullptr &&
                  dv != nullptr,
              "attn_masked_bwd: null argument");
  const size_t need = static_cast<size_t>(batch * q_heads * seq_q) * sizeof(float);
  NMB_REQUIRE(workspace != nullptr && workspace_bytes >= need,
              "attn_masked_bwd: workspace of %zu bytes is smaller than the %zu required", workspace_bytes,
              need);
  kv.dk[0] = dk;
  kv.dv[0] = dv;
  if (batch == 0) return NMB_OK;
  float* delta = static_cast<float*>(workspace);
  float* norm = mask_kind == 2 && workspace_bytes >= 2 * need ? delta + batch * q_heads * seq_q : nullptr;
  if (nmb::mfma_shape(p, head_dim, dtype, {q, k, v, o, dout, dq}))
    nmb::mfma_bwd_launch(p, mr, dp, mask_kind, dropout_p > 0.f, static_cast<int>(head_dim), q, k, v, o, dout, lse,
                         delta, norm, dq, dk, dv, stream);
  else if (dtype == NMB_BF16)
    nmb::f32_bwd_launch<nmb::bf16>(p, kv, mr, dp, mask_kind, dropout_p > 0.f, q, o, dout, lse, delta, norm, dq,
                                   static_cast<int>(head_dim), stream);
  else
    nmb::f32_bwd_launch<float>(p, kv, mr, dp, mask_kind, dropout_p > 0.f, q, o, dout, lse, delta, norm, dq,
                               static_cast<int>(head_dim), stream);
  NMB_CHECK_LAUNCH("attn_masked_bwd");
  return NMB_OK;
}

