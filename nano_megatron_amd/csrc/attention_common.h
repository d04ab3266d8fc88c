// Shapes, tile streaming and argument checks shared by the attention kernels.
#pragma once

#include <math.h>

#include "common.h"
#include "lds_dma.h"

namespace nmb {
namespace {

constexpr int kMaxBlocks = 8;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct KVBlocks {
  const void* k[kMaxBlocks];
  const void* v[kMaxBlocks];
  void* dk[kMaxBlocks];
  void* dv[kMaxBlocks];
  int64_t koff[kMaxBlocks];
};

struct AttnShape {
  int B, Hq, Hkv, Sq, Sk, nblk, causal;
  int64_t q_sb, q_ss, q_sh;
  int64_t kv_sb, kv_ss, kv_sh;
  int64_t o_sb, o_ss, o_sh;
  int64_t q_offset;
  float scale;       // softmax scale
  float scale_log2;  // scale * log2(e)
};

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = static_cast<bf16>(0.f);
  return z;
}

__device__ __forceinline__ bf16x8 ld8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// exp2 as the raw v_exp_f32: results below 2^-126 flush to 0, which is
// immaterial for softmax weights (the library exp2 adds a 5-instruction
// denormal range fix-up around every exponential).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Number of 64-key tiles of a block that any query up to absolute position
// q_last can see.
__device__ __forceinline__ int visible_key_tiles(const AttnShape& p, int64_t koff, int64_t q_last) {
  int n = (p.Sk + 63) >> 6;
  if (p.causal) {
    const int64_t lim = q_last - koff;
    if (lim < 0) return 0;
    const int64_t t = (lim >> 6) + 1;
    if (t < n) n = static_cast<int>(t);
  }
  return n;
}

// Blocks are dispatched round-robin over the 8 XCDs (block L runs on XCD L % 8,
// each XCD with its own L2).  Work item w = (L % 8) * per_xcd + L / 8 puts
// consecutive items -- the q-tiles of one head, which read the same K/V -- on
// the same XCD.  Returns -1 for the padding blocks of the last round.
__device__ __forceinline__ int xcd_item(int items, int per_xcd) {
  const int L = static_cast<int>(blockIdx.x);
  const int w = (L % 8) * per_xcd + L / 8;
  return w < items ? w : -1;
}

// Advance (blk, kt) to the next visible K/V tile of the concatenated blocks;
// nt holds the visible tile count of block blk (recomputed only when the
// block changes).
__device__ __forceinline__ void next_tile(const AttnShape& p, const KVBlocks& kv, int64_t q_last,
                                          int& blk, int& kt, int& nt) {
  if (++kt < nt) return;
  kt = 0;
  for (++blk; blk < p.nblk; ++blk) {
    nt = visible_key_tiles(p, kv.koff[blk], q_last);
    if (nt > 0) return;
  }
}

__device__ __forceinline__ int first_block(const AttnShape& p, const KVBlocks& kv, int64_t q_last,
                                           int& nt) {
  int blk = 0;
  nt = 0;
  for (; blk < p.nblk; ++blk) {
    nt = visible_key_tiles(p, kv.koff[blk], q_last);
    if (nt > 0) break;
  }
  return blk;
}

// Largest tile-relative key index (key = k0 + index) visible to a query at
// absolute position qa: keys beyond Sk are never visible, and with causal
// masking key position koff + k0 + index must not exceed qa.
__device__ __forceinline__ int mask_limit(const AttnShape& p, int64_t koff, int k0, int64_t qa) {
  int64_t lim = static_cast<int64_t>(p.Sk) - 1 - k0;
  if (p.causal) {
    const int64_t c = qa - koff - k0;
    if (c < lim) lim = c;
  }
  if (lim < -1) lim = -1;
  if (lim > 1 << 20) lim = 1 << 20;
  return static_cast<int>(lim);
}

// 64-row x D bf16 tiles (K, V, Q, dO) stream from HBM straight into LDS
// (buffer_load ... lds: no register round trip), kStages deep, so kStages - 1
// tiles are in flight while one is computed.  A tile keeps the row-major
// layout with its 16-byte chunks swizzled: chunk c of row r in slot
// c ^ swz(r).  The swizzle serves both fragment kinds without bank conflicts
// (SQ_LDS_BANK_CONFLICT reads zero for each kind alone on gfx950):
//  * row fragments (an MFMA operand holding 8 consecutive columns of a row per
//    lane; 16 rows per lane group): one ds_read_b128;
//  * column fragments (8 rows of one column per lane: rows r0 + 4g .. +3 and
//    r0 + 16 + 4g .. +3 of a 32-row chunk, the key/query order in which the
//    score accumulators hold P and dS): two ds_read_b64_tr_b16.
// (2 ((r >> 1) & 3) + ((r >> 3) & 1) at D 64 and 2 (r & 7) + ((r >> 3) & 1) at
// D 128 keep the column reads conflict-free but give every row read a two-way
// conflict; r & 15 at D 128 the reverse.)
template <int D>
struct Tile64 {
  static constexpr int kElems = 64 * D;
  __device__ static int swz(int r) { return D == 64 ? (r & 7) : 2 * (r & 7); }
  __device__ static int at(int r, int col) { return r * D + 8 * ((col >> 3) ^ swz(r)) + (col & 7); }
  // row r, columns col .. col + 7 (col a multiple of 8)
  __device__ static bf16x8 row8(const bf16* t, int r, int col) { return ld8(t + at(r, col)); }
  // lane (l16, g): column c0 + l16, rows r0 + 4g .. +3 then r0 + 16 + 4g .. +3
  __device__ static bf16x8 col8(const bf16* t, int r0, int c0, int l16, int g) {
    const int r = r0 + 4 * g + (l16 >> 2), cc = c0 + 4 * (l16 & 3);
    return ld_tr(t + at(r, cc), t + at(r + 16, cc));
  }
};

// One wave's share (of NW waves) of the direct loads of a 64-row tile: load j
// fills LDS bytes [1024 (wave P + j), + 1024) of the tile; lane l's 16 bytes
// are chunk slot s of row r there, read from global chunk s ^ swz(r).
template <int D, int NW = 4>
struct TileStream {
  using Tile = Tile64<D>;
  static constexpr int P = Tile::kElems * 2 / 1024 / NW;  // 1 KB loads per wave per tile
  static_assert(P >= 1 && Tile::kElems * 2 % (1024 * NW) == 0, "a tile splits evenly over the waves");
  uint32_t off[P];  // byte offset from row 0 of the tile
  int row[P];

  __device__ void init(int64_t row_stride, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const int e = (1024 * (wave * P + j) + 16 * lane) / 2;  // element offset within the tile
      const int r = e / D, sl = (e % D) / 8;
      row[j] = r;
      off[j] = static_cast<uint32_t>(r * row_stride * 2) + 16u * static_cast<uint32_t>(sl ^ Tile::swz(r));
    }
  }

  // rows r0 .. r0 + 63 (r0 * row bytes = r0_bytes) of a matrix of nrows rows;
  // rows at and past nrows read as zeros
  __device__ __forceinline__ void issue(const i32x4& rs, bf16* dst, int r0, int nrows, uint32_t r0_bytes,
                                        int wave) const {
#pragma unroll
    for (int j = 0; j < P; ++j)
      load_lds16(rs, dst + 512 * (wave * P + j), r0 + row[j] < nrows ? r0_bytes + off[j] : kOOB);
  }
};

// ---------------------------------------------------------------- host side
int fill_shape(AttnShape* p, KVBlocks* kv, const void* q, const void* const* kb,
               const void* const* vb, const int64_t* koff, int nblk, int64_t B, int64_t Hq,
               int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D, const int64_t* qs,
               const int64_t* kvs, const int64_t* os, int causal, int64_t q_offset, float scale,
               int dtype) {
  NMB_REQUIRE(q != nullptr && kb != nullptr && vb != nullptr && koff != nullptr && qs != nullptr &&
                  kvs != nullptr && os != nullptr,
              "attention: null argument");
  NMB_REQUIRE(nblk >= 1 && nblk <= kMaxBlocks, "attention: n_blocks must be in [1, %d], got %d",
              kMaxBlocks, nblk);
  NMB_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Sq >= 0 && Sk >= 0 && D > 0,
              "attention: invalid shape");
  NMB_REQUIRE(Hq % Hkv == 0, "query heads (%lld) must be divisible by KV heads (%lld)",
              (long long)Hq, (long long)Hkv);
  NMB_REQUIRE(B <= 65535 && Hq <= 65535 && Sq <= 0x3fffffff && Sk <= 0x3fffffff,
              "attention: shape exceeds the launch grid");
  if (dtype == NMB_BF16) {
    NMB_REQUIRE_SUPPORTED(D == 64 || D == 128, "attention (bf16): head_dim must be 64 or 128, got %lld",
                          (long long)D);
    for (int i = 0; i < 3; ++i)
      NMB_REQUIRE_SUPPORTED(qs[i] % 8 == 0 && kvs[i] % 8 == 0 && os[i] % 8 == 0,
                            "attention (bf16): strides must be multiples of 8 elements");
    NMB_REQUIRE(aligned16(q), "attention: q must be 16-byte aligned");
  } else if (dtype == NMB_F32) {
    NMB_REQUIRE_SUPPORTED(D <= 128, "attention (fp32): head_dim must be <= 128, got %lld",
                          (long long)D);
  } else {
    NMB_REQUIRE_SUPPORTED(false, "attention: unsupported dtype code %d", dtype);
  }
  for (int i = 0; i < nblk; ++i) {
    NMB_REQUIRE(kb[i] != nullptr && vb[i] != nullptr, "attention: null K/V block %d", i);
    NMB_REQUIRE(dtype != NMB_BF16 || (aligned16(kb[i]) && aligned16(vb[i])),
                "attention: K/V blocks must be 16-byte aligned");
    kv->k[i] = kb[i];
    kv->v[i] = vb[i];
    kv->koff[i] = koff[i];
    kv->dk[i] = nullptr;
    kv->dv[i] = nullptr;
  }
  p->B = static_cast<int>(B);
  p->Hq = static_cast<int>(Hq);
  p->Hkv = static_cast<int>(Hkv);
  p->Sq = static_cast<int>(Sq);
  p->Sk = static_cast<int>(Sk);
  p->nblk = nblk;
  p->causal = causal ? 1 : 0;
  p->q_sb = qs[0];
  p->q_ss = qs[1];
  p->q_sh = qs[2];
  p->kv_sb = kvs[0];
  p->kv_ss = kvs[1];
  p->kv_sh = kvs[2];
  p->o_sb = os[0];
  p->o_ss = os[1];
  p->o_sh = os[2];
  p->q_offset = q_offset;
  p->scale = scale > 0.f ? scale : static_cast<float>(1.0 / sqrt(static_cast<double>(D)));
  p->scale_log2 = p->scale * kLog2e;
  return NMB_OK;
}

// Launch geometry of the XCD-mapped kernels: a 1-D grid of 8 * per_xcd blocks.
void xcd_grid(int64_t items, int* per_xcd, unsigned* blocks) {
  const int64_t per = (items + 7) / 8;
  *per_xcd = static_cast<int>(per);
  *blocks = static_cast<unsigned>(per * 8);
}
}  // namespace
}  // namespace nmb
