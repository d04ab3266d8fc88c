// Token embedding forward and backward for gfx950.
//
// Follows VocabParallelEmbedding.forward at TP=1 (reference
// tensor_parallel/embedding.py:60-74: F.embedding, a row gather of the [V, H]
// table) and its backward, the scatter-add of the output gradient rows into
// the table gradient.  An id outside [0, V) yields a zero row and adds nothing
// to the table gradient (embedding.py:63-68 masks ids outside the partition).  The table is tied to the LM head (models/gpt/model.py:
// 125-142), so the backward can take the LM head's table gradient and return
// the sum, in the order autograd accumulates them: bf16(lm + bf16(rows)).
//
// Backward without atomics (deterministic: a row's gradients are added in token
// order in fp32, and rounded once).  A first launch lists, for every 32 to 256
// table rows and every 8,192 tokens, the tokens whose id falls in the rows, in token
// order (one workgroup each: 8 ids per thread, a prefix sum of the hits).  In
// the second each wavefront owns 4 table rows x 256 columns and adds up rows
// of few tokens by itself, all their gradient rows in flight together; rows of
// more than 24 tokens are added by their workgroup, 64 gradient rows (32 KB) at
// a time through LDS.  What bounds it: writing the table gradient, and for a
// frequent token (6% of the tokens of text, or the padding of a batch) the
// latency of its stages, since its additions stay in order.
// Measured, bf16, us (before: one launch whose workgroups each walked every id
// for their 16 rows and added 16 gradient rows at a time):
// 8,192 Zipf tokens x 768, vocabulary 50,304: 43 (99); 8,192 x 1024, vocabulary
// 8,192: uniform 18 (18), Zipf 40 (93); 16,384 x 1024 of which two thirds one
// padding token: 370 (1,461); 65,536 Zipf x 1024, vocabulary 50,304: 289 (723).
#include <type_traits>

#include "common.h"
#include "vec.h"

namespace nmb {
namespace {

constexpr int RV = 4;           // table rows per wavefront, one after the other
constexpr int CW = 256;         // columns per wavefront (4 per lane)
constexpr int kSegment = 8192;  // tokens per list
constexpr int kHot = 24;        // more tokens than this: the row is added by the whole workgroup
constexpr int kTokens = 1024;   // such a row's tokens held in LDS
constexpr int kFewTokens = 64;  // no lists up to here
// Without a workspace every wavefront scans the ids up to here, else workgroups
// walk them (hidden 768, vocabulary 50,304: 65 tokens 22.6 against 29.5 us, 200
// 28.1 and 29.7, 8,192 746 and 99)
constexpr int kScanTokens = 192;

template <typename T>
__global__ __launch_bounds__(256) void embedding_fwd_kernel(const T* __restrict__ table,
                                                            const int64_t* __restrict__ ids,
                                                            T* __restrict__ out, int64_t n_tokens,
                                                            int64_t vocab, int64_t hidden) {
  constexpr int V = VecTraits<T>::N;
  const int64_t vecs = hidden / V;
  const int64_t total = n_tokens * vecs;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t t = i / vecs;
    const int64_t c = (i - t * vecs) * V;
    const int64_t id = ids[t];
    float v[V];
    if (id >= 0 && id < vocab) {
      load_vec<T>(table + id * hidden + c, v);
    } else {
      // an id outside the table's [0, vocab) gives a zero row and reads
      // nothing, as the reference masks ids outside its partition
      // (tensor_parallel/embedding.py:63-68; at TP=1 the partition is the table)
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = 0.f;
    }
    store_vec<T>(out + t * hidden + c, v);
  }
}

// List (segment blockIdx.y, group blockIdx.x): the segment's tokens whose id is
// in the group's rows, in token order.  A segment's lists stand one after the
// other in its kSegment entries (a token is in one list at most): list g at
// [starts[segment][g], starts[segment][g + 1]), the start being the number of
// ids below the group's rows, which the workgroup counts as it goes over them.
__global__ __launch_bounds__(1024) void embedding_list_kernel(const int64_t* __restrict__ ids, int64_t n_tokens,
                                                              int64_t vocab, int* __restrict__ starts,
                                                              int* __restrict__ lists, int row_bits) {
  constexpr int kPer = kSegment / 1024;
  __shared__ int totals[16], below[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t v0 = static_cast<int64_t>(blockIdx.x) << row_bits;
  const int64_t v1 = min(v0 + (int64_t{1} << row_bits), vocab);
  const int64_t base = static_cast<int64_t>(blockIdx.y) * kSegment;
  const int t0 = static_cast<int>(threadIdx.x) * kPer;
  int64_t id[kPer];
  int hits = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) id[j] = base + t0 + j < n_tokens ? ids[base + t0 + j] : -1;
#pragma unroll
  for (int j = 0; j < kPer; ++j) hits += id[j] >= v0 && id[j] < v1;
  int incl = hits;  // inclusive prefix over the wavefront
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  int lower = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) lower += static_cast<int>(__popcll(__ballot(id[j] >= 0 && id[j] < v0)));
  if (lane == 63) {
    totals[wave] = incl;
    below[wave] = lower;
  }
  __syncthreads();
  int pos = incl - hits;
  for (int w = 0; w < wave; ++w) pos += totals[w];
  for (int w = 0; w < 16; ++w) pos += below[w];
  int* start = starts + static_cast<int64_t>(blockIdx.y) * (gridDim.x + 1) + blockIdx.x;
  if (threadIdx.x == 0) start[0] = pos;
  if (threadIdx.x == 1023 && blockIdx.x + 1 == gridDim.x) start[1] = pos + hits;
  int* out = lists + base;
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if (id[j] >= v0 && id[j] < v1) out[pos++] = (t0 + j) << row_bits | static_cast<int>(id[j] - v0);
}

// four consecutive elements
template <typename T>
struct Quad;
template <>
struct Quad<bf16> {
  using Raw = uint2;
};
template <>
struct Quad<float> {
  using Raw = uint4;
};

template <typename T>
__device__ __forceinline__ void unpack4(const typename Quad<T>::Raw& raw, float (&v)[4]) {
  T e[4];
  __builtin_memcpy(e, &raw, sizeof(e));
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = to_f32(e[i]);
}

// LISTS: the tokens come from embedding_list_kernel's lists; else every
// wavefront scans the ids, 64 at a step (up to kScanTokens).
template <typename T, bool LISTS>
__global__ __launch_bounds__(256) void embedding_bwd_kernel(const T* __restrict__ dout,
                                                            const int64_t* __restrict__ ids,
                                                            const T* __restrict__ grad_in,
                                                            T* __restrict__ grad_out, int64_t n_tokens,
                                                            int64_t vocab, int64_t hidden,
                                                            const int* __restrict__ starts,
                                                            const int* __restrict__ lists, int groups, int row_bits,
                                                            int chunks) {
  using Raw = typename Quad<T>::Raw;
  constexpr int kStage = 128 / static_cast<int>(sizeof(T));  // gradient rows per stage of a hot row: 32 KB
  constexpr int kPer = kStage / 4;                           // of one wavefront
  __shared__ __attribute__((aligned(16))) T stage[kStage * CW];
  __shared__ int tok[kTokens];
  __shared__ int hot_rows[4], hot_state[2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t w0 = static_cast<int64_t>(blockIdx.x) / chunks * (4 * RV);  // the workgroup's rows
  const int64_t v0 = w0 + RV * wave;                                        // the wavefront's
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) % chunks * CW;
  const bool in = c0 + 4 * lane < hidden;
  const uint32_t col = in ? 4u * lane : 0u;  // (a lane past the columns loads the first ones, unused)
  const int rows = static_cast<int>(max<int64_t>(0, min<int64_t>(RV, vocab - v0)));
  const char* base = reinterpret_cast<const char*>(dout + c0);
  const int64_t row_bytes = hidden * static_cast<int64_t>(sizeof(T));
  auto grad_row = [&](int token) {
    return *reinterpret_cast<const Raw*>(base + token * row_bytes + col * static_cast<uint32_t>(sizeof(T)));
  };
  // the embedding's own gradient is rounded to the table dtype before the tied
  // LM-head gradient is added (autograd adds two gradient tensors)
  auto finished = [&](float sum, float prior) {
    const float mine = round_as<T>(sum);
    return from_f32<T>(grad_in != nullptr ? add_rn(prior, mine) : mine);
  };

  Raw prior[RV];  // the tied LM head's rows of this wavefront
  if (grad_in != nullptr) {
#pragma unroll
    for (int r = 0; r < RV; ++r)
      prior[r] = *reinterpret_cast<const Raw*>(grad_in + min<int64_t>(v0 + r, vocab - 1) * hidden + c0 + col);
  }

  // Entry k + lane of list s of the group's rows: the row within the group
  // (negative: none) and its token.
  const int group = static_cast<int>(w0 >> row_bits);
  const int64_t g0 = static_cast<int64_t>(group) << row_bits;
  const int r0 = static_cast<int>(v0 - g0);
  const int segments = LISTS ? static_cast<int>((n_tokens + kSegment - 1) / kSegment) : 1;
  struct List {
    int start, n;
  };
  auto entries = [&](int s) {
    if constexpr (!LISTS) return List{0, static_cast<int>(n_tokens)};
    const int* st = starts + static_cast<int64_t>(s) * (groups + 1) + group;
    return List{st[0], st[1] - st[0]};
  };
  auto fetch = [&](int s, const List& l, int k, int& row, int& token) {
    row = -1;
    token = 0;
    if (k + lane >= l.n) return;
    if constexpr (LISTS) {
      const int e = lists[static_cast<int64_t>(s) * kSegment + l.start + k + lane];
      row = e & ((1 << row_bits) - 1);
      token = s * kSegment + (e >> row_bits);
    } else {
      const int64_t id = ids[k + lane];  // (the last group's rows may end past the table)
      if (id >= g0 && id < min<int64_t>(g0 + (1 << row_bits), vocab)) row = static_cast<int>(id - g0);
      token = k + lane;
    }
  };

  // how many tokens each row has
  int cnt[RV];
#pragma unroll
  for (int r = 0; r < RV; ++r) cnt[r] = 0;
  const List first = segments > 0 ? entries(0) : List{0, 0};
  int row0 = -1, token0 = 0;  // the first entries, kept
  fetch(0, first, 0, row0, token0);
  for (int s = 0; s < segments; ++s) {
    const List l = s == 0 ? first : entries(s);
    for (int k = 0; k < l.n; k += 64) {
      int row = row0, token;
      if (s != 0 || k != 0) fetch(s, l, k, row, token);
#pragma unroll
      for (int r = 0; r < RV; ++r) cnt[r] += __popcll(__ballot(row == r0 + r));
    }
  }
  int hot = 0;
  float acc[RV][4];
#pragma unroll
  for (int r = 0; r < RV; ++r) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[r][e] = 0.f;
    if (cnt[r] > kHot) {
      hot |= 1 << r;
      cnt[r] = 0;
    }
  }
  auto add = [&](float (&a)[4], const Raw& raw) {
    float v[4];
    unpack4<T>(raw, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] += v[e];
  };
  // the first U tokens of the mask (bit: the lane holding the token), in order
  auto take = [&](auto width, uint64_t& mask, int token, Raw (&raw)[decltype(width)::value]) {
    int at = 0;
#pragma unroll
    for (int u = 0; u < decltype(width)::value; ++u) {
      if (mask == 0) break;
      at = __ffsll(static_cast<unsigned long long>(mask)) - 1;
      mask &= mask - 1;
      raw[u] = grad_row(__builtin_amdgcn_readlane(token, at));
    }
  };
  using W4 = std::integral_constant<int, 4>;
  using W8 = std::integral_constant<int, 8>;
  // rows of up to kHot tokens, 64 entries at a time: the first four tokens of
  // every row loaded together
  int left = (cnt[0] + cnt[1]) + (cnt[2] + cnt[3]);
  for (int s = 0; s < segments && left > 0; ++s) {
    const List l = s == 0 ? first : entries(s);
    for (int k = 0; k < l.n && left > 0; k += 64) {
      int row = row0, token = token0;
      if (s != 0 || k != 0) fetch(s, l, k, row, token);
      uint64_t mask[RV];
      int n4[RV];
      Raw raw[RV][4];
#pragma unroll
      for (int r = 0; r < RV; ++r) {
        mask[r] = cnt[r] > 0 ? __ballot(row == r0 + r) : 0;
        n4[r] = min(4, static_cast<int>(__popcll(mask[r])));
        left -= static_cast<int>(__popcll(mask[r]));
        take(W4{}, mask[r], token, raw[r]);
      }
#pragma unroll
      for (int r = 0; r < RV; ++r) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (u < n4[r]) add(acc[r], raw[r][u]);
        while (mask[r] != 0) {
          Raw more[8];
          const int m = min(8, static_cast<int>(__popcll(mask[r])));
          take(W8{}, mask[r], token, more);
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (u < m) add(acc[r], more[u]);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RV; ++r) {
    if (r >= rows || !in || (hot >> r & 1)) continue;
    float p[4] = {0.f, 0.f, 0.f, 0.f};
    if (grad_in != nullptr) unpack4<T>(prior[r], p);
    T out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = finished(acc[r][e], p[e]);
    Raw raw;
    __builtin_memcpy(&raw, out, sizeof(out));
    *reinterpret_cast<Raw*>(grad_out + (v0 + r) * hidden + c0 + col) = raw;
  }

  // Rows of many tokens, by the whole workgroup: wavefront 0 gathers their
  // tokens, all four load a stage of gradient rows into LDS (the next stage's
  // loads in flight meanwhile), and each thread adds up one column in order.
  if (lane == 0) hot_rows[wave] = hot;
  __syncthreads();
  int todo = hot_rows[0] | hot_rows[1] << RV | hot_rows[2] << (2 * RV) | hot_rows[3] << (3 * RV);
  while (todo != 0) {
    const int hr = __ffs(todo) - 1;
    todo &= todo - 1;
    const int64_t v = w0 + hr;
    const int row_in_group = static_cast<int>(v - g0);
    const int64_t cell = v * hidden + c0 + threadIdx.x;
    const bool mine = c0 + threadIdx.x < hidden;
    float sum = 0.f;
    int s = 0, k = 0;  // wavefront 0's place in the lists
    for (bool last = false; !last;) {
      if (wave == 0) {
        int n = 0;
        while (s < segments && n <= kTokens - 64) {
          const List l = entries(s);
          for (; k < l.n && n <= kTokens - 64; k += 64) {
            int row, token;
            fetch(s, l, k, row, token);
            const uint64_t mask = __ballot(row == row_in_group);
            if (row == row_in_group) tok[n + __popcll(mask & ((1ull << lane) - 1))] = token;
            n += static_cast<int>(__popcll(mask));
          }
          if (k >= l.n) {
            ++s;
            k = 0;
          }
        }
        if (lane == 0) {
          hot_state[0] = n;
          hot_state[1] = s >= segments;
        }
      }
      __syncthreads();
      const int n = hot_state[0];
      last = hot_state[1] != 0;
      Raw next[kPer];
      auto load = [&](int at) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) next[j] = grad_row(tok[min(at + wave * kPer + j, n - 1)]);
      };
      if (n > 0) load(0);
      for (int at = 0; at < n; at += kStage) {
#pragma unroll
        for (int j = 0; j < kPer; ++j)
          *reinterpret_cast<Raw*>(&stage[(wave * kPer + j) * CW + 4 * lane]) = next[j];
        __syncthreads();
        if (at + kStage < n) load(at + kStage);
        const int m = min(kStage, n - at);
        if (m == kStage) {
#pragma unroll 16
          for (int i = 0; i < kStage; ++i) sum += to_f32(stage[i * CW + threadIdx.x]);
        } else {
          for (int i = 0; i < m; ++i) sum += to_f32(stage[i * CW + threadIdx.x]);
        }
        __syncthreads();
      }
    }
    if (mine) grad_out[cell] = finished(sum, grad_in != nullptr ? to_f32(grad_in[cell]) : 0.f);
    // a last gather that found nothing passed no barrier since hot_state was
    // read, and wavefront 0 writes it again for the next row
    __syncthreads();
  }
}

// Backward of a caller without a workspace for the lists: a workgroup owns 16
// table rows x 1,024 columns, goes over the ids in rounds of 2,048 (8 consecutive
// ones per thread, loaded together), lists the tokens of its rows in token order
// (a workgroup prefix sum of each thread's hits), and once the ids are done (or
// the list is full) adds their gradient rows, sixteen in flight, to fp32
// accumulators in LDS in list order.  The ids (8 bytes a token) are read by
// every workgroup from L2, which bounds it for many tokens.
constexpr int kWalkRows = 16, kWalkCols = 1024;
constexpr int kWalkPer = 8, kWalkRound = 256 * kWalkPer;
constexpr int kWalkList = 3072;  // listed tokens held before their rows are added (12 KB of LDS)
constexpr int kWalkBatch = 16;   // gradient rows loaded together

template <typename T>
__device__ __forceinline__ void load4(const T* p, float (&v)[4]) {
  unpack4<T>(*reinterpret_cast<const typename Quad<T>::Raw*>(p), v);
}

template <typename T>
__global__ __launch_bounds__(256, 2) void embedding_bwd_walk_kernel(const T* __restrict__ dout,
                                                                    const int64_t* __restrict__ ids,
                                                                    const T* __restrict__ grad_in,
                                                                    T* __restrict__ grad_out, int64_t n_tokens,
                                                                    int64_t vocab, int64_t hidden) {
  __shared__ float4 acc[kWalkRows * kWalkCols / 4];  // 64 KB: row r, this thread's 4 columns at [r * kWalkCols / 4 + thread]
  __shared__ int list[kWalkList];          // matching tokens in token order: token * kWalkRows + row
  __shared__ int wave_total[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row_blocks = (vocab + kWalkRows - 1) / kWalkRows;
  const int64_t v0 = (blockIdx.x % row_blocks) * kWalkRows;
  const int64_t c0 = (blockIdx.x / row_blocks) * kWalkCols;
  const int cols = static_cast<int>(min<int64_t>(kWalkCols, hidden - c0));
  const int c = threadIdx.x * 4;  // this thread's 4 columns
  const int cc = c < cols ? c : 0;  // (a thread past the chunk's columns loads column 0, unused)
#pragma unroll
  for (int r = 0; r < kWalkRows; ++r) acc[r * (kWalkCols / 4) + threadIdx.x] = make_float4(0.f, 0.f, 0.f, 0.f);

  // the tied LM head's rows of this block, loaded first: nothing depends on
  // them until the end (rows past the table read its last row, not stored)
  float prior[kWalkRows][4];
#pragma unroll
  for (int r = 0; r < kWalkRows; ++r) {
    if (grad_in != nullptr) {
      load4(grad_in + min(v0 + r, vocab - 1) * hidden + c0 + cc, prior[r]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) prior[r][e] = 0.f;
    }
  }

  // the listed gradient rows, in token order, into the accumulators: all of
  // a batch's loads in flight together
  int listed = 0;  // workgroup-uniform
  auto add_listed = [&]() {
    if (c < cols) {
      for (int k0 = 0; k0 < listed; k0 += kWalkBatch) {
        float v[kWalkBatch][4];
        int row[kWalkBatch];
#pragma unroll
        for (int u = 0; u < kWalkBatch; ++u) {
          const int e = list[min(k0 + u, listed - 1)];
          row[u] = e % kWalkRows;
          load4(dout + static_cast<int64_t>(e / kWalkRows) * hidden + c0 + c, v[u]);
        }
#pragma unroll
        for (int u = 0; u < kWalkBatch; ++u) {
          if (k0 + u < listed) {  // (no break: the loaded rows stay in registers)
            float4& a = acc[row[u] * (kWalkCols / 4) + threadIdx.x];
            float4 t = a;
            t.x += v[u][0];
            t.y += v[u][1];
            t.z += v[u][2];
            t.w += v[u][3];
            a = t;
          }
        }
      }
    }
    listed = 0;
  };

  // the ids in rounds of kWalkPer consecutive tokens per thread, the next round's
  // in flight while this round's are listed; the rows are added once the
  // list is full or the ids are done, so that their loads are not spread
  // over the rounds one latency each
  int64_t id[kWalkPer], next[kWalkPer];
#pragma unroll
  for (int j = 0; j < kWalkPer; ++j) next[j] = -1;
  auto load_ids = [&](int64_t base, int64_t (&dst)[kWalkPer]) {
    const int64_t t0 = base + threadIdx.x * kWalkPer;
#pragma unroll
    for (int j = 0; j < kWalkPer; ++j) dst[j] = t0 + j < n_tokens ? ids[t0 + j] : -1;
  };
  load_ids(0, id);
  for (int64_t base = 0; base < n_tokens; base += kWalkRound) {
    if (listed > kWalkList - kWalkRound) {
      // a full round may not fit: add what is listed first (every thread is
      // past the previous round's list writes: second barrier below)
      add_listed();
      __syncthreads();  // every thread is done reading the list
    }
    const int t_off = static_cast<int>(base) + threadIdx.x * kWalkPer;
    int hits = 0;
#pragma unroll
    for (int j = 0; j < kWalkPer; ++j) hits += id[j] >= v0 && id[j] < v0 + kWalkRows;
    // exclusive prefix of the hits over the workgroup (thread order = token order)
    int incl = hits;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d, 64);
      if (lane >= d) incl += y;
    }
    if (lane == 63) wave_total[wave] = incl;
    __syncthreads();  // wave totals ready
    int pos = listed + incl - hits;
    for (int w = 0; w < wave; ++w) pos += wave_total[w];
    const int total = wave_total[0] + wave_total[1] + wave_total[2] + wave_total[3];
#pragma unroll
    for (int j = 0; j < kWalkPer; ++j)
      if (id[j] >= v0 && id[j] < v0 + kWalkRows) list[pos++] = (t_off + j) * kWalkRows + static_cast<int>(id[j] - v0);
    listed += total;
    __syncthreads();  // the round's list entries are visible; wave totals read
    if (base + kWalkRound < n_tokens) load_ids(base + kWalkRound, next);
#pragma unroll
    for (int j = 0; j < kWalkPer; ++j) id[j] = next[j];
  }
  add_listed();
  __syncthreads();
  if (c >= cols) return;
#pragma unroll
  for (int r = 0; r < kWalkRows; ++r) {
    if (v0 + r >= vocab) break;
    const int64_t o = (v0 + r) * hidden + c0 + c;
    const float4 a4 = acc[r * (kWalkCols / 4) + threadIdx.x];
    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
    T out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float mine = round_as<T>(av[e]);  // as in embedding_bwd_kernel
      out[e] = from_f32<T>(grad_in != nullptr ? add_rn(prior[r][e], mine) : mine);
    }
    typename Quad<T>::Raw raw;
    __builtin_memcpy(&raw, out, sizeof(out));
    *reinterpret_cast<typename Quad<T>::Raw*>(grad_out + o) = raw;
  }
}

// Rows per list as a power of two: lists as short as 256 of them allow (a
// wavefront scans its rows' list 64 entries at a time), 32 rows at least; an
// entry holds a token of 13 bits and a row of at most 18.
int list_row_bits(int64_t vocab) {
  int bits = 5;
  while (bits < 18 && ((vocab - 1) >> bits) + 1 > 256) ++bits;
  return bits;
}

// Bytes of the starts (rounded up to 256) and lists of n_tokens ids: 4 bytes per
// token and at most 1 KB per 8,192.  Up to 64 tokens every wavefront scans the
// ids itself (one step) instead of a launch for the lists (64 tokens x 768,
// vocabulary 50,304, forward and backward replayed: 30.5 us, with lists 34).
int64_t starts_bytes(int64_t n_tokens, int64_t groups) {
  return ((n_tokens + kSegment - 1) / kSegment * (groups + 1) * 4 + 255) / 256 * 256;
}
int64_t list_bytes(int64_t n_tokens, int64_t vocab) {
  if (n_tokens <= kFewTokens) return 0;
  return starts_bytes(n_tokens, ((vocab - 1) >> list_row_bits(vocab)) + 1) + n_tokens * 4;
}

template <typename T>
int fwd_impl(const void* table, const int64_t* ids, void* out, int64_t n_tokens, int64_t vocab,
             int64_t hidden, hipStream_t stream) {
  constexpr int V = VecTraits<T>::N;
  NMB_REQUIRE_SUPPORTED(hidden % V == 0, "embedding: hidden (%lld) must be a multiple of %d",
                        (long long)hidden, V);
  NMB_REQUIRE(aligned16(table) && aligned16(out), "embedding: tensors must be 16-byte aligned");
  const int64_t total = n_tokens * (hidden / V);
  if (total == 0) return NMB_OK;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((embedding_fwd_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     stream, static_cast<const T*>(table), ids, static_cast<T*>(out), n_tokens,
                     vocab, hidden);
  NMB_CHECK_LAUNCH("embedding_fwd");
  return NMB_OK;
}

template <typename T>
int bwd_impl(const void* dout, const int64_t* ids, const void* grad_in, void* grad_out,
             int64_t n_tokens, int64_t vocab, int64_t hidden, void* workspace, int64_t workspace_bytes,
             hipStream_t stream) {
  NMB_REQUIRE_SUPPORTED(hidden % 4 == 0, "embedding_bwd: hidden (%lld) must be a multiple of 4",
                        (long long)hidden);
  const int64_t chunks = (hidden + CW - 1) / CW;
  const int64_t blocks = (vocab + 4 * RV - 1) / (4 * RV) * chunks;
  const int row_bits = list_row_bits(vocab);
  const int64_t groups = ((vocab - 1) >> row_bits) + 1;
  NMB_REQUIRE(blocks < (int64_t{1} << 31) && chunks < (int64_t{1} << 31), "embedding_bwd: table too large");
  NMB_REQUIRE_SUPPORTED(n_tokens < (int64_t{1} << 27), "embedding_bwd: %lld tokens exceed the supported 2^27",
                        (long long)n_tokens);
  // rows of 4 elements: one alignment for every dtype's accesses
  const uintptr_t align = 4 * sizeof(T) - 1;
  NMB_REQUIRE((reinterpret_cast<uintptr_t>(dout) & align) == 0 &&
                  (reinterpret_cast<uintptr_t>(grad_out) & align) == 0 &&
                  (grad_in == nullptr || (reinterpret_cast<uintptr_t>(grad_in) & align) == 0),
              "embedding_bwd: dout, grad_in and grad_out must be aligned to %d bytes",
              static_cast<int>(align + 1));
  if (blocks == 0) return NMB_OK;
  const int64_t bytes = workspace != nullptr ? list_bytes(n_tokens, vocab) : 0;
  int* starts = nullptr;
  int* lists = nullptr;
  if (bytes > 0) {
    NMB_REQUIRE(workspace_bytes >= bytes, "embedding_bwd: workspace of %lld bytes is smaller than the %lld required",
                (long long)workspace_bytes, (long long)bytes);
    const int64_t segments = (n_tokens + kSegment - 1) / kSegment;
    starts = static_cast<int*>(workspace);
    lists = starts + starts_bytes(n_tokens, groups) / 4;
    hipLaunchKernelGGL(embedding_list_kernel, dim3(static_cast<unsigned>(groups), static_cast<unsigned>(segments)),
                       dim3(1024), 0, stream, ids, n_tokens, vocab, starts, lists, row_bits);
    NMB_CHECK_LAUNCH("embedding_bwd(lists)");
    hipLaunchKernelGGL((embedding_bwd_kernel<T, true>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,
                       static_cast<const T*>(dout), ids, static_cast<const T*>(grad_in), static_cast<T*>(grad_out),
                       n_tokens, vocab, hidden, starts, lists, static_cast<int>(groups), row_bits,
                       static_cast<int>(chunks));
  } else if (n_tokens <= kScanTokens) {
    hipLaunchKernelGGL((embedding_bwd_kernel<T, false>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,
                       static_cast<const T*>(dout), ids, static_cast<const T*>(grad_in), static_cast<T*>(grad_out),
                       n_tokens, vocab, hidden, starts, lists, static_cast<int>(groups), row_bits,
                       static_cast<int>(chunks));
  } else {
    const int64_t walkers = ((vocab + kWalkRows - 1) / kWalkRows) * ((hidden + kWalkCols - 1) / kWalkCols);
    hipLaunchKernelGGL(embedding_bwd_walk_kernel<T>, dim3(static_cast<unsigned>(walkers)), dim3(256), 0, stream,
                       static_cast<const T*>(dout), ids, static_cast<const T*>(grad_in), static_cast<T*>(grad_out),
                       n_tokens, vocab, hidden);
  }
  NMB_CHECK_LAUNCH("embedding_bwd");
  return NMB_OK;
}

int bwd(const void* dout, const int64_t* ids, const void* grad_in, void* grad_out, int64_t n_tokens, int64_t vocab,
        int64_t hidden, void* workspace, int64_t workspace_bytes, int dtype, hipStream_t stream) {
  NMB_REQUIRE(dout != nullptr && ids != nullptr && grad_out != nullptr, "embedding_bwd: null argument");
  NMB_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden > 0, "embedding_bwd: invalid shape");
  if (dtype == NMB_BF16)
    return bwd_impl<bf16>(dout, ids, grad_in, grad_out, n_tokens, vocab, hidden, workspace, workspace_bytes, stream);
  if (dtype == NMB_F32)
    return bwd_impl<float>(dout, ids, grad_in, grad_out, n_tokens, vocab, hidden, workspace, workspace_bytes, stream);
  NMB_REQUIRE_SUPPORTED(false, "embedding_bwd: unsupported dtype %d", dtype);
  return NMB_EUNSUPPORTED;
}

}  // namespace
}  // namespace nmb

extern "C" int nmb_embedding_fwd(const void* table, const int64_t* ids, void* out, int64_t n_tokens,
                                 int64_t vocab, int64_t hidden, int dtype, hipStream_t stream) {
  NMB_REQUIRE(table != nullptr && ids != nullptr && out != nullptr, "embedding_fwd: null argument");
  NMB_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden > 0, "embedding_fwd: invalid shape");
  if (dtype == NMB_BF16) return nmb::fwd_impl<nmb::bf16>(table, ids, out, n_tokens, vocab, hidden, stream);
  if (dtype == NMB_F32) return nmb::fwd_impl<float>(table, ids, out, n_tokens, vocab, hidden, stream);
  NMB_REQUIRE_SUPPORTED(false, "embedding_fwd: unsupported dtype %d", dtype);
  return NMB_EUNSUPPORTED;
}

extern "C" int nmb_embedding_bwd(const void* dout, const int64_t* ids, const void* grad_in,
                                 void* grad_out, int64_t n_tokens, int64_t vocab, int64_t hidden,
                                 int dtype, hipStream_t stream) {
  return nmb::bwd(dout, ids, grad_in, grad_out, n_tokens, vocab, hidden, nullptr, 0, dtype, stream);
}

extern "C" int nmb_embedding_bwd_workspace_bytes(int64_t n_tokens, int64_t vocab, int64_t* bytes) {
  NMB_REQUIRE(bytes != nullptr && n_tokens >= 0 && vocab > 0, "embedding_bwd_workspace_bytes: bad args");
  *bytes = nmb::list_bytes(n_tokens, vocab);
  return NMB_OK;
}

extern "C" int nmb_embedding_bwd_ws(const void* dout, const int64_t* ids, const void* grad_in, void* grad_out,
                                    int64_t n_tokens, int64_t vocab, int64_t hidden, void* workspace,
                                    int64_t workspace_bytes, int dtype, hipStream_t stream) {
  return nmb::bwd(dout, ids, grad_in, grad_out, n_tokens, vocab, hidden, workspace, workspace_bytes, dtype, stream);
}
