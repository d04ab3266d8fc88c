// The transformer block's launch sequences (reference GPTLayer.forward,
// models/gpt/layer.py:91-137, and its autograd): host code that enqueues the
// kernels of the other files one after the other, so that a block costs its
// caller one call forward and two backward.  Driven one C call per kernel from
// Python, every launch cost about 29 us of host time and short sequences waited
// for the host: a smoke-configuration step (4 fp32 layers, 4 x 128 tokens) took
// 4.44 ms against 1.4 ms of kernels (1.92 ms so), the logits of a 193-token
// prefix through 24 layers of hidden 1024 4.69 ms (2.02 ms so), one layer of
// hidden 768 on 3 x 709 tokens forward and backward 0.87 ms (0.41 ms so).
//
// Weight gradients on a second stream: the block's weight gradients feed
// nothing else in its backward, and beside the dX chain they fill the CUs that
// its launches leave idle.  The MLP's two run there; the out projection's and
// the QKV projection's stay on the main stream (on the side the first's overlap
// would fall on the attention backward, whose workgroups it then displaces,
// the second's on the norm backward only: each measured slower).  Where the
// two are queued depends on the launch, as measured on whole config-3 steps.
// Launched from the host, the gate/up weight gradient is queued after the dX
// product that follows the fused MLP backward (before it, it takes that
// product's CUs: 2.2% slower), and the post-attention norm's dw column sum runs
// on the side.  Captured in a HIP graph, where every cross-stream wait is an
// edge that costs device time at each replay, both products are queued behind
// one wait and the column sum stays on the main stream (1.75% faster).
#include <algorithm>

#include "common.h"

namespace {

struct Dims {
  int64_t T, H, Nq, Nk, N, F;  // tokens, hidden, q / k columns, q|k|v columns, ffn
  bool bf16;
  int64_t es;
};

int block_dims(const nmb_block* b, Dims* d) {
  NMB_REQUIRE(b != nullptr, "block: null description");
  NMB_REQUIRE_SUPPORTED(b->dtype == NMB_BF16 || b->dtype == NMB_F32, "block: unsupported dtype code %d", b->dtype);
  NMB_REQUIRE(b->batch >= 0 && b->seq >= 0 && b->hidden > 0 && b->q_heads > 0 && b->kv_heads > 0 &&
                  b->head_dim > 0 && b->ffn > 0,
              "block: invalid shape");
  NMB_REQUIRE_SUPPORTED(b->dtype == NMB_F32 || b->head_dim == 64 || b->head_dim == 128,
                        "block (bf16): head_dim must be 64 or 128, got %lld", (long long)b->head_dim);
  d->T = b->batch * b->seq;
  d->H = b->hidden;
  d->Nq = b->q_heads * b->head_dim;
  d->Nk = b->kv_heads * b->head_dim;
  d->N = d->Nq + 2 * d->Nk;
  d->F = b->ffn;
  d->bf16 = b->dtype == NMB_BF16;
  d->es = d->bf16 ? 2 : 4;
  return NMB_OK;
}

#define NMB_TRY(call)              \
  do {                             \
    const int _st = (call);        \
    if (_st != NMB_OK) return _st; \
  } while (0)

int gemm_ws(const Dims& d, int la, int lb, int64_t m, int64_t n, int64_t k, int64_t* bytes) {
  if (d.bf16) return nmb_gemm_bf16_workspace_bytes(la, lb, m, n, k, bytes);
  return nmb_gemm_f32_workspace_bytes(m, n, k, bytes);
}

// out = op(a) op(b) (+ c), row-major out of leading dimension n
int gemm(const Dims& d, int la, int lb, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda, const void* b,
         int64_t ldb, const void* c, void* out, void* ws, int64_t ws_bytes, hipStream_t s) {
  int64_t need = 0;
  NMB_TRY(gemm_ws(d, la, lb, m, n, k, &need));
  NMB_REQUIRE(need <= ws_bytes, "block: product workspace too small");
  const float beta = c != nullptr ? 1.f : 0.f;
  if (d.bf16)
    return nmb_gemm_bf16(la, lb, m, n, k, 1.f, a, lda, b, ldb, beta, c, n, out, n, need ? ws : nullptr, need, s);
  return nmb_gemm_f32_split(la, lb, m, n, k, 1.f, static_cast<const float*>(a), lda, static_cast<const float*>(b),
                            ldb, beta, static_cast<const float*>(c), n, static_cast<float*>(out), n,
                            need ? ws : nullptr, need, s);
}

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

int forward_ws(const Dims& d, int64_t* bytes) {
  int64_t o = 0, down = 0, qkv = 0, gu = 0;
  NMB_TRY(gemm_ws(d, 0, 0, d.T, d.H, d.Nq, &o));
  NMB_TRY(gemm_ws(d, 0, 0, d.T, d.H, d.F, &down));
  if (!d.bf16) {
    NMB_TRY(gemm_ws(d, 0, 0, d.T, d.N, d.H, &qkv));
    NMB_TRY(gemm_ws(d, 0, 0, d.T, 2 * d.F, d.H, &gu));
  }
  *bytes = std::max(std::max(o, down), std::max(qkv, gu));
  return NMB_OK;
}

// The backward's scratch: byte offsets of its parts in one buffer.  What only
// the main stream reads and writes shares its place with what comes before or
// after it there: dn2 (until the post-attention norm) with dqkv, do2 (until the
// attention) with dn1, fp32's [g|u] and ds (until the SwiGLU backward) with all
// of these, and the workspaces of the main stream's products, the attention and
// the input norm with each other.  The second stream reads dgu, act, ws_side
// and ws_post until it is joined, so those keep theirs.  (All parts side by
// side: 374 MB against 338 for 16 x 512 tokens of hidden 1024, 635 against 499
// for 4 x 2048 of hidden 2048.)
struct BwdScratch {
  int64_t dgu, act, dn2, dh, do2, dqkv, dn1, gu, ds, attn, ws_main, ws_side, ws_post, ws_in, total;
  int64_t main_bytes, side_bytes, attn_bytes, norm_bytes;
};

int backward_scratch(const nmb_block* b, const Dims& d, BwdScratch* s) {
  int64_t m[6] = {0, 0, 0, 0, 0, 0}, side[2] = {0, 0};
  NMB_TRY(gemm_ws(d, 1, 1, d.H, d.F, d.T, &side[0]));
  NMB_TRY(gemm_ws(d, 1, 1, 2 * d.F, d.H, d.T, &side[1]));
  NMB_TRY(gemm_ws(d, 0, 1, d.T, d.H, 2 * d.F, &m[0]));
  NMB_TRY(gemm_ws(d, 0, 1, d.T, d.Nq, d.H, &m[1]));
  NMB_TRY(gemm_ws(d, 1, 1, d.H, d.Nq, d.T, &m[2]));
  NMB_TRY(gemm_ws(d, 0, 1, d.T, d.H, d.N, &m[3]));
  NMB_TRY(gemm_ws(d, 1, 1, d.N, d.H, d.T, &m[4]));
  if (!d.bf16) {
    int64_t gu = 0, ds = 0;
    NMB_TRY(gemm_ws(d, 0, 0, d.T, 2 * d.F, d.H, &gu));
    NMB_TRY(gemm_ws(d, 0, 1, d.T, d.F, d.H, &ds));
    m[5] = std::max(gu, ds);
  }
  size_t attn = 0, norm = 0;
  NMB_TRY(nmb_attn_bwd_workspace_bytes_split(b->batch, b->q_heads, b->kv_heads, b->seq, b->seq, b->head_dim, 1,
                                             b->dtype, &attn));
  NMB_TRY(nmb_rmsnorm_bwd_workspace_bytes(d.T, d.H, &norm));
  s->main_bytes = *std::max_element(m, m + 6);
  s->side_bytes = std::max(side[0], side[1]);
  s->attn_bytes = static_cast<int64_t>(attn);
  s->norm_bytes = static_cast<int64_t>(norm);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t off = at;
    at += align256(bytes);
    return off;
  };
  s->dgu = take(d.T * 2 * d.F * d.es);
  s->act = take(d.T * d.F * d.es);
  s->gu = at;
  s->ds = s->gu + align256(d.T * 2 * d.F * d.es);
  s->dh = take(d.T * d.H * d.es);
  s->do2 = s->dn1 = take(d.T * std::max(d.Nq, d.H) * d.es);
  s->dqkv = s->dn2 = take(d.T * std::max(d.N, d.H) * d.es);
  if (!d.bf16) at = std::max(at, s->ds + align256(d.T * d.F * d.es));
  s->attn = s->ws_main = s->ws_in = take(std::max(std::max(s->attn_bytes, s->main_bytes), s->norm_bytes));
  s->ws_side = take(s->side_bytes);
  s->ws_post = take(s->norm_bytes);
  s->total = at;
  return NMB_OK;
}

// `waiter` waits for what `other` holds so far
int stream_wait(hipStream_t waiter, hipStream_t other) {
  hipEvent_t ev = nullptr;
  hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e == hipSuccess) {
    e = hipEventRecord(ev, other);
    if (e == hipSuccess) e = hipStreamWaitEvent(waiter, ev, 0);
    const hipError_t e2 = hipEventDestroy(ev);
    if (e == hipSuccess) e = e2;
  }
  if (e != hipSuccess) {
    nmb::set_error("block: ordering two streams failed: %s", hipGetErrorString(e));
    return NMB_EHIP;
  }
  return NMB_OK;
}

const char* at(const void* p, int64_t bytes) { return static_cast<const char*>(p) + bytes; }
char* at(void* p, int64_t bytes) { return static_cast<char*>(p) + bytes; }

}  // namespace

extern "C" int nmb_block_sizes(const nmb_block* b, int64_t* forward_workspace, int64_t* backward_bytes) {
  Dims d;
  NMB_TRY(block_dims(b, &d));
  if (forward_workspace != nullptr) NMB_TRY(forward_ws(d, forward_workspace));
  if (backward_bytes != nullptr) {
    BwdScratch s;
    NMB_TRY(backward_scratch(b, d, &s));
    *backward_bytes = s.total;
  }
  return NMB_OK;
}

extern "C" int nmb_block_attention(const nmb_block* b, const void* n1, void* qkv, void* o, float* lse,
                                   void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  Dims d;
  NMB_TRY(block_dims(b, &d));
  NMB_REQUIRE(qkv != nullptr, "block: null tensor");
  const int64_t heads = b->q_heads + b->kv_heads;
  const int64_t qs[3] = {b->seq * d.N, d.N, b->head_dim}, os[3] = {b->seq * d.Nq, d.Nq, b->head_dim};
  if (d.bf16) {
    NMB_TRY(nmb_gemm_bf16_rope(0, d.T, d.N, d.H, n1, d.H, b->w_qkv, d.H, qkv, d.N, b->cos_table, b->sin_table,
                               b->n_pos, b->positions, b->pos_batch_stride, b->pos_offset, b->seq, b->head_dim,
                               heads * b->head_dim, stream));
  } else {
    NMB_TRY(gemm(d, 0, 0, d.T, d.N, d.H, n1, d.H, b->w_qkv, d.H, nullptr, qkv, workspace, workspace_bytes, stream));
    NMB_TRY(nmb_rope_apply(qkv, qkv, b->cos_table, b->sin_table, b->n_pos, b->positions, b->pos_batch_stride,
                           b->pos_offset, b->batch, b->seq, heads, b->head_dim, qs, qs, 0, b->dtype, stream));
  }
  const void* k[1] = {at(qkv, d.Nq * d.es)};
  const void* v[1] = {at(qkv, (d.Nq + d.Nk) * d.es)};
  const int64_t koff[1] = {0};
  return nmb_attn_fwd(qkv, k, v, koff, 1, o, lse, b->batch, b->q_heads, b->kv_heads, b->seq, b->seq, b->head_dim, qs,
                      qs, os, 1, b->q_offset, 0.f, b->dtype, stream);
}

extern "C" int nmb_block_forward(const nmb_block* b, const void* x, void* n1, void* qkv, void* o, float* lse, void* h,
                                 void* n2, void* gu, void* act, void* y, void* workspace, int64_t workspace_bytes,
                                 hipStream_t stream) {
  Dims d;
  NMB_TRY(block_dims(b, &d));
  NMB_REQUIRE(y == nullptr || act != nullptr, "block_forward: y needs the activation");
  NMB_REQUIRE(d.bf16 || act == nullptr || gu != nullptr, "block_forward (fp32): the activation needs gu");
  NMB_TRY(nmb_rmsnorm_fwd(x, b->w_in, n1, nullptr, d.T, d.H, b->eps, b->dtype, stream));
  NMB_TRY(nmb_block_attention(b, n1, qkv, o, lse, workspace, workspace_bytes, stream));
  NMB_TRY(gemm(d, 0, 0, d.T, d.H, d.Nq, o, d.Nq, b->w_o, d.Nq, x, h, workspace, workspace_bytes, stream));
  NMB_TRY(nmb_rmsnorm_fwd(h, b->w_post, n2, nullptr, d.T, d.H, b->eps, b->dtype, stream));
  if (gu == nullptr && act == nullptr) return NMB_OK;
  if (d.bf16) {
    NMB_TRY(nmb_gemm_bf16_swiglu(d.T, d.F, d.H, n2, d.H, b->w_gu, d.H, act, d.F, gu, 2 * d.F, stream));
  } else {
    NMB_TRY(gemm(d, 0, 0, d.T, 2 * d.F, d.H, n2, d.H, b->w_gu, d.H, nullptr, gu, workspace, workspace_bytes, stream));
    if (act != nullptr)
      NMB_TRY(nmb_swiglu_fwd(gu, 2 * d.F, at(gu, d.F * d.es), 2 * d.F, act, d.F, d.T, d.F, b->dtype, stream));
  }
  if (y == nullptr) return NMB_OK;
  return gemm(d, 0, 0, d.T, d.H, d.F, act, d.F, b->w_d, d.F, h, y, workspace, workspace_bytes, stream);
}

extern "C" int nmb_block_backward_mlp(const nmb_block* b, const void* dy, const void* o, const void* h, const void* n2,
                                      const void* gu, void* dw_o, void* dw_post, void* dw_gu, void* dw_d,
                                      void* scratch, int64_t scratch_bytes, int captured, hipStream_t stream,
                                      hipStream_t side) {
  Dims d;
  BwdScratch s;
  NMB_TRY(block_dims(b, &d));
  NMB_TRY(backward_scratch(b, d, &s));
  NMB_REQUIRE(scratch != nullptr && scratch_bytes >= s.total, "block_backward: scratch of %lld bytes is too small",
              (long long)scratch_bytes);
  void *dgu = at(scratch, s.dgu), *act = at(scratch, s.act), *dn2 = at(scratch, s.dn2), *dh = at(scratch, s.dh);
  void *ws = at(scratch, s.ws_main), *ws_post = at(scratch, s.ws_post), *ws_side = at(scratch, s.ws_side);
  const bool two = side != stream;
  // MLP: y = h + s Wd^T, s = silu(g) * u, [g|u] = n2 [Wg;Wu]^T.  ds = dY Wd and
  // the SwiGLU backward in one product (bf16; without a kept [g|u] the same
  // kernel first forms it for its tile, with the forward's bits).
  if (d.bf16) {
    if (gu != nullptr)
      NMB_TRY(nmb_gemm_bf16_swiglu_bwd(1, d.T, d.F, d.H, dy, d.H, b->w_d, d.F, gu, 2 * d.F, dgu, 2 * d.F, act, d.F,
                                       stream));
    else
      NMB_TRY(nmb_gemm_bf16_gate_up_swiglu_bwd(d.T, d.F, d.H, n2, d.H, b->w_gu, d.H, d.H, dy, d.H, 1, b->w_d, d.F,
                                               dgu, 2 * d.F, act, d.F, stream));
  } else {
    if (gu == nullptr) {
      void* g = at(scratch, s.gu);
      NMB_TRY(gemm(d, 0, 0, d.T, 2 * d.F, d.H, n2, d.H, b->w_gu, d.H, nullptr, g, ws, s.main_bytes, stream));
      gu = g;
    }
    void* ds = at(scratch, s.ds);
    NMB_TRY(gemm(d, 0, 1, d.T, d.F, d.H, dy, d.H, b->w_d, d.F, nullptr, ds, ws, s.main_bytes, stream));
    NMB_TRY(nmb_swiglu_bwd(gu, 2 * d.F, at(gu, d.F * d.es), 2 * d.F, ds, d.F, dgu, 2 * d.F, at(dgu, d.F * d.es),
                           2 * d.F, act, d.F, d.T, d.F, b->dtype, stream));
  }
  auto weight_gu = [&]() {
    return gemm(d, 1, 1, 2 * d.F, d.H, d.T, dgu, 2 * d.F, n2, d.H, nullptr, dw_gu, ws_side, s.side_bytes, side);
  };
  if (two) NMB_TRY(stream_wait(side, stream));
  NMB_TRY(gemm(d, 1, 1, d.H, d.F, d.T, dy, d.H, act, d.F, nullptr, dw_d, ws_side, s.side_bytes, side));
  if (captured) NMB_TRY(weight_gu());
  NMB_TRY(gemm(d, 0, 1, d.T, d.H, 2 * d.F, dgu, 2 * d.F, b->w_gu, d.H, nullptr, dn2, ws, s.main_bytes, stream));
  if (!captured) {
    if (two) NMB_TRY(stream_wait(side, stream));
    NMB_TRY(weight_gu());
  }
  NMB_TRY(nmb_rmsnorm_bwd_rows(h, b->w_post, dn2, dy, dh, ws_post, s.norm_bytes, d.T, d.H, b->eps, b->dtype, stream));
  const bool sum_on_side = two && !captured;
  if (sum_on_side) NMB_TRY(stream_wait(side, stream));
  NMB_TRY(nmb_rmsnorm_bwd_dw(ws_post, s.norm_bytes, d.T, d.H, dw_post, b->dtype, sum_on_side ? side : stream));
  // attention: h = x + o Wo^T
  NMB_TRY(gemm(d, 0, 1, d.T, d.Nq, d.H, dh, d.H, b->w_o, d.Nq, nullptr, at(scratch, s.do2), ws, s.main_bytes,
               stream));
  return gemm(d, 1, 1, d.H, d.Nq, d.T, dh, d.H, o, d.Nq, nullptr, dw_o, ws, s.main_bytes, stream);
}

extern "C" int nmb_block_backward_attention(const nmb_block* b, const void* x, const void* n1, const void* qkv,
                                            const void* o, const float* lse, void* dx, void* dw_in, void* dw_qkv,
                                            void* scratch, int64_t scratch_bytes, hipStream_t stream) {
  Dims d;
  BwdScratch s;
  NMB_TRY(block_dims(b, &d));
  NMB_TRY(backward_scratch(b, d, &s));
  NMB_REQUIRE(scratch != nullptr && scratch_bytes >= s.total, "block_backward: scratch of %lld bytes is too small",
              (long long)scratch_bytes);
  void *dqkv = at(scratch, s.dqkv), *dn1 = at(scratch, s.dn1), *ws = at(scratch, s.ws_main);
  const void* k = at(qkv, d.Nq * d.es);
  const void* v = at(qkv, (d.Nq + d.Nk) * d.es);
  void *dk = at(dqkv, d.Nq * d.es), *dv = at(dqkv, (d.Nq + d.Nk) * d.es);
  const int64_t qs[3] = {b->seq * d.N, d.N, b->head_dim}, os[3] = {b->seq * d.Nq, d.Nq, b->head_dim};
  // attention backward with the RoPE backward of q and k (bf16: in its stores)
  if (d.bf16) {
    NMB_TRY(nmb_attn_bwd_rope(qkv, k, v, o, at(scratch, s.do2), lse, dqkv, dk, dv, at(scratch, s.attn),
                              static_cast<size_t>(s.attn_bytes), b->batch, b->q_heads, b->kv_heads, b->seq,
                              b->head_dim, qs, qs, os, 1, b->q_offset, 0.f, b->cos_table, b->sin_table, b->n_pos,
                              b->positions, b->pos_batch_stride, b->pos_offset, stream));
  } else {
    const void *kb[1] = {k}, *vb[1] = {v};
    void *dkb[1] = {dk}, *dvb[1] = {dv};
    const int64_t koff[1] = {0};
    NMB_TRY(nmb_attn_bwd(qkv, kb, vb, koff, 1, o, at(scratch, s.do2), lse, dqkv, dkb, dvb, at(scratch, s.attn),
                         static_cast<size_t>(s.attn_bytes), b->batch, b->q_heads, b->kv_heads, b->seq, b->seq,
                         b->head_dim, qs, qs, os, 1, b->q_offset, 0.f, b->dtype, stream));
    NMB_TRY(nmb_rope_apply(dqkv, dqkv, b->cos_table, b->sin_table, b->n_pos, b->positions, b->pos_batch_stride,
                           b->pos_offset, b->batch, b->seq, b->q_heads + b->kv_heads, b->head_dim, qs, qs, 1,
                           b->dtype, stream));
  }
  NMB_TRY(gemm(d, 0, 1, d.T, d.H, d.N, dqkv, d.N, b->w_qkv, d.H, nullptr, dn1, ws, s.main_bytes, stream));
  NMB_TRY(gemm(d, 1, 1, d.N, d.H, d.T, dqkv, d.N, n1, d.H, nullptr, dw_qkv, ws, s.main_bytes, stream));
  return nmb_rmsnorm_bwd(x, b->w_in, dn1, at(scratch, s.dh), dx, dw_in, at(scratch, s.ws_in),
                         static_cast<size_t>(s.norm_bytes), d.T, d.H, b->eps, b->dtype, stream);
}

extern "C" int nmb_stream_join(hipStream_t stream, hipStream_t other) {
  if (stream == other) return NMB_OK;
  return stream_wait(stream, other);
}
