// fp32 GEMM on the fp32 MFMA (v_mfma_f32_16x16x4_f32) for gfx950.
//
// The dense projections of the fp32 parity configuration (reference
// nn.Linear / F.linear at nn/kernels/torch_backend.py:19-20 and
// tensor_parallel/layers.py:214, and their autograd products, in fp32):
//   D[M, N] = alpha * op(A)[M, K] * op(B)[K, N] + beta * C[M, N]   (row-major)
// with the operand layouts of nmb_gemm_bf16 (A [M, K] or [K, M]; B [N, K] or
// [K, N]), any shape, leading dimension and alignment.  Every product is an
// exact fp32 product accumulated in fp32 by the matrix core, so results agree
// with an fp32 reference GEMM to the rounding of the summation order.
//
// Workgroup tile 64 x 64, four wavefronts of 32 x 32 (2 x 2 MFMA tiles), K
// tiles of 32 double-buffered in LDS, the next tile's global loads in flight
// during the current one's 32 MFMAs per wave.  Both operands are kept as rows
// of 32 k (36 floats apart, so the rows of a fragment read spread over the
// banks), and a lane reads four consecutive k at once: lane group q supplies
// k = 16 j + 4 q + e to the e-th MFMA of step j for A and B alike, which sums
// the same products in a fixed order.  M/N-contiguous operands are transposed
// on the way into LDS.  Each MFMA computes a D^T tile (B fragment as the A
// operand), so a lane holds four consecutive columns of one row of D.
//
// What bounds it: the smoke configuration's products (512 tokens, K 256 to
// 8192) are a few tens of tiles of 64 x 64, so launch and memory latency and
// idle CUs, not the 256 FLOP per clock and CU of the fp32 matrix core.  The K
// range is therefore split over workgroups until about two per CU run, with
// the partial products (caller's workspace) summed in split order by a second
// launch.  Over the 64 products of one smoke-configuration step (4 x 128
// tokens, forward and backward): 0.62 ms and 0.27 ms of sums, against 4.95 ms
// with 16-deep single-buffered tiles of element loads and no split (512 x 256
// x 8192 alone 1.4 ms on its 32 workgroups).
#include <algorithm>

#include "common.h"

namespace nmb {
namespace {

constexpr int kTile = 64;
constexpr int kKT = 32;
constexpr int kRow = kKT + 4;  // floats between rows in LDS

struct GemmF32Args {
  const float* a;
  const float* b;
  const float* c;
  float* d;
  float* partial;  // split K: [splits][M][N]
  int64_t lda, ldb, ldc, ldd;
  int M, N, K;
  float alpha, beta;
  int kps;               // K range of a split (a multiple of kKT, or K)
  int vec_a, vec_b;      // 16-byte loads allowed (base and leading dimension)
  int vec_c, vec_d;      // the same for C and D (and the partial rows: vec_p)
  int vec_p;
};

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// One thread's 2 x 4 consecutive elements of a 64 x 32 operand tile: rows r0
// .. (valid up to rows), k range [k0, k_end).  KC: stored [row][k], each group
// of 4 along k; else stored [k][row], along the row dimension.  Elements
// outside read as zeros.
template <bool KC>
struct TileLoad {
  f32x4 v[2];
  __device__ __forceinline__ void load(const float* p, int64_t ld, int r0, int rows, int k0, int k_end, bool vec) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int idx = static_cast<int>(threadIdx.x) + 256 * j;
      if (KC) {
        const int r = r0 + idx / (kKT / 4), k = k0 + 4 * (idx % (kKT / 4));
        v[j] = group(p + static_cast<int64_t>(r) * ld + k, r < rows ? k_end - k : 0, vec);
      } else {
        const int k = k0 + idx / (kTile / 4), r = r0 + 4 * (idx % (kTile / 4));
        v[j] = group(p + static_cast<int64_t>(k) * ld + r, k < k_end ? rows - r : 0, vec);
      }
    }
  }
  // p[0..3], the first n of them (n may be negative or above 4)
  __device__ static f32x4 group(const float* p, int n, bool vec) {
    if (vec && n >= 4) return *reinterpret_cast<const f32x4*>(p);
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) o[e] = p[e];
    return o;
  }
  __device__ __forceinline__ void store(float (*s)[kRow]) const {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int idx = static_cast<int>(threadIdx.x) + 256 * j;
      if (KC) {
        *reinterpret_cast<f32x4*>(&s[idx / (kKT / 4)][4 * (idx % (kKT / 4))]) = v[j];
      } else {
        const int k = idx / (kTile / 4), r = 4 * (idx % (kTile / 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) s[r + e][k] = v[j][e];
      }
    }
  }
};

// row[n .. n + 3] = v (+ beta * c[..]), the columns below N
__device__ __forceinline__ void store_row(float* row, const float* crow, float beta, f32x4 v, int n, int N, bool vec,
                                          bool vec_c) {
  if (n >= N) return;
  if (n + 3 < N && vec && (crow == nullptr || vec_c)) {
    if (crow != nullptr) {
      const f32x4 c = *reinterpret_cast<const f32x4*>(crow + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += beta * c[e];
    }
    *reinterpret_cast<f32x4*>(row + n) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) row[n + e] = crow != nullptr ? v[e] + beta * crow[n + e] : v[e];
}

// A_KC: A stored [M, K] (K contiguous), else [K, M].  B_KC: B stored [N, K],
// else [K, N].  blockIdx: (column tile, row tile, split).
template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmF32Args g) {
  __shared__ __attribute__((aligned(16))) float sA[2][kTile][kRow];
  __shared__ __attribute__((aligned(16))) float sB[2][kTile][kRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  const int m0 = static_cast<int>(blockIdx.y) * kTile;
  const int n0 = static_cast<int>(blockIdx.x) * kTile;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int k_begin = static_cast<int>(blockIdx.z) * g.kps;
  const int k_end = min(g.K, k_begin + g.kps);

  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  TileLoad<A_KC> la;
  TileLoad<B_KC> lb;
  la.load(g.a, g.lda, m0, g.M, k_begin, k_end, g.vec_a);
  lb.load(g.b, g.ldb, n0, g.N, k_begin, k_end, g.vec_b);
  int buf = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += kKT, buf ^= 1) {
    // the buffer last read two tiles ago: every wave has passed the barrier since
    la.store(sA[buf]);
    lb.store(sB[buf]);
    __syncthreads();
    if (k0 + kKT < k_end) {
      la.load(g.a, g.lda, m0, g.M, k0 + kKT, k_end, g.vec_a);
      lb.load(g.b, g.ldb, n0, g.N, k0 + kKT, k_end, g.vec_b);
    }
#pragma unroll
    for (int j16 = 0; j16 < kKT; j16 += 16) {
      f32x4 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[i] = *reinterpret_cast<const f32x4*>(&sA[buf][wm + 16 * i + l16][j16 + 4 * q]);
        fb[i] = *reinterpret_cast<const f32x4*>(&sB[buf][wn + 16 * i + l16][j16 + 4 * q]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f32(fb[j][e], fa[i][e], acc[i][j]);
    }
  }

  // acc[i][j][e] = D[m0 + wm + 16 i + l16][n0 + wn + 16 j + 4 q + e]
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm + 16 * i + l16;
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn + 16 * j + 4 * q;
      if (g.partial != nullptr) {
        float* row = g.partial + (static_cast<int64_t>(blockIdx.z) * g.M + m) * g.N;
        store_row(row, nullptr, 0.f, acc[i][j], n, g.N, g.vec_p, false);
      } else {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = g.alpha * acc[i][j][e];
        const float* crow = g.beta != 0.f ? g.c + static_cast<int64_t>(m) * g.ldc : nullptr;
        store_row(g.d + static_cast<int64_t>(m) * g.ldd, crow, g.beta, v, n, g.N, g.vec_d, g.vec_c);
      }
    }
  }
}

// D = alpha * (sum of the splits' partials, in order) + beta * C; a thread
// takes four columns.
__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(GemmF32Args g, int splits) {
  const int groups = (g.N + 3) / 4;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<int64_t>(g.M) * groups) return;
  const int m = static_cast<int>(idx / groups), n = 4 * static_cast<int>(idx % groups);
  const int cnt = min(4, g.N - n);
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) {
    const float* p = g.partial + (static_cast<int64_t>(s) * g.M + m) * g.N + n;
    const f32x4 t = TileLoad<true>::group(p, cnt, g.vec_p);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += t[e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= g.alpha;
  const float* crow = g.beta != 0.f ? g.c + static_cast<int64_t>(m) * g.ldc : nullptr;
  store_row(g.d + static_cast<int64_t>(m) * g.ldd, crow, g.beta, v, n, g.N, g.vec_d, g.vec_c);
}

// K range of a split: with fewer than 512 tiles (two workgroups per CU) as
// many splits as bring the launch near that, each of 64 k at least (two K
// tiles: shorter ones spend more on the partials than the idle CUs cost) and
// 32 at most (the reduction reads one partial per split one after the other).
int split_k(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + kTile - 1) / kTile) * ((n + kTile - 1) / kTile);
  int64_t want = tiles > 0 ? std::min<int64_t>(512 / tiles, 32) : 1;
  want = std::min(want, k / 64);
  if (want <= 1) return static_cast<int>(k);
  const int64_t kps = ((k + want - 1) / want + kKT - 1) / kKT * kKT;
  return static_cast<int>(kps);
}

bool vec_ok(const float* p, int64_t ld) { return aligned16(p) && ld % 4 == 0; }

int gemm_f32(int a_layout, int b_layout, int64_t m, int64_t n, int64_t k, float alpha, const float* a, int64_t lda,
             const float* b, int64_t ldb, float beta, const float* c, int64_t ldc, float* d, int64_t ldd,
             float* workspace, int64_t workspace_bytes, hipStream_t stream) {
  NMB_REQUIRE(a_layout == 0 || a_layout == 1, "gemm_f32: a_layout must be 0 ([M,K]) or 1 ([K,M])");
  NMB_REQUIRE(b_layout == 0 || b_layout == 1, "gemm_f32: b_layout must be 0 ([N,K]) or 1 ([K,N])");
  NMB_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m < (1 << 30) && n < (1 << 30) && k < (1 << 30),
              "gemm_f32: invalid shape %lld x %lld x %lld", (long long)m, (long long)n, (long long)k);
  NMB_REQUIRE(d != nullptr && (k == 0 || (a != nullptr && b != nullptr)), "gemm_f32: null operand");
  NMB_REQUIRE(beta == 0.f || c != nullptr, "gemm_f32: beta != 0 needs C");
  const bool a_kc = a_layout == 0, b_kc = b_layout == 0;
  NMB_REQUIRE(lda >= (a_kc ? k : m) && ldb >= (b_kc ? k : n) && ldd >= n && (beta == 0.f || ldc >= n),
              "gemm_f32: leading dimension too small");
  if (m == 0 || n == 0) return NMB_OK;
  const int64_t gy = (m + kTile - 1) / kTile, gx = (n + kTile - 1) / kTile;
  NMB_REQUIRE(gy <= 65535 && gx < (int64_t{1} << 31), "gemm_f32: problem too large for one launch");
  GemmF32Args g{};
  g.a = a;
  g.b = b;
  g.c = c;
  g.d = d;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.ldd = ldd;
  g.M = static_cast<int>(m);
  g.N = static_cast<int>(n);
  g.K = static_cast<int>(k);
  g.alpha = alpha;
  g.beta = beta;
  g.kps = workspace != nullptr ? split_k(m, n, k) : static_cast<int>(k);
  const int splits = g.kps > 0 ? static_cast<int>((k + g.kps - 1) / g.kps) : 1;
  if (splits > 1) {
    NMB_REQUIRE(workspace_bytes >= static_cast<int64_t>(splits) * m * n * 4 && aligned16(workspace),
                "gemm_f32: workspace of %lld bytes is too small or not 16-byte aligned", (long long)workspace_bytes);
    g.partial = workspace;
  }
  g.vec_a = vec_ok(a, lda);
  g.vec_b = vec_ok(b, ldb);
  g.vec_c = vec_ok(c, ldc);
  g.vec_d = vec_ok(d, ldd);
  g.vec_p = n % 4 == 0;
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy), static_cast<unsigned>(splits));
  if (a_kc && b_kc) hipLaunchKernelGGL((gemm_f32_kernel<true, true>), grid, dim3(256), 0, stream, g);
  else if (a_kc) hipLaunchKernelGGL((gemm_f32_kernel<true, false>), grid, dim3(256), 0, stream, g);
  else if (b_kc) hipLaunchKernelGGL((gemm_f32_kernel<false, true>), grid, dim3(256), 0, stream, g);
  else hipLaunchKernelGGL((gemm_f32_kernel<false, false>), grid, dim3(256), 0, stream, g);
  if (splits > 1) {
    const int64_t blocks = (m * ((n + 3) / 4) + 255) / 256;
    hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, g, splits);
  }
  NMB_CHECK_LAUNCH("gemm_f32");
  return NMB_OK;
}

}  // namespace
}  // namespace nmb

extern "C" int nmb_gemm_f32(int a_layout, int b_layout, int64_t m, int64_t n, int64_t k, float alpha,
                            const float* a, int64_t lda, const float* b, int64_t ldb, float beta,
                            const float* c, int64_t ldc, float* d, int64_t ldd, hipStream_t stream) {
  return nmb::gemm_f32(a_layout, b_layout, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, d, ldd, nullptr, 0, stream);
}

extern "C" int nmb_gemm_f32_workspace_bytes(int64_t m, int64_t n, int64_t k, int64_t* bytes) {
  NMB_REQUIRE(bytes != nullptr, "gemm_f32_workspace_bytes: null output");
  NMB_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m < (1 << 30) && n < (1 << 30) && k < (1 << 30),
              "gemm_f32: invalid shape %lld x %lld x %lld", (long long)m, (long long)n, (long long)k);
  const int64_t kps = nmb::split_k(m, n, k);
  const int64_t splits = kps > 0 ? (k + kps - 1) / kps : 1;
  *bytes = splits > 1 ? splits * m * n * 4 : 0;
  return NMB_OK;
}

extern "C" int nmb_gemm_f32_split(int a_layout, int b_layout, int64_t m, int64_t n, int64_t k, float alpha,
                                  const float* a, int64_t lda, const float* b, int64_t ldb, float beta,
                                  const float* c, int64_t ldc, float* d, int64_t ldd, void* workspace,
                                  int64_t workspace_bytes, hipStream_t stream) {
  return nmb::gemm_f32(a_layout, b_layout, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, d, ldd,
                       static_cast<float*>(workspace), workspace_bytes, stream);
}
