// Learned collision surrogate for gfx950: Hermite-mode encoder/decoder of
// velocity distributions, a 4-layer spectral network (forward, backward and
// Adam in HIP, GEMMs on MFMA with BF16 operands and FP32 accumulation), and
// the surrogate-with-fallback evaluation of Q(f).
//
// Representation.  A point's distribution f on the Nv^3 grid is described in
// the frame of its own Maxwellian M[f] (density rho, velocity u, temperature
// T from the discrete moments; DGFS convention M = rho (pi T)^-3/2
// exp(-|c-u|^2/T), so the per-axis variance is s^2 = T/2).  With
// c' = (c - u)/s and the probabilists' Hermite polynomials He_n, the 8^3
// retained modes a_n (n = (nx, ny, nz), n_d < 8) are the coefficients of f/M0
// (M0 the Gaussian factor of M) in the grid-orthonormal basis phi_n spanned by
// psi_n = prod_d He_{n_d}(c'_d)/sqrt(n_d!) exp(-c'_d^2/2) (the span of Grad's
// expansion f ~ M sum_n b_n psi_n; equilibrium maps to a = 0).  The basis
// decays like M, so round-off far in the tails never reaches the modes, and
// the modes' Euclidean norm is the grid L2 norm of the represented field.  The collision
// operator's modes b_n (same projection of Q) scale as prefac rho T^{gamma/2}
// in the continuum, so the network maps the dimensionless a to
// b^ = b / (prefac rho T^{gamma/2}).
// Network (8^3 = 512 modes m, width 32 channels c, activations Z[m][p][c]):
//   Z0[m][p][c] = P0[c] x[p][m] + P1[c] log T[p] + E[m][c]
//   U_l = K_l Z_l            (mode mixing, K_l 512x512, one GEMM over all points)
//   V_l = U_l W_l + Z_l R_l + bias_l     (channel mixing, W_l, R_l 32x32)
//   Z_{l+1} = GELU(V_l) for l < 3, Z_4 = V_3
//   out[p][m] = sum_c Z_4[m][p][c] Pout[c] + bout[m]
// Fallback: points whose non-equilibrium indicator ||f - M[f]|| / ||f||
// exceeds a threshold are evaluated by the exact spectral operator.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <optional>
#include <vector>

#include "common.hpp"
#include "spectral.hpp"

namespace dgfs {

constexpr int kSurD = 8;                    // Hermite degrees per axis
constexpr int kSurModes = kSurD * kSurD * kSurD;
constexpr int kSurWidth = 32;
constexpr int kSurLayers = 4;
constexpr long kSurLayerSize = static_cast<long>(kSurModes) * kSurModes + 2L * kSurWidth * kSurWidth + kSurWidth;
constexpr long kSurOffP0 = 0, kSurOffP1 = kSurWidth, kSurOffE = 2 * kSurWidth;
constexpr long kSurOffLayers = kSurOffE + static_cast<long>(kSurModes) * kSurWidth;
constexpr long kSurOffPout = kSurOffLayers + kSurLayers * kSurLayerSize;
constexpr long kSurOffBout = kSurOffPout + kSurWidth;
constexpr long kSurParams = kSurOffBout + kSurModes;

// ---------------------------------------------------------------------------
// GEMM  C[M][N] = alpha op(A)[M][K] op(B)[K][N] + beta C, row-major FP32
// storage; op(A)[m][k] = A[m*lda + k] or (transA) A[k*lda + m], likewise B.
// BF16: operands rounded to bfloat16, v_mfma_f32_16x16x16bf16_1k; else FP32
// operands on v_mfma_f32_16x16x4f32.  64x64 block tile, 4 waves of 32x32,
// K staged through LDS 32 at a time.  Split-K writes raw partial products to
// part[z][M][N] (reduced by k_gemm_reduce).
// ---------------------------------------------------------------------------
struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  float* part;
  long lda, ldb, ldc;
  int transA, transB, M, N, K, kchunk;
  float alpha, beta;
};

typedef short sh4 __attribute__((ext_vector_type(4)));
typedef float fl4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short to_bf16(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return static_cast<short>(u >> 16);
}

constexpr int kGT = 64, kGK = 32, kGPad = kGT + 4;

template <bool BF16>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ float As[kGK][kGPad];
  __shared__ float Bs[kGK][kGPad];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.y * kGT, n0 = blockIdx.x * kGT;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int kbeg = blockIdx.z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  fl4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = fl4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = kbeg; k0 < kend; k0 += kGK) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = tid + 256 * i;
      int mm, kk;
      if (g.transA) { mm = e & 63; kk = e >> 6; } else { kk = e & 31; mm = e >> 5; }
      const int gm = m0 + mm, gk = k0 + kk;
      float v = 0.f;
      if (gm < g.M && gk < kend) v = g.transA ? g.A[static_cast<long>(gk) * g.lda + gm] : g.A[static_cast<long>(gm) * g.lda + gk];
      As[kk][mm] = v;
      int nn, kb;
      if (g.transB) { kb = e & 31; nn = e >> 5; } else { nn = e & 63; kb = e >> 6; }
      const int gn = n0 + nn, gkb = k0 + kb;
      float w = 0.f;
      if (gn < g.N && gkb < kend) w = g.transB ? g.B[static_cast<long>(gn) * g.ldb + gkb] : g.B[static_cast<long>(gkb) * g.ldb + gn];
      Bs[kb][nn] = w;
    }
    __syncthreads();
    if constexpr (BF16) {
#pragma unroll
      for (int s = 0; s < kGK / 16; ++s) {
        sh4 av[2], bv[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            av[t][j] = to_bf16(As[s * 16 + 4 * lg + j][wm + t * 16 + li]);
            bv[t][j] = to_bf16(Bs[s * 16 + 4 * lg + j][wn + t * 16 + li]);
          }
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[a], bv[b], acc[a][b], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int s = 0; s < kGK / 4; ++s) {
        float av[2], bv[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          av[t] = As[s * 4 + lg][wm + t * 16 + li];
          bv[t] = Bs[s * 4 + lg][wn + t * 16 + li];
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a], bv[b], acc[a][b], 0, 0, 0);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + a * 16 + 4 * lg + r, col = n0 + wn + b * 16 + li;
        if (row < g.M && col < g.N) {
          if (g.part) {
            g.part[(static_cast<long>(blockIdx.z) * g.M + row) * g.N + col] = acc[a][b][r];
          } else {
            float* cp = g.C + static_cast<long>(row) * g.ldc + col;
            const float v = g.alpha * acc[a][b][r];
            *cp = (g.beta == 0.f) ? v : v + g.beta * *cp;
          }
        }
      }
}

// Large-tile BF16 variant: 128x128 block tile, 4 waves of 64x64 (4 x 4 MFMA
// tiles each), K staged 32 at a time as BF16 in K-contiguous LDS rows
// (As[m][k], Bs[n][k]) so every MFMA operand is one 8-byte LDS read.  Used
// when both output dimensions are >= 128.
constexpr int kBT = 128, kBK = 32, kBKP = kBK + 4;

template <int UNUSED>
__global__ __launch_bounds__(256) void k_gemm_bf16_big(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) short As[kBT][kBKP];
  __shared__ __attribute__((aligned(16))) short Bs[kBT][kBKP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.y * kBT, n0 = blockIdx.x * kBT;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const int kbeg = blockIdx.z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  fl4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = fl4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = kbeg; k0 < kend; k0 += kBK) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = tid + 256 * i;  // 4096 elements of each tile
      int mm, kk;
      if (g.transA) { mm = e & 127; kk = e >> 7; } else { kk = e & 31; mm = e >> 5; }
      const int gm = m0 + mm, gk = k0 + kk;
      float v = 0.f;
      if (gm < g.M && gk < kend)
        v = g.transA ? g.A[static_cast<long>(gk) * g.lda + gm] : g.A[static_cast<long>(gm) * g.lda + gk];
      As[mm][kk] = to_bf16(v);
      int nn, kb;
      if (g.transB) { kb = e & 31; nn = e >> 5; } else { nn = e & 127; kb = e >> 7; }
      const int gn = n0 + nn, gkb = k0 + kb;
      float w = 0.f;
      if (gn < g.N && gkb < kend)
        w = g.transB ? g.B[static_cast<long>(gn) * g.ldb + gkb] : g.B[static_cast<long>(gkb) * g.ldb + gn];
      Bs[nn][kb] = to_bf16(w);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kBK / 16; ++s) {
      sh4 av[4], bv[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        av[t] = *reinterpret_cast<const sh4*>(&As[wm + t * 16 + li][s * 16 + 4 * lg]);
        bv[t] = *reinterpret_cast<const sh4*>(&Bs[wn + t * 16 + li][s * 16 + 4 * lg]);
      }
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[a], bv[b], acc[a][b], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + a * 16 + 4 * lg + r, col = n0 + wn + b * 16 + li;
        if (row < g.M && col < g.N) {
          if (g.part) {
            g.part[(static_cast<long>(blockIdx.z) * g.M + row) * g.N + col] = acc[a][b][r];
          } else {
            float* cp = g.C + static_cast<long>(row) * g.ldc + col;
            const float v = g.alpha * acc[a][b][r];
            *cp = (g.beta == 0.f) ? v : v + g.beta * *cp;
          }
        }
      }
}

// Large-tile FP32 variant: 128 x 64 block tile, 4 waves of 64 x 32 (4 x 2 MFMA
// tiles), K 32 at a time in K-contiguous LDS rows (As[m][k], Bs[n][k], padded
// to 36 floats), double buffered: the next tile is in flight in registers
// while one is multiplied, one barrier per tile.  A lane reads four
// consecutive k of a row as one 16-byte value and gives MFMA step j the value
// k = 4 g + j of its lane group g, for A and B alike, so the four steps of a
// read cover 16 k in another order than step by step.  Two workgroups (55 KB of
// LDS each) share a CU.  For outputs of at least 128 x 64 with 16-byte
// aligned operands; the 64 x 64 kernel above stages every value through a
// bounds-checked scalar load and two barriers per 32 k and ran the network's
// products (512 x 32 P x 512) at 39 TFLOP/s on MI355X, this one at 83 (P =
// 256) to 86 (P = 1000), 71 with op(A) = A^T.
constexpr int kFM = 128, kFN = 64, kFK = 32, kFP = kFK + 4;

// this thread's share of an R x 32 operand tile (R rows of op(A) or columns of
// op(B)): R * 32 / 4 / 256 vectors of 4 consecutive k of one row.  KC: k is the
// contiguous index in memory, read as vectors; else the lanes run along the
// rows and read k by k, so that the LDS stores are 16-byte rows either way
// (vectors along the rows would be scattered into LDS with 16-way conflicts).
template <int R, bool KC>
__device__ __forceinline__ void gemm_load(const float* __restrict__ X, long ld, int r0, int rows, int k0, int kend,
                                          fl4 (&v)[R / 32]) {
#pragma unroll
  for (int i = 0; i < R / 32; ++i) {
    const int e = threadIdx.x + 256 * i;
    const int r = KC ? e >> 3 : e % R, k = KC ? (e & 7) * 4 : (e / R) * 4;
    const int gr = r0 + r, gk = k0 + k;
    const float* p = KC ? X + static_cast<long>(gr) * ld + gk : X + static_cast<long>(gk) * ld + gr;
    const int left = gr < rows ? kend - gk : 0;  // values of k that exist
    if (left >= 4) {
      if constexpr (KC) {
        v[i] = *reinterpret_cast<const fl4*>(p);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = p[j * ld];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = (j < left) ? p[KC ? j : j * ld] : 0.f;
    }
  }
}
template <int R, bool KC>
__device__ __forceinline__ void gemm_store(float (*T)[kFP], const fl4 (&v)[R / 32]) {
#pragma unroll
  for (int i = 0; i < R / 32; ++i) {
    const int e = threadIdx.x + 256 * i;
    const int r = KC ? e >> 3 : e % R, k = KC ? (e & 7) * 4 : (e / R) * 4;
    *reinterpret_cast<fl4*>(&T[r][k]) = v[i];
  }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void k_gemm_f32_big(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float As[2][kFM][kFP];
  __shared__ __attribute__((aligned(16))) float Bs[2][kFN][kFP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.y * kFM, n0 = blockIdx.x * kFN;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 32;
  const int kbeg = blockIdx.z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  fl4 acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = fl4{0.f, 0.f, 0.f, 0.f};
  fl4 va[kFM / 32], vb[kFN / 32];
  gemm_load<kFM, !TA>(g.A, g.lda, m0, g.M, kbeg, kend, va);
  gemm_load<kFN, TB>(g.B, g.ldb, n0, g.N, kbeg, kend, vb);
  gemm_store<kFM, !TA>(As[0], va);
  gemm_store<kFN, TB>(Bs[0], vb);
  __syncthreads();
  int cur = 0;
  for (int k0 = kbeg; k0 < kend; k0 += kFK, cur ^= 1) {
    const bool more = k0 + kFK < kend;
    if (more) {
      gemm_load<kFM, !TA>(g.A, g.lda, m0, g.M, k0 + kFK, kend, va);
      gemm_load<kFN, TB>(g.B, g.ldb, n0, g.N, k0 + kFK, kend, vb);
    }
#pragma unroll
    for (int s = 0; s < kFK / 16; ++s) {
      fl4 av[4], bv[2];
#pragma unroll
      for (int t = 0; t < 4; ++t) av[t] = *reinterpret_cast<const fl4*>(&As[cur][wm + t * 16 + li][s * 16 + 4 * lg]);
#pragma unroll
      for (int t = 0; t < 2; ++t) bv[t] = *reinterpret_cast<const fl4*>(&Bs[cur][wn + t * 16 + li][s * 16 + 4 * lg]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a][j], bv[b][j], acc[a][b], 0, 0, 0);
    }
    if (more) {  // the other buffer: its readers passed the last barrier
      gemm_store<kFM, !TA>(As[cur ^ 1], va);
      gemm_store<kFN, TB>(Bs[cur ^ 1], vb);
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + a * 16 + 4 * lg + r, col = n0 + wn + b * 16 + li;
        if (row < g.M && col < g.N) {
          if (g.part) {
            g.part[(static_cast<long>(blockIdx.z) * g.M + row) * g.N + col] = acc[a][b][r];
          } else {
            float* cp = g.C + static_cast<long>(row) * g.ldc + col;
            const float v = g.alpha * acc[a][b][r];
            *cp = (g.beta == 0.f) ? v : v + g.beta * *cp;
          }
        }
      }
}

__global__ __launch_bounds__(256) void k_gemm_reduce(const float* __restrict__ part, int splits, int M, int N,
                                                     float alpha, float beta, float* C, long ldc) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<long>(M) * N) return;
  float s = 0.f;
  for (int z = 0; z < splits; ++z) s += part[static_cast<long>(z) * M * N + i];
  const int row = static_cast<int>(i / N), col = static_cast<int>(i % N);
  float* cp = C + static_cast<long>(row) * ldc + col;
  *cp = (beta == 0.f) ? alpha * s : alpha * s + beta * *cp;
}

// split-K partials: up to 256 / tiles splits of an M x N output; the weight
// gradients (512 x 512 from K = 32 * batch, 32 x 32 from K = 512 * batch)
// need at most 16 M floats.  Allocated once at that size and never resized
// while work may be in flight; a split that would not fit runs unsplit.
constexpr size_t kGemmPartFloats = size_t{1} << 24;
constexpr int kGemmSplitK = 512;  // shortest reduction that any shape splits
struct GemmWs {
  float* part = nullptr;
  // a workspace that calls on several streams and threads share: a product
  // waits on the device for the reduction of the one before (event `done`),
  // and the mutex keeps wait, launches and record of one call together
  bool shared = false;
  std::mutex mu;
  hipEvent_t done = nullptr;
  int init() {
    if (!part) DGFS_HIP_TRY(hipMalloc(&part, kGemmPartFloats * sizeof(float)));
    if (shared && !done) DGFS_HIP_TRY(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    return DGFS_OK;
  }
  ~GemmWs() {
    (void)hipFree(part);
    if (done) (void)hipEventDestroy(done);
  }
};

// one split product's hold on the workspace, from before its launch to after
// its reduction's
class GemmWsUse {
 public:
  GemmWsUse(GemmWs* ws, hipStream_t st) : ws_(ws), st_(st) {
    if (ws_->shared) lock_ = std::unique_lock<std::mutex>(ws_->mu);
  }
  GemmWsUse(const GemmWsUse&) = delete;
  GemmWsUse& operator=(const GemmWsUse&) = delete;
  int begin() {
    int rc = ws_->init();
    if (rc || !ws_->shared) return rc;
    DGFS_HIP_TRY(hipStreamWaitEvent(st_, ws_->done, 0));
    held_ = true;
    return DGFS_OK;
  }
  ~GemmWsUse() {
    if (held_ && hipEventRecord(ws_->done, st_) != hipSuccess) (void)hipStreamSynchronize(st_);
  }

 private:
  GemmWs* ws_;
  hipStream_t st_;
  std::unique_lock<std::mutex> lock_;
  bool held_ = false;
};

// the current device's workspace for products without a handle, or null on a
// stream under capture: the replays of the graph would not be ordered against
// other calls, so a captured product runs unsplit
static GemmWs* shared_gemm_ws(hipStream_t st) {
  constexpr int kMaxDev = 64;
  static std::mutex mu;
  static GemmWs* table[kMaxDev] = {};  // process-lifetime (released by the driver at exit)
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  int dev = 0;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess || hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (cap != hipStreamCaptureStatusNone || dev < 0 || dev >= kMaxDev) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!table[dev]) {
    table[dev] = new (std::nothrow) GemmWs();
    if (table[dev]) table[dev]->shared = true;
  }
  return table[dev];
}

static int gemm(GemmWs* ws, int transA, int transB, int M, int N, int K, float alpha, const float* A, long lda,
                const float* B, long ldb, float beta, float* C, long ldc, bool bf16, hipStream_t st) {
  if (M <= 0 || N <= 0) return DGFS_OK;
  if (bf16 && M >= kBT && N >= kBT) {
    // large outputs: 128x128 tiles; split K when the output has few tiles
    GemmArgs g{A, B, C, nullptr, lda, ldb, ldc, transA, transB, M, N, K, K, alpha, beta};
    const int gx = (N + kBT - 1) / kBT, gy = (M + kBT - 1) / kBT, tiles = gx * gy;
    int splits = 1;
    if (tiles < 256 && K > 4096) splits = std::min(256 / tiles, (K + 2047) / 2048);
    if (splits > 1 && ws) {
      int kchunk = (K + splits - 1) / splits;
      kchunk = (kchunk + kBK - 1) / kBK * kBK;
      splits = (K + kchunk - 1) / kchunk;
      if (static_cast<size_t>(splits) * M * N > kGemmPartFloats) splits = 1;
      else {
        GemmWsUse use(ws, st);
        int rc = use.begin();
        if (rc) return rc;
        g.kchunk = kchunk;
        g.part = ws->part;
        hipLaunchKernelGGL(k_gemm_bf16_big<0>, dim3(gx, gy, splits), dim3(256), 0, st, g);
        DGFS_LAUNCH_CHECK("gemm_big(split)");
        const long tot = static_cast<long>(M) * N;
        hipLaunchKernelGGL(k_gemm_reduce, dim3(static_cast<unsigned>((tot + 255) / 256)), dim3(256), 0, st,
                           ws->part, splits, M, N, alpha, beta, C, ldc);
        DGFS_LAUNCH_CHECK("gemm_reduce");
        return DGFS_OK;
      }
    }
    hipLaunchKernelGGL(k_gemm_bf16_big<0>, dim3(gx, gy, 1), dim3(256), 0, st, g);
    DGFS_LAUNCH_CHECK("gemm_big");
    return DGFS_OK;
  }
  GemmArgs g{A, B, C, nullptr, lda, ldb, ldc, transA, transB, M, N, K, K, alpha, beta};
  const bool aligned = reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 &&
                       lda % 4 == 0 && ldb % 4 == 0;
  if (!bf16 && M >= kFM && N >= kFN && aligned && (M + kFM - 1) / kFM <= 65535) {
    // large FP32 outputs; K is split while the tiles are fewer than two per
    // CU, into chunks of at least 256 (the reduction then reads the partials)
    const int bx = (N + kFN - 1) / kFN, by = (M + kFM - 1) / kFM;
    const long tl = static_cast<long>(bx) * by, want = 2L * cu_count();
    int splits = 1;
    std::optional<GemmWsUse> use;
    if (ws && tl < want && K >= kGemmSplitK) splits = static_cast<int>(std::min<long>(want / tl, K / 256));
    if (splits > 1) {
      int kchunk = (K + splits - 1) / splits;
      kchunk = (kchunk + kFK - 1) / kFK * kFK;
      splits = (K + kchunk - 1) / kchunk;
      if (splits > 1 && static_cast<size_t>(splits) * M * N <= kGemmPartFloats) {
        use.emplace(ws, st);
        int rc = use->begin();
        if (rc) return rc;
        g.kchunk = kchunk;
        g.part = ws->part;
      } else {
        splits = 1;
      }
    }
    const dim3 grid(bx, by, splits);
    if (transA && transB)
      hipLaunchKernelGGL((k_gemm_f32_big<true, true>), grid, dim3(256), 0, st, g);
    else if (transA)
      hipLaunchKernelGGL((k_gemm_f32_big<true, false>), grid, dim3(256), 0, st, g);
    else if (transB)
      hipLaunchKernelGGL((k_gemm_f32_big<false, true>), grid, dim3(256), 0, st, g);
    else
      hipLaunchKernelGGL((k_gemm_f32_big<false, false>), grid, dim3(256), 0, st, g);
    DGFS_LAUNCH_CHECK("gemm_f32");
    if (splits > 1) {
      const long tot = static_cast<long>(M) * N;
      hipLaunchKernelGGL(k_gemm_reduce, dim3(static_cast<unsigned>((tot + 255) / 256)), dim3(256), 0, st, ws->part,
                         splits, M, N, alpha, beta, C, ldc);
      DGFS_LAUNCH_CHECK("gemm_reduce");
    }
    return DGFS_OK;
  }
  const int gx = (N + kGT - 1) / kGT, gy = (M + kGT - 1) / kGT;
  // split the reduction when the output has few tiles and K is long
  int splits = 1;
  const int tiles = gx * gy;
  if (tiles < 256 && K > 4096) splits = std::min(256 / tiles, (K + 2047) / 2048);
  if (splits > 1 && ws) {
    int kchunk = (K + splits - 1) / splits;
    kchunk = (kchunk + kGK - 1) / kGK * kGK;
    splits = (K + kchunk - 1) / kchunk;
    if (static_cast<size_t>(splits) * M * N > kGemmPartFloats)
      return fail(DGFS_ERR_INVALID_VALUE, "split-K workspace too small");
    GemmWsUse use(ws, st);
    int rc = use.begin();
    if (rc) return rc;
    g.kchunk = kchunk;
    g.part = ws->part;
    if (bf16)
      hipLaunchKernelGGL(k_gemm<true>, dim3(gx, gy, splits), dim3(256), 0, st, g);
    else
      hipLaunchKernelGGL(k_gemm<false>, dim3(gx, gy, splits), dim3(256), 0, st, g);
    DGFS_LAUNCH_CHECK("gemm(split)");
    const long tot = static_cast<long>(M) * N;
    hipLaunchKernelGGL(k_gemm_reduce, dim3(static_cast<unsigned>((tot + 255) / 256)), dim3(256), 0, st,
                       ws->part, splits, M, N, alpha, beta, C, ldc);
    DGFS_LAUNCH_CHECK("gemm_reduce");
    return DGFS_OK;
  }
  if (bf16)
    hipLaunchKernelGGL(k_gemm<true>, dim3(gx, gy, 1), dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL(k_gemm<false>, dim3(gx, gy, 1), dim3(256), 0, st, g);
  DGFS_LAUNCH_CHECK("gemm");
  return DGFS_OK;
}

// ---------------------------------------------------------------------------
// network elementwise kernels (activations Z[m][p][c], c fastest)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float gelu(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  return 0.5f * x * (1.f + tanhf(k0 * (x + k1 * x * x * x)));
}
__device__ __forceinline__ float gelu_d(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  const float t = tanhf(k0 * (x + k1 * x * x * x));
  return 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * k0 * (1.f + 3.f * k1 * x * x);
}

__global__ __launch_bounds__(256) void k_lift_fwd(const float* __restrict__ th, const float* __restrict__ x,
                                                  const float* __restrict__ lt, float* __restrict__ Z, int P) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const long tot = static_cast<long>(kSurModes) * P * kSurWidth;
  if (i >= tot) return;
  const int c = static_cast<int>(i % kSurWidth);
  const long mp = i / kSurWidth;
  const int p = static_cast<int>(mp % P), m = static_cast<int>(mp / P);
  Z[i] = th[kSurOffP0 + c] * x[static_cast<long>(p) * kSurModes + m] + th[kSurOffP1 + c] * lt[p] +
         th[kSurOffE + m * kSurWidth + c];
}

// V += bias; Z = act(V) (act = GELU or identity); V keeps the pre-activation
__global__ __launch_bounds__(256) void k_bias_act(float* __restrict__ V, const float* __restrict__ bias,
                                                  float* __restrict__ Z, long tot, int act) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= tot) return;
  const float v = V[i] + bias[i % kSurWidth];
  V[i] = v;
  Z[i] = act ? gelu(v) : v;
}

__global__ __launch_bounds__(256) void k_head_fwd(const float* __restrict__ th, const float* __restrict__ Z,
                                                  float* __restrict__ out, int P) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;  // over (m, p)
  if (i >= static_cast<long>(kSurModes) * P) return;
  const int p = static_cast<int>(i % P), m = static_cast<int>(i / P);
  const float* z = Z + i * kSurWidth;
  float s = th[kSurOffBout + m];
#pragma unroll
  for (int c = 0; c < kSurWidth; ++c) s += z[c] * th[kSurOffPout + c];
  out[static_cast<long>(p) * kSurModes + m] = s;
}

__global__ __launch_bounds__(256) void k_head_bwd(const float* __restrict__ th, const float* __restrict__ dout,
                                                  float* __restrict__ dZ, int P) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const long tot = static_cast<long>(kSurModes) * P * kSurWidth;
  if (i >= tot) return;
  const int c = static_cast<int>(i % kSurWidth);
  const long mp = i / kSurWidth;
  const int p = static_cast<int>(mp % P), m = static_cast<int>(mp / P);
  dZ[i] = dout[static_cast<long>(p) * kSurModes + m] * th[kSurOffPout + c];
}

__global__ __launch_bounds__(256) void k_act_bwd(const float* __restrict__ V, float* __restrict__ dZ, long tot) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= tot) return;
  dZ[i] *= gelu_d(V[i]);
}

// One layer's channel mixing with FP32 operands, fused:
//   V = U W + Z R + bias, Znext = act(V)
// over the rows (m, p) of U and Z.  A wave takes 32 rows: the rows are the A
// operand of v_mfma_f32_16x16x4f32 (lane i of a group holds row i, channels
// 16 h + 4 g + j as one 16-byte load), W and R stay in registers as B.  Bound by
// reading U, Z and writing V, Znext once; as two products and an elementwise
// pass V was written three times and read twice (P = 256: 42 -> 16 us per
// layer on MI355X).
constexpr int kLayRows = 32;

// B operand values of a 32 x 32 matrix X (transposed: X^T) for column tile t:
// step (h, j) takes row 16 h + 4 g + j
template <bool TR>
__device__ __forceinline__ void chan_operand(const float* __restrict__ X, int li, int lg, float (&b)[2][8]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int row = 16 * (k >> 2) + 4 * lg + (k & 3), col = 16 * t + li;
      b[t][k] = TR ? X[col * kSurWidth + row] : X[row * kSurWidth + col];
    }
}

__global__ __launch_bounds__(256) void k_layer_fwd(const float* __restrict__ U, const float* __restrict__ Z,
                                                   const float* __restrict__ W, const float* __restrict__ R,
                                                   const float* __restrict__ bias, float* __restrict__ V,
                                                   float* __restrict__ Zn, long rows, int act) {
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  float bw[2][8], br[2][8], bb[2];
  chan_operand<false>(W, li, lg, bw);
  chan_operand<false>(R, li, lg, br);
#pragma unroll
  for (int t = 0; t < 2; ++t) bb[t] = bias[16 * t + li];
  const long nw = static_cast<long>(gridDim.x) * 4, nt = rows / kLayRows;
  for (long w = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6); w < nt; w += nw) {
    const long r0 = w * kLayRows;
    fl4 u[2][2], z[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const long o = (r0 + 16 * a + li) * kSurWidth + 16 * h + 4 * lg;
        u[a][h] = *reinterpret_cast<const fl4*>(U + o);
        z[a][h] = *reinterpret_cast<const fl4*>(Z + o);
      }
    // U W and Z R in sums of their own, added last: one chain through both was 5 %
    // further from 64 bits (forward of 256 points 6.8e-7 against 6.5e-7)
    fl4 acc[2][2], acz[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[a][t] = acz[a][t] = fl4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[a][k >> 2][k & 3], bw[t][k], acc[a][t], 0, 0, 0);
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acz[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(z[a][k >> 2][k & 3], br[t][k], acz[a][t], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const long o = (r0 + 16 * a + 4 * lg + r) * kSurWidth + 16 * t + li;
          const float v = (acc[a][t][r] + acz[a][t][r]) + bb[t];
          V[o] = v;
          Zn[o] = act ? gelu(v) : v;
        }
  }
}

// The same layer backward, fused: with dV = dZ act'(V) (act = 0: dV = dZ)
//   dU = dV W^T, dZn = dV R^T, and the block's partial sums of
//   gW = U^T dV, gR = Z^T dV, gb = sum dV over its rows.
// dV is formed twice in registers, as A operand (rows on lanes) for dU and dZn
// and as B operand (channels on lanes) for the weight gradients; nothing but
// dU and dZn is written per row.  part[block][2 * 32 * 32 + 32]; the partials
// are summed by k_sum_parts, in a fixed order.  As separate kernels the weight
// gradients were 32 x 32 products over 512 P rows on 64 workgroups: 670 us per
// layer at P = 256 on MI355X, 39 us fused.
constexpr int kLayPart = 2 * kSurWidth * kSurWidth + kSurWidth;

__global__ __launch_bounds__(256) void k_layer_bwd(const float* __restrict__ dZ, const float* __restrict__ V,
                                                   const float* __restrict__ U, const float* __restrict__ Z,
                                                   const float* __restrict__ W, const float* __restrict__ R,
                                                   float* __restrict__ dU, float* __restrict__ dZn,
                                                   float* __restrict__ part, long rows, int act) {
  __shared__ float red[kLayPart];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4, wave = threadIdx.x >> 6;
  float bw[2][8], br[2][8];
  chan_operand<true>(W, li, lg, bw);
  chan_operand<true>(R, li, lg, br);
  fl4 gw[2][2], gr[2][2];  // [channel tile of U / Z][channel tile of dV]
  float gb[2] = {0.f, 0.f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < 2; ++t) gw[a][t] = gr[a][t] = fl4{0.f, 0.f, 0.f, 0.f};
  const long nw = static_cast<long>(gridDim.x) * 4, nt = rows / kLayRows;
  for (long w = static_cast<long>(blockIdx.x) * 4 + wave; w < nt; w += nw) {
    const long r0 = w * kLayRows;
    {
      fl4 dv[2][2];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const long o = (r0 + 16 * a + li) * kSurWidth + 16 * h + 4 * lg;
          dv[a][h] = *reinterpret_cast<const fl4*>(dZ + o);
          if (act) {
            const fl4 v = *reinterpret_cast<const fl4*>(V + o);
#pragma unroll
            for (int j = 0; j < 4; ++j) dv[a][h][j] *= gelu_d(v[j]);
          }
        }
      fl4 au[2][2], az[2][2];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t) au[a][t] = az[a][t] = fl4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const float d = dv[a][k >> 2][k & 3];
            au[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(d, bw[t][k], au[a][t], 0, 0, 0);
            az[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(d, br[t][k], az[a][t], 0, 0, 0);
          }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const long o = (r0 + 16 * a + 4 * lg + r) * kSurWidth + 16 * t + li;
            dU[o] = au[a][t][r];
            dZn[o] = az[a][t][r];
          }
    }
    // rows 4 s + g on the k index, channels on the lanes
#pragma unroll
    for (int s = 0; s < kLayRows / 4; ++s) {
      float d[2], u[2], z[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const long o = (r0 + 4 * s + lg) * kSurWidth + 16 * t + li;
        d[t] = dZ[o];
        if (act) d[t] *= gelu_d(V[o]);
        u[t] = U[o];
        z[t] = Z[o];
        gb[t] += d[t];
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          gw[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[a], d[t], gw[a][t], 0, 0, 0);
          gr[a][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(z[a], d[t], gr[a][t], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    gb[t] += __shfl_xor(gb[t], 16);
    gb[t] += __shfl_xor(gb[t], 32);
  }
  for (int w = 0; w < 4; ++w) {  // the waves in turn
    if (wave == w) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int o = (16 * a + 4 * lg + r) * kSurWidth + 16 * t + li;
            red[o] = (w ? red[o] : 0.f) + gw[a][t][r];
            red[kSurWidth * kSurWidth + o] = (w ? red[kSurWidth * kSurWidth + o] : 0.f) + gr[a][t][r];
          }
      if (lg == 0)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int o = 2 * kSurWidth * kSurWidth + 16 * t + li;
          red[o] = (w ? red[o] : 0.f) + gb[t];
        }
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < kLayPart; i += 256) part[static_cast<long>(blockIdx.x) * kLayPart + i] = red[i];
}

// Per-channel and per-mode reductions of the backward pass, two stages
// (block partials, then one block) so the sums are deterministic.
//   kind 0: out[c]     = sum_{m,p} X[m][p][c]                 (bias)
//   kind 1: out[c]     = sum_{m,p} X[m][p][c] Y[m][p][c]      (Pout)
//   kind 2: out[c]     = sum_{m,p} X[m][p][c] x[p][m]          (P0)
//   kind 3: out[c]     = sum_{m,p} X[m][p][c] lt[p]            (P1)
struct ChanRedArgs {
  const float* X;
  const float* Y;   // kind 1
  const float* xin; // kind 2: [P][512]
  const float* lt;  // kind 3: [P]
  const float* dout; // unused
  float* part;      // [gridDim.x][32]
  int P, kind;
};

__global__ __launch_bounds__(256) void k_chan_reduce(ChanRedArgs a) {
  __shared__ float red[8][kSurWidth];
  const int c = threadIdx.x & 31, row = threadIdx.x >> 5;  // 8 rows of 32 channels
  const long rows = static_cast<long>(kSurModes) * a.P;
  float s = 0.f;
  for (long r = static_cast<long>(blockIdx.x) * 8 + row; r < rows; r += static_cast<long>(gridDim.x) * 8) {
    const long i = r * kSurWidth + c;
    float v = a.X[i];
    if (a.kind == 1) {
      v *= a.Y[i];
    } else if (a.kind == 2) {
      const int p = static_cast<int>(r % a.P), m = static_cast<int>(r / a.P);
      v *= a.xin[static_cast<long>(p) * kSurModes + m];
    } else if (a.kind == 3) {
      v *= a.lt[r % a.P];
    }
    s += v;
  }
  red[row][c] = s;
  __syncthreads();
  if (row == 0) {
    float t = 0.f;
    for (int k = 0; k < 8; ++k) t += red[k][c];
    a.part[static_cast<long>(blockIdx.x) * kSurWidth + c] = t;
  }
}

// out[c] = sum_k part[k][c]: 32 columns per block, 32 rows of threads over k,
// then the rows in order (one thread per column summed 240 partials one after
// another: 54 us, 5 us this way)
__global__ __launch_bounds__(1024) void k_sum_parts(const float* __restrict__ part, int nparts, int width,
                                                   float* __restrict__ out) {
  __shared__ float red[32][33];
  const int lc = threadIdx.x & 31, row = threadIdx.x >> 5, c = blockIdx.x * 32 + lc;
  float s = 0.f;
  if (c < width)
    for (int k = row; k < nparts; k += 32) s += part[static_cast<long>(k) * width + c];
  red[row][lc] = s;
  __syncthreads();
  if (row == 0 && c < width) {
    float t = 0.f;
    for (int k = 0; k < 32; ++k) t += red[k][lc];
    out[c] = t;
  }
}

// dE[m][c] = sum_p dZ0[m][p][c]: a block per mode, 8 rows of threads over p
__global__ __launch_bounds__(256) void k_mode_reduce(const float* __restrict__ dZ, float* __restrict__ out, int P) {
  __shared__ float red[8][kSurWidth];
  const int c = threadIdx.x & 31, row = threadIdx.x >> 5, m = blockIdx.x;
  float s = 0.f;
  for (int p = row; p < P; p += 8) s += dZ[(static_cast<long>(m) * P + p) * kSurWidth + c];
  red[row][c] = s;
  __syncthreads();
  if (row == 0) {
    float t = 0.f;
    for (int k = 0; k < 8; ++k) t += red[k][c];
    out[m * kSurWidth + c] = t;
  }
}

// dbout[m] = sum_p dout[p][m]: 32 modes per block, 32 rows of threads over p
__global__ __launch_bounds__(1024) void k_bout_reduce(const float* __restrict__ dout, float* __restrict__ out, int P) {
  __shared__ float red[32][33];
  const int lm = threadIdx.x & 31, row = threadIdx.x >> 5, m = blockIdx.x * 32 + lm;
  float s = 0.f;
  for (int p = row; p < P; p += 32) s += dout[static_cast<long>(p) * kSurModes + m];
  red[row][lm] = s;
  __syncthreads();
  if (row == 0) {
    float t = 0.f;
    for (int k = 0; k < 32; ++k) t += red[k][lm];
    out[m] = t;
  }
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ th, const float* __restrict__ g,
                                              float* __restrict__ m1, float* __restrict__ m2, long n, float lr,
                                              float b1, float b2, float eps, float c1, float c2) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  th[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// dst = BF16 rounding (nearest even) of src, kept in FP32 storage: the
// network's BF16 weights, used with FP32 activations on the FP32 MFMA
__global__ __launch_bounds__(256) void k_round_bf16(const float* __restrict__ src, float* __restrict__ dst, long n) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned u = static_cast<unsigned>(static_cast<unsigned short>(to_bf16(src[i]))) << 16;
  dst[i] = __uint_as_float(u);
}

// ---------------------------------------------------------------------------
// Hermite encoder / decoder (FP64), one workgroup per point
// ---------------------------------------------------------------------------
struct EncArgs {
  const double* f;  // [npts][n]
  double* mom;      // [npts][8]: rho, ux, uy, uz, T, indicator, high-mode indicator, 0
  float* x;         // [npts][512] a_n (a_000 replaced by 0), or null
  float* lt;        // [npts] log T, or null
  double L, cw;
  int npts;
};

// 1/sqrt(a!): the basis uses He_a / sqrt(a!), which keeps the per-axis Gram
// matrices well conditioned (about 1e3 instead of 4e4 at degree 7)
__constant__ double kInvSqrtFact[kSurD] = {1.0, 1.0, 0.70710678118654752, 0.40824829046386302,
                                           0.20412414523193151, 0.091287092917527686, 0.037267799624996495,
                                           0.014085904245475275};

// V[i*8 + a] = He_a(x_i) / sqrt(a!) exp(-x_i^2 / 2), x_i = (c0 + i h - u) / s:
// the 1D factors of the basis functions (exp(-x^2/2) = exp(-(c-u)^2/T))
__device__ __forceinline__ void herm_table(double* V, double c0, double h, double u, double s, int N) {
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    const double x = (c0 + i * h - u) / s, w = exp(-0.5 * x * x);
    double p0 = 1.0, p1 = x;
    V[i * kSurD + 0] = w * p0 * kInvSqrtFact[0];
    V[i * kSurD + 1] = w * p1 * kInvSqrtFact[1];
    for (int a = 1; a + 1 < kSurD; ++a) {
      const double p2 = x * p1 - a * p0;
      V[i * kSurD + a + 1] = w * p2 * kInvSqrtFact[a + 1];
      p0 = p1;
      p1 = p2;
    }
  }
}

// totals of NQ values per thread over a workgroup of NT threads; red holds
// NT / 64 * NQ doubles and is free on return
template <int NQ, int NT>
__device__ __forceinline__ void block_sums(double (&s)[NQ], double* red) {
#pragma unroll
  for (int j = 0; j < NQ; ++j)
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s[j] += __shfl_xor(s[j], d);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int j = 0; j < NQ; ++j) red[(threadIdx.x >> 6) * NQ + j] = s[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) t += red[w * NQ + j];
    s[j] = t;
  }
  __syncthreads();
}

// Linv[d] = L_d^{-1}, L_d the Cholesky factor of the per-axis Gram matrix
// G_d = (h/s) V_d^T V_d (work holds 3 x 8 x 8 doubles).  The Gram sums take a
// thread each; the 8 x 8 factorisation is one thread per axis in registers
// (with its operands in LDS every step waited for the one before: the encoder
// spent a third of its time there).
// The 1D functions V_d L_d^{-T} are orthonormal on the grid with the measure
// dx' = h/s, so their tensor products are orthonormal in 3D.
template <int N>
__device__ void herm_chol_inv(const double* V, double hs, double* Linv, double* work) {
  for (int e = threadIdx.x; e < 3 * kSurD * kSurD; e += blockDim.x) {
    const int d = e / (kSurD * kSurD), a = (e / kSurD) % kSurD, b = e % kSurD;
    if (b > a) continue;
    const double* Vd = V + d * N * kSurD;
    double s = 0.0;
    for (int i = 0; i < N; ++i) s += Vd[i * kSurD + a] * Vd[i * kSurD + b];
    work[e] = s * hs;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double G[kSurD][kSurD], rd[kSurD];
#pragma unroll
    for (int a = 0; a < kSurD; ++a)
#pragma unroll
      for (int b = 0; b <= a; ++b) G[a][b] = work[threadIdx.x * kSurD * kSurD + a * kSurD + b];
#pragma unroll
    for (int b = 0; b < kSurD; ++b) {
#pragma unroll
      for (int k = 0; k < b; ++k) G[b][b] -= G[b][k] * G[b][k];
      rd[b] = 1.0 / sqrt(fmax(G[b][b], 1e-300));
#pragma unroll
      for (int a = b + 1; a < kSurD; ++a) {
#pragma unroll
        for (int k = 0; k < b; ++k) G[a][b] -= G[a][k] * G[b][k];
        G[a][b] *= rd[b];
      }
    }
    // forward substitution for the inverse of the lower triangle
    double* Li = Linv + threadIdx.x * kSurD * kSurD;
#pragma unroll
    for (int c = 0; c < kSurD; ++c) {
      double x[kSurD];
#pragma unroll
      for (int a = 0; a < kSurD; ++a) {
        double t = (a == c) ? 1.0 : 0.0;
#pragma unroll
        for (int k = c; k < a; ++k) t -= G[a][k] * x[k];
        x[a] = (a < c) ? 0.0 : t * rd[a];
        Li[a * kSurD + c] = x[a];
      }
    }
  }
  __syncthreads();
}

// Apply A_x (x) A_y (x) A_z to the 8^3 block `in` (A_d = Linv_d, or its
// transpose when `transpose`), through `tmp`; result in `out` (may alias in).
__device__ void kron3(const double* Linv, bool transpose, double* in, double* tmp, double* out) {
  auto A = [&](int d, int r, int c) {
    return transpose ? Linv[d * kSurD * kSurD + c * kSurD + r] : Linv[d * kSurD * kSurD + r * kSurD + c];
  };
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x) {
    const int a = e / (kSurD * kSurD), bc = e % (kSurD * kSurD);
    double s = 0.0;
    for (int q = 0; q < kSurD; ++q) s += A(0, a, q) * in[q * kSurD * kSurD + bc];
    tmp[e] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x) {
    const int a = e / (kSurD * kSurD), b = (e / kSurD) % kSurD, c = e % kSurD;
    double s = 0.0;
    for (int q = 0; q < kSurD; ++q) s += A(1, b, q) * tmp[(a * kSurD + q) * kSurD + c];
    in[e] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x) {
    const int ab = e / kSurD, c = e % kSurD;
    double s = 0.0;
    for (int q = 0; q < kSurD; ++q) s += A(2, c, q) * in[ab * kSurD + q];
    tmp[e] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x) out[e] = tmp[e];
  __syncthreads();
}

// Coefficients of g / C in the grid-orthonormal basis phi_n (tensor products
// of V_d L_d^{-T}), divided by `scale`:
//   c = (Lx^-1 (x) Ly^-1 (x) Lz^-1) (h/s)^3 sum_r g(r) V_x V_y V_z / (C scale).
// ||c|| is the grid L2 norm (measure dx'^3) of the part of g / (C scale) in
// the span, so the modes stay bounded and a mean-square error of the modes is
// the L2 error of the decoded field.
template <int N>
__device__ void herm_project_rest(const double* V, const double* Linv, double* t1, double* t2, double* b3,
                                  double factor, float* out, float shift0);

template <int N>
__device__ void herm_project(const double* __restrict__ g, const double* V, const double* Linv, double* t1,
                             double* t2, double* b3, double factor, float* out, float shift0) {
  constexpr int NN = N * N;
  const double* Vx = V;
  // t1[a][j][k]: each thread owns columns jk and reads every g value once,
  // accumulating all kSurD x-modes of it
  for (int jk = threadIdx.x; jk < NN; jk += blockDim.x) {
    double acc[kSurD];
#pragma unroll
    for (int a = 0; a < kSurD; ++a) acc[a] = 0.0;
    for (int i = 0; i < N; ++i) {
      const double gv = g[i * NN + jk];
#pragma unroll
      for (int a = 0; a < kSurD; ++a) acc[a] += gv * Vx[i * kSurD + a];
    }
#pragma unroll
    for (int a = 0; a < kSurD; ++a) t1[a * NN + jk] = acc[a];
  }
  herm_project_rest<N>(V, Linv, t1, t2, b3, factor, out, shift0);
}

// the other two axes of the projection, from t1[a][j][k] (not yet synchronised)
template <int N>
__device__ void herm_project_rest(const double* V, const double* Linv, double* t1, double* t2, double* b3,
                                  double factor, float* out, float shift0) {
  constexpr int NN = N * N;
  const double* Vy = V + N * kSurD;
  const double* Vz = V + 2 * N * kSurD;
  __syncthreads();
  for (int e = threadIdx.x; e < kSurD * kSurD * N; e += blockDim.x) {  // t2[a][b][k]
    const int a = e / (kSurD * N), rem = e - a * kSurD * N, b = rem / N, k = rem - b * N;
    double s = 0.0;
    for (int j = 0; j < N; ++j) s += t1[a * NN + j * N + k] * Vy[j * kSurD + b];
    t2[e] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x) {  // B[a][b][c] -> b3
    const int ab = e / kSurD, c = e % kSurD;
    double s = 0.0;
    for (int k = 0; k < N; ++k) s += t2[ab * N + k] * Vz[k * kSurD + c];
    b3[e] = s * factor;
  }
  __syncthreads();
  kron3(Linv, false, b3, t1, b3);
  for (int e = threadIdx.x; e < kSurModes; e += blockDim.x)
    out[e] = static_cast<float>(b3[e] - (e == 0 ? static_cast<double>(shift0) : 0.0));
  __syncthreads();
}

// LDS of the encoder / target kernels: t1 (8 N^2), t2 (64 N), V (24 N),
// Linv (192), work (192), b3 (512), red (256) doubles
template <int N>
constexpr size_t enc_lds_doubles() {
  return static_cast<size_t>(kSurD) * N * N + kSurD * kSurD * N + 3 * N * kSurD + 3 * kSurD * kSurD +
         3 * kSurD * kSurD + kSurModes + 256;
}

// A thread owns columns (j, k) and walks along x, so a value's abscissae and
// basis factors are one LDS row for all of its columns; f is read twice, once
// for the moments (the frame) and once for the x-modes and the indicator
// together.  The Maxwellian is the product of the tables' order-0 columns, not
// an exp per velocity.  Bound by reading f (2 x 8 n bytes per point) and by the
// 8 FP64 multiply-adds per value: 1000 points at 32^3, 704 -> 253 us on MI355X.
// MODES = false is for calls that want the moments and the indicator alone (no
// x): the same sums without the x-modes, the basis tables and their LDS.
constexpr int kEncThreads = 512;

template <int N>
constexpr size_t enc_moments_lds_doubles() {
  return 3 * N * kSurD + kEncThreads / 64 * 5;
}

template <int N, bool MODES>
__global__ __launch_bounds__(kEncThreads) void k_sur_encode(EncArgs a) {
  constexpr int n = N * N * N, NN = N * N, NT = kEncThreads;
  extern __shared__ double sm[];
  double* t1 = sm;                          // kSurD * N * N
  double* t2 = t1 + kSurD * NN;             // kSurD * kSurD * N
  double* V = MODES ? t2 + kSurD * kSurD * N : sm;  // 3 * N * kSurD
  double* Linv = V + 3 * N * kSurD;         // 3 * 64
  double* work = Linv + 3 * kSurD * kSurD;  // 3 * 64
  double* b3 = work + 3 * kSurD * kSurD;    // 512
  double* red = MODES ? b3 + kSurModes : V + 3 * N * kSurD;  // 256 (without the modes 40)
  const double hh = 2.0 * a.L / N, c0 = -a.L + 0.5 * hh;
  const double pi = 3.14159265358979323846;
  for (int pt = blockIdx.x; pt < a.npts; pt += gridDim.x) {
    const double* f = a.f + static_cast<size_t>(pt) * n;
    double m[5] = {0, 0, 0, 0, 0};
    for (int jk = threadIdx.x; jk < NN; jk += NT) {
      const double cy = c0 + (jk / N) * hh, cz = c0 + (jk % N) * hh;
      double a0 = 0, a1 = 0, a2 = 0;
#pragma unroll 8
      for (int i = 0; i < N; ++i) {
        const double v = f[i * NN + jk], cx = c0 + i * hh, vc = v * cx;
        a0 += v;
        a1 += vc;
        a2 += vc * cx;
      }
      m[0] += a0;
      m[1] += a1;
      m[2] += a0 * cy;
      m[3] += a0 * cz;
      m[4] += a2 + a0 * (cy * cy + cz * cz);
    }
    block_sums<5, NT>(m, red);
    const double rho = m[0] * a.cw;
    const double ux = m[1] * a.cw / rho, uy = m[2] * a.cw / rho, uz = m[3] * a.cw / rho;
    const double T = (2.0 / 3.0) * (m[4] * a.cw / rho - (ux * ux + uy * uy + uz * uz));
    const double Mn = rho / pow(pi * T, 1.5);
    const double s = sqrt(0.5 * T), hs = hh / s;
    if constexpr (MODES) {
      herm_table(V, c0, hh, ux, s, N);
      herm_table(V + N * kSurD, c0, hh, uy, s, N);
      herm_table(V + 2 * N * kSurD, c0, hh, uz, s, N);
    } else {  // the order-0 columns
      for (int e = threadIdx.x; e < 3 * N; e += NT) {
        const double x = (c0 + (e % N) * hh - (e < N ? ux : e < 2 * N ? uy : uz)) / s;
        V[e * kSurD] = exp(-0.5 * x * x) * kInvSqrtFact[0];
      }
    }
    __syncthreads();
    double ds[2] = {0, 0};  // sums of (f - M)^2 and f^2
    for (int jk = threadIdx.x; jk < NN; jk += NT) {
      const double My = Mn * V[(N + jk / N) * kSurD] * V[(2 * N + jk % N) * kSurD];
      double acc[kSurD];
#pragma unroll
      for (int q = 0; q < kSurD; ++q) acc[q] = 0.0;
#pragma unroll 8
      for (int i = 0; i < N; ++i) {
        const double v = f[i * NN + jk];
        const double* Vi = V + i * kSurD;
        const double d = v - My * Vi[0];
        ds[0] += d * d;
        ds[1] += v * v;
        if constexpr (MODES) {
#pragma unroll
          for (int q = 0; q < kSurD; ++q) acc[q] += v * Vi[q];
        }
      }
      if constexpr (MODES) {
#pragma unroll
        for (int q = 0; q < kSurD; ++q) t1[q * NN + jk] = acc[q];
      }
    }
    block_sums<2, NT>(ds, red);
    if (threadIdx.x == 0) {
      double* mo = a.mom + static_cast<size_t>(pt) * 8;
      mo[0] = rho; mo[1] = ux; mo[2] = uy; mo[3] = uz; mo[4] = T; mo[5] = sqrt(ds[0] / ds[1]); mo[6] = 0; mo[7] = 0;
      if (a.lt) a.lt[pt] = static_cast<float>(log(T));
    }
    if constexpr (MODES) {
      herm_chol_inv<N>(V, hs, Linv, work);
      // f = M is the 000 basis function: its coefficient is prod_d L_d[0][0],
      // subtracted so that equilibrium maps to zero
      const double c000 = 1.0 / (Linv[0] * Linv[kSurD * kSurD] * Linv[2 * kSurD * kSurD]);
      herm_project_rest<N>(V, Linv, t1, t2, b3, hs * hs * hs / Mn, a.x + static_cast<size_t>(pt) * kSurModes,
                           static_cast<float>(c000));
      // second indicator: the share of f's norm in the modes of total degree
      // >= 4 (zero for Maxwellians carrying the heat-flux and stress modes of
      // Grad's 13-moment description)
      double hv[2] = {0, 0};
      for (int e = threadIdx.x; e < kSurModes; e += NT) {
        const int deg = e / (kSurD * kSurD) + (e / kSurD) % kSurD + e % kSurD;
        const double v = b3[e];
        hv[1] += v * v;
        if (deg >= 4) hv[0] += v * v;
      }
      block_sums<2, NT>(hv, red);
      if (threadIdx.x == 0) a.mom[static_cast<size_t>(pt) * 8 + 6] = sqrt(hv[0] / hv[1]);
    }
    __syncthreads();
  }
}

// targets: b^ = (orthonormal-basis coefficients of Q in the frame of mom) / (prefac rho T^{gamma/2})
struct TgtArgs {
  const double* Q;
  const double* mom;
  float* y;
  double L, cw, gamma, prefac;
  int npts;
};

template <int N>
__global__ __launch_bounds__(256) void k_sur_targets(TgtArgs a) {
  constexpr int n = N * N * N, NN = N * N;
  extern __shared__ double sm[];
  double* t1 = sm;
  double* t2 = t1 + kSurD * NN;
  double* V = t2 + kSurD * kSurD * N;
  double* Linv = V + 3 * N * kSurD;
  double* work = Linv + 3 * kSurD * kSurD;
  double* b3 = work + 3 * kSurD * kSurD;
  const double hh = 2.0 * a.L / N, c0 = -a.L + 0.5 * hh;
  const double pi = 3.14159265358979323846;
  for (int pt = blockIdx.x; pt < a.npts; pt += gridDim.x) {
    const double* mo = a.mom + static_cast<size_t>(pt) * 8;
    const double rho = mo[0], T = mo[4], s = sqrt(0.5 * T), hs = hh / s;
    herm_table(V, c0, hh, mo[1], s, N);
    herm_table(V + N * kSurD, c0, hh, mo[2], s, N);
    herm_table(V + 2 * N * kSurD, c0, hh, mo[3], s, N);
    __syncthreads();
    herm_chol_inv<N>(V, hs, Linv, work);
    const double Mn = rho / pow(pi * T, 1.5);
    const double factor = hs * hs * hs / (Mn * a.prefac * rho * pow(T, 0.5 * a.gamma));
    herm_project<N>(a.Q + static_cast<size_t>(pt) * n, V, Linv, t1, t2, b3, factor,
                    a.y + static_cast<size_t>(pt) * kSurModes, 0.0f);
  }
}

// decode: the network output y holds orthonormal-basis coefficients; the
// Hermite-basis coefficients are b = prefac rho T^{gamma/2} (Lx^-T (x) Ly^-T
// (x) Lz^-T) y, the mass, momentum and energy modes are removed
// (b_000 = b_100 = b_010 = b_001 = 0, b_200 + b_020 + b_002 = 0) and
// Q[idx[i]] = M sum_n b_n psi_n(c')
struct DecArgs {
  const float* y;    // [nidx][512] network outputs, row i for point idx[i]
  const double* mom; // [npts][8]
  const int* idx;    // [nidx] point index of row i (null: identity)
  double* Q;         // [npts][n]
  double L, gamma, prefac;
  int nidx;
  // FP64 projection onto the collision invariants, or none
  int project;
  double cw;
  double Ainv[25];
};

// A thread owns columns (j, k): the y and z sums of a column's eight x-modes
// stay in its registers and the x sum gives its Q values.  With the projection
// the values are formed twice, first for the moments and then, corrected, to
// be written: Q is written once and never read (decode and the separate
// projection moved 4 x 8 n bytes per point: 402 -> 145 us per 1000 points at
// 32^3 on MI355X).
template <int N>
__global__ __launch_bounds__(256, 2) void k_sur_decode(DecArgs a) {
  constexpr int n = N * N * N, NN = N * N, NT = 256, CPT = (NN + NT - 1) / NT;
  extern __shared__ double sm[];
  double* s1 = sm;                      // kSurD * kSurD * N [a][b][k] (>= 512)
  double* V = s1 + kSurD * kSurD * N;   // 3 * N * kSurD
  double* bb = V + 3 * N * kSurD;       // 512
  double* Linv = bb + kSurModes;        // 3 * 64
  double* work = Linv + 3 * kSurD * kSurD;  // 3 * 64
  double* red = work + 3 * kSurD * kSurD;   // NT / 64 * 5
  const double hh = 2.0 * a.L / N, c0 = -a.L + 0.5 * hh;
  const double pi = 3.14159265358979323846;
  for (int i = blockIdx.x; i < a.nidx; i += gridDim.x) {
    const int pt = a.idx ? a.idx[i] : i;
    const double* mo = a.mom + static_cast<size_t>(pt) * 8;
    const double rho = mo[0], ux = mo[1], uy = mo[2], uz = mo[3], T = mo[4], s = sqrt(0.5 * T);
    herm_table(V, c0, hh, ux, s, N);
    herm_table(V + N * kSurD, c0, hh, uy, s, N);
    herm_table(V + 2 * N * kSurD, c0, hh, uz, s, N);
    const double scale = a.prefac * rho * pow(T, 0.5 * a.gamma);
    const float* yi = a.y + static_cast<size_t>(i) * kSurModes;
    for (int e = threadIdx.x; e < kSurModes; e += NT) bb[e] = scale * static_cast<double>(yi[e]);
    __syncthreads();
    herm_chol_inv<N>(V, hh / s, Linv, work);
    kron3(Linv, true, bb, s1, bb);
    if (threadIdx.x == 0) {
      constexpr int e200 = 2 * kSurD * kSurD, e020 = 2 * kSurD, e002 = 2;
      const double tr = (bb[e200] + bb[e020] + bb[e002]) / 3.0;
      bb[e200] -= tr; bb[e020] -= tr; bb[e002] -= tr;
      bb[0] = 0.0; bb[kSurD * kSurD] = 0.0; bb[kSurD] = 0.0; bb[1] = 0.0;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kSurD * kSurD * N; e += NT) {  // s1[a][b][k]
      const int ab = e / N, k = e - ab * N;
      double t = 0.0;
      for (int c = 0; c < kSurD; ++c) t += bb[ab * kSurD + c] * V[2 * N * kSurD + k * kSurD + c];
      s1[e] = t;
    }
    __syncthreads();
    // the tables carry the per-axis Gaussian factors of M
    const double Mn = rho / pow(pi * T, 1.5);
    double x[CPT][kSurD];  // x-modes of the thread's columns
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int jk = threadIdx.x + c * NT;
      if (jk < NN) {
        const int j = jk / N, k = jk - j * N;
#pragma unroll
        for (int q = 0; q < kSurD; ++q) {
          double t = 0.0;
#pragma unroll
          for (int b = 0; b < kSurD; ++b) t += s1[(q * kSurD + b) * N + k] * V[(N + j) * kSurD + b];
          x[c][q] = Mn * t;
        }
      } else {
#pragma unroll
        for (int q = 0; q < kSurD; ++q) x[c][q] = 0.0;
      }
    }
    double m[5] = {0, 0, 0, 0, 0};
    if (a.project) {
      double a0[CPT] = {}, a1 = 0.0, a2 = 0.0;
#pragma unroll 2
      for (int ii = 0; ii < N; ++ii) {
        const double cx = c0 + ii * hh;
        double qs = 0.0;
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
          double t = 0.0;
#pragma unroll
          for (int q = 0; q < kSurD; ++q) t += x[c][q] * V[ii * kSurD + q];
          a0[c] += t;
          qs += t;
        }
        a1 += qs * cx;
        a2 += qs * (cx * cx);
      }
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        const int jk = threadIdx.x + c * NT;
        const double cy = c0 + (jk / N) * hh, cz = c0 + (jk % N) * hh;
        m[0] += a0[c];
        m[2] += a0[c] * cy;
        m[3] += a0[c] * cz;
        m[4] += a0[c] * (cy * cy + cz * cz);
      }
      m[1] = a1;
      m[4] += a2;
      block_sums<5, NT>(m, red);
      double lam[5];
#pragma unroll
      for (int p = 0; p < 5; ++p) {
        lam[p] = 0.0;
#pragma unroll
        for (int k = 0; k < 5; ++k) lam[p] += a.Ainv[p * 5 + k] * (m[k] * a.cw);
      }
#pragma unroll
      for (int p = 0; p < 5; ++p) m[p] = a.cw * lam[p];
    }
    double* Q = a.Q + static_cast<size_t>(pt) * n;
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int jk = threadIdx.x + c * NT;
      if (jk >= NN) continue;
      const double cy = c0 + (jk / N) * hh, cz = c0 + (jk % N) * hh;
      const double l0 = m[0] + m[2] * cy + m[3] * cz + m[4] * (cy * cy + cz * cz);
#pragma unroll 4
      for (int ii = 0; ii < N; ++ii) {
        const double cx = c0 + ii * hh;
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < kSurD; ++q) t += x[c][q] * V[ii * kSurD + q];
        Q[ii * NN + jk] = t - (l0 + cx * (m[1] + m[4] * cx));
      }
    }
    __syncthreads();
  }
}

// rows of src [*][n] -> dst [nidx][n] (gather) or back (scatter)
__global__ __launch_bounds__(256) void k_rows_copy(const double* __restrict__ src, double* __restrict__ dst,
                                                   const int* __restrict__ idx, int nidx, int n, int gather) {
  const int i = blockIdx.y;
  if (i >= nidx) return;
  const long s = gather ? idx[i] : i, d = gather ? i : idx[i];
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x)
    dst[d * n + r] = src[s * n + r];
}

__global__ __launch_bounds__(256) void k_rows_copy_f(const float* __restrict__ src, float* __restrict__ dst,
                                                     const int* __restrict__ idx, int nidx, int n) {
  const int i = blockIdx.y;
  if (i >= nidx) return;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x)
    dst[static_cast<long>(i) * n + r] = src[static_cast<long>(idx[i]) * n + r];
}

// out[2i] = ||Q[idx[i]] - R[i]||^2, out[2i+1] = ||R[i]||^2 over the n
// velocities of row i (one workgroup per row)
__global__ __launch_bounds__(256) void k_row_err(const double* __restrict__ Q, const int* __restrict__ idx,
                                                 const double* __restrict__ R, int nrows, int n,
                                                 double* __restrict__ out) {
  __shared__ double red[2][256];
  const int i = blockIdx.x;
  if (i >= nrows) return;
  const double* q = Q + static_cast<long>(idx[i]) * n;
  const double* r = R + static_cast<long>(i) * n;
  double e = 0.0, m = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) {
    const double d = q[k] - r[k];
    e += d * d;
    m += r[k] * r[k];
  }
  red[0][threadIdx.x] = e;
  red[1][threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s) {
      red[0][threadIdx.x] += red[0][threadIdx.x + s];
      red[1][threadIdx.x] += red[1][threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * i] = red[0][0];
    out[2 * i + 1] = red[1][0];
  }
}

// out[i] = ||Q[i]||^2 (one workgroup per row)
__global__ __launch_bounds__(256) void k_row_norm2(const double* __restrict__ Q, int nrows, int n,
                                                   double* __restrict__ out) {
  __shared__ double red[256];
  const int i = blockIdx.x;
  if (i >= nrows) return;
  const double* q = Q + static_cast<long>(i) * n;
  double m = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) m += q[k] * q[k];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[i] = red[0];
}

// ---------------------------------------------------------------------------
// handle
// ---------------------------------------------------------------------------
struct SurHandle {
  int magic = 0x73757231;
  int N = 0, n = 0, max_batch = 0;
  double L = 0, cw = 0, gamma = 0, prefac = 0;
  double Ainv[25] = {};
  GemmWs ws;
  // activations of the last forward (capacity max_batch points)
  float* Z[kSurLayers + 1] = {};
  float* U[kSurLayers] = {};
  float* Vv[kSurLayers] = {};
  float* dA = nullptr;
  float* dB = nullptr;
  float* dU = nullptr;
  float* part = nullptr;  // channel-reduction partials
  const float* x_last = nullptr;
  const float* lt_last = nullptr;
  int P_last = 0;
  int bf16_last = 1;
  // evaluation workspace
  size_t cap_pts = 0;
  double* mom = nullptr;
  float* xin = nullptr;
  float* ltin = nullptr;
  float* yout = nullptr;
  float* xg = nullptr;
  float* ltg = nullptr;
  int* idx_d = nullptr;
  double* fb_f = nullptr;
  double* fb_Q = nullptr;
  size_t cap_fb = 0;
  double* mom_h = nullptr;  // pinned copy of the moments
  // sampled spectral check: per-row squared errors and norms, and their
  // pinned host copy ([3][cap_pts])
  double* chk_d = nullptr;
  double* chk_h = nullptr;
  ~SurHandle() {
    for (auto* p : Z) (void)hipFree(p);
    for (auto* p : U) (void)hipFree(p);
    for (auto* p : Vv) (void)hipFree(p);
    (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dU); (void)hipFree(part);
    (void)hipFree(mom); (void)hipFree(xin); (void)hipFree(ltin); (void)hipFree(yout);
    (void)hipFree(xg); (void)hipFree(ltg); (void)hipFree(idx_d); (void)hipFree(fb_f); (void)hipFree(fb_Q);
    (void)hipHostFree(mom_h);
    (void)hipFree(chk_d);
    (void)hipHostFree(chk_h);
  }
};

static SurHandle* as_sur(void* p) {
  auto* h = static_cast<SurHandle*>(p);
  if (!h || h->magic != 0x73757231) return nullptr;
  return h;
}

static inline unsigned nblk(long tot) { return static_cast<unsigned>((tot + 255) / 256); }
constexpr int kRedBlocks = 240;
// workgroups of the fused layer kernels: four waves of kLayRows rows each, and
// at most two per CU backward, whose partial sums are read back per workgroup
constexpr unsigned kLayBwdBlocks = 512;
static unsigned lay_blocks(int P) {
  static_assert(kSurModes % (4 * kLayRows) == 0, "whole rows for every wave");
  return static_cast<unsigned>(static_cast<long>(kSurModes) * P / (4 * kLayRows));
}

static int chan_reduce(SurHandle* h, int kind, const float* X, const float* Y, const float* xin, const float* lt,
                       int P, float* out, hipStream_t st) {
  ChanRedArgs ca{X, Y, xin, lt, nullptr, h->part, P, kind};
  hipLaunchKernelGGL(k_chan_reduce, dim3(kRedBlocks), dim3(256), 0, st, ca);
  DGFS_LAUNCH_CHECK("chan_reduce");
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(1024), 0, st, h->part, kRedBlocks, kSurWidth, out);
  DGFS_LAUNCH_CHECK("sum_parts");
  return DGFS_OK;
}

static int sur_forward(SurHandle* h, const float* th, const float* x, const float* lt, int P, float* out, bool bf16,
                       hipStream_t st) {
  const long act = static_cast<long>(kSurModes) * P * kSurWidth;
  hipLaunchKernelGGL(k_lift_fwd, dim3(nblk(act)), dim3(256), 0, st, th, x, lt, h->Z[0], P);
  DGFS_LAUNCH_CHECK("lift_fwd");
  for (int l = 0; l < kSurLayers; ++l) {
    const float* K = th + kSurOffLayers + l * kSurLayerSize;
    const float* W = K + static_cast<long>(kSurModes) * kSurModes;
    const float* R = W + kSurWidth * kSurWidth;
    const float* bias = R + kSurWidth * kSurWidth;
    int rc = gemm(&h->ws, 0, 0, kSurModes, kSurWidth * P, kSurModes, 1.f, K, kSurModes, h->Z[l],
                  static_cast<long>(kSurWidth) * P, 0.f, h->U[l], static_cast<long>(kSurWidth) * P, bf16, st);
    if (!rc && !bf16) {
      hipLaunchKernelGGL(k_layer_fwd, dim3(lay_blocks(P)), dim3(256), 0, st, h->U[l], h->Z[l], W, R, bias, h->Vv[l],
                         h->Z[l + 1], static_cast<long>(kSurModes) * P, l + 1 < kSurLayers ? 1 : 0);
      DGFS_LAUNCH_CHECK("layer_fwd");
      continue;
    }
    if (!rc) rc = gemm(&h->ws, 0, 0, kSurModes * P, kSurWidth, kSurWidth, 1.f, h->U[l], kSurWidth, W, kSurWidth, 0.f,
                       h->Vv[l], kSurWidth, bf16, st);
    if (!rc) rc = gemm(&h->ws, 0, 0, kSurModes * P, kSurWidth, kSurWidth, 1.f, h->Z[l], kSurWidth, R, kSurWidth, 1.f,
                       h->Vv[l], kSurWidth, bf16, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_bias_act, dim3(nblk(act)), dim3(256), 0, st, h->Vv[l], bias, h->Z[l + 1], act,
                       l + 1 < kSurLayers ? 1 : 0);
    DGFS_LAUNCH_CHECK("bias_act");
  }
  hipLaunchKernelGGL(k_head_fwd, dim3(nblk(static_cast<long>(kSurModes) * P)), dim3(256), 0, st, th,
                     h->Z[kSurLayers], out, P);
  DGFS_LAUNCH_CHECK("head_fwd");
  h->x_last = x;
  h->lt_last = lt;
  h->P_last = P;
  h->bf16_last = bf16 ? 1 : 0;
  return DGFS_OK;
}

static int sur_backward(SurHandle* h, const float* th, const float* dout, float* grad, hipStream_t st) {
  const int P = h->P_last;
  const bool bf16 = h->bf16_last != 0;
  const long act = static_cast<long>(kSurModes) * P * kSurWidth;
  const long ld = static_cast<long>(kSurWidth) * P;
  // head
  hipLaunchKernelGGL(k_head_bwd, dim3(nblk(act)), dim3(256), 0, st, th, dout, h->dA, P);
  DGFS_LAUNCH_CHECK("head_bwd");
  {
    // dPout[c] = sum_{m,p} Z4[m][p][c] dout[p][m] (kind 2 with xin = dout)
    int rc = chan_reduce(h, 2, h->Z[kSurLayers], nullptr, dout, nullptr, P, grad + kSurOffPout, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_bout_reduce, dim3(kSurModes / 32), dim3(1024), 0, st, dout, grad + kSurOffBout, P);
    DGFS_LAUNCH_CHECK("bout_reduce");
  }
  float* dZ = h->dA;    // gradient w.r.t. Z_{l+1}
  float* dZn = h->dB;   // gradient w.r.t. Z_l
  for (int l = kSurLayers - 1; l >= 0; --l) {
    const float* K = th + kSurOffLayers + l * kSurLayerSize;
    const float* W = K + static_cast<long>(kSurModes) * kSurModes;
    const float* R = W + kSurWidth * kSurWidth;
    float* gK = grad + kSurOffLayers + l * kSurLayerSize;
    float* gW = gK + static_cast<long>(kSurModes) * kSurModes;
    float* gR = gW + kSurWidth * kSurWidth;
    float* gb = gR + kSurWidth * kSurWidth;
    if (!bf16) {
      const unsigned nb = std::min<unsigned>(lay_blocks(P), kLayBwdBlocks);
      hipLaunchKernelGGL(k_layer_bwd, dim3(nb), dim3(256), 0, st, dZ, h->Vv[l], h->U[l], h->Z[l], W, R, h->dU, dZn,
                         h->part, static_cast<long>(kSurModes) * P, l + 1 < kSurLayers ? 1 : 0);
      DGFS_LAUNCH_CHECK("layer_bwd");
      // gW, gR and gb follow each other in the parameter vector as in a partial
      hipLaunchKernelGGL(k_sum_parts, dim3((kLayPart + 31) / 32), dim3(1024), 0, st, h->part, static_cast<int>(nb),
                         kLayPart, gW);
      DGFS_LAUNCH_CHECK("layer_grads");
      int rc = gemm(&h->ws, 0, 1, kSurModes, kSurModes, kSurWidth * P, 1.f, h->dU, ld, h->Z[l], ld, 0.f, gK,
                    kSurModes, false, st);
      if (!rc) rc = gemm(&h->ws, 1, 0, kSurModes, kSurWidth * P, kSurModes, 1.f, K, kSurModes, h->dU, ld, 1.f, dZn, ld,
                         false, st);
      if (rc) return rc;
      std::swap(dZ, dZn);
      continue;
    }
    if (l + 1 < kSurLayers) {
      hipLaunchKernelGGL(k_act_bwd, dim3(nblk(act)), dim3(256), 0, st, h->Vv[l], dZ, act);
      DGFS_LAUNCH_CHECK("act_bwd");
    }
    // dZ now holds dV
    int rc = chan_reduce(h, 0, dZ, nullptr, nullptr, nullptr, P, gb, st);
    if (!rc) rc = gemm(&h->ws, 1, 0, kSurWidth, kSurWidth, kSurModes * P, 1.f, h->U[l], kSurWidth, dZ, kSurWidth, 0.f,
                       gW, kSurWidth, bf16, st);
    if (!rc) rc = gemm(&h->ws, 1, 0, kSurWidth, kSurWidth, kSurModes * P, 1.f, h->Z[l], kSurWidth, dZ, kSurWidth, 0.f,
                       gR, kSurWidth, bf16, st);
    if (!rc) rc = gemm(&h->ws, 0, 1, kSurModes * P, kSurWidth, kSurWidth, 1.f, dZ, kSurWidth, W, kSurWidth, 0.f,
                       h->dU, kSurWidth, bf16, st);
    if (!rc) rc = gemm(&h->ws, 0, 1, kSurModes * P, kSurWidth, kSurWidth, 1.f, dZ, kSurWidth, R, kSurWidth, 0.f,
                       dZn, kSurWidth, bf16, st);
    if (!rc) rc = gemm(&h->ws, 0, 1, kSurModes, kSurModes, kSurWidth * P, 1.f, h->dU, ld, h->Z[l], ld, 0.f, gK,
                       kSurModes, bf16, st);
    if (!rc) rc = gemm(&h->ws, 1, 0, kSurModes, kSurWidth * P, kSurModes, 1.f, K, kSurModes, h->dU, ld, 1.f, dZn, ld,
                       bf16, st);
    if (rc) return rc;
    std::swap(dZ, dZn);
  }
  // lift
  int rc = chan_reduce(h, 2, dZ, nullptr, h->x_last, nullptr, P, grad + kSurOffP0, st);
  if (!rc) rc = chan_reduce(h, 3, dZ, nullptr, nullptr, h->lt_last, P, grad + kSurOffP1, st);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mode_reduce, dim3(kSurModes), dim3(256), 0, st, dZ, grad + kSurOffE, P);
  DGFS_LAUNCH_CHECK("mode_reduce");
  return DGFS_OK;
}

template <int N>
static size_t enc_lds() {
  return enc_lds_doubles<N>() * sizeof(double);
}
template <int N>
static size_t dec_lds() {
  return (static_cast<size_t>(kSurD) * kSurD * N + 3 * N * kSurD + kSurModes + 6 * kSurD * kSurD + 20) *
         sizeof(double);
}

template <int N>
static int launch_encode(const EncArgs& ea, hipStream_t st) {
  const dim3 grid(std::min(ea.npts, 4 * cu_count()));
  if (!ea.x) {
    hipLaunchKernelGGL((k_sur_encode<N, false>), grid, dim3(kEncThreads), enc_moments_lds_doubles<N>() * sizeof(double),
                       st, ea);
    DGFS_LAUNCH_CHECK("sur_encode(moments)");
    return DGFS_OK;
  }
  const size_t lds = enc_lds<N>();
  DGFS_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sur_encode<N, true>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  hipLaunchKernelGGL((k_sur_encode<N, true>), grid, dim3(kEncThreads), lds, st, ea);
  DGFS_LAUNCH_CHECK("sur_encode");
  return DGFS_OK;
}
template <int N>
static int launch_targets(const TgtArgs& ta, hipStream_t st) {
  const size_t lds = enc_lds<N>();
  DGFS_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sur_targets<N>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  hipLaunchKernelGGL(k_sur_targets<N>, dim3(std::min(ta.npts, 4 * cu_count())), dim3(256), lds, st, ta);
  DGFS_LAUNCH_CHECK("sur_targets");
  return DGFS_OK;
}
template <int N>
static int launch_decode(const DecArgs& da, hipStream_t st) {
  const size_t lds = dec_lds<N>();
  DGFS_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sur_decode<N>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  hipLaunchKernelGGL(k_sur_decode<N>, dim3(std::min(da.nidx, 4 * cu_count())), dim3(256), lds, st, da);
  DGFS_LAUNCH_CHECK("sur_decode");
  return DGFS_OK;
}

static int do_encode(SurHandle* h, const EncArgs& ea, hipStream_t st) {
  switch (h->N) {
    case 8: return launch_encode<8>(ea, st);
    case 12: return launch_encode<12>(ea, st);
    case 16: return launch_encode<16>(ea, st);
    case 24: return launch_encode<24>(ea, st);
    case 32: return launch_encode<32>(ea, st);
    default: return fail(DGFS_ERR_UNSUPPORTED, "Nv=%d not built for the surrogate", h->N);
  }
}
static int do_targets(SurHandle* h, const TgtArgs& ta, hipStream_t st) {
  switch (h->N) {
    case 8: return launch_targets<8>(ta, st);
    case 12: return launch_targets<12>(ta, st);
    case 16: return launch_targets<16>(ta, st);
    case 24: return launch_targets<24>(ta, st);
    case 32: return launch_targets<32>(ta, st);
    default: return fail(DGFS_ERR_UNSUPPORTED, "Nv=%d not built for the surrogate", h->N);
  }
}
// unprojected decode of rows of y into the points idx (null: row i, point i)
static DecArgs dec_args(const SurHandle* h, const float* y, const double* mom, const int* idx, double* Q, int nidx) {
  DecArgs da{};
  da.y = y; da.mom = mom; da.idx = idx; da.Q = Q;
  da.L = h->L; da.gamma = h->gamma; da.prefac = h->prefac;
  da.nidx = nidx;
  return da;
}

static int do_decode(SurHandle* h, const DecArgs& da, hipStream_t st) {
  switch (h->N) {
    case 8: return launch_decode<8>(da, st);
    case 12: return launch_decode<12>(da, st);
    case 16: return launch_decode<16>(da, st);
    case 24: return launch_decode<24>(da, st);
    case 32: return launch_decode<32>(da, st);
    default: return fail(DGFS_ERR_UNSUPPORTED, "Nv=%d not built for the surrogate", h->N);
  }
}

static int ensure_eval_ws(SurHandle* h, int npts) {
  if (static_cast<size_t>(npts) <= h->cap_pts) return DGFS_OK;
  (void)hipFree(h->mom); (void)hipFree(h->xin); (void)hipFree(h->ltin); (void)hipFree(h->yout);
  (void)hipFree(h->xg); (void)hipFree(h->ltg); (void)hipFree(h->idx_d); (void)hipHostFree(h->mom_h);
  (void)hipFree(h->chk_d); (void)hipHostFree(h->chk_h);
  h->mom = nullptr; h->xin = h->ltin = h->yout = h->xg = h->ltg = nullptr; h->idx_d = nullptr; h->mom_h = nullptr;
  h->chk_d = h->chk_h = nullptr;
  h->cap_pts = 0;
  DGFS_HIP_TRY(hipMalloc(&h->mom, static_cast<size_t>(npts) * 8 * sizeof(double)));
  DGFS_HIP_TRY(hipMalloc(&h->xin, static_cast<size_t>(npts) * kSurModes * sizeof(float)));
  DGFS_HIP_TRY(hipMalloc(&h->ltin, static_cast<size_t>(npts) * sizeof(float)));
  DGFS_HIP_TRY(hipMalloc(&h->yout, static_cast<size_t>(npts) * kSurModes * sizeof(float)));
  DGFS_HIP_TRY(hipMalloc(&h->xg, static_cast<size_t>(npts) * kSurModes * sizeof(float)));
  DGFS_HIP_TRY(hipMalloc(&h->ltg, static_cast<size_t>(npts) * sizeof(float)));
  DGFS_HIP_TRY(hipMalloc(&h->idx_d, static_cast<size_t>(npts) * 4 * sizeof(int)));
  DGFS_HIP_TRY(hipHostMalloc(&h->mom_h, static_cast<size_t>(npts) * 8 * sizeof(double)));
  DGFS_HIP_TRY(hipMalloc(&h->chk_d, static_cast<size_t>(npts) * 3 * sizeof(double)));
  DGFS_HIP_TRY(hipHostMalloc(&h->chk_h, static_cast<size_t>(npts) * 3 * sizeof(double)));
  h->cap_pts = npts;
  return DGFS_OK;
}

}  // namespace dgfs

using namespace dgfs;

extern "C" long dgfs_sur_param_count(void) { return kSurParams; }

extern "C" int dgfs_nn_gemm(int transA, int transB, int M, int N, int K, float alpha, const float* A, long lda,
                            const float* B, long ldb, float beta, float* C, long ldc, int bf16, void* stream) {
  if (!A || !B || !C) return fail(DGFS_ERR_INVALID_VALUE, "null GEMM operand");
  if (M < 0 || N < 0 || K < 1) return fail(DGFS_ERR_INVALID_VALUE, "bad GEMM sizes %d %d %d", M, N, K);
  if (lda < (transA ? M : K) || ldb < (transB ? K : N) || ldc < N)
    return fail(DGFS_ERR_INVALID_VALUE, "leading dimension too small");
  if ((M + kGT - 1) / kGT > 65535) return fail(DGFS_ERR_INVALID_VALUE, "M = %d exceeds the grid (65535 row tiles)", M);
  auto st = static_cast<hipStream_t>(stream);
  // no shape splits a reduction shorter than kGemmSplitK
  return gemm(K >= kGemmSplitK ? shared_gemm_ws(st) : nullptr, transA ? 1 : 0, transB ? 1 : 0, M, N, K, alpha, A,
              lda, B, ldb, beta, C, ldc, bf16 != 0, st);
}

extern "C" int dgfs_sur_create(const dgfs_sur_desc* d, void** out) {
  if (!d || !out) return fail(DGFS_ERR_INVALID_VALUE, "null descriptor or handle pointer");
  *out = nullptr;
  switch (d->Nv) {
    case 8: case 12: case 16: case 24: case 32: break;
    default: return fail(DGFS_ERR_UNSUPPORTED, "surrogate Nv=%d unsupported (built: 8 12 16 24 32)", d->Nv);
  }
  // the channel GEMMs have 512 * batch rows, one 64-row tile per grid row
  if (d->max_batch < 1 || d->max_batch > 4096) return fail(DGFS_ERR_INVALID_VALUE, "max_batch must be 1..4096");
  if (!(d->L > 0) || !(d->cw > 0) || !(d->prefac > 0)) return fail(DGFS_ERR_INVALID_VALUE, "L, cw, prefac must be positive");
  auto h = std::make_unique<SurHandle>();
  h->N = d->Nv;
  h->n = d->Nv * d->Nv * d->Nv;
  h->max_batch = d->max_batch;
  h->L = d->L;
  h->cw = d->cw;
  h->gamma = d->gamma;
  h->prefac = d->prefac;
  int rc = invariant_gram_inverse(h->N, h->L, h->cw, h->Ainv);
  if (rc) return rc;
  const size_t act = static_cast<size_t>(kSurModes) * d->max_batch * kSurWidth * sizeof(float);
  for (int l = 0; l <= kSurLayers; ++l) DGFS_HIP_TRY(hipMalloc(&h->Z[l], act));
  for (int l = 0; l < kSurLayers; ++l) {
    DGFS_HIP_TRY(hipMalloc(&h->U[l], act));
    DGFS_HIP_TRY(hipMalloc(&h->Vv[l], act));
  }
  DGFS_HIP_TRY(hipMalloc(&h->dA, act));
  DGFS_HIP_TRY(hipMalloc(&h->dB, act));
  DGFS_HIP_TRY(hipMalloc(&h->dU, act));
  DGFS_HIP_TRY(hipMalloc(&h->part, std::max(static_cast<size_t>(kRedBlocks) * kSurWidth,
                                            static_cast<size_t>(kLayBwdBlocks) * kLayPart) * sizeof(float)));
  // the products of any batch may split their reduction: no call allocates later
  rc = h->ws.init();
  if (rc) return rc;
  *out = h.release();
  return DGFS_OK;
}

extern "C" int dgfs_sur_destroy(void* p) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  (void)hipDeviceSynchronize();
  h->magic = 0;
  delete h;
  return DGFS_OK;
}

extern "C" int dgfs_sur_forward(void* p, const float* params, const float* x, const float* lt, int P, float* out,
                                int bf16, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!params || !x || !lt || !out) return fail(DGFS_ERR_INVALID_VALUE, "null network operand");
  if (P < 1 || P > h->max_batch) return fail(DGFS_ERR_INVALID_VALUE, "batch %d outside 1..%d", P, h->max_batch);
  return sur_forward(h, params, x, lt, P, out, bf16 != 0, static_cast<hipStream_t>(stream));
}

extern "C" int dgfs_sur_backward(void* p, const float* params, const float* dout, float* grad, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!params || !dout || !grad) return fail(DGFS_ERR_INVALID_VALUE, "null network operand");
  if (h->P_last < 1) return fail(DGFS_ERR_INVALID_VALUE, "backward needs a preceding forward");
  return sur_backward(h, params, dout, grad, static_cast<hipStream_t>(stream));
}

extern "C" int dgfs_sur_adam(long n, float* params, const float* grad, float* m1, float* m2, float lr, float b1,
                             float b2, float eps, int step, void* stream) {
  if (!params || !grad || !m1 || !m2) return fail(DGFS_ERR_INVALID_VALUE, "null Adam operand");
  if (n < 1 || step < 1) return fail(DGFS_ERR_INVALID_VALUE, "Adam needs n >= 1 and step >= 1");
  const float c1 = 1.f - std::pow(b1, static_cast<float>(step));
  const float c2 = 1.f - std::pow(b2, static_cast<float>(step));
  hipLaunchKernelGGL(k_adam, dim3(nblk(n)), dim3(256), 0, static_cast<hipStream_t>(stream), params, grad, m1, m2, n,
                     lr, b1, b2, eps, c1, c2);
  DGFS_LAUNCH_CHECK("adam");
  return DGFS_OK;
}

extern "C" int dgfs_sur_encode(void* p, const double* f, int npts, double* mom, float* x, float* lt, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!f || !mom) return fail(DGFS_ERR_INVALID_VALUE, "null encode operand");
  if (npts < 0) return fail(DGFS_ERR_INVALID_VALUE, "npts must be >= 0");
  if (npts == 0) return DGFS_OK;
  EncArgs ea{f, mom, x, lt, h->L, h->cw, npts};
  return do_encode(h, ea, static_cast<hipStream_t>(stream));
}

extern "C" int dgfs_sur_targets(void* p, const double* Q, const double* mom, int npts, float* y, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!Q || !mom || !y) return fail(DGFS_ERR_INVALID_VALUE, "null target operand");
  if (npts < 0) return fail(DGFS_ERR_INVALID_VALUE, "npts must be >= 0");
  if (npts == 0) return DGFS_OK;
  TgtArgs ta{Q, mom, y, h->L, h->cw, h->gamma, h->prefac, npts};
  return do_targets(h, ta, static_cast<hipStream_t>(stream));
}

extern "C" int dgfs_sur_decode(void* p, const float* y, const double* mom, const int* idx, int nidx, double* Q,
                               int project, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!y || !mom || !Q) return fail(DGFS_ERR_INVALID_VALUE, "null decode operand");
  if (nidx < 0) return fail(DGFS_ERR_INVALID_VALUE, "nidx must be >= 0");
  if (nidx == 0) return DGFS_OK;
  if (project && idx) return fail(DGFS_ERR_INVALID_VALUE, "projection of an index subset: project the rows afterwards");
  auto st = static_cast<hipStream_t>(stream);
  DecArgs da = dec_args(h, y, mom, idx, Q, nidx);
  if (project) {
    da.project = 1;
    da.cw = h->cw;
    std::memcpy(da.Ainv, h->Ainv, sizeof(da.Ainv));
  }
  return do_decode(h, da, st);
}

namespace dgfs {

// checks shared by the evaluation entry points; the exact operator runs on
// row buffers sized for this surrogate's grid
static int check_eval_args(SurHandle* h, void* vhs, const float* params, const double* f, double* Q, int npts) {
  if (!vhs || !params || !f || !Q) return fail(DGFS_ERR_INVALID_VALUE, "null operand");
  if (npts < 0) return fail(DGFS_ERR_INVALID_VALUE, "npts must be >= 0");
  int vN = 0;
  double vL = 0.0;
  const int rc0 = dgfs_vhs_get_dims(vhs, &vN, nullptr, nullptr, nullptr, &vL);
  if (rc0) return rc0;
  if (vN != h->N || std::fabs(vL - h->L) > 1e-12 * h->L)
    return fail(DGFS_ERR_INVALID_VALUE, "surrogate (N=%d, L=%g) and exact operator (N=%d, L=%g) grids differ",
                h->N, h->L, vN, vL);
  return DGFS_OK;
}

// encode every point and read the moments and indicators on the host
static int encode_and_read(SurHandle* h, const double* f, int npts, hipStream_t st) {
  int rc = ensure_eval_ws(h, npts);
  if (rc) return rc;
  EncArgs ea{f, h->mom, h->xin, h->ltin, h->L, h->cw, npts};
  rc = do_encode(h, ea, st);
  if (rc) return rc;
  DGFS_HIP_TRY(hipMemcpyAsync(h->mom_h, h->mom, static_cast<size_t>(npts) * 8 * sizeof(double),
                              hipMemcpyDeviceToHost, st));
  DGFS_HIP_TRY(hipStreamSynchronize(st));
  return DGFS_OK;
}

// row buffers for `rows` exact/projected rows, sized before any launch that
// reads them (the stream is drained before a buffer is replaced)
static int ensure_rows(SurHandle* h, int rows, hipStream_t st) {
  const size_t need = static_cast<size_t>(std::max(rows, 1)) * h->n;
  if (need <= h->cap_fb) return DGFS_OK;
  DGFS_HIP_TRY(hipStreamSynchronize(st));
  (void)hipFree(h->fb_f); (void)hipFree(h->fb_Q);
  h->fb_f = h->fb_Q = nullptr;
  h->cap_fb = 0;
  DGFS_HIP_TRY(hipMalloc(&h->fb_f, need * sizeof(double)));
  DGFS_HIP_TRY(hipMalloc(&h->fb_Q, need * sizeof(double)));
  h->cap_fb = need;
  return DGFS_OK;
}

static dim3 rows_grid(const SurHandle* h, int nrows) { return dim3(std::max(1, std::min(64, h->n / 256)), nrows); }

// exact operator on the rows idx[0..nr) of f: results in fb_Q[0..nr), and
// scattered into Q when scatter is set
static int exact_rows(SurHandle* h, void* vhs, const double* f, double* Q, const int* idx, int nr, bool scatter,
                      hipStream_t st) {
  if (nr == 0) return DGFS_OK;
  hipLaunchKernelGGL(k_rows_copy, rows_grid(h, nr), dim3(256), 0, st, f, h->fb_f, idx, nr, h->n, 1);
  DGFS_LAUNCH_CHECK("rows_gather");
  int rc = dgfs_vhs_eval_contig(vhs, h->fb_f, h->fb_Q, nr, st);
  if (rc) return rc;
  if (scatter) {
    hipLaunchKernelGGL(k_rows_copy, rows_grid(h, nr), dim3(256), 0, st, h->fb_Q, Q, idx, nr, h->n, 0);
    DGFS_LAUNCH_CHECK("rows_scatter");
  }
  return DGFS_OK;
}

// network, decoder and FP64 projection on the rows idx[0..ns) of Q (uses
// fb_Q as the projection's row buffer)
static int network_rows(SurHandle* h, const float* params, double* Q, const int* idx, int ns, bool bf16,
                        hipStream_t st) {
  if (ns == 0) return DGFS_OK;
  for (int b0 = 0; b0 < ns; b0 += h->max_batch) {
    const int nb = std::min(h->max_batch, ns - b0);
    hipLaunchKernelGGL(k_rows_copy_f, dim3(2, nb), dim3(256), 0, st, h->xin, h->xg, idx + b0, nb, kSurModes);
    DGFS_LAUNCH_CHECK("x_gather");
    hipLaunchKernelGGL(k_rows_copy_f, dim3(1, nb), dim3(256), 0, st, h->ltin, h->ltg, idx + b0, nb, 1);
    DGFS_LAUNCH_CHECK("lt_gather");
    int rc = sur_forward(h, params, h->xg, h->ltg, nb, h->yout, bf16, st);
    if (rc) return rc;
    const DecArgs da = dec_args(h, h->yout, h->mom, idx + b0, Q, nb);
    rc = do_decode(h, da, st);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(k_rows_copy, rows_grid(h, ns), dim3(256), 0, st, Q, h->fb_Q, idx, ns, h->n, 1);
  DGFS_LAUNCH_CHECK("rows_gather");
  int rc = launch_invariant_projection(h->fb_Q, h->Ainv, h->L, h->cw, h->N, ns, st);
  if (rc) return rc;
  hipLaunchKernelGGL(k_rows_copy, rows_grid(h, ns), dim3(256), 0, st, h->fb_Q, Q, idx, ns, h->n, 0);
  DGFS_LAUNCH_CHECK("rows_scatter");
  return DGFS_OK;
}

// indicator routing: points within both thresholds are surrogate candidates
static void route(const SurHandle* h, int npts, double threshold, double threshold_hi, std::vector<int>& sur,
                  std::vector<int>& fb) {
  sur.clear();
  fb.clear();
  for (int i = 0; i < npts; ++i) {
    const double ind = h->mom_h[static_cast<size_t>(i) * 8 + 5];
    const double ind_hi = h->mom_h[static_cast<size_t>(i) * 8 + 6];
    const bool ok = ind <= threshold && std::isfinite(ind) && (threshold_hi <= 0.0 || ind_hi <= threshold_hi);
    (ok ? sur : fb).push_back(i);
  }
}

static int upload_idx(int* dst, const std::vector<int>& v, hipStream_t st) {
  if (!v.empty()) DGFS_HIP_TRY(hipMemcpyAsync(dst, v.data(), v.size() * sizeof(int), hipMemcpyHostToDevice, st));
  return DGFS_OK;
}

}  // namespace dgfs

// Surrogate with fallback: encode every point, evaluate the network on the
// points whose indicator is <= threshold (and, if threshold_hi > 0, whose
// high-mode indicator is <= threshold_hi), decode and project them; run the
// exact operator (a dgfs_vhs handle) on the rest.  One host synchronisation
// reads the indicators.  nfallback (optional) receives the fallback count.
extern "C" int dgfs_sur_eval(void* p, void* vhs, const float* params, const double* f, double* Q, int npts,
                             double threshold, double threshold_hi, int bf16, int* nfallback, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  int rc = check_eval_args(h, vhs, params, f, Q, npts);
  if (rc) return rc;
  if (npts == 0) {
    if (nfallback) *nfallback = 0;
    return DGFS_OK;
  }
  auto st = static_cast<hipStream_t>(stream);
  rc = encode_and_read(h, f, npts, st);
  if (rc) return rc;
  std::vector<int> sur, fb;
  route(h, npts, threshold, threshold_hi, sur, fb);
  if (nfallback) *nfallback = static_cast<int>(fb.size());
  const int ns = static_cast<int>(sur.size()), nf = static_cast<int>(fb.size());
  int* idx_s = h->idx_d;
  int* idx_f = h->idx_d + npts;
  rc = upload_idx(idx_s, sur, st);
  if (!rc) rc = upload_idx(idx_f, fb, st);
  if (!rc) rc = ensure_rows(h, std::max(nf, ns), st);
  if (!rc) rc = exact_rows(h, vhs, f, Q, idx_f, nf, true, st);
  if (!rc) rc = network_rows(h, params, Q, idx_s, ns, bf16 != 0, st);
  return rc;
}

// Surrogate with fallback and a sampled spectral check.  After the indicator
// routing, the surrogate candidates are ranked by indicator and cut into bins
// of equal count, and a stratified sample of every bin is evaluated both by
// the network and by the exact operator (with the indicator fallback points
// in the same exact call).  In each bin the sample's squared errors, and the
// exact |Q|^2, are taken proportional to the squared indicator (a ratio
// estimator with the indicator as the auxiliary variable), which predicts the
// unsampled points' error and |Q|^2 from their own indicators.  Whole bins,
// the largest predicted error per point first, then fall back until the
// predicted error of the points the network keeps is within safety * tol of
// the batch's |Q|.  The rejected points take one more exact call, the kept
// ones the network; sampled points keep their exact Q.  Two host
// synchronisations: the indicators, the sample.
extern "C" int dgfs_sur_eval_checked(void* p, void* vhs, const float* params, const double* f, double* Q,
                                     int npts, double threshold, double threshold_hi, const dgfs_sur_check* chk,
                                     int bf16, dgfs_sur_check_stats* stats, void* stream) {
  SurHandle* h = as_sur(p);
  if (!h) return fail(DGFS_ERR_NOT_INITIALIZED, "invalid surrogate handle");
  if (!chk) return fail(DGFS_ERR_INVALID_VALUE, "null check settings");
  if (!(chk->tol > 0) || !(chk->safety > 0) || chk->safety > 1 || chk->nbins < 1 || chk->min_per_bin < 1 ||
      !(chk->sample_frac >= 0) || chk->sample_frac > 1)
    return fail(DGFS_ERR_INVALID_VALUE, "check settings: tol > 0, 0 < safety <= 1, nbins >= 1, min_per_bin >= 1, "
                                        "0 <= sample_frac <= 1");
  int rc = check_eval_args(h, vhs, params, f, Q, npts);
  if (rc) return rc;
  dgfs_sur_check_stats out{};
  if (npts == 0) {
    if (stats) *stats = out;
    return DGFS_OK;
  }
  auto st = static_cast<hipStream_t>(stream);
  rc = encode_and_read(h, f, npts, st);
  if (rc) return rc;
  auto ind = [&](int i) { return h->mom_h[static_cast<size_t>(i) * 8 + 5]; };
  std::vector<int> cand, fb;
  route(h, npts, threshold, threshold_hi, cand, fb);
  // rank the candidates by indicator, largest first, and cut equal bins
  std::stable_sort(cand.begin(), cand.end(), [&](int a, int b) { return ind(a) > ind(b); });
  const int nc = static_cast<int>(cand.size());
  const int nbins = std::max(1, std::min(chk->nbins, nc));
  std::vector<int> bin_lo(nbins + 1);
  for (int b = 0; b <= nbins; ++b) bin_lo[b] = static_cast<int>((static_cast<long>(nc) * b) / nbins);
  // stratified sample: s_b evenly spaced ranks in each bin, offset by a
  // seeded fraction of the spacing
  std::vector<int> samp, samp_bin;
  std::vector<char> in_sample(nc, 0);
  unsigned long long x = chk->seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
  auto unif = [&]() {  // splitmix64 -> [0, 1)
    x += 0x9E3779B97F4A7C15ull;
    unsigned long long z = x;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return static_cast<double>(z >> 11) * (1.0 / 9007199254740992.0);
  };
  for (int b = 0; b < nbins; ++b) {
    const int nb = bin_lo[b + 1] - bin_lo[b];
    if (nb == 0) continue;
    const int sb = std::min(nb, std::max(chk->min_per_bin, static_cast<int>(std::ceil(chk->sample_frac * nb))));
    const double u = unif();
    for (int j = 0; j < sb; ++j) {
      const int r = bin_lo[b] + std::min(nb - 1, static_cast<int>((j + u) * nb / sb));
      if (in_sample[r]) continue;
      in_sample[r] = 1;
      samp.push_back(cand[r]);
      samp_bin.push_back(b);
    }
  }
  const int nsamp = static_cast<int>(samp.size()), nf = static_cast<int>(fb.size());
  // device index lists: [sample | fallback + sample | rejected | kept]
  int* idx_s = h->idx_d;
  int* idx_e = h->idx_d + npts;
  int* idx_r = h->idx_d + 2 * npts;
  int* idx_k = h->idx_d + 3 * npts;
  std::vector<int> exact(fb);
  exact.insert(exact.end(), samp.begin(), samp.end());
  const int ne = static_cast<int>(exact.size());
  rc = upload_idx(idx_s, samp, st);
  if (!rc) rc = upload_idx(idx_e, exact, st);
  if (!rc) rc = ensure_rows(h, std::max(ne, nc), st);
  // the network on the sample, then the exact operator on the fallback and
  // sampled rows; the sample's errors and every exact row's |Q|^2
  if (!rc) rc = network_rows(h, params, Q, idx_s, nsamp, bf16 != 0, st);
  if (!rc) rc = exact_rows(h, vhs, f, Q, idx_e, ne, false, st);
  if (rc) return rc;
  if (nsamp) {
    hipLaunchKernelGGL(k_row_err, dim3(nsamp), dim3(256), 0, st, Q, idx_s, h->fb_Q + static_cast<size_t>(nf) * h->n,
                       nsamp, h->n, h->chk_d);
    DGFS_LAUNCH_CHECK("row_err");
  }
  if (ne) {
    hipLaunchKernelGGL(k_row_norm2, dim3(ne), dim3(256), 0, st, h->fb_Q, ne, h->n,
                       h->chk_d + 2 * static_cast<size_t>(npts));
    DGFS_LAUNCH_CHECK("row_norm2");
    hipLaunchKernelGGL(k_rows_copy, rows_grid(h, ne), dim3(256), 0, st, h->fb_Q, Q, idx_e, ne, h->n, 0);
    DGFS_LAUNCH_CHECK("rows_scatter");
  }
  DGFS_HIP_TRY(hipMemcpyAsync(h->chk_h, h->chk_d, static_cast<size_t>(npts) * 3 * sizeof(double),
                              hipMemcpyDeviceToHost, st));
  DGFS_HIP_TRY(hipStreamSynchronize(st));
  // ratio estimates per bin: squared error and |Q|^2 per unit squared
  // indicator, from the sample
  constexpr double kTiny = 1e-300;
  std::vector<double> e_b(nbins, 0.0), q_b(nbins, 0.0), i_b(nbins, 0.0), cnt_b(nbins, 0.0);
  for (int s = 0; s < nsamp; ++s) {
    const int b = samp_bin[s];
    e_b[b] += h->chk_h[2 * s];
    q_b[b] += h->chk_h[2 * s + 1];
    i_b[b] += ind(samp[s]) * ind(samp[s]);
    cnt_b[b] += 1.0;
  }
  std::vector<double> rest_b(nbins, 0.0), nrest_b(nbins, 0.0);  // unsampled: sum of ind^2, count
  for (int b = 0; b < nbins; ++b)
    for (int r = bin_lo[b]; r < bin_lo[b + 1]; ++r)
      if (!in_sample[r]) {
        rest_b[b] += ind(cand[r]) * ind(cand[r]);
        nrest_b[b] += 1.0;
      }
  double qnorm2 = 0.0;
  for (int i = 0; i < ne; ++i) qnorm2 += h->chk_h[2 * static_cast<size_t>(npts) + i];
  std::vector<double> est(nbins, 0.0), per_pt(nbins, 0.0);
  double kept = 0.0;
  for (int b = 0; b < nbins; ++b) {
    if (cnt_b[b] == 0 || nrest_b[b] == 0) continue;
    // with no indicator spread to scale by (all zero), the sample mean
    const bool ratio = i_b[b] > kTiny;
    est[b] = ratio ? e_b[b] / i_b[b] * rest_b[b] : e_b[b] / cnt_b[b] * nrest_b[b];
    qnorm2 += ratio ? q_b[b] / i_b[b] * rest_b[b] : q_b[b] / cnt_b[b] * nrest_b[b];
    per_pt[b] = est[b] / nrest_b[b];
    kept += est[b];
  }
  // drop bins, largest predicted error per point first, until the kept
  // estimate fits the budget
  const double budget = (chk->safety * chk->tol) * (chk->safety * chk->tol) * qnorm2;
  std::vector<int> order(nbins);
  for (int b = 0; b < nbins; ++b) order[b] = b;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return per_pt[a] > per_pt[b]; });
  std::vector<char> reject(nbins, 0);
  for (int k = 0; k < nbins && kept > budget; ++k) {
    if (nrest_b[order[k]] == 0) continue;
    reject[order[k]] = 1;
    kept -= est[order[k]];
    out.nrejected_bins += 1;
  }
  std::vector<int> rej, keep;
  for (int b = 0; b < nbins; ++b)
    for (int r = bin_lo[b]; r < bin_lo[b + 1]; ++r)
      if (!in_sample[r]) (reject[b] ? rej : keep).push_back(cand[r]);
  const int nr = static_cast<int>(rej.size()), nk = static_cast<int>(keep.size());
  rc = upload_idx(idx_r, rej, st);
  if (!rc) rc = upload_idx(idx_k, keep, st);
  if (!rc) rc = exact_rows(h, vhs, f, Q, idx_r, nr, true, st);
  if (!rc) rc = network_rows(h, params, Q, idx_k, nk, bf16 != 0, st);
  if (rc) return rc;
  out.nfallback = nf + nr;
  out.nsampled = nsamp;
  out.nsurrogate = nk;
  out.est_rel_err = qnorm2 > 0 ? std::sqrt(std::max(kept, 0.0) / qnorm2) : 0.0;
  if (stats) *stats = out;
  return DGFS_OK;
}

extern "C" int dgfs_sur_round_bf16(long n, const float* src, float* dst, void* stream) {
  if (!src || !dst || n < 0) return fail(DGFS_ERR_INVALID_VALUE, "bad rounding operands");
  if (n == 0) return DGFS_OK;
  hipLaunchKernelGGL(k_round_bf16, dim3(nblk(n)), dim3(256), 0, static_cast<hipStream_t>(stream), src, dst, n);
  DGFS_LAUNCH_CHECK("round_bf16");
  return DGFS_OK;
}
