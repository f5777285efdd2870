// Gain of the VHS operator for planar half-sphere designs, on the matrix
// cores of gfx950.
//
// exp(i a_pq) F is the spectrum of f moved by (qz_p / 2) sigma_q, so P+- are
// trigonometric interpolations of f on moved grids, and a move along one axis
// is a circulant N x N matrix: S(s) = R(s) + i beta(s) w w^T, with R real,
// w_j = (-1)^j and beta = -sin(theta N/2) / N the part of the unpaired Nyquist
// mode.  A design is planar when every direction has exactly one zero
// component and comes with its mirror image, (a, b) and (a, -b) on an axis
// pair (u, v): nothing then moves along the third axis, every plane of it is
// an independent 2D problem, and the two directions share the move along u.
//
// One plane of one such group costs three "pair moves": f -> X+- = R(+-a) f
// along u, then X+ and X- by +-b along v each, for
//   S += Z(+,+) Z(-,-) + Z(+,-) Z(-,+).
// R(-s) = J R(s) J with J the index reversal, so with f = e + o (even and
// odd under J) R(+-s) f needs only the products G = R e and H = R o of half
// length: R(s) f = G + H, R(-s) f = J (G - H).  Rows are kept in two tiles,
// idx and N-1-idx, so that J is a swap of the tiles.
//
// A plane is one wave's work and never leaves its registers: the first move
// takes the plane as the A operand of v_mfma 16x16x4 and R as B, which leaves
// the rows of v in the result registers, where the second move reads them as
// its B operand with R as A.  No LDS exchange and no barrier lies between.
//
// Exactness of the Nyquist modes.  Re(P+ P-) = R+ R- - I+ I-:
//   R+- carry -beta_a beta_b w_u w_v f^_uv (f^_uv = sum w_u w_v f, one number
//   per plane), set as the initial value of the G accumulators of the second
//   move; and over the two directions
//   -sum I+ I- = eU(v) + eV(u) - dU(v) dV(u), eU = 2 beta_a^2 U+ U-,
//   dU = beta_b w_v (U+ - U-), U+- = R_v(+-b) f^_u, and eV, dV alike with u
//   and v, a and b exchanged: lines that four waves form per group in LDS.
//
// S_p is collected in LDS over the three axis pairs (each element has one
// writer between two barriers, so the order is fixed), transformed along y
// and z two real planes at a time, and stored as
//   T[point][p][slot][ky][kz], slot s the planes x1(s) + i x2(s);
// k_planar_xfwd finishes the transform along x for half of the (ky, kz) (the
// rest follows from the symmetry of a real field) and sums over p.
//
// Why: the FFT form does K 3D complex transforms per point, each through two
// exchanges of the field in LDS, and reached 61 % VALU issue; FP32 and FP64
// MFMA share the VALU's multipliers on MI355X (an MFMA wave starves a VALU
// wave of the same SIMD), so what counts is the sum of both.  Per direction
// and grid point the planar form takes 1.5 N multiply-adds on the matrix
// cores, and about 5 VALU operations instead of 49.  Gain and x transform per
// 4096 points at 32^3 FP32 (M = 12, Nrho = 16): 29.5 ms against 62.5 ms for
// k_vhs_gain_rr with its Nyquist planes; 601 points FP64: 12.3 against 27.1 ms
// for the slab kernel; 24^3 (Nrho = 12), 576 points: 1.8 against 2.9 ms FP32,
// 3.7 against 9.3 ms FP64.  The matrix cores are busy 62 % of the FP32 32^3
// gain's cycles, the VALU about 20 %.
#pragma once
#include <hip/hip_runtime.h>

#include "cplx.hpp"
#include "spectral.hpp"

namespace dgfs {

template <typename T>
struct MmaTile;
// result row of register r in lane group g = lane / 16 is index 4 r + g; col()
// and valid() give the index of lane i = lane % 16 (operand row or column)
template <>
struct MmaTile<float> {
  typedef float V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V4 mma(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ __forceinline__ int col(int i) { return 4 * (i & 3) + (i >> 2); }
  static __host__ __device__ __forceinline__ bool valid(int i, int RN) { return (i & 3) < RN; }
};
template <>
struct MmaTile<double> {
  typedef double V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V4 mma(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ __forceinline__ int col(int i) { return i; }
  static __host__ __device__ __forceinline__ bool valid(int i, int RN) { return i < 4 * RN; }
};

constexpr int kPlanarMaxGroups = 32;
constexpr int kPlanarMaxShifts = 16;
struct PlanarGroup {
  int pair;    // 0: (x, y), 1: (x, z), 2: (y, z)
  int ia, ib;  // shifts (indices of |component|) along u and v
};

template <typename T, int N>
struct PlanarShape {
  static constexpr int HN = N / 2, RN = N / 8, NN = N * N, n = NN * N;
  static constexpr int NR = 4 * RN;  // operand values per lane of one shift's matrices
  // x-halves per work item: the FP64 32^3 field (256 KB) does not fit in LDS
  // in one piece.  The halves repeat the first move of the pairs (x, .): 22
  // pair moves per p for 18.
  static constexpr int XH = (sizeof(T) == 8 && N == 32) ? 2 : 1;
  static constexpr int NX = N / XH;
  // waves per workgroup: two per SIMD where the registers of a plane allow it
  static constexpr int NW = (sizeof(T) == 8 || N < 32) ? 4 : 8;
  static constexpr int WPE = (sizeof(T) == 8 && N >= 24) ? 1 : 2;  // waves per SIMD the registers are budgeted for
  // LDS strides: rows padded to N + 1, planes to 4 banks more than a multiple
  // of 32, so that the lanes of each axis pair's accesses spread over the banks
  static constexpr int PY = N + 1;
  static constexpr int PX = N * PY + ((N == 16) ? 20 : 4);
  static constexpr int s_elems = NX * PX;
  static constexpr int ln_elems = (XH == 2) ? 3 * NN : 4 * NN;
  static constexpr size_t lds_bytes = (static_cast<size_t>(s_elems) + ln_elems) * sizeof(T);
  static constexpr size_t per_point = 3 * static_cast<size_t>(n) + 6 * NN + 3 * N;  // operand values of one point
  static constexpr int nslots = N / 2;  // real-plane pairs of T
  // planes of slot s
  static __host__ __device__ __forceinline__ constexpr int x1(int s) {
    if (XH == 1) return s;
    return s < N / 4 ? s : N - 1 - (s - N / 4);
  }
  static __host__ __device__ __forceinline__ constexpr int x2(int s) {
    if (XH == 1) return s + N / 2;
    return s < N / 4 ? s + N / 4 : N - 1 - s;
  }
  static_assert(N % 8 == 0 && N <= 32, "tiles of N/2 <= 16 rows");
};

// ---------------------------------------------------------------------------
// Operand form of the points: per axis pair and plane of the third axis the
// even / odd parts of f along both axes, stored so that a wave of the gain
// reads its 64 lanes' operand registers as one contiguous block:
//   [pair][s][v index][lane group][r][u even/odd][v even/odd], u index 4 r + g,
// followed by the six Nyquist sums (same form, the plane index as lanes) and
// the three lines f^_uv(s).  A workgroup takes a point; N/4 x-planes at a time
// (both mirror images of every fourth x) pass through LDS, read once from f.
// Bound by its stores (3 n values per point).
// ---------------------------------------------------------------------------
template <typename T>
struct PlanarPrepArgs {
  const double* f;  // [npts][n]
  T* op;            // [npts][per_point]
  int npts;
};

template <typename T, int N>
__global__ __launch_bounds__(256) void k_planar_prep(PlanarPrepArgs<T> a) {
  using PS = PlanarShape<T, N>;
  constexpr int HN = PS::HN, RN = PS::RN, NN = PS::NN, n = PS::n, NR = PS::NR, PP = N * (N + 1), Q = 2 * RN;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* pl = reinterpret_cast<T*>(smem_raw);  // [Q][N][N + 1]
  T* fx = pl + Q * PP;                     // Nyquist sums over x: [y][z]
  T* fy = fx + PP;                         // over y: [x][z]
  T* fz = fy + PP;                         // over z: [x][y]
  const int tid = threadIdx.x;
  auto combine = [](T* o, T a0, T b0, T c0, T d0) {
    const double s = static_cast<double>(a0) + b0, d = static_cast<double>(a0) - b0;
    const double t = static_cast<double>(c0) + d0, e = static_cast<double>(c0) - d0;
    o[0] = static_cast<T>(0.25 * (s + t));
    o[1] = static_cast<T>(0.25 * (s - t));
    o[2] = static_cast<T>(0.25 * (d + e));
    o[3] = static_cast<T>(0.25 * (d - e));
  };
  for (int pt = xcd_slot(); pt < a.npts; pt += gridDim.x) {
    const double* f = a.f + static_cast<size_t>(pt) * n;
    T* op = a.op + static_cast<size_t>(pt) * PS::per_point;
    for (int e = tid; e < PP; e += 256) fx[e] = T(0);
    for (int g = 0; g < 4; ++g) {
      __syncthreads();
      for (int e = tid; e < Q * NN; e += 256) {
        const int q = e / NN, rem = e - q * NN, y = rem / N, z = rem - y * N;
        const int k = 4 * (q >> 1) + g, x = (q & 1) ? N - 1 - k : k;
        pl[q * PP + y * (N + 1) + z] = static_cast<T>(f[x * NN + rem]);
      }
      __syncthreads();
      for (int e = tid; e < NN; e += 256) {
        const int y = e / N, z = e - y * N;
        double s = 0.0;
        for (int q = 0; q < Q; ++q) {
          const double v = pl[q * PP + y * (N + 1) + z];
          s += ((g + q) & 1) ? -v : v;  // x = 4 r + g, or its mirror image
        }
        fx[y * (N + 1) + z] = static_cast<T>(static_cast<double>(fx[y * (N + 1) + z]) + s);
      }
      for (int e = tid; e < Q * N; e += 256) {
        const int q = e / N, i = e - q * N;
        const int k = 4 * (q >> 1) + g, x = (q & 1) ? N - 1 - k : k;
        double s = 0.0, t = 0.0;
        for (int j = 0; j < N; ++j) {
          const double v = pl[q * PP + j * (N + 1) + i], w = pl[q * PP + i * (N + 1) + j];
          s += (j & 1) ? -v : v;
          t += (j & 1) ? -w : w;
        }
        fy[x * (N + 1) + i] = static_cast<T>(s);
        fz[x * (N + 1) + i] = static_cast<T>(t);
      }
      T o[NR];
      for (int e = tid; e < HN * N; e += 256) {  // (x, y), plane z = s
        const int j = e / N, s = e - j * N;
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          const T* p0 = pl + 2 * r * PP;
          combine(o + 4 * r, p0[j * (N + 1) + s], p0[PP + j * (N + 1) + s], p0[(N - 1 - j) * (N + 1) + s],
                  p0[PP + (N - 1 - j) * (N + 1) + s]);
        }
        T* d = op + static_cast<size_t>(s) * NN + (j * 4 + g) * NR;
#pragma unroll
        for (int k = 0; k < NR; ++k) d[k] = o[k];
      }
      for (int e = tid; e < HN * N; e += 256) {  // (x, z), plane y = s
        const int s = e / HN, j = e - s * HN;
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          const T* p0 = pl + 2 * r * PP + s * (N + 1);
          combine(o + 4 * r, p0[j], p0[PP + j], p0[N - 1 - j], p0[PP + N - 1 - j]);
        }
        T* d = op + static_cast<size_t>(N + s) * NN + (j * 4 + g) * NR;
#pragma unroll
        for (int k = 0; k < NR; ++k) d[k] = o[k];
      }
      for (int e = tid; e < Q * HN * 4; e += 256) {  // (y, z), plane x
        const int j = e % HN, lg = (e / HN) % 4, q = e / (HN * 4);
        const int kx = 4 * (q >> 1) + g, x = (q & 1) ? N - 1 - kx : kx;
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          const int y = 4 * r + lg;
          const T *pa = pl + q * PP + y * (N + 1), *pb = pl + q * PP + (N - 1 - y) * (N + 1);
          combine(o + 4 * r, pa[j], pb[j], pa[N - 1 - j], pb[N - 1 - j]);
        }
        T* d = op + static_cast<size_t>(2 * N + x) * NN + (j * 4 + lg) * NR;
#pragma unroll
        for (int k = 0; k < NR; ++k) d[k] = o[k];
      }
    }
    __syncthreads();
    T* ny = op + 3 * static_cast<size_t>(n);
    // contraction index k, plane index s of the six sums
    auto src = [&](int w, int k, int s) -> double {
      switch (w) {
        case 0: return fx[k * (N + 1) + s];
        case 1: return fy[k * (N + 1) + s];
        case 2: return fx[s * (N + 1) + k];
        case 3: return fz[k * (N + 1) + s];
        case 4: return fy[s * (N + 1) + k];
        default: return fz[s * (N + 1) + k];
      }
    };
    for (int e = tid; e < 6 * NN; e += 256) {
      const int w = e / NN, rem = e - w * NN;
      const int st = rem & 1, eo = (rem >> 1) & 1, rg = rem >> 2, r = rg % RN, lg = (rg / RN) & 3, j = rg / (4 * RN);
      const int k = 4 * r + lg, s = st ? N - 1 - j : j;
      const double va = src(w, k, s), vb = src(w, N - 1 - k, s);
      ny[e] = static_cast<T>(0.5 * (eo ? va - vb : va + vb));
    }
    T* line = ny + 6 * NN;
    for (int e = tid; e < 3 * N; e += 256) {
      const int w = e / N, s = e - w * N;
      double acc = 0.0;
      for (int j = 0; j < N; ++j) {
        const double v = (w == 0) ? fx[j * (N + 1) + s] : (w == 1) ? fx[s * (N + 1) + j] : fy[s * (N + 1) + j];
        acc += (j & 1) ? -v : v;
      }
      line[e] = static_cast<T>(acc);
    }
    __syncthreads();
  }
}

template <typename T>
struct PlanarGainArgs {
  const T* op;        // [npts][per_point]
  const T* smat;      // [Nrho][nshift][64][NR] operand values of R(shift), per lane
  const double* beta; // [Nrho][nshift]
  cpx<T>* Tb;         // [npts][Nrho][N/2][N][N]
  int nitems, ngroups, ppg, Nrho, nshift, ngr;
  PlanarGroup gr[kPlanarMaxGroups];
};

// G = R e and H = R o of both row tiles; DATA_A: the data is the A operand
// (its lanes become the result's rows), else the B operand.  The accumulators
// start at c1, c2 (G) and zero (H).
template <typename T, int RN, bool DATA_A>
__device__ __forceinline__ void pair_move(const T (&e)[RN], const T (&o)[RN], const T (&S)[4 * RN],
                                          typename MmaTile<T>::V4 c1, typename MmaTile<T>::V4 c2,
                                          typename MmaTile<T>::V4& G1, typename MmaTile<T>::V4& G2,
                                          typename MmaTile<T>::V4& H1, typename MmaTile<T>::V4& H2) {
  using M = MmaTile<T>;
  G1 = c1;
  G2 = c2;
  H1 = H2 = typename M::V4{T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    if constexpr (DATA_A) {
      G1 = M::mma(e[r], S[r], G1);
      G2 = M::mma(e[r], S[RN + r], G2);
      H1 = M::mma(o[r], S[2 * RN + r], H1);
      H2 = M::mma(o[r], S[3 * RN + r], H2);
    } else {
      G1 = M::mma(S[r], e[r], G1);
      G2 = M::mma(S[RN + r], e[r], G2);
      H1 = M::mma(S[2 * RN + r], o[r], H1);
      H2 = M::mma(S[3 * RN + r], o[r], H2);
    }
  }
}

// the planes of one group: PAIR fixes which axes u, v and the plane index are.
// The operand values of the next plane are in flight during the second move,
// and the group's lines and the previous sum of S are read ahead of the
// products that use them.
template <typename T, int N, int PAIR>
__device__ __forceinline__ void planar_planes(const T* op, const T (&Sa)[4 * (N / 8)], const T (&Sb)[4 * (N / 8)],
                                              T bab, T* S, const T* ln, int half, bool first) {
  using PS = PlanarShape<T, N>;
  using M = MmaTile<T>;
  using V4 = typename M::V4;
  constexpr int RN = PS::RN, HN = PS::HN, NN = PS::NN, NR = PS::NR, XH = PS::XH, NX = PS::NX, NW = PS::NW;
  constexpr bool HALF_U = XH == 2 && PAIR < 2;       // only the u tile of this x-half is wanted
  constexpr int NT = HALF_U ? 1 : 2;                 // u tiles
  constexpr int NS = (XH == 2 && PAIR == 2) ? NX : N;  // planes of the item
  constexpr int NU = HALF_U ? HN : N;                  // u values of the lines
  // strides of S along u, v and the plane index
  constexpr int TU = PAIR == 2 ? PS::PY : PS::PX, TV = PAIR == 0 ? PS::PY : 1;
  constexpr int TS = PAIR == 0 ? 1 : PAIR == 1 ? PS::PY : PS::PX;
  const int lane = threadIdx.x & 63, lg = lane >> 4, i = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ci = M::col(i);
  const bool ok = (RN == 4) || M::valid(i, RN);
  const int cc = ok ? ci : 0;
  const T* eU = ln + lg * RN;
  const T* dU = eU + NS * N;
  const T* eV = ln + 2 * NS * N + (cc & 3) * RN + (cc >> 2);  // this lane's u
  const T* dV = eV + NS * NU;
  const T* line = op + 3 * PS::n + 6 * NN + PAIR * N;
  const T sg = ((ci + lg) & 1) ? -bab : bab;
  T* Su[2] = {S + cc * TU, S + (N - 1 - cc) * TU};
  const T* P0 = op + static_cast<size_t>(PAIR * N) * NN + (cc * 4 + lg) * NR;
  auto plane = [&](int sl) { return (PAIR == 2 && XH == 2 && half) ? N - 1 - sl : sl; };
  T fr[NR], c0;
  {
    const int s = plane(w);
    const T* P = P0 + static_cast<size_t>(s) * NN;
#pragma unroll
    for (int k = 0; k < NR; ++k) fr[k] = P[k];
    c0 = line[s];
  }
#pragma unroll 1
  for (int sl = w; sl < NS; sl += NW) {
    const T ck = sg * c0;
    // move along u: X+-[tile][v even / odd][r], lanes u, registers v
    T Xp[NT][2][RN], Xm[NT][2][RN];
    const V4 z4{T(0), T(0), T(0), T(0)};
    {
      V4 G1[2], G2[2], H1[2], H2[2];
#pragma unroll
      for (int vt = 0; vt < 2; ++vt) {
        T e[RN], o[RN];
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          e[r] = fr[4 * r + vt];
          o[r] = fr[4 * r + 2 + vt];
        }
        pair_move<T, RN, true>(e, o, Sa, z4, z4, G1[vt], G2[vt], H1[vt], H2[vt]);
      }
#pragma unroll
      for (int vt = 0; vt < 2; ++vt)
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          if constexpr (HALF_U) {
            Xp[0][vt][r] = half ? G2[vt][r] + H2[vt][r] : G1[vt][r] + H1[vt][r];
            Xm[0][vt][r] = half ? G1[vt][r] - H1[vt][r] : G2[vt][r] - H2[vt][r];
          } else {
            Xp[0][vt][r] = G1[vt][r] + H1[vt][r];
            Xm[0][vt][r] = G2[vt][r] - H2[vt][r];
            Xp[NT - 1][vt][r] = G2[vt][r] + H2[vt][r];
            Xm[NT - 1][vt][r] = G1[vt][r] - H1[vt][r];
          }
        }
    }
    {  // the next plane (the last iteration reads its own again)
      const int s = plane(sl + NW < NS ? sl + NW : sl);
      const T* P = P0 + static_cast<size_t>(s) * NN;
#pragma unroll
      for (int k = 0; k < NR; ++k) fr[k] = P[k];
      c0 = line[s];
    }
    T u1[RN], u2[RN], d1[RN], d2[RN];
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      u1[r] = eU[sl * N + r];
      u2[r] = eU[sl * N + HN + r];
      d1[r] = dU[sl * N + r];
      d2[r] = dU[sl * N + HN + r];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // S at (u of the tile, v = 4 r + lg) and its mirror images in v, lowest address first
      T* S1 = Su[t] + sl * TS + lg * TV;
      T* S2 = Su[t] + sl * TS + (N - 1 - 4 * (RN - 1) - lg) * TV;
      T p1[RN], p2[RN];
#pragma unroll
      for (int r = 0; r < RN; ++r) p1[r] = p2[r] = T(0);
      if (!first) {
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          p1[r] = S1[4 * r * TV];
          p2[r] = S2[4 * (RN - 1 - r) * TV];
        }
      }
      const bool mirror = HALF_U ? half != 0 : t != 0;  // u = N - 1 - ci
      const T ct = mirror ? -ck : ck;
      const V4 cp{ct, ct, ct, ct}, cn{-ct, -ct, -ct, -ct};
      V4 G1p, G2p, H1p, H2p, G1m, G2m, H1m, H2m;
      pair_move<T, RN, false>(Xp[t][0], Xp[t][1], Sb, cn, cp, G1p, G2p, H1p, H2p);
      pair_move<T, RN, false>(Xm[t][0], Xm[t][1], Sb, cp, cn, G1m, G2m, H1m, H2m);
      const T ev = eV[sl * NU + (t ? HN : 0)], dv = dV[sl * NU + (t ? HN : 0)];
      T q1[RN], q2[RN];
#pragma unroll
      for (int r = 0; r < RN; ++r) {
        const T a1 = (G1p[r] + H1p[r]) * (G2m[r] - H2m[r]) + (G2p[r] - H2p[r]) * (G1m[r] + H1m[r]);
        const T a2 = (G2p[r] + H2p[r]) * (G1m[r] - H1m[r]) + (G1p[r] - H1p[r]) * (G2m[r] + H2m[r]);
        q1[r] = p1[r] + (a1 + (u1[r] + ev - d1[r] * dv));
        q2[r] = p2[r] + (a2 + (u2[r] + ev - d2[r] * dv));
      }
      if (ok) {
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          S1[4 * r * TV] = q1[r];
          S2[4 * (RN - 1 - r) * TV] = q2[r];
        }
      }
    }
  }
}

template <typename T, int N>
__global__ __launch_bounds__((PlanarShape<T, N>::NW * 64), (PlanarShape<T, N>::WPE)) void k_vhs_gain_planar(
    PlanarGainArgs<T> a) {
  using PS = PlanarShape<T, N>;
  using M = MmaTile<T>;
  using V4 = typename M::V4;
  constexpr int RN = PS::RN, HN = PS::HN, NN = PS::NN, NR = PS::NR, XH = PS::XH, NX = PS::NX, NW = PS::NW;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* S = reinterpret_cast<T*>(smem_raw);
  T* ln = S + PS::s_elems;
  const int lane = threadIdx.x & 63, lg = lane >> 4, i = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ci = M::col(i);
  const bool ok = M::valid(i, RN);
  const int cc = ok ? ci : 0;
  for (int item = xcd_slot(); item < a.nitems; item += gridDim.x) {
    const int half = (XH == 2) ? item % 2 : 0, pg = item / XH;
    const int pt = pg / a.ngroups, grp = pg - pt * a.ngroups;
    const int p0 = grp * a.ppg, p1 = min(p0 + a.ppg, a.Nrho);
    const T* op = a.op + static_cast<size_t>(pt) * PS::per_point;
    for (int p = p0; p < p1; ++p) {
      for (int gi = 0; gi < a.ngr; ++gi) {
        const int pair = a.gr[gi].pair, ia = a.gr[gi].ia, ib = a.gr[gi].ib;
        T Sa[NR], Sb[NR];
        {
          const T* sa = a.smat + (static_cast<size_t>(p * a.nshift + ia) * 64 + lane) * NR;
          const T* sb = a.smat + (static_cast<size_t>(p * a.nshift + ib) * 64 + lane) * NR;
#pragma unroll
          for (int k = 0; k < NR; ++k) Sa[k] = sa[k];
#pragma unroll
          for (int k = 0; k < NR; ++k) Sb[k] = sb[k];
        }
        const T ba = static_cast<T>(a.beta[p * a.nshift + ia]), bb = static_cast<T>(a.beta[p * a.nshift + ib]);
        const bool half_s = XH == 2 && pair == 2, half_u = XH == 2 && pair < 2;
        const int NS = half_s ? NX : N, NU = half_u ? HN : N;
        __syncthreads();  // the previous group's (or p's) readers of the lines and of S are done
        if (w < 4) {
          // lines of the group: wave 2 * (V line) + (mirrored plane tile)
          const bool vline = w & 2;
          const int st = w & 1;
          if (!half_s || st == half) {
            const T* P = op + 3 * PS::n + (2 * pair + (vline ? 1 : 0)) * NN + (cc * 4 + lg) * NR;
            T de[RN], dd[RN];
#pragma unroll
            for (int r = 0; r < RN; ++r) {
              de[r] = P[4 * r + st];
              dd[r] = P[4 * r + 2 + st];
            }
            const V4 z4{T(0), T(0), T(0), T(0)};
            V4 G1, G2, H1, H2;
            if (vline)
              pair_move<T, RN, true>(de, dd, Sa, z4, z4, G1, G2, H1, H2);
            else
              pair_move<T, RN, true>(de, dd, Sb, z4, z4, G1, G2, H1, H2);
            const T e2 = vline ? T(2) * bb * bb : T(2) * ba * ba;
            const T ds = ((ci & 1) ? T(-1) : T(1)) * (vline ? ba : bb);
            const int NL = vline ? NU : N;
            T* e = ln + (vline ? 2 * NS * N : 0);
            T* d = e + NS * NL;
            const int pos = (cc & 3) * RN + (cc >> 2);
#pragma unroll
            for (int r = 0; r < RN; ++r) {
              const int si = 4 * r + lg, s = (st && !half_s) ? N - 1 - si : si;
              const T a1 = G1[r] + H1[r], b1 = G2[r] - H2[r];  // index ci: shift +, -
              const T a2 = G2[r] + H2[r], b2 = G1[r] - H1[r];  // index N - 1 - ci
              if (ok) {
                if (vline && half_u) {
                  e[s * NL + pos] = half ? e2 * a2 * b2 : e2 * a1 * b1;
                  d[s * NL + pos] = half ? -ds * (a2 - b2) : ds * (a1 - b1);
                } else {
                  e[s * NL + pos] = e2 * a1 * b1;
                  e[s * NL + HN + pos] = e2 * a2 * b2;
                  d[s * NL + pos] = ds * (a1 - b1);
                  d[s * NL + HN + pos] = -ds * (a2 - b2);
                }
              }
            }
          }
        }
        __syncthreads();
        const bool first = gi == 0;
        if (pair == 0)
          planar_planes<T, N, 0>(op, Sa, Sb, ba * bb, S, ln, half, first);
        else if (pair == 1)
          planar_planes<T, N, 1>(op, Sa, Sb, ba * bb, S, ln, half, first);
        else
          planar_planes<T, N, 2>(op, Sa, Sb, ba * bb, S, ln, half, first);
      }
      __syncthreads();
      // y, z forward transform of two real planes at a time, in place: N lanes
      // per pair of planes (its rows along z, then its columns along y)
      constexpr int PPW = 64 / N, NPP = NX / 2;
      const int sub = lane / N, l = lane - sub * N;
      for (int pp = w * PPW + sub; pp - sub < NPP; pp += NW * PPW) {
        const bool act = sub < PPW && pp < NPP;
        T* A = S + (act ? pp : 0) * PS::PX;
        T* B = A + NPP * PS::PX;
        cpx<T> v[N];
        if (act) {
#pragma unroll
          for (int z = 0; z < N; ++z) v[z] = cpx<T>{A[l * PS::PY + z], B[l * PS::PY + z]};
        }
        FFT<T, N, -1>::run(v);
        if (act) {
#pragma unroll
          for (int z = 0; z < N; ++z) {
            A[l * PS::PY + z] = v[z].x;
            B[l * PS::PY + z] = v[z].y;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // rows are in LDS: the columns are read by the same wave
        if (act) {
#pragma unroll
          for (int y = 0; y < N; ++y) v[y] = cpx<T>{A[y * PS::PY + l], B[y * PS::PY + l]};
        }
        FFT<T, N, -1>::run(v);
        if (act) {
          cpx<T>* t = a.Tb + ((static_cast<size_t>(pt) * a.Nrho + p) * PS::nslots + half * NPP + pp) * NN + l;
#pragma unroll
          for (int y = 0; y < N; ++y) t[y * N] = v[y];
        }
      }
    }
  }
}

// x-forward transform and the weighted sum over p:
// G^[pt](k) = sum_p w_p b1_p(k) FFT_x(T_p)(k).  A thread takes the pencil
// (ky, kz) with ky <= N/2 and, as S_p is real, writes its mirror image
// (-ky, -kz) too.  HV of the N kx sums are kept per pass (all in FP32, half in
// FP64, whose waves share a pencil), in registers over p.  Bound by reading T.
template <typename T>
struct PlanarXfwdArgs {
  const cpx<T>* Tb;
  const T* b1;        // [Nrho][n]
  const double* wgt;  // [Nrho]
  cpx<T>* Ghat;       // [npts][n]
  int npts, Nrho;
};

template <typename T, int N, int K0, int KN>
__device__ __forceinline__ void planar_xfwd_part(const PlanarXfwdArgs<T>& a, int pt, int ky, int kz) {
  using PS = PlanarShape<T, N>;
  constexpr int NN = N * N, n = NN * N;
  const int i1 = ky * N + kz, my = (N - ky) % N, mz = (N - kz) % N, i2 = my * N + mz;
  cpx<T> acc[KN];
#pragma unroll
  for (int k = 0; k < KN; ++k) acc[k] = cpx<T>{T(0), T(0)};
  for (int p = 0; p < a.Nrho; ++p) {
    const cpx<T>* Tp = a.Tb + (static_cast<size_t>(pt) * a.Nrho + p) * PS::nslots * NN;
    cpx<T> A[N / 2], B[N / 2];
#pragma unroll
    for (int s = 0; s < N / 2; ++s) {
      A[s] = Tp[s * NN + i1];
      B[s] = Tp[s * NN + i2];
    }
    cpx<T> v[N];
#pragma unroll
    for (int s = 0; s < N / 2; ++s) {
      // the transforms of the two real planes from that of x1 + i x2
      v[PS::x1(s)] = cpx<T>{T(0.5) * (A[s].x + B[s].x), T(0.5) * (A[s].y - B[s].y)};
      v[PS::x2(s)] = cpx<T>{T(0.5) * (A[s].y + B[s].y), T(0.5) * (B[s].x - A[s].x)};
    }
    FFT<T, N, -1>::run(v);
    const T wp = static_cast<T>(a.wgt[p]);
    const T* b = a.b1 + static_cast<size_t>(p) * n + i1;
#pragma unroll
    for (int k = 0; k < KN; ++k) acc[k] = acc[k] + (wp * b[static_cast<size_t>(k + K0) * NN]) * v[k + K0];
  }
  cpx<T>* G = a.Ghat + static_cast<size_t>(pt) * n;
#pragma unroll
  for (int k = 0; k < KN; ++k) G[static_cast<size_t>(k + K0) * NN + i1] = acc[k];
  if (i1 != i2) {
#pragma unroll
    for (int k = 0; k < KN; ++k) {
      const int mk = (N - (k + K0)) % N;
      G[static_cast<size_t>(mk) * NN + i2] = conj(acc[k]);
    }
  }
}

template <typename T, int N>
__global__ __launch_bounds__(256) void k_planar_xfwd(PlanarXfwdArgs<T> a) {
  constexpr int NV = (N / 2 + 1) * N, SPLIT = sizeof(T) == 8 ? 2 : 1, PER = 256 / SPLIT;
  const int w = threadIdx.x / 64, lane = threadIdx.x & 63;
  const long col = static_cast<long>(blockIdx.x) * PER + (w / SPLIT) * 64 + lane;
  if (col >= static_cast<long>(a.npts) * NV) return;
  const int pt = static_cast<int>(col / NV), idx = static_cast<int>(col - static_cast<long>(pt) * NV);
  const int ky = idx / N, kz = idx - (idx / N) * N;
  // on the self-conjugate rows ky = 0 and N/2 the second half of kz is the
  // mirror image of the first
  if ((ky == 0 || ky == N / 2) && kz > N / 2) return;
  if constexpr (SPLIT == 1) {
    planar_xfwd_part<T, N, 0, N>(a, pt, ky, kz);
  } else {
    if (w & 1)
      planar_xfwd_part<T, N, N / 2, N / 2>(a, pt, ky, kz);
    else
      planar_xfwd_part<T, N, 0, N / 2>(a, pt, ky, kz);
  }
}

}  // namespace dgfs
