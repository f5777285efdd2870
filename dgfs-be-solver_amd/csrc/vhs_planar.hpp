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
// Two splits cut a pair move from 2 N^2 to N^2 / 2 multiply-adds per line:
//   c_j = (f_j + f_{j+M}) / 2, d_j = (f_j - f_{j+M}) / 2, M = N/2: a circulant
//   of N is a circulant R^c of M on c and a skew circulant R^d on d, with
//   (R f)_j = c'_j + d'_j and (R f)_{j+M} = c'_j - d'_j;
//   R^{c,d}(-s) = K R^{c,d}(s) K with K the index reversal of M, so with even
//   and odd parts under K, R(s) = G + H and R(-s) = K (G - H), G and H the
//   products with the even and the odd half.
// The four parts ce, co, de, do of N/4 values each are the K index of the
// products, the M outputs the rows of one 16 x 16 tile; K is a swap of result
// registers (rows) or of neighbouring lanes (columns), because every output
// and its mirror image share a lane group.  At N = 16 the tile has room for
// both j and j + M (the d rows negated).
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
// and grid point the planar form takes 0.75 N multiply-adds on the matrix
// cores, and about 14 VALU operations instead of 49.  Gain and x transform per
// 4096 points at 32^3 FP32 (M = 12, Nrho = 16): 22.6 ms against 62.5 ms for
// k_vhs_gain_rr with its Nyquist planes (29.5 ms with the even/odd split
// alone); 601 points FP64: 8.7 against 27.1 ms for the slab kernel (12.3); 24^3
// (Nrho = 12), 576 points: 1.7 against 2.9 ms FP32, 3.6 against 9.3 ms FP64,
// where 6 of 8 K steps of a part are filled.  The matrix cores are busy 42 % of
// the FP32 32^3 gain's cycles; 440 VALU instructions for 48 MFMA of a plane take
// about as long.
#pragma once
#include <hip/hip_runtime.h>

#include "cplx.hpp"
#include "spectral.hpp"

namespace dgfs {

template <typename T>
struct MmaTile;
// Row or column i of a tile belongs to register reg(i) of lane group grp(i) in
// the result layout (FP32: row 4 g + r, FP64: row 4 r + g).  mirror<RQ>(x):
// the value of the lane whose register index differs by ^ RQ.
template <>
struct MmaTile<float> {
  typedef float V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V4 mma(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ __forceinline__ constexpr int reg(int i) { return i & 3; }
  static __host__ __device__ __forceinline__ constexpr int grp(int i) { return i >> 2; }
  static __host__ __device__ __forceinline__ constexpr int at(int r, int g) { return 4 * g + r; }
  template <int RQ>
  static __device__ __forceinline__ float mirror(float x) {  // i ^ RQ within each quad
    constexpr int ctrl = RQ == 2 ? 0x4E : 0xB1;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xF, 0xF, true));
  }
};
template <>
struct MmaTile<double> {
  typedef double V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V4 mma(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ __forceinline__ constexpr int reg(int i) { return i >> 2; }
  static __host__ __device__ __forceinline__ constexpr int grp(int i) { return i & 3; }
  static __host__ __device__ __forceinline__ constexpr int at(int r, int g) { return 4 * r + g; }
  template <int RQ>
  static __device__ __forceinline__ double mirror(double x) {  // i ^ (4 RQ) within each 16
    int lo = __double2loint(x), hi = __double2hiint(x);
    if constexpr (RQ == 2) {  // row rotation by 8
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x128, 0xF, 0xF, true);
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x128, 0xF, 0xF, true);
    } else {  // half-row mirror (7 - i), then each quad reversed
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x141, 0xF, 0xF, true);
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x141, 0xF, 0xF, true);
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x1B, 0xF, 0xF, true);
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x1B, 0xF, 0xF, true);
    }
    return __hiloint2double(hi, lo);
  }
};

constexpr int kPlanarMaxGroups = 32;
constexpr int kPlanarMaxShifts = 16;
struct PlanarGroup {
  int pair;    // 0: (x, y), 1: (x, z), 2: (y, z)
  int ia, ib;  // shifts (indices of |component|) along u and v
};

template <typename T, int N>
struct PlanarShape {
  static constexpr int M = N / 2, Q = N / 4, NN = N * N, n = NN * N;
  static constexpr int RQ = (Q + 3) / 4;         // K steps (registers) of one part
  static constexpr int NT = (N == 16) ? 1 : 2;   // 16-wide tiles of an axis: j and j + M, or both in one
  static constexpr int NR = 4 * RQ;              // operand values per lane of one shift's matrices
  static constexpr int ND = NR * NT;             // operand values per lane of a plane
  static constexpr int plane = 64 * ND;
  static constexpr int LN = 16 * NT;             // values of a line, in tile order
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
  static constexpr int ln_elems = (XH == 2) ? 3 * N * LN : 4 * N * LN;
  static constexpr size_t lds_bytes = (static_cast<size_t>(s_elems) + ln_elems) * sizeof(T);
  // operand values of one point: the planes, the six Nyquist sums, three lines
  static constexpr size_t per_point = static_cast<size_t>(3 * N + 6) * plane + 4 * N;
  static constexpr int nslots = N / 2;  // real-plane pairs of T
  // planes of slot s
  static __host__ __device__ __forceinline__ constexpr int x1(int s) {
    return (XH == 1 || s < N / 4) ? s : s + N / 4;
  }
  static __host__ __device__ __forceinline__ constexpr int x2(int s) {
    return x1(s) + ((XH == 1) ? N / 2 : N / 4);
  }
  // index of output register r in lane group g; the mirror image (M - 1 - j,
  // in the same half of N) is register r ^ RQ of the same group
  static __host__ __device__ __forceinline__ constexpr int slot(int r, int g) {
    if (RQ == 2) return r < 2 ? 4 * r + g : M - 1 - 4 * (r - 2) - g;
    return ((r & 1) ? M - 1 - g : g) + ((r & 2) ? M : 0);
  }
  // whether the register holds anything (Q = 6 at N = 24 leaves gaps)
  static __host__ __device__ __forceinline__ constexpr bool filled(int r, int g) {
    return RQ == 1 || 4 * (r & 1) + g < Q;
  }
  // tile and register of part `sub` (ce, co, de, do), index 4 q + g, on the
  // lane axis of a plane
  static __host__ __device__ __forceinline__ constexpr int part_tile(int sub) { return NT == 2 ? sub >> 1 : 0; }
  static __host__ __device__ __forceinline__ constexpr int part_reg(int sub, int q) {
    return NT == 2 ? 2 * (sub & 1) + q : sub;
  }
  static_assert(N == 16 || N == 24 || N == 32, "tiles of N/2 <= 16 rows");
};

// ---------------------------------------------------------------------------
// Operand form of the points: per axis pair and plane of the third axis the
// parts (ce, co, de, do) x (ce, co, de, do) of f along both axes, stored as the
// gain's lanes hold them:
//   [pair][s][lane][K step q][v tile][u part], u index 4 q + lane / 16, v by lane % 16,
// followed by the six Nyquist sums (same form, the plane index on the lanes) and
// the three lines f^_uv(s).  A workgroup takes a point; the x-planes with one
// residue of their part index modulo 4 (four mirror and half-shift images of
// each) pass through LDS at a time, read once from f.  Bound by its stores (3 n
// values per point).
// ---------------------------------------------------------------------------
template <typename T>
struct PlanarPrepArgs {
  const double* f;  // [npts][n]
  T* op;            // [npts][per_point]
  int npts;
};

template <typename T, int N, int NTH>
__global__ __launch_bounds__(NTH, NTH / 128) void k_planar_prep(PlanarPrepArgs<T> a) {
  using PS = PlanarShape<T, N>;
  using MT = MmaTile<T>;
  constexpr int M = PS::M, Q = PS::Q, RQ = PS::RQ, NT = PS::NT, NN = PS::NN, n = PS::n, ND = PS::ND, PLN = PS::plane;
  constexpr int PP = N * (N + 1), NQ = 4 * RQ, KP = 4 * RQ;  // staged planes, part indices (with gaps)
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* pl = reinterpret_cast<T*>(smem_raw);  // [NQ][N][N + 1]
  T* fx = pl + NQ * PP;                    // Nyquist sums over x: [y][z]
  T* fy = fx + PP;                         // over y: [x][z]
  T* fz = fy + PP;                         // over z: [x][y]
  const int tid = threadIdx.x;
  // image m of part index k: k, M - 1 - k, k + M, N - 1 - k
  auto image = [](int k, int m) { return ((m & 1) ? M - 1 - k : k) + ((m & 2) ? M : 0); };
  auto parts = [](double p0, double p1, double p2, double p3, double* o) {
    const double s = p0 + p2, t = p1 + p3, d = p0 - p2, e = p1 - p3;
    o[0] = s + t;
    o[1] = s - t;
    o[2] = d + e;
    o[3] = d - e;
  };
  // the 4 x 4 parts of f(image(ku, .), image(kv, .)) into a plane; get(mu, mv)
  // gives the value, `on` whether the indices exist
  auto put = [&](T* P, int ku, int kv, bool on, auto&& get) {
    double h[4][4];  // [v image][u part]
#pragma unroll
    for (int mv = 0; mv < 4; ++mv) {
      if (on)
        parts(get(0, mv), get(1, mv), get(2, mv), get(3, mv), h[mv]);
      else
        h[mv][0] = h[mv][1] = h[mv][2] = h[mv][3] = 0.0;
    }
    double o[4][4];  // [u part][v part]
#pragma unroll
    for (int su = 0; su < 4; ++su) parts(h[0][su], h[1][su], h[2][su], h[3][su], o[su]);
#pragma unroll
    for (int sv = 0; sv < 4; ++sv) {
      const int i = MT::at(PS::part_reg(sv, kv >> 2), kv & 3);
      T* d = P + (16 * (ku & 3) + i) * ND + ((ku >> 2) * NT + PS::part_tile(sv)) * 4;
#pragma unroll
      for (int su = 0; su < 4; ++su) d[su] = static_cast<T>(0.0625 * o[su][sv]);
    }
  };
  for (int pt = xcd_slot(); pt < a.npts; pt += gridDim.x) {
    const double* f = a.f + static_cast<size_t>(pt) * n;
    T* op = a.op + static_cast<size_t>(pt) * PS::per_point;
    for (int e = tid; e < PP; e += NTH) fx[e] = T(0);
    for (int g = 0; g < 4; ++g) {
      const int nq = (4 * (RQ - 1) + g < Q) ? NQ : NQ - 4;  // planes whose part index exists
      __syncthreads();
      for (int e = tid; e < nq * NN; e += NTH) {
        const int q = e / NN, rem = e - q * NN, y = rem / N, z = rem - y * N;
        pl[q * PP + y * (N + 1) + z] = static_cast<T>(f[image(4 * (q >> 2) + g, q & 3) * NN + rem]);
      }
      __syncthreads();
      // what is formed of the staged planes, as one range of tasks: the three
      // axis pairs' parts (whole waves each), then the Nyquist sums
      constexpr int EA = RQ * KP * N, EB = 2 * EA;
      static_assert(EA % 64 == 0, "a wave's tasks are of one kind");
      const int EC = EB + nq * KP * KP, ED = EC + NN, EE = ED + nq * N;
      for (int e = tid; e < EE; e += NTH) {
        if (e < EA) {  // (x, y), plane z = s
          const int s = e % N, kv = (e / N) % KP, r = e / (N * KP), ku = 4 * r + g;
          const T* p0 = pl + 4 * r * PP;
          put(op + static_cast<size_t>(s) * PLN, ku, kv, ku < Q && kv < Q,
              [&](int mu, int mv) -> double { return p0[mu * PP + image(kv, mv) * (N + 1) + s]; });
        } else if (e < EB) {  // (x, z), plane y = s
          const int t = e - EA, kv = t % KP, s = (t / KP) % N, r = t / (N * KP), ku = 4 * r + g;
          const T* p0 = pl + 4 * r * PP + s * (N + 1);
          put(op + static_cast<size_t>(N + s) * PLN, ku, kv, ku < Q && kv < Q,
              [&](int mu, int mv) -> double { return p0[mu * PP + image(kv, mv)]; });
        } else if (e < EC) {  // (y, z), plane x
          const int t = e - EB, kv = t % KP, ku = (t / KP) % KP, q = t / (KP * KP);
          const int x = image(4 * (q >> 2) + g, q & 3);
          const T* p0 = pl + q * PP;
          put(op + static_cast<size_t>(2 * N + x) * PLN, ku, kv, ku < Q && kv < Q,
              [&](int mu, int mv) -> double { return p0[image(ku, mu) * (N + 1) + image(kv, mv)]; });
        } else if (e < ED) {
          const int t = e - EC, y = t / N, z = t - y * N;
          double s = 0.0;
          for (int q = 0; q < nq; ++q) {
            const double v = pl[q * PP + y * (N + 1) + z];
            s += ((g + q) & 1) ? -v : v;  // images 1 and 3 have the other parity (M is even)
          }
          fx[y * (N + 1) + z] = static_cast<T>(static_cast<double>(fx[y * (N + 1) + z]) + s);
        } else {
          const int d = e - ED, q = d / N, i = d - q * N, x = image(4 * (q >> 2) + g, q & 3);
          double s = 0.0, t = 0.0;
          for (int j = 0; j < N; ++j) {
            const double v = pl[q * PP + j * (N + 1) + i], w = pl[q * PP + i * (N + 1) + j];
            s += (j & 1) ? -v : v;
            t += (j & 1) ? -w : w;
          }
          fy[x * (N + 1) + i] = static_cast<T>(s);
          fz[x * (N + 1) + i] = static_cast<T>(t);
        }
      }
    }
    __syncthreads();
    T* ny = op + static_cast<size_t>(3 * N) * PLN;
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
    for (int e = tid; e < 6 * 64 * RQ * NT; e += NTH) {
      const int t = e % NT, r = (e / NT) % RQ, lane = (e / (NT * RQ)) & 63, w = e / (64 * RQ * NT);
      const int g = lane >> 4, i = lane & 15, k = 4 * r + g;
      const int s = PS::slot(MT::reg(i), MT::grp(i)) + t * M;
      double o[4] = {0.0, 0.0, 0.0, 0.0};
      if (k < Q && PS::filled(MT::reg(i), MT::grp(i)))
        parts(src(w, image(k, 0), s), src(w, image(k, 1), s), src(w, image(k, 2), s), src(w, image(k, 3), s), o);
      T* d = ny + w * PLN + lane * ND + (r * NT + t) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = static_cast<T>(0.25 * o[j]);
    }
    T* line = ny + 6 * PLN;
    for (int e = tid; e < 3 * N; e += NTH) {
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
  const T* smat;      // [Nrho][nshift][64][NR] operand values of R(shift), per lane [part][K step]
  const double* beta; // [Nrho][nshift]
  cpx<T>* Tb;         // [npts][Nrho][gsplit][N/2][N][N]
  int nitems, ngroups, ppg, Nrho, nshift, ngr;
  int gsplit;  // parts of the groups, each a work item of its own
  PlanarGroup gr[kPlanarMaxGroups];
};

// products of the four parts with their matrices: Gc, Hc from ce, co and Gd, Hd
// from de, do; x and S are indexed [part][K step].  DATA_A: the data is the A
// operand (its lanes become the result's rows), else the B operand.  Gc
// starts at `init`, the others at zero.
template <typename T, int RQ, bool DATA_A>
__device__ __forceinline__ void pair_move(const T (&x)[4 * RQ], const T (&S)[4 * RQ], typename MmaTile<T>::V4 init,
                                          typename MmaTile<T>::V4 (&o)[4]) {
  using MT = MmaTile<T>;
  o[0] = init;
  o[1] = o[2] = o[3] = typename MT::V4{T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int p = 0; p < 4; ++p)
      o[p] = DATA_A ? MT::mma(x[p * RQ + q], S[p * RQ + q], o[p]) : MT::mma(S[p * RQ + q], x[p * RQ + q], o[p]);
}

// the two moves of one register from its four products: pa, pb at j and j + M
// for the shift, ma, mb at the mirror images of j and j + M for the opposite
// shift (NT = 1: j + M is in the products' rows, pb and mb are not formed)
template <typename T, int NT>
__device__ __forceinline__ void pair_sums(T gc, T hc, T gd, T hd, T& pa, T& pb, T& ma, T& mb) {
  const T c = gc + hc, d = gd + hd, e = gc - hc, f = gd - hd;
  pa = c + d;
  ma = e + f;
  if constexpr (NT == 2) {
    pb = c - d;
    mb = e - f;
  }
}

// the planes of one group: PAIR fixes which axes u, v and the plane index are.
// The operand values of the next plane are in flight during the second move,
// and the group's lines and the previous sum of S are read ahead of the
// products that use them.
template <typename T, int N, int PAIR>
__device__ __forceinline__ void planar_planes(const T* op, const T (&Sa)[PlanarShape<T, N>::NR],
                                              const T (&Sb)[PlanarShape<T, N>::NR], T bab, T* S, const T* ln, int half,
                                              bool first) {
  using PS = PlanarShape<T, N>;
  using MT = MmaTile<T>;
  using V4 = typename MT::V4;
  constexpr int RQ = PS::RQ, M = PS::M, NT = PS::NT, ND = PS::ND, XH = PS::XH, NX = PS::NX, NW = PS::NW, LN = PS::LN;
  constexpr bool HALF_U = XH == 2 && PAIR < 2;         // only the u tile of this x-half is wanted
  constexpr int NU = HALF_U ? 1 : NT;                  // u tiles
  constexpr int NS = (XH == 2 && PAIR == 2) ? NX : N;  // planes of the item
  constexpr int LU = HALF_U ? 16 : LN;                 // u values of the lines
  // strides of S along u, v and the plane index
  constexpr int TU = PAIR == 2 ? PS::PY : PS::PX, TV = PAIR == 0 ? PS::PY : 1;
  constexpr int TS = PAIR == 0 ? 1 : PAIR == 1 ? PS::PY : PS::PX;
  const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ri = MT::reg(i), gi = MT::grp(i);
  const bool ok = PS::filled(ri, gi);
  const int cu = ok ? PS::slot(ri, gi) : 0;  // this lane's u (in its tile)
  const T* eU = ln + 4 * g;                  // [s][LN]: tile, lane group, register
  const T* dU = eU + NS * LN;
  const T* eV = ln + 2 * NS * LN + 4 * gi + ri;  // [s][LU]
  const T* dV = eV + NS * LU;
  const T* line = op + static_cast<size_t>(3 * N + 6) * PS::plane + PAIR * N;
  // -w_u w_v beta_a beta_b of register 0: the sign changes with the mirror images
  const T sg = (((gi + g) & 1) != ((ri & RQ) != 0)) ? bab : -bab;
  T* S0 = S + cu * TU;
  // register r of v: the rows 4 r + g (or g, M + g) from one base, their mirror
  // images from another
  auto vrow = [&](T* b, int r) -> T* {
    const bool mir = (r & RQ) != 0;
    const int off = (RQ == 2) ? (mir ? 4 * (3 - r) : 4 * r) : ((r & 2) ? M : 0);
    return b + (mir ? (M - 1 - 4 * (RQ - 1) - g) * TV : g * TV) + off * TV;
  };
  const T* P0 = op + static_cast<size_t>(PAIR * N) * PS::plane + lane * ND;
  auto plane = [&](int sl) { return (PAIR == 2 && XH == 2 && half) ? sl + M : sl; };
  T fr[ND], l0;
  {
    const int s = plane(w);
    const T* P = P0 + static_cast<size_t>(s) * PS::plane;
#pragma unroll
    for (int k = 0; k < ND; ++k) fr[k] = P[k];
    l0 = line[s];
  }
#pragma unroll 1
  for (int sl = w; sl < NS; sl += NW) {
    const T ck = sg * l0;
    // move along u: lanes u, registers v.  Xp[u tile] at u, Xm[u tile] at the
    // mirror image of u; both [v part][K step] as the second move reads them
    T Xp[NU][PS::NR], Xm[NU][PS::NR];
    const V4 z4{T(0), T(0), T(0), T(0)};
    V4 o1[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      T x[PS::NR];
#pragma unroll
      for (int q = 0; q < RQ; ++q)
#pragma unroll
        for (int p = 0; p < 4; ++p) x[p * RQ + q] = fr[(q * NT + t) * 4 + p];
      pair_move<T, RQ, true>(x, Sa, z4, o1[t]);
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int t = PS::part_tile(p), r = PS::part_reg(p, q);
        T pa, pb = T(0), ma, mb = T(0);
        pair_sums<T, NT>(o1[t][0][r], o1[t][1][r], o1[t][2][r], o1[t][3][r], pa, pb, ma, mb);
        if constexpr (HALF_U) {
          Xp[0][p * RQ + q] = half ? pb : pa;
          Xm[0][p * RQ + q] = half ? mb : ma;
        } else {
          Xp[0][p * RQ + q] = pa;
          Xm[0][p * RQ + q] = ma;
          Xp[NU - 1][p * RQ + q] = NT == 2 ? pb : pa;
          Xm[NU - 1][p * RQ + q] = NT == 2 ? mb : ma;
        }
      }
    {  // the next plane (the last iteration reads its own again)
      const int s = plane(sl + NW < NS ? sl + NW : sl);
      const T* P = P0 + static_cast<size_t>(s) * PS::plane;
#pragma unroll
      for (int k = 0; k < ND; ++k) fr[k] = P[k];
      l0 = line[s];
    }
    T ul[NT][4], dl[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ul[t][r] = eU[sl * LN + 16 * t + r];
        dl[t][r] = dU[sl * LN + 16 * t + r];
      }
#pragma unroll
    for (int t = 0; t < NU; ++t) {
      T* B = S0 + sl * TS + t * M * TU;
      T prev[NT][4];
#pragma unroll
      for (int v = 0; v < NT; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) prev[v][r] = T(0);
      if (!first) {
#pragma unroll
        for (int v = 0; v < NT; ++v)
#pragma unroll
          for (int r = 0; r < 4; ++r) prev[v][r] = vrow(B + v * M * TV, r)[0];
      }
      const V4 init = (RQ == 2) ? V4{ck, ck, -ck, -ck} : V4{ck, -ck, ck, -ck};
      V4 op2[4], om2[4];
      pair_move<T, RQ, false>(Xp[t], Sb, init, op2);
      pair_move<T, RQ, false>(Xm[t], Sb, init, om2);
      // Z(+,+) = pp, Z(+,-) = pm (rows mirrored), Z(-,+) = mp (lanes mirrored),
      // Z(-,-) = mm (both)
      T pp[2][4], pm[2][4], mp[2][4], mm[2][4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pair_sums<T, NT>(op2[0][r], op2[1][r], op2[2][r], op2[3][r], pp[0][r], pp[1][r], pm[0][r], pm[1][r]);
        pair_sums<T, NT>(om2[0][r], om2[1][r], om2[2][r], om2[3][r], mp[0][r], mp[1][r], mm[0][r], mm[1][r]);
      }
      const T ev = eV[sl * LU + 16 * t], dv = dV[sl * LU + 16 * t];
      T q[NT][4];
#pragma unroll
      for (int v = 0; v < NT; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T x = ul[v][r] + ev - dl[v][r] * dv;
          x += MT::template mirror<RQ>(mm[v][r ^ RQ]) * pp[v][r];
          x += MT::template mirror<RQ>(mp[v][r]) * pm[v][r ^ RQ];
          q[v][r] = prev[v][r] + x;
        }
      if (ok) {
#pragma unroll
        for (int v = 0; v < NT; ++v)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (PS::filled(r, g)) vrow(B + v * M * TV, r)[0] = q[v][r];
      }
    }
  }
}

template <typename T, int N>
__global__ __launch_bounds__((PlanarShape<T, N>::NW * 64), (PlanarShape<T, N>::WPE)) void k_vhs_gain_planar(
    PlanarGainArgs<T> a) {
  using PS = PlanarShape<T, N>;
  using MT = MmaTile<T>;
  using V4 = typename MT::V4;
  constexpr int RQ = PS::RQ, M = PS::M, NT = PS::NT, NN = PS::NN, NR = PS::NR, ND = PS::ND, LN = PS::LN;
  constexpr int XH = PS::XH, NX = PS::NX, NW = PS::NW;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* S = reinterpret_cast<T*>(smem_raw);
  T* ln = S + PS::s_elems;
  const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ri = MT::reg(i), gi = MT::grp(i);
  for (int item = xcd_slot(); item < a.nitems; item += gridDim.x) {
    const int half = (XH == 2) ? item % 2 : 0, part = (item / XH) % a.gsplit, pg = item / (XH * a.gsplit);
    const int pt = pg / a.ngroups, grp = pg - pt * a.ngroups;
    const int gr0 = part * a.ngr / a.gsplit, gr1 = (part + 1) * a.ngr / a.gsplit;
    const int p0 = grp * a.ppg, p1 = min(p0 + a.ppg, a.Nrho);
    const T* op = a.op + static_cast<size_t>(pt) * PS::per_point;
    for (int p = p0; p < p1; ++p) {
      for (int gr = gr0; gr < gr1; ++gr) {
        const int pair = a.gr[gr].pair, ia = a.gr[gr].ia, ib = a.gr[gr].ib;
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
        const int NS = half_s ? NX : N, LU = half_u ? 16 : LN;
        __syncthreads();  // the previous group's (or p's) readers of the lines and of S are done
        if (w < 4) {
          // lines of the group: wave 2 * (V line) + (tile of the plane index)
          const bool vline = w & 2;
          const int st = w & 1;
          if (st < NT && (!half_s || st == half)) {
            const T* P = op + static_cast<size_t>(3 * N + 2 * pair + (vline ? 1 : 0)) * PS::plane + lane * ND;
            T x[NR];
#pragma unroll
            for (int q = 0; q < RQ; ++q)
#pragma unroll
              for (int p4 = 0; p4 < 4; ++p4) x[p4 * RQ + q] = P[(q * NT + st) * 4 + p4];
            const V4 z4{T(0), T(0), T(0), T(0)};
            V4 o[4];
            if (vline)
              pair_move<T, RQ, true>(x, Sa, z4, o);
            else
              pair_move<T, RQ, true>(x, Sb, z4, o);
            const T e2 = vline ? T(2) * bb * bb : T(2) * ba * ba;
            // w of this lane's index (the same at j + M) times the other shift's beta
            const T ds = (((gi & 1) != ((ri & RQ) != 0)) ? T(-1) : T(1)) * (vline ? ba : bb);
            const int LL = vline ? LU : LN;
            T* e = ln + (vline ? 2 * NS * LN : 0) + 4 * gi + ri;
            T* d = e + NS * LL;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              T pa, pb = T(0), ma, mb = T(0);
              pair_sums<T, NT>(o[0][r], o[1][r], o[2][r], o[3][r], pa, pb, ma, mb);
              ma = MT::template mirror<RQ>(ma);
              mb = MT::template mirror<RQ>(mb);
              const int s = PS::slot(r, g) + ((half_s || NT == 1) ? 0 : st * M);
              if (PS::filled(r, g) && PS::filled(ri, gi)) {
                if (vline && half_u) {
                  e[s * LL] = half ? e2 * pb * mb : e2 * pa * ma;
                  d[s * LL] = half ? ds * (pb - mb) : ds * (pa - ma);
                } else {
                  e[s * LL] = e2 * pa * ma;
                  d[s * LL] = ds * (pa - ma);
                  if constexpr (NT == 2) {
                    e[s * LL + 16] = e2 * pb * mb;
                    d[s * LL + 16] = ds * (pb - mb);
                  }
                }
              }
            }
          }
        }
        __syncthreads();
        const bool first = gr == gr0;
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
          cpx<T>* t = a.Tb + (((static_cast<size_t>(pt) * a.Nrho + p) * a.gsplit + part) * PS::nslots + half * NPP + pp) * NN + l;
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
// (-ky, -kz) too.  The kx sums are kept in registers over p: all in FP32, half
// of them per wave in FP64.  Bound by reading T where the pencils fill the
// chip; PW > 1 spreads the sum over p of 64 pencils over PW waves for batches
// that leave it idle (one point at 24^3 FP32: 51 us with one wave per pencil
// block, whose 12 reads of T follow one another; the whole call went from 179
// to 112 us with both splits).
template <typename T>
struct PlanarXfwdArgs {
  const cpx<T>* Tb;
  const T* b1;        // [Nrho][n]
  const double* wgt;  // [Nrho]
  cpx<T>* Ghat;       // [npts][n]
  int npts, Nrho, gsplit;
};

template <typename T, int N, int K0, int KN>
__device__ __forceinline__ void planar_xfwd_sum(const PlanarXfwdArgs<T>& a, int pt, int i1, int i2, int q0, int dq,
                                                cpx<T> (&acc)[KN]) {
  using PS = PlanarShape<T, N>;
  constexpr int NN = N * N, n = NN * N;
#pragma unroll
  for (int k = 0; k < KN; ++k) acc[k] = cpx<T>{T(0), T(0)};
  for (int q = q0; q < a.Nrho * a.gsplit; q += dq) {
    const int p = q / a.gsplit;
    const cpx<T>* Tp = a.Tb + (static_cast<size_t>(pt) * a.Nrho * a.gsplit + q) * PS::nslots * NN;
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
}

template <typename T, int N, int K0, int KN, int PW>
__device__ __forceinline__ void planar_xfwd_part(const PlanarXfwdArgs<T>& a, cpx<T>* red, int col, int w) {
  constexpr int NN = N * N, n = NN * N, NV = (N / 2 + 1) * N;
  const int lane = threadIdx.x & 63;
  bool act = col < a.npts * NV;
  const int pt = act ? col / NV : 0, i1 = act ? col - pt * NV : 0, ky = i1 / N, kz = i1 - ky * N;
  const int i2 = ((N - ky) % N) * N + (N - kz) % N;
  // on the self-conjugate rows ky = 0 and N/2 the second half of kz is the
  // mirror image of the first
  if ((ky == 0 || ky == N / 2) && kz > N / 2) act = false;
  if (PW == 1 && !act) return;
  cpx<T> acc[KN];
  if (act) planar_xfwd_sum<T, N, K0, KN>(a, pt, i1, i2, PW > 1 ? w : 0, PW, acc);
  if constexpr (PW > 1) {
    wave_tree_sum<T, KN, PW>(acc, red, w, lane, act);
    if (w) return;
  }
  if (!act) return;
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

// threads of a workgroup
template <int PW>
constexpr int xfwd_threads() {
  return PW > 1 ? 64 * PW : 256;
}
// pencils per workgroup (FP64: two waves, or two workgroups, per 64 pencils)
template <typename T, int PW>
constexpr int xfwd_pencils() {
  return PW > 1 ? 64 : (sizeof(T) == 8 ? 128 : 256);
}

template <typename T, int N, int PW>
__global__ __launch_bounds__((xfwd_threads<PW>()), (PW == 1 && sizeof(T) == 4 ? 3 : 1)) void k_planar_xfwd(PlanarXfwdArgs<T> a) {
  constexpr int SPLIT = sizeof(T) == 8 ? 2 : 1, KN = N / SPLIT;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x & 63;
  if constexpr (PW > 1) {
    __shared__ cpx<T> red[PW / 2 * KN * 64];
    const int col = static_cast<int>(blockIdx.x / SPLIT) * 64 + lane;
    if (SPLIT == 2 && (blockIdx.x & 1))
      planar_xfwd_part<T, N, N - KN, KN, PW>(a, red, col, w);
    else
      planar_xfwd_part<T, N, 0, KN, PW>(a, red, col, w);
  } else {
    const int col = static_cast<int>(blockIdx.x) * xfwd_pencils<T, 1>() + (w / SPLIT) * 64 + lane;
    if (SPLIT == 2 && (w & 1))
      planar_xfwd_part<T, N, N - KN, KN, 1>(a, nullptr, col, 0);
    else
      planar_xfwd_part<T, N, 0, KN, 1>(a, nullptr, col, 0);
  }
}

}  // namespace dgfs
