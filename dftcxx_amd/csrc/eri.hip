// Analytic two-electron integrals and the Coulomb matrix from them, the
// reference's alternative Hartree path (hartree_evaluation =
// two_electron_integrals): DFT::calculate_two_electron_integrals
// (src/dft.cpp:254-288) computes every unique (ij|kl) once, and
// DFT::calculate_hartree_potential_te_int (src/dft.cpp:452-477) forms
// J_ij = sum_kl P_kl (ij|kl) every iteration.
//
// Here the integrals come from the McMurchie-Davidson scheme (Hermite
// expansion of each product Gaussian, Hermite Coulomb integrals R_tuv by the
// recursion on the Boys function) rather than the reference's
// Taketa-Huzinaga-O-ohata sums (src/integrals.cpp:389-468); both are exact, so
// they agree to rounding.  The prefactor 2 pi^(5/2) and the primitive norms
// use the reference's pi = 3.14159265359 (src/integrals.cpp:394, src/cgf.cpp:103),
// and the Boys argument is clamped to >= 1e-8 as src/gamma.cpp:41-46 does.
//
// Layout: function pairs IJ = i(i+1)/2 + j (i >= j) and integrals at
// IJ(IJ+1)/2 + KL (IJ >= KL), the reference's teindex (src/integrals.cpp:470-486).
//
// Quartets of s and p shells (every shipped basis) are evaluated by shell: a team of
// lanes forms all integrals of one shell quartet, so the Boys function and the R_tuv
// of a primitive quartet are computed once for its 1 to 81 integrals and stay in
// registers (k_eri_shell).  Integrals with a d function go one thread each through
// records of every function pair's Hermite coefficients (k_eri).  Benzene / 6-31G,
// 2.4 million integrals: one thread per integral for all of them took 31 ms, bound by
// repeated Boys series and by R arrays in scratch memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/dftgrid.h"
#include "device_math.h"
#include "grid_tables.h"
#include "unroll.h"

namespace {

using dg::rsqrt64;
using dg::static_for;

constexpr int kRec = 20;         // doubles per primitive-pair record
constexpr int kMaxLsum = 8;      // (dd|dd): four Cartesian d functions
constexpr double kPiTrunc = 3.14159265359;

int fail(int code, const std::string& msg) {
  dg::set_last_error(msg);
  return code;
}

#define ERI_HIP(expr)                                                                     \
  do {                                                                                    \
    hipError_t _e = (expr);                                                               \
    if (_e != hipSuccess) return fail(DG_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
  } while (0)

const int kCart[3][6][3] = {{{0, 0, 0}},
                            {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}},
                            {{2, 0, 0}, {1, 1, 0}, {1, 0, 1}, {0, 2, 0}, {0, 1, 1}, {0, 0, 2}}};

// Hermite expansion coefficients E^{ij}_t (t = 0..i+j) of x_A^i x_B^j exp(-a x_A^2 - b x_B^2)
// about the product centre, E^{00}_0 = exp(-ab/(a+b) X_AB^2); i, j <= 2.
void hermite_1d(int i, int j, double a, double b, double xa, double xb, double* E /* [5] */) {
  double e[3][3][5];
  std::memset(e, 0, sizeof(e));
  const double p = a + b, xp = (a * xa + b * xb) / p;
  const double xpa = xp - xa, xpb = xp - xb, o2p = 0.5 / p;
  e[0][0][0] = std::exp(-a * b / p * (xa - xb) * (xa - xb));
  for (int ii = 0; ii <= i; ++ii)
    for (int jj = 0; jj <= j; ++jj) {
      if (ii == 0 && jj == 0) continue;
      const double(*s)[5] = ii > 0 ? e[ii - 1] : e[ii];
      const double* src = ii > 0 ? s[jj] : s[jj - 1];
      const double x = ii > 0 ? xpa : xpb;
      for (int t = 0; t <= ii + jj; ++t)
        e[ii][jj][t] = x * src[t] + (t + 1 <= 4 ? (t + 1) * src[t + 1] : 0.0) + (t > 0 ? o2p * src[t - 1] : 0.0);
    }
  for (int t = 0; t < 5; ++t) E[t] = t <= i + j ? e[i][j][t] : 0.0;
}

// Boys function F_n(T), n = 0..nmax, T clamped to >= 1e-8 (src/gamma.cpp:41-46):
// series e^{-T} sum_k (2T)^k / ((2n+1)(2n+3)...(2n+2k+1)) and downward recursion
// below T = 40, F_0 = sqrt(pi/T)/2 and upward recursion above.
__device__ void boys_dev(int nmax, double T, double* F) {
  T = fmax(fabs(T), 1e-8);
  const double et = exp(-T);
  if (T < 40.0) {
    double term = 1.0 / (2 * nmax + 1), sum = term;
    for (int k = 1; k < 400; ++k) {
      term *= 2.0 * T / (2 * nmax + 2 * k + 1);
      sum += term;
      if (term < 1e-17 * sum) break;
    }
    F[nmax] = et * sum;
    for (int n = nmax; n > 0; --n) F[n - 1] = (2.0 * T * F[n] + et) / (2 * n - 1);
  } else {
    F[0] = 0.5 * sqrt(3.14159265358979323846 / T);
    for (int n = 0; n < nmax; ++n) F[n + 1] = ((2 * n + 1) * F[n] - et) / (2.0 * T);
  }
}

// index of (t, u, v), t + u + v = s, in the Hermite tetrahedron
__device__ __forceinline__ int tuv(int t, int u, int v) {
  const int s = t + u + v, m = u + v;
  return s * (s + 1) * (s + 2) / 6 + m * (m + 1) / 2 + v;
}

// One unique contracted integral (IJ|KL) per thread, IJ >= KL, written at
// IJ(IJ+1)/2 + KL, where one of its four functions is a d function (pair_d).  pair_off: primitive-pair records of pair IJ are
// [pair_off[IJ], pair_off[IJ+1]); pair_l: per pair the Hermite orders
// (lx_i + lx_j, ly_i + ly_j, lz_i + lz_j).  LMAX bounds the total order.
template <int LMAX>
__global__ __launch_bounds__(256) void k_eri(long nints, const int* __restrict__ pair_off,
                                             const int* __restrict__ pair_l, const int* __restrict__ pair_d,
                                             const double* __restrict__ rec, double* ints) {
  constexpr int NT = (LMAX + 1) * (LMAX + 2) * (LMAX + 3) / 6;
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nints) return;
  long IJ = (long)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
  while (IJ * (IJ + 1) / 2 > q) --IJ;
  while ((IJ + 1) * (IJ + 2) / 2 <= q) ++IJ;
  const long KL = q - IJ * (IJ + 1) / 2;
  if (!(pair_d[IJ] | pair_d[KL])) return;
  const int ax = pair_l[3 * IJ], ay = pair_l[3 * IJ + 1], az = pair_l[3 * IJ + 2];
  const int cx = pair_l[3 * KL], cy = pair_l[3 * KL + 1], cz = pair_l[3 * KL + 2];
  const int L = ax + ay + az + cx + cy + cz;
  double Ra[NT], Rb[NT], F[LMAX + 1];
  double total = 0.0;
  for (int ab = pair_off[IJ]; ab < pair_off[IJ + 1]; ++ab) {
    const double* A = rec + (long)ab * kRec;
    const double p = A[0];
    for (int cd = pair_off[KL]; cd < pair_off[KL + 1]; ++cd) {
      const double* C = rec + (long)cd * kRec;
      const double qe = C[0];
      const double X = A[1] - C[1], Y = A[2] - C[2], Z = A[3] - C[3];
      const double al = p * qe / (p + qe);
      boys_dev(L, al * (X * X + Y * Y + Z * Z), F);
      // R^n_tuv from n = L down to 0 (two levels in Ra / Rb)
      double* cur = Ra;
      double* nxt = Rb;
      double m2a = 1.0;
      for (int k = 0; k < L; ++k) m2a *= -2.0 * al;
      cur[0] = m2a * F[L];
      for (int n = L - 1; n >= 0; --n) {
        m2a /= -2.0 * al;
        const int lev = L - n;
        for (int s = 0; s <= lev; ++s)
          for (int t = s; t >= 0; --t)
            for (int v = 0; v <= s - t; ++v) {
              const int u = s - t - v;
              double r;
              if (s == 0)
                r = m2a * F[n];
              else if (t > 0)
                r = (t > 1 ? (t - 1) * cur[tuv(t - 2, u, v)] : 0.0) + X * cur[tuv(t - 1, u, v)];
              else if (u > 0)
                r = (u > 1 ? (u - 1) * cur[tuv(t, u - 2, v)] : 0.0) + Y * cur[tuv(t, u - 1, v)];
              else
                r = (v > 1 ? (v - 1) * cur[tuv(t, u, v - 2)] : 0.0) + Z * cur[tuv(t, u, v - 1)];
              nxt[tuv(t, u, v)] = r;
            }
        double* tmp = cur;
        cur = nxt;
        nxt = tmp;
      }
      double val = 0.0;
      for (int t = 0; t <= ax; ++t)
        for (int u = 0; u <= ay; ++u)
          for (int v = 0; v <= az; ++v) {
            const double eab = A[5 + t] * A[10 + u] * A[15 + v];
            double inner = 0.0;
            for (int tt = 0; tt <= cx; ++tt)
              for (int uu = 0; uu <= cy; ++uu)
                for (int vv = 0; vv <= cz; ++vv) {
                  const double ecd = C[5 + tt] * C[10 + uu] * C[15 + vv];
                  const double r = cur[tuv(t + tt, u + uu, v + vv)];
                  inner += ((tt + uu + vv) & 1) ? -ecd * r : ecd * r;
                }
            val += eab * inner;
          }
      const double pref = 2.0 * pow(kPiTrunc, 2.5) / (p * qe * sqrt(p + qe));
      total += pref * A[4] * C[4] * val;
    }
  }
  ints[q] = total;
}

// --- quartets of s and p shells ------------------------------------------------

enum { kSS = 0, kSP = 1, kPP = 2 };  // shell-pair types; also their Hermite order

// One primitive pair of a shell pair.
struct PairRec {
  double p, P[3];  // exponent sum, centre
  double K;        // c_a N_a c_b N_b exp(-ab/(a+b) |A-B|^2) / p
  double h;        // 1 / 2p
  double A[3];     // SP: P - (the p shell's centre); PP: P - A
  double B[3];     // PP: P - B
};

struct ShellPair {
  int rec, n;    // primitive pairs rec[0..n)
  int i0, j0;    // first function of each shell, i0 >= j0
  int p_first;   // SP: 1 if the p shell is the one at i0
  int pad;
};

// Ket pairs one work-group takes: [first, first + n), 1 << lg lanes to a quartet.
struct KetBlock {
  int first, n, lg;
};

// Boys function F_n at T0 = row / 16 for the Taylor expansion of boys_tab: columns
// 0..11 F_n, column 15 exp(-T0).
constexpr int kBoysRows = 801, kBoysCols = 16;
constexpr double kBoysEnd = 50.0;
__global__ void k_boys_table(double* tab) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= kBoysRows) return;
  const double T = row / 16.0;
  double F[12];
  boys_dev(11, T, F);
  for (int n = 0; n < 12; ++n) tab[row * kBoysCols + n] = row ? F[n] : 1.0 / (2 * n + 1);  // (boys_dev clamps T)
  for (int n = 12; n < 15; ++n) tab[row * kBoysCols + n] = 0.0;
  tab[row * kBoysCols + 15] = exp(-T);
}

// F_n(T), n = 0..L, T clamped to >= 1e-8 (src/gamma.cpp:41-46).  Below T = 50, F_L by
// eight Taylor terms about the nearest table row (|d| <= 1/32: the ninth is below
// 3e-17 of the first) and downward recursion; above, F_0 = sqrt(pi/T)/2 and upward
// recursion without exp(-T), which is below 2e-17 of every F_n, n <= 4, there.
template <int L>
__device__ __forceinline__ void boys_tab(double T, const double* __restrict__ tab, double (&F)[L + 1]) {
  T = fmax(fabs(T), 1e-8);
  if (T < kBoysEnd) {
    const int row = (int)(T * 16.0 + 0.5);
    const double* t = tab + row * kBoysCols;
    const double d = row * (1.0 / 16.0) - T;
    double f = t[L + 7];
    static_for<0, 7>([&](auto k) { f = __fma_rn(f, d * (1.0 / (7 - k)), t[L + 6 - k]); });
    F[L] = f;
    if constexpr (L > 0) {
      double e = 1.0;  // exp(d)
      static_for<0, 8>([&](auto k) { e = __fma_rn(e, d * (1.0 / (8 - k)), 1.0); });
      e *= t[15];
      static_for<0, L>([&](auto k) {
        constexpr int n = L - k;
        F[n - 1] = __fma_rn(2.0 * T, F[n], e) * (1.0 / (2 * n - 1));
      });
    }
  } else {
    const double rs = rsqrt64(T), it = 0.5 * rs * rs;
    F[0] = 0.88622692545275801365 * rs;  // sqrt(pi)/2
    static_for<0, L>([&](auto n) { F[n + 1] = (2 * n + 1) * F[n] * it; });
  }
}

constexpr int hermite_count(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
constexpr int hermite_index(int t, int u, int v) {
  return (t + u + v) * (t + u + v + 1) * (t + u + v + 2) / 6 + (u + v) * (u + v + 1) / 2 + v;
}
struct Tuv {
  int t, u, v;
};
constexpr Tuv hermite_tuv(int idx) {
  int s = 0;
  while (hermite_count(s) <= idx) ++s;
  int r = idx - (s ? hermite_count(s - 1) : 0), m = 0;
  while ((m + 1) * (m + 2) / 2 <= r) ++m;
  const int v = r - m * (m + 1) / 2;
  return {s - m, m - v, v};
}

// R_tuv, t + u + v <= L, in place: level n+1 holds orders up to L - n - 1; level n's
// order s needs level n+1's s-1 and s-2, so descending s overwrites nothing needed.
template <int L>
__device__ __forceinline__ void hermite_coulomb(double al, double X, double Y, double Z, const double (&F)[L + 1],
                                                double (&R)[hermite_count(L)]) {
  double g[L + 1];
  double m2 = 1.0;
  static_for<0, L + 1>([&](auto n) {
    g[n] = m2 * F[n];
    m2 *= -2.0 * al;
  });
  R[0] = g[L];
  static_for<1, L + 1>([&](auto lev) {
    static_for<0, hermite_count(lev) - 1>([&](auto k) {
      constexpr int idx = hermite_count(lev) - 1 - k;
      constexpr Tuv c = hermite_tuv(idx);
      double r;
      if constexpr (c.t > 0) {
        r = X * R[hermite_index(c.t - 1, c.u, c.v)];
        if constexpr (c.t > 1) r = __fma_rn((double)(c.t - 1), R[hermite_index(c.t - 2, c.u, c.v)], r);
      } else if constexpr (c.u > 0) {
        r = Y * R[hermite_index(c.t, c.u - 1, c.v)];
        if constexpr (c.u > 1) r = __fma_rn((double)(c.u - 1), R[hermite_index(c.t, c.u - 2, c.v)], r);
      } else {
        r = Z * R[hermite_index(c.t, c.u, c.v - 1)];
        if constexpr (c.v > 1) r = __fma_rn((double)(c.v - 1), R[hermite_index(c.t, c.u, c.v - 2)], r);
      }
      R[idx] = r;
    });
    R[0] = g[L - lev];
  });
}

constexpr int hermite_add(int idx, int x, int y) {  // index of tuv(idx) + e_x + e_y (x, y = -1: none)
  const Tuv c = hermite_tuv(idx);
  return hermite_index(c.t + (x == 0) + (y == 0), c.u + (x == 1) + (y == 1), c.v + (x == 2) + (y == 2));
}

// sum over the Hermite functions of one function pair of type T of E_tuv sign^(t+u+v)
// V[tuv + base]: SS; SP with p component a; PP with components a, b.
template <int T, int SIGN, int A, int B, int BASE, int N>
__device__ __forceinline__ double hermite_sum(const PairRec& r, const double (&V)[N]) {
  if constexpr (T == kSS) return V[BASE];
  const double h = SIGN * r.h;
  if constexpr (T == kSP) return __fma_rn(h, V[hermite_add(BASE, A, -1)], r.A[A] * V[BASE]);
  if constexpr (T == kPP) {
    const double e0 = A == B ? __fma_rn(r.A[A], r.B[B], r.h) : r.A[A] * r.B[B];
    double s = e0 * V[BASE];
    if constexpr (A == B) {
      s = __fma_rn(h * (r.A[A] + r.B[B]), V[hermite_add(BASE, A, -1)], s);
    } else {
      s = __fma_rn(h * r.B[B], V[hermite_add(BASE, A, -1)], s);
      s = __fma_rn(h * r.A[A], V[hermite_add(BASE, B, -1)], s);
    }
    return __fma_rn(r.h * r.h, V[hermite_add(BASE, A, B)], s);
  }
  return 0.0;
}

constexpr int pair_functions(int T) { return T == kSS ? 1 : T == kSP ? 3 : 9; }

// All integrals of the shell quartets (bra pair | ket pairs), bra type BT <= ket type
// KT; with BT = KT the ket index runs up to the bra's.  One work-group: one bra pair
// (and for PP bras one of its first shell's three components, which keeps 27 sums per
// lane instead of 81) and the ket pairs of one KetBlock, one lane team each, the ket's
// primitive pairs dealt over the team.  The block's lists are sorted by descending
// primitive count, so a wave's teams run about equally long.  (pp|pp) keeps 27 sums,
// 35 R and 10 half-transformed values in registers; nothing is in scratch.
template <int BT, int KT>
__global__ __launch_bounds__(256) void k_eri_shell(const ShellPair* __restrict__ bras, int b0,
                                                   const ShellPair* __restrict__ kets,
                                                   const KetBlock* __restrict__ blocks, int nblocks,
                                                   const PairRec* __restrict__ rec, const double* __restrict__ tab,
                                                   double* __restrict__ ints) {
  constexpr int L = BT + KT, NB = BT == kSS ? 1 : 3, NK = pair_functions(KT);
  const KetBlock kb = blocks[blockIdx.x % nblocks];
  const int b = b0 + (int)(blockIdx.x / nblocks);
  const int lg = kb.lg, kt = kb.first + (int)(threadIdx.x >> lg), sub = threadIdx.x & ((1 << lg) - 1);
  if (kt >= kb.first + kb.n || (BT == KT && kt > b)) return;  // whole teams leave together
  const ShellPair bra = bras[b], ket = kets[kt];
  const int a = BT == kPP ? (int)blockIdx.y : 0;
  double acc[NB][NK];
  static_for<0, NB>([&](auto f) { static_for<0, NK>([&](auto k) { acc[f][k] = 0.0; }); });
  for (int cd = sub; cd < ket.n; cd += 1 << lg) {
    const PairRec C = rec[ket.rec + cd];
    for (int ab = 0; ab < bra.n; ++ab) {
      const PairRec A = rec[bra.rec + ab];
      const double X = A.P[0] - C.P[0], Y = A.P[1] - C.P[1], Z = A.P[2] - C.P[2];
      const double rs = rsqrt64(A.p + C.p), al = A.p * C.p * rs * rs;
      double F[L + 1], R[hermite_count(L)];
      boys_tab<L>(al * (X * X + Y * Y + Z * Z), tab, F);
      const double pre = A.K * C.K * rs;
      static_for<0, L + 1>([&](auto n) { F[n] *= pre; });
      hermite_coulomb<L>(al, X, Y, Z, F, R);
      static_for<0, NB>([&](auto f) {
        double V[hermite_count(KT)];
        if constexpr (BT == kPP) {
          // component a of the first shell is the work-group's: rotate it into place
          static_for<0, hermite_count(KT)>([&](auto t) {
            V[t] = a == 0   ? hermite_sum<BT, 1, 0, f, t>(A, R)
                   : a == 1 ? hermite_sum<BT, 1, 1, f, t>(A, R)
                            : hermite_sum<BT, 1, 2, f, t>(A, R);
          });
        } else {
          static_for<0, hermite_count(KT)>([&](auto t) { V[t] = hermite_sum<BT, 1, f, 0, t>(A, R); });
        }
        static_for<0, NK>([&](auto k) {
          acc[f][k] += KT == kPP ? hermite_sum<KT, -1, k / 3, k % 3, 0>(C, V) : hermite_sum<KT, -1, k % 3, 0, 0>(C, V);
        });
      });
    }
  }
  for (int o = (1 << lg) >> 1; o > 0; o >>= 1)
    static_for<0, NB>([&](auto f) { static_for<0, NK>([&](auto k) { acc[f][k] += __shfl_xor(acc[f][k], o); }); });
  if (sub) return;
  constexpr double c = 34.986836655255488;  // 2 pi^(5/2), pi = kPiTrunc
  auto function_pair = [](const ShellPair& s, int type, int x, int y) -> long {  // -1: i < j, the mirror is written
    const long i = s.i0 + (type == kPP || (type == kSP && s.p_first) ? x : 0);
    const long j = s.j0 + (type == kPP ? y : type == kSP && !s.p_first ? x : 0);
    return i < j ? -1 : i * (i + 1) / 2 + j;
  };
  static_for<0, NB>([&](auto f) {
    const long IJ = BT == kPP ? function_pair(bra, BT, a, f) : function_pair(bra, BT, f, 0);
    static_for<0, NK>([&](auto k) {
      const long KL = KT == kPP ? function_pair(ket, KT, k / 3, k % 3) : function_pair(ket, KT, k, 0);
      if (IJ < 0 || KL < 0 || (BT == KT && kt == b && IJ < KL)) return;
      const long hi = IJ > KL ? IJ : KL, lo = IJ > KL ? KL : IJ;
      ints[hi * (hi + 1) / 2 + lo] = c * acc[f][k];
    });
  });
}

// v_KL = P_kl (k == l) or P_kl + P_lk: J_IJ = sum_KL (IJ|KL) v_KL.
__global__ void k_eri_vec(const double* __restrict__ P, int n, const int* __restrict__ pij, int npair, double* v) {
  const int IJ = blockIdx.x * blockDim.x + threadIdx.x;
  if (IJ >= npair) return;
  const int i = pij[2 * IJ], j = pij[2 * IJ + 1];
  v[IJ] = (i == j) ? P[i + (long)i * n] : P[i + (long)j * n] + P[j + (long)i * n];
}

// Both halves of J in one launch.  The first npair work-groups:
// Jp[IJ] = sum_{KL <= IJ} (IJ|KL) v_KL, the row of the packed lower triangle read
// contiguously.  The others: part[chunk][IJ] = sum_{KL > IJ, KL in chunk} (KL|IJ) v_KL
// for 64 pairs IJ, the four waves taking every fourth KL of the chunk (64 consecutive
// integrals of row KL each).  Chunks are short enough that the column blocks fill the
// chip (benzene, 2211 pairs: 105 one-wave blocks of 1024 rows took 335 us).
// Fixed-order sums.
__global__ __launch_bounds__(256) void k_eri_partial(const double* __restrict__ ints, const double* __restrict__ v,
                                                     int npair, int chunk, double* Jp, double* part) {
  __shared__ double red[256];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < npair) {
    const long IJ = blockIdx.x;
    const double* row = ints + IJ * (IJ + 1) / 2;
    double s = 0.0;
    for (long KL = tid; KL <= IJ; KL += 256) s += row[KL] * v[KL];
    red[tid] = s;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (tid < st) red[tid] += red[tid + st];
      __syncthreads();
    }
    if (tid == 0) Jp[IJ] = red[0];
    return;
  }
  const int ncol = (npair + 63) / 64, cb = (int)blockIdx.x - npair;
  const long IJ0 = 64L * (cb % ncol), IJ = IJ0 + (tid & 63), ch = cb / ncol;
  const long k0 = ch * chunk, k1 = std::min<long>(k0 + chunk, npair);
  if (k1 <= IJ0) return;  // below the chunks k_eri_unpack takes for these pairs, (IJ + 1) / chunk and up
  double s = 0.0;
  if (IJ < npair) {
    long KL = k0 + (tid >> 6);
    if (KL <= IJ) KL += (IJ - KL) / 4 * 4 + 4;
#pragma unroll 4
    for (; KL < k1; KL += 4) s += ints[KL * (KL + 1) / 2 + IJ] * v[KL];
  }
  red[tid] = s;
  __syncthreads();
  if (tid < 64 && IJ < npair)
    part[ch * npair + IJ] = ((red[tid] + red[tid + 64]) + red[tid + 128]) + red[tid + 192];
}

// J_ij = J_ji = Jp[IJ] + sum over chunks of part (in chunk order).
__global__ void k_eri_unpack(const double* __restrict__ Jp, const double* __restrict__ part, int nchunk, int chunk,
                             const int* __restrict__ pij, int npair, int n, double* J) {
  const int IJ = blockIdx.x * blockDim.x + threadIdx.x;
  if (IJ >= npair) return;
  double s = Jp[IJ];
  for (int c = (IJ + 1) / chunk; c < nchunk; ++c) s += part[(long)c * npair + IJ];
  const int i = pij[2 * IJ], j = pij[2 * IJ + 1];
  J[i + (long)j * n] = s;
  J[j + (long)i * n] = s;
}

unsigned nb(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

struct dg_eri {
  int nbf = 0, npair = 0, nchunk = 0, chunk = 0;
  long nints = 0;
  hipStream_t stream = nullptr;
  double* ints = nullptr;
  char* work = nullptr;  // every other array, carved from one allocation
  double *v = nullptr, *Jp = nullptr, *part = nullptr, *P = nullptr, *J = nullptr;
  int* pij = nullptr;
  ~dg_eri() {
    if (stream) (void)hipStreamSynchronize(stream);
    if (ints) (void)hipFree(ints);
    if (work) (void)hipFree(work);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

// Offsets of arrays carved from one allocation; upload() queues their copies.
struct Carve {
  size_t size = 0;
  size_t add(size_t bytes) {
    const size_t at = size;
    size += (bytes + 255) & ~(size_t)255;
    return at;
  }
};

// Lanes per quartet for a ket pair of n primitive pairs: about three rounds of the
// longest pairs (36), so that a core-core quartet (36 x 36 primitive quartets) is not
// one lane's chain; none for the short pairs, which are most.
int team_lg(int n) { return n >= 24 ? 4 : n >= 9 ? 2 : n >= 4 ? 1 : 0; }

struct ShellQuartets {
  std::vector<PairRec> rec;
  std::vector<ShellPair> pairs[3];
  std::vector<KetBlock> blocks[3];
};

template <int BT, int KT>
void launch_quartets(const ShellQuartets& sq, const ShellPair* const (&pairs)[3], const KetBlock* const (&blocks)[3],
                     const PairRec* rec, const double* tab, double* ints, hipStream_t st) {
  const long nb = (long)sq.blocks[KT].size(), nbra = (long)sq.pairs[BT].size();
  if (nb == 0) return;
  const long per = std::max(1L, (1L << 23) / nb);  // bra pairs per launch: under 2^32 threads
  for (long b0 = 0; b0 < nbra; b0 += per)
    hipLaunchKernelGGL((k_eri_shell<BT, KT>), dim3((unsigned)(nb * std::min(per, nbra - b0)), BT == kPP ? 3 : 1),
                       dim3(256), 0, st, pairs[BT], (int)b0, pairs[KT], blocks[KT], (int)nb, rec, tab, ints);
}

}  // namespace

extern "C" {

int dg_eri_create(const dg_molecule* mol, const dg_basis* basis, dg_eri** out) {
  if (!mol || !basis || !out) return fail(DG_ERR_INVALID, "dg_eri_create: null argument");
  *out = nullptr;
  if (mol->natoms < 1 || !mol->xyz) return fail(DG_ERR_INVALID, "dg_eri_create: empty molecule");
  if (basis->nshell < 1 || !basis->atom || !basis->L || !basis->nprim || !basis->offset || !basis->alpha ||
      !basis->coef)
    return fail(DG_ERR_INVALID, "dg_eri_create: empty basis");
  // functions: shell, centre, Cartesian powers, normalised coefficients
  struct Fn {
    int shell;
    const double* A;
    const int* l;
    std::vector<double> cn;
  };
  std::vector<Fn> fn;
  std::vector<int> first(basis->nshell);
  int lmax = 0;
  for (int s = 0; s < basis->nshell; ++s) {
    const int L = basis->L[s], at = basis->atom[s];
    if (L < 0 || L > 2) return fail(DG_ERR_INVALID, "dg_eri_create: shell L must be 0, 1 or 2");
    if (at < 0 || at >= mol->natoms) return fail(DG_ERR_INVALID, "dg_eri_create: shell atom out of range");
    if (basis->nprim[s] < 1 || basis->offset[s] < 0) return fail(DG_ERR_INVALID, "dg_eri_create: bad primitive range");
    lmax = std::max(lmax, L);
    first[s] = (int)fn.size();
    for (int c = 0; c < (L + 1) * (L + 2) / 2; ++c) {
      Fn f{s, mol->xyz + 3 * at, kCart[L][c], {}};
      for (int k = 0; k < basis->nprim[s]; ++k) {
        const double a = basis->alpha[basis->offset[s] + k];
        if (!(a > 0.0)) return fail(DG_ERR_INVALID, "dg_eri_create: primitive exponent must be positive");
        f.cn.push_back(basis->coef[basis->offset[s] + k] * dg::gto_norm(a, f.l[0], f.l[1], f.l[2]));
      }
      fn.push_back(std::move(f));
    }
  }
  const int n = (int)fn.size();
  std::unique_ptr<dg_eri> e(new dg_eri);
  e->nbf = n;
  e->npair = n * (n + 1) / 2;
  e->nints = (long)e->npair * (e->npair + 1) / 2;
  if (e->nints > (1L << 36)) return fail(DG_ERR_UNSUPPORTED, "dg_eri_create: more than 2^36 integrals");
  ERI_HIP(hipStreamCreate(&e->stream));
  ERI_HIP((hipError_t)dg::device_malloc((void**)&e->ints, sizeof(double) * std::max<long>(e->nints, 1)));
  std::vector<int> pij(2 * (size_t)e->npair);
  for (int i = 0, IJ = 0; i < n; ++i)
    for (int j = 0; j <= i; ++j, ++IJ) {
      pij[2 * IJ] = i;
      pij[2 * IJ + 1] = j;
    }
  // shell pairs without d shells
  ShellQuartets sq;
  for (int s = 0; s < basis->nshell; ++s)
    for (int t = 0; t <= s; ++t) {
      const int ls = basis->L[s], lt = basis->L[t];
      if (ls > 1 || lt > 1) continue;
      ShellPair pr{(int)sq.rec.size(), basis->nprim[s] * basis->nprim[t], first[s], first[t], ls > lt, 0};
      const double *A = mol->xyz + 3 * basis->atom[s], *B = mol->xyz + 3 * basis->atom[t];
      const double r2 = (A[0] - B[0]) * (A[0] - B[0]) + (A[1] - B[1]) * (A[1] - B[1]) + (A[2] - B[2]) * (A[2] - B[2]);
      for (int x = 0; x < basis->nprim[s]; ++x)
        for (int y = 0; y < basis->nprim[t]; ++y) {
          const double a = basis->alpha[basis->offset[s] + x], b = basis->alpha[basis->offset[t] + y], p = a + b;
          PairRec r;
          r.p = p;
          r.h = 0.5 / p;
          r.K = fn[first[s]].cn[x] * fn[first[t]].cn[y] * std::exp(-a * b / p * r2) / p;
          for (int d = 0; d < 3; ++d) {
            r.P[d] = (a * A[d] + b * B[d]) / p;
            r.A[d] = r.P[d] - (ls >= lt ? A[d] : B[d]);
            r.B[d] = r.P[d] - B[d];
          }
          sq.rec.push_back(r);
        }
      sq.pairs[ls + lt].push_back(pr);
    }
  for (int t = 0; t < 3; ++t) {
    std::vector<ShellPair>& p = sq.pairs[t];
    std::stable_sort(p.begin(), p.end(), [](const ShellPair& a, const ShellPair& b) { return a.n > b.n; });
    for (int i = 0, m = (int)p.size(); i < m;) {
      const int lg = team_lg(p[i].n);
      int len = 1;
      while (len < (256 >> lg) && i + len < m && team_lg(p[i + len].n) == lg) ++len;
      sq.blocks[t].push_back({i, len, lg});
      i += len;
    }
  }
  // function-pair records of the integrals with a d function
  std::vector<double> rec;
  std::vector<int> off, pl, pd;
  if (lmax > 1) {
    off.assign(e->npair + 1, 0);
    pl.resize(3 * (size_t)e->npair);
    pd.resize(e->npair);
    for (int IJ = 0; IJ < e->npair; ++IJ) {
      const Fn &fi = fn[pij[2 * IJ]], &fj = fn[pij[2 * IJ + 1]];
      const int si = fi.shell, sj = fj.shell;
      for (int d = 0; d < 3; ++d) pl[3 * IJ + d] = fi.l[d] + fj.l[d];
      pd[IJ] = basis->L[si] > 1 || basis->L[sj] > 1;
      off[IJ] = (int)(rec.size() / kRec);
      for (int ka = 0; ka < basis->nprim[si]; ++ka)
        for (int kb = 0; kb < basis->nprim[sj]; ++kb) {
          const double a = basis->alpha[basis->offset[si] + ka], b = basis->alpha[basis->offset[sj] + kb], p = a + b;
          double r[kRec];
          r[0] = p;
          for (int d = 0; d < 3; ++d) r[1 + d] = (a * fi.A[d] + b * fj.A[d]) / p;
          r[4] = fi.cn[ka] * fj.cn[kb];
          for (int d = 0; d < 3; ++d) hermite_1d(fi.l[d], fj.l[d], a, b, fi.A[d], fj.A[d], r + 5 + 5 * d);
          rec.insert(rec.end(), r, r + kRec);
        }
    }
    off[e->npair] = (int)(rec.size() / kRec);
  }
  e->chunk = std::max(128, (e->npair + 4095) / 4096 * 64);
  e->nchunk = (e->npair + e->chunk - 1) / e->chunk;
  // one allocation for everything but the integrals; the uploaded arrays come first
  // and are gathered into one copy
  Carve c;
  const size_t o_rec = c.add(sq.rec.size() * sizeof(PairRec)), o_pij = c.add(pij.size() * 4);
  size_t o_pairs[3], o_blocks[3];
  for (int t = 0; t < 3; ++t) {
    o_pairs[t] = c.add(sq.pairs[t].size() * sizeof(ShellPair));
    o_blocks[t] = c.add(sq.blocks[t].size() * sizeof(KetBlock));
  }
  const size_t o_drec = c.add(rec.size() * 8), o_off = c.add(off.size() * 4), o_pl = c.add(pl.size() * 4),
               o_pd = c.add(pd.size() * 4), uploaded = c.size;
  const size_t o_tab = c.add(sizeof(double) * kBoysRows * kBoysCols), o_v = c.add(8 * (size_t)e->npair),
               o_jp = c.add(8 * (size_t)e->npair), o_part = c.add(8 * (size_t)e->nchunk * e->npair),
               o_p = c.add(8 * (size_t)n * n), o_j = c.add(8 * (size_t)n * n);
  std::vector<char> host(uploaded);
  auto put = [&](size_t o, const void* p, size_t bytes) {
    if (bytes) std::memcpy(host.data() + o, p, bytes);
  };
  put(o_rec, sq.rec.data(), sq.rec.size() * sizeof(PairRec));
  put(o_pij, pij.data(), pij.size() * 4);
  for (int t = 0; t < 3; ++t) {
    put(o_pairs[t], sq.pairs[t].data(), sq.pairs[t].size() * sizeof(ShellPair));
    put(o_blocks[t], sq.blocks[t].data(), sq.blocks[t].size() * sizeof(KetBlock));
  }
  put(o_drec, rec.data(), rec.size() * 8);
  put(o_off, off.data(), off.size() * 4);
  put(o_pl, pl.data(), pl.size() * 4);
  put(o_pd, pd.data(), pd.size() * 4);
  ERI_HIP((hipError_t)dg::device_malloc((void**)&e->work, c.size));
  char* w = e->work;
  double* tab = (double*)(w + o_tab);
  e->pij = (int*)(w + o_pij);
  e->v = (double*)(w + o_v);
  e->Jp = (double*)(w + o_jp);
  e->part = (double*)(w + o_part);
  e->P = (double*)(w + o_p);
  e->J = (double*)(w + o_j);
  hipLaunchKernelGGL(k_boys_table, dim3(nb(kBoysRows, 64)), dim3(64), 0, e->stream, tab);
  ERI_HIP(hipMemcpyAsync(w, host.data(), uploaded, hipMemcpyHostToDevice, e->stream));
  const ShellPair* pairs[3];
  const KetBlock* blocks[3];
  for (int t = 0; t < 3; ++t) {
    pairs[t] = (const ShellPair*)(w + o_pairs[t]);
    blocks[t] = (const KetBlock*)(w + o_blocks[t]);
  }
  const PairRec* prec = (const PairRec*)(w + o_rec);
  launch_quartets<kSS, kSS>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  launch_quartets<kSS, kSP>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  launch_quartets<kSP, kSP>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  launch_quartets<kSS, kPP>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  launch_quartets<kSP, kPP>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  launch_quartets<kPP, kPP>(sq, pairs, blocks, prec, tab, e->ints, e->stream);
  if (lmax > 1)
    hipLaunchKernelGGL(k_eri<kMaxLsum>, dim3(nb(e->nints, 256)), dim3(256), 0, e->stream, e->nints,
                       (const int*)(w + o_off), (const int*)(w + o_pl), (const int*)(w + o_pd),
                       (const double*)(w + o_drec), e->ints);
  ERI_HIP(hipGetLastError());
  ERI_HIP(hipStreamSynchronize(e->stream));
  *out = e.release();
  return DG_OK;
}

int dg_eri_destroy(dg_eri* e) {
  delete e;
  return DG_OK;
}

int dg_eri_count(const dg_eri* e, long* nints, int* nbf) {
  if (!e) return fail(DG_ERR_INVALID, "dg_eri_count: null object");
  if (nints) *nints = e->nints;
  if (nbf) *nbf = e->nbf;
  return DG_OK;
}

int dg_eri_get(dg_eri* e, double* ints) {
  if (!e || !ints) return fail(DG_ERR_INVALID, "dg_eri_get: null argument");
  ERI_HIP(hipMemcpyAsync(ints, e->ints, sizeof(double) * e->nints, hipMemcpyDeviceToHost, e->stream));
  ERI_HIP(hipStreamSynchronize(e->stream));
  return DG_OK;
}

int dg_eri_coulomb_device(dg_eri* e, const double* dP, double* dJ, void* stream) {
  if (!e || !dP || !dJ) return fail(DG_ERR_INVALID, "dg_eri_coulomb_device: null argument");
  hipStream_t st = stream ? (hipStream_t)stream : e->stream;
  const int np = e->npair;
  hipLaunchKernelGGL(k_eri_vec, dim3(nb(np, 256)), dim3(256), 0, st, dP, e->nbf, e->pij, np, e->v);
  hipLaunchKernelGGL(k_eri_partial, dim3(np + nb(np, 64) * e->nchunk), dim3(256), 0, st, e->ints, e->v, np, e->chunk,
                     e->Jp, e->part);
  hipLaunchKernelGGL(k_eri_unpack, dim3(nb(np, 256)), dim3(256), 0, st, e->Jp, e->part, e->nchunk, e->chunk, e->pij,
                     np, e->nbf, dJ);
  ERI_HIP(hipGetLastError());
  return DG_OK;
}

int dg_eri_coulomb(dg_eri* e, const double* P, double* J) {
  if (!e || !P || !J) return fail(DG_ERR_INVALID, "dg_eri_coulomb: null argument");
  const size_t bytes = sizeof(double) * (size_t)e->nbf * e->nbf;
  ERI_HIP(hipMemcpyAsync(e->P, P, bytes, hipMemcpyHostToDevice, e->stream));
  const int rc = dg_eri_coulomb_device(e, e->P, e->J, nullptr);
  if (rc != DG_OK) return rc;
  ERI_HIP(hipMemcpyAsync(J, e->J, bytes, hipMemcpyDeviceToHost, e->stream));
  ERI_HIP(hipStreamSynchronize(e->stream));
  return DG_OK;
}

}  // extern "C"
