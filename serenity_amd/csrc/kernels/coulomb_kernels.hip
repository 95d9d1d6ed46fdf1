// Density-fitted Coulomb matrix on the GPU ("J engine"), the Coulomb part of
// the SCF around the XC build (Serenity's densFitJ = RI: RI_J_IntegralController,
// src/integrals/RI_J_IntegralController.cpp:41-121, with libint2's 3-centre
// integrals).  No 3-centre integral is stored.  Every significant primitive
// pair q of the orbital basis is a sum of Hermite Gaussians,
//   phi_a phi_b = K_q sum_tuv E^ab_tuv Lambda_tuv(p_q, P_q),
// and meets an auxiliary primitive (exponent a, centre C) through
//   (Lambda_tuv | Lambda_tau,nu,phi) = 2 pi^(5/2) / (p a sqrt(p + a)) (-1)^(tau+nu+phi)
//                                      R_(t+tau, u+nu, v+phi)(p a / (p + a), P - C)
// (McMurchie-Davidson Hermite Coulomb integrals, Boys function).  Per SCF
// iteration:
//   1. D_q = K_q sum_ij Pc_ij E^ij         (Hermite density of each primitive pair)
//   2. b_k = sum_q (D_q | aux k)           (fitting right-hand side, Cartesian aux)
//   3. M c = b                             (two triangular solves with M's factor; the host's where it
//                                           is not resident)
//   4. V_q = sum_k c_k (Lambda_q | aux k)  (Hermite potential of each pair)
//   5. J_ab = K_q sum_tuv V_q,tuv E^ab_tuv (then the shells' angular transforms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "xc_internal.h"

namespace sxc {

namespace {

// Packed Hermite indices of order <= kJMaxL (all orders below s = t + u + v first, then t descending,
// u descending) as tables: (t, u, v) of index i, and the recursion of
// i >= 1 in its first non-zero direction dir: R_i = x_dir R_m1 + mul R_m2 (m2 = m1 where mul = 0).
// Read with constant indices in unrolled loops only, so that the arrays they index stay in registers.
struct HermiteTable {
  int t[kJMaxH], u[kJMaxH], v[kJMaxH], dir[kJMaxH], m1[kJMaxH], m2[kJMaxH], mul[kJMaxH];
};
constexpr int hidx_c(int t, int u, int v) {
  return (t + u + v) * (t + u + v + 1) * (t + u + v + 2) / 6 + (u + v) * (u + v + 1) / 2 + v;
}
constexpr int hcount_c(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
constexpr HermiteTable make_hermite_table() {
  HermiteTable h{};
  int i = 0;
  for (int s = 0; s <= kJMaxL; ++s)
    for (int t = s; t >= 0; --t)
      for (int u = s - t; u >= 0; --u, ++i) {
        const int v = s - t - u;
        h.t[i] = t;
        h.u[i] = u;
        h.v[i] = v;
        const int d = t > 0 ? 0 : u > 0 ? 1 : 2, e = d == 0 ? t : d == 1 ? u : v;
        h.dir[i] = d;
        h.mul[i] = e > 1 ? e - 1 : 0;
        h.m1[i] = i == 0 ? 0 : hidx_c(t - (d == 0), u - (d == 1), v - (d == 2));
        h.m2[i] = e > 1 ? hidx_c(t - 2 * (d == 0), u - 2 * (d == 1), v - 2 * (d == 2)) : h.m1[i];
      }
  return h;
}
__device__ constexpr HermiteTable kHerm = make_hermite_table();

// Boys functions F_0..F_M at T.  Below kBoysEnd: F_M by its Taylor expansion about the nearest node
// of a table (dF_m/dT = -F_(m+1); |T - T_i| <= 0.05, nine terms: truncation below 1e-17 F_M) and
// downward recursion, with e^-T from the same node.  Above: F_0 = sqrt(pi / T) / 2 (its
// complement is below 1e-16 there) and upward recursion.
template <int M>
__device__ __forceinline__ void boys_table(double T, const double* __restrict__ tab, double (&F)[M + 1]) {
  if (T < kBoysEnd) {
    const int i = (int)(T * kBoysPerUnit + 0.5);
    const double d = i * (1.0 / kBoysPerUnit) - T;
    const gmem<const double>* row = to_global(tab) + i * kBoysCols;
    double f = row[1 + M + 8], e = 1.0;
#pragma unroll
    for (int k = 8; k >= 1; --k) {
      f = row[M + k] + f * (d * (1.0 / k));
      e = 1.0 + e * (d * (1.0 / k));
    }
    e *= row[0];
    F[M] = f;
#pragma unroll
    for (int j = M; j > 0; --j) F[j - 1] = (2.0 * T * F[j] + e) * (1.0 / (2 * j - 1));
  } else {
    const double r = rsqrt(T), o2t = 0.5 * r * r;
    const double e = T < 100.0 ? exp(-T) : 0.0;  // beyond: below 1e-26 of every F_m kept
    F[0] = 0.88622692545275801365 * r;           // sqrt(pi) / 2
#pragma unroll
    for (int j = 0; j < M; ++j) F[j + 1] = ((2 * j + 1) * F[j] - e) * o2t;
  }
}

// One level n of the Hermite Coulomb recursion, in place: entries of order <= M - n from those of
// level n + 1 (descending, so an entry's sources of lower order are still of that level).
template <int M, int N>
__device__ __forceinline__ void r_level(const double (&x)[3], const double (&F)[M + 1], double (&R)[hcount_c(M)]) {
#pragma unroll
  for (int i = hcount_c(M - N) - 1; i >= 1; --i) {
    double val = x[kHerm.dir[i]] * R[kHerm.m1[i]];
    if (kHerm.mul[i] > 0) val += (double)kHerm.mul[i] * R[kHerm.m2[i]];
    R[i] = val;
  }
  R[0] = F[N];
  if constexpr (N > 0) r_level<M, N - 1>(x, F, R);
}

// scale R_tuv(alpha, x) for t + u + v <= M, packed, in registers.
template <int M>
__device__ __forceinline__ void r_tensor(double alpha, double scale, const double (&x)[3],
                                         const double* __restrict__ tab, double (&R)[hcount_c(M)]) {
  double F[M + 1];
  boys_table<M>(alpha * (x[0] * x[0] + x[1] * x[1] + x[2] * x[2]), tab, F);
  double pw = scale;
#pragma unroll
  for (int n = 0; n <= M; ++n) {
    F[n] *= pw;
    pw *= -2.0 * alpha;
  }
  r_level<M, M>(x, F, R);
}

// Hermite expansion E[i][j][t] (i <= LA, j <= LB, t <= i + j) of one direction.
template <int LA, int LB>
__device__ __forceinline__ void hermite_E(double p, double XPA, double XPB,
                                          double (&E)[LA + 1][LB + 1][LA + LB + 1]) {
  const double o2p = 0.5 / p;
#pragma unroll
  for (int i = 0; i <= LA; ++i)
#pragma unroll
    for (int j = 0; j <= LB; ++j)
#pragma unroll
      for (int t = 0; t <= LA + LB; ++t) {
        double v = 0.0;
        if (i + j == 0) {
          v = t == 0 ? 1.0 : 0.0;
        } else if (t <= i + j) {
          const double* old = i > 0 ? E[i > 0 ? i - 1 : 0][j] : E[i][j > 0 ? j - 1 : 0];
          v = (i > 0 ? XPA : XPB) * old[t];
          if (t > 0) v += o2p * old[t - 1];
          if (t + 1 <= i + j - 1) v += (t + 1) * old[t + 1];
        }
        E[i][j][t] = v;
      }
}

// Cartesian exponents of every component up to the auxiliary shells, as tables for unrolled loops.
struct CartTable {
  int x[kJMaxLAux + 1][kJMaxNcartAux], y[kJMaxLAux + 1][kJMaxNcartAux], z[kJMaxLAux + 1][kJMaxNcartAux];
};
constexpr CartTable make_cart_table() {
  CartTable c{};
  for (int l = 0; l <= kJMaxLAux; ++l) {
    int k = 0;
    for (int a = l; a >= 0; --a)
      for (int b = l - a; b >= 0; --b, ++k) {
        c.x[l][k] = a;
        c.y[l][k] = b;
        c.z[l][k] = l - a - b;
      }
  }
  return c;
}
__device__ constexpr CartTable kCart = make_cart_table();

// x^n exp(-a x^2) = sum_t c[n][t] (2a)^(-(n + t) / 2) Lambda_t about its own centre,
// c[n][t] = n! / (t! m! 2^m) with 2 m = n - t (zero for odd n - t).
struct AuxTable {
  double c[kJMaxLAux + 1][kJMaxLAux + 1];
};
constexpr AuxTable make_aux_table() {
  AuxTable a{};
  a.c[0][0] = 1.0;
  for (int n = 1; n <= kJMaxLAux; ++n)
    for (int t = 0; t <= n; ++t)
      a.c[n][t] = (t > 0 ? a.c[n - 1][t - 1] : 0.0) + (t + 1 <= n - 1 ? (t + 1) * a.c[n - 1][t + 1] : 0.0);
  return a;
}
__device__ constexpr AuxTable kAux = make_aux_table();

// Cartesian functions of a class's shells and Hermite functions of their pairs.  A wavefront's pairs
// are of one class, so the angular transforms are the same for every lane (scalar loads).
template <int LA, int LB>
struct PairDims {
  static constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2, H = hcount_c(LA + LB);
  typedef double ETab[LA + 1][LB + 1][LA + LB + 1];
};

// One Cartesian function I of A at a time (recursion instead of a loop, which for f shells would be
// too long to unroll): the row's part of the Hermite density, or the row of J from the potential.
template <int LA, int LB, int I>
__device__ __forceinline__ void hermite_row_in(const typename PairDims<LA, LB>::ETab& Ex,
                                               const typename PairDims<LA, LB>::ETab& Ey,
                                               const typename PairDims<LA, LB>::ETab& Ez,
                                               const double (&Pc)[PairDims<LA, LB>::NA][PairDims<LA, LB>::NB],
                                               double (&out)[PairDims<LA, LB>::H]) {
  using Dim = PairDims<LA, LB>;
  constexpr int ax = kCart.x[LA][I], ay = kCart.y[LA][I], az = kCart.z[LA][I];
#pragma unroll
  for (int j = 0; j < Dim::NB; ++j) {
    const int bx = kCart.x[LB][j], by = kCart.y[LB][j], bz = kCart.z[LB][j];
#pragma unroll
    for (int k = 0; k < Dim::H; ++k) {
      const int t = kHerm.t[k], u = kHerm.u[k], v = kHerm.v[k];
      if (t <= ax + bx && u <= ay + by && v <= az + bz)
        out[k] += Pc[I][j] * (Ex[ax][bx][t] * (Ey[ay][by][u] * Ez[az][bz][v]));
    }
  }
  if constexpr (I + 1 < Dim::NA) hermite_row_in<LA, LB, I + 1>(Ex, Ey, Ez, Pc, out);
}
template <int LA, int LB, int I>
__device__ __forceinline__ void hermite_row_out(const typename PairDims<LA, LB>::ETab& Ex,
                                                const typename PairDims<LA, LB>::ETab& Ey,
                                                const typename PairDims<LA, LB>::ETab& Ez,
                                                const double (&in)[PairDims<LA, LB>::H],
                                                double (&Jc)[PairDims<LA, LB>::NA][PairDims<LA, LB>::NB]) {
  using Dim = PairDims<LA, LB>;
  constexpr int ax = kCart.x[LA][I], ay = kCart.y[LA][I], az = kCart.z[LA][I];
#pragma unroll
  for (int j = 0; j < Dim::NB; ++j) {
    const int bx = kCart.x[LB][j], by = kCart.y[LB][j], bz = kCart.z[LB][j];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < Dim::H; ++k) {
      const int t = kHerm.t[k], u = kHerm.u[k], v = kHerm.v[k];
      if (t <= ax + bx && u <= ay + by && v <= az + bz) s += in[k] * (Ex[ax][bx][t] * (Ey[ay][by][u] * Ez[az][bz][v]));
    }
    Jc[I][j] = s;
  }
  if constexpr (I + 1 < Dim::NA) hermite_row_out<LA, LB, I + 1>(Ex, Ey, Ez, in, Jc);
}

// 1. Hermite density of each primitive pair, over the pair's exponent (step 2 wants D / p)
template <int LA, int LB>
__device__ __forceinline__ void jdens_pair(const JPair& pr, const DevShell& A, const DevShell& B,
                                           const double* __restrict__ angA, const double* __restrict__ angB,
                                           const double* __restrict__ P, int n, double* __restrict__ D) {
  using Dim = PairDims<LA, LB>;
  double Pc[Dim::NA][Dim::NB];
#pragma unroll
  for (int i = 0; i < Dim::NA; ++i)
#pragma unroll
    for (int j = 0; j < Dim::NB; ++j) Pc[i][j] = 0.0;
  const gmem<const double>* Pg = to_global(P) + A.ao_off + (int64_t)n * B.ao_off;
  const int nfa = A.nfunc, nfb = B.nfunc;
  for (int f = 0; f < nfa; ++f) {
    double row[Dim::NB];
#pragma unroll
    for (int j = 0; j < Dim::NB; ++j) row[j] = 0.0;
    for (int h = 0; h < nfb; ++h) {
      const double v = Pg[f + (int64_t)n * h];
#pragma unroll
      for (int j = 0; j < Dim::NB; ++j) row[j] += v * angB[h * Dim::NB + j];
    }
#pragma unroll
    for (int i = 0; i < Dim::NA; ++i)
#pragma unroll
      for (int j = 0; j < Dim::NB; ++j) Pc[i][j] += angA[f * Dim::NA + i] * row[j];
  }
  double Ex[LA + 1][LB + 1][LA + LB + 1], Ey[LA + 1][LB + 1][LA + LB + 1], Ez[LA + 1][LB + 1][LA + LB + 1];
  hermite_E<LA, LB>(pr.p, pr.PA[0], pr.PB[0], Ex);
  hermite_E<LA, LB>(pr.p, pr.PA[1], pr.PB[1], Ey);
  hermite_E<LA, LB>(pr.p, pr.PA[2], pr.PB[2], Ez);
  double out[Dim::H];
#pragma unroll
  for (int k = 0; k < Dim::H; ++k) out[k] = 0.0;
  hermite_row_in<LA, LB, 0>(Ex, Ey, Ez, Pc, out);
  const double scale = pr.sym * pr.K / pr.p;
  gmem<double>* dst = to_global(D) + pr.herm_off;
#pragma unroll
  for (int k = 0; k < Dim::H; ++k) dst[k] = scale * out[k];
}

// 5. J block of each primitive pair from its Hermite potential, added to both triangles of J
template <int LA, int LB>
__device__ __forceinline__ void jassemble_pair(const JPair& pr, const DevShell& A, const DevShell& B,
                                               const double* __restrict__ angA, const double* __restrict__ angB,
                                               const gmem<const double>* __restrict__ V, int64_t stride, int n,
                                               double* __restrict__ J) {
  using Dim = PairDims<LA, LB>;
  double Ex[LA + 1][LB + 1][LA + LB + 1], Ey[LA + 1][LB + 1][LA + LB + 1], Ez[LA + 1][LB + 1][LA + LB + 1];
  hermite_E<LA, LB>(pr.p, pr.PA[0], pr.PB[0], Ex);
  hermite_E<LA, LB>(pr.p, pr.PA[1], pr.PB[1], Ey);
  hermite_E<LA, LB>(pr.p, pr.PA[2], pr.PB[2], Ez);
  double in[Dim::H];
#pragma unroll
  for (int k = 0; k < Dim::H; ++k) in[k] = pr.K * V[k * stride];
  double Jc[Dim::NA][Dim::NB];
  hermite_row_out<LA, LB, 0>(Ex, Ey, Ez, in, Jc);
  const int nfa = A.nfunc, nfb = B.nfunc;
  const bool off = pr.A != pr.B;
  for (int f = 0; f < nfa; ++f) {
    double row[Dim::NB];
#pragma unroll
    for (int j = 0; j < Dim::NB; ++j) {
      row[j] = 0.0;
#pragma unroll
      for (int i = 0; i < Dim::NA; ++i) row[j] += angA[f * Dim::NA + i] * Jc[i][j];
    }
    for (int h = 0; h < nfb; ++h) {
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < Dim::NB; ++j) s += row[j] * angB[h * Dim::NB + j];
      const int mu = A.ao_off + f, nu = B.ao_off + h;
      atomicAdd(&J[mu + (int64_t)n * nu], s);
      if (off) atomicAdd(&J[nu + (int64_t)n * mu], s);
    }
  }
}

// One wavefront per item: up to 64 primitive pairs of one (l_A, l_B), shells of one kind each.
// Straight-line code per class keeps the expansions in registers (with run-time angular momenta
// they were 3.5 KB of private memory per lane: 1.04 and 0.86 ms at (H2O)32/def2-TZVP).
template <bool Dens, int Lo, int Hi>
__global__ __launch_bounds__(64) void jpair_kernel(const JPairItem* __restrict__ items, const JPair* __restrict__ pairs,
                                                   const DevShell* __restrict__ shells,
                                                   const double* __restrict__ ang, JView Jv,
                                                   const double* __restrict__ in, int n, double* __restrict__ out) {
  const JPairItem it = items[blockIdx.x];
  const double* angA = ang + it.angA;
  const double* angB = ang + it.angB;
  const int q = it.q0 + threadIdx.x;
  if ((int)threadIdx.x >= it.nq) return;
  const JPair pr = pairs[q];
  DevShell A = shells[pr.A], B = shells[pr.B];
  A.nfunc = it.nfa;  // the class's own, the same for every lane
  B.nfunc = it.nfb;
#define SXC_P(LA_, LB_)                                                                                       \
  if constexpr (LA_ + LB_ >= Lo && LA_ + LB_ <= Hi)                                                           \
    if (it.la == LA_ && it.lb == LB_) {                                                                       \
      if constexpr (Dens) {                                                                                   \
        jdens_pair<LA_, LB_>(pr, A, B, angA, angB, in, n, out);                                               \
      } else {                                                                                                \
        constexpr int L_ = LA_ + LB_;                                                                         \
        jassemble_pair<LA_, LB_>(pr, A, B, angA, angB, to_global(in) + Jv.herm0[L_] + (q - Jv.pair0[L_]),     \
                                 Jv.pair0[L_ + 1] - Jv.pair0[L_], n, out);                                    \
      }                                                                                                       \
      return;                                                                                                 \
    }
#define SXC_PL(LA_) SXC_P(LA_, 0) SXC_P(LA_, 1) SXC_P(LA_, 2) SXC_P(LA_, 3)
  static_assert(kJMaxLPrim == 3, "one case per (l_A, l_B)");
  SXC_PL(0) SXC_PL(1) SXC_PL(2) SXC_PL(3)
#undef SXC_PL
#undef SXC_P
}

// Steps 2 and 4 meet every primitive pair with every auxiliary primitive.  Work items are one
// wavefront each, of one (L, l) class (pair and auxiliary angular momentum), so that the recursion
// and the contraction are straight-line code on registers: per meeting a Boys evaluation, about
// 3 sum_(n <= L + l) hcount(n) operations of the recursion and 2 hcount(L) hcount(l) of the
// contraction, all FP64 vector work.  What does not change in a lane's loop is read once, what is the
// same for all lanes (the pair's density, the auxiliary's coefficients) comes through scalar loads,
// and no lane meets another before an item's end.  The classes are bundled in three kernels by L + l
// (<= 3, <= 6, above), because a kernel holds the registers of its widest class (128, 256, 512 and
// spills: the last hold 0.4 % of the meetings).  At (H2O)32/def2-TZVP (160 297 pairs x 1280
// auxiliary primitives) step 2 takes 1.5 ms and step 4 1.2 ms, the three kernels side by side: 73 GFLOP
// at 27 TFLOP/s (FP64 vector peak 78).  Alone the kernels run at 22 to 29 TFLOP/s with the vector units
// busy 40 to 72 % of the time (the widest 11 and 21, 17 and 24 %): a tenth (L + l of 4 to 6) to a
// fifth (<= 3) of their vector instructions are not FP64, a third to two fifths of the FP64 ones are
// single multiplies or additions, and a wavefront waits 26 to 47 % of its time, the narrow classes
// with one vector load in 15 instructions, the rows of the Boys table.  With run-time angular
// momenta, whose arrays live in private memory, and one thread per pair steps 2 and 4 took 50 and 263 ms.

// acc[j] += sum over i >= I of c[i] R(index i + index j), i < NI, j < NJ (recursion over i: one loop
// over both would be too long to unroll for the widest classes).
template <int NI, int NJ, int I, typename Ptr, int NR>
__device__ __forceinline__ void meet_contract(Ptr c, const double (&R)[NR], double (&acc)[NJ]) {
  const double d = c[I];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    acc[j] += d * R[hidx_c(kHerm.t[I] + kHerm.t[j], kHerm.u[I] + kHerm.u[j], kHerm.v[I] + kHerm.v[j])];
  if constexpr (I + 1 < NI) meet_contract<NI, NJ, I + 1>(c, R, acc);
}

// 2. W_tau of the auxiliary primitives: lanes are auxiliary primitives (where a class has fewer than
// 64, groups of lanes take different pairs), the loop runs over the item's pairs.
template <int L, int l>
__device__ __forceinline__ void jrhs_item(const JItem& it, const JView& J, const double* __restrict__ D,
                                          double* __restrict__ W) {
  constexpr int M = L + l, HL = hcount_c(L), Hl = hcount_c(l);
  const int lane = threadIdx.x;
  const int width = it.na;  // lanes per pair: a power of two for the grouped classes
  const int g = l >= kJGroupL ? lane / width : 0;
  const int step = l >= kJGroupL ? 64 / width : 1;
  const int aw = l >= kJGroupL ? lane - g * width : lane;
  const int a = min(it.a0 + aw, J.aux0[l + 1] - 1);
  const bool live = it.a0 + aw < J.aux0[l + 1] && aw < width;
  const gmem<const double>* A = to_global(J.aux) + 4 * (int64_t)a;
  const double cx = A[0], cy = A[1], cz = A[2], ea = A[3];
  double acc[Hl];
#pragma unroll
  for (int j = 0; j < Hl; ++j) acc[j] = 0.0;
  const double* D0 = D + J.herm0[L];
  const int q1 = it.q0 + it.nq;
  for (int q = it.q0 + g; q < q1; q += step) {
    const double* Q = J.pair + 4 * (int64_t)q;
    const double p = Q[3];
    const double* Dq = D0 + (int64_t)(q - J.pair0[L]) * HL;
    const double r = rsqrt(p + ea);
    const double x[3] = {Q[0] - cx, Q[1] - cy, Q[2] - cz};
    double R[hcount_c(M)];
    r_tensor<M>(p * ea * r * r, r, x, J.boys, R);
    meet_contract<HL, Hl, 0>(Dq, R, acc);
  }
  if (!live) return;
  const int nal = J.aux0[l + 1] - J.aux0[l];
  double* out = W + J.aherm0[l] + (a - J.aux0[l]);
#pragma unroll
  for (int j = 0; j < Hl; ++j) atomicAdd(out + (int64_t)j * nal, acc[j]);
}

// 4. Hermite potential of the pairs: lanes are pairs, the loop runs over the item's auxiliary
// primitives, whose Hermite coefficients U are the same for every lane.
template <int L, int l>
__device__ __forceinline__ void jpot_item(const JItem& it, const JView& J, const double* __restrict__ U,
                                          double* __restrict__ V) {
  constexpr int M = L + l, HL = hcount_c(L), Hl = hcount_c(l);
  const int lane = threadIdx.x;
  const int q = it.q0 + min(lane, it.nq - 1);
  const gmem<const double>* Q = to_global(J.pair) + 4 * (int64_t)q;
  const double px = Q[0], py = Q[1], pz = Q[2], p = Q[3];
  double acc[HL];
#pragma unroll
  for (int i = 0; i < HL; ++i) acc[i] = 0.0;
  for (int k = 0; k < it.na; ++k) {
    const int a = it.a0 + k;
    const double* A = J.aux + 4 * (int64_t)a;
    const double* Ua = U + J.aherm0[l] + (int64_t)(a - J.aux0[l]) * Hl;
    const double ea = A[3], r = rsqrt(p + ea);
    const double x[3] = {px - A[0], py - A[1], pz - A[2]};
    double R[hcount_c(M)];
    r_tensor<M>(p * ea * r * r, r, x, J.boys, R);
    meet_contract<Hl, HL, 0>(Ua, R, acc);
  }
  if (lane >= it.nq) return;
  const double ip = 1.0 / p;
  const int nql = J.pair0[L + 1] - J.pair0[L];
  double* out = V + J.herm0[L] + (q - J.pair0[L]);
#pragma unroll
  for (int i = 0; i < HL; ++i) atomicAdd(out + (int64_t)i * nql, acc[i] * ip);
}

template <bool Rhs, int Lo, int Hi>
__device__ __forceinline__ void jmeet(const JItem& it, const JView& J, const double* __restrict__ in,
                                      double* __restrict__ out) {
#define SXC_J(L_, l_)                                                              \
  if constexpr (L_ + l_ >= Lo && L_ + l_ <= Hi)                                    \
    if (it.L == L_ && it.l == l_) {                                                \
      if constexpr (Rhs)                                                           \
        jrhs_item<L_, l_>(it, J, in, out);                                         \
      else                                                                         \
        jpot_item<L_, l_>(it, J, in, out);                                         \
      return;                                                                      \
    }
#define SXC_JL(L_) SXC_J(L_, 0) SXC_J(L_, 1) SXC_J(L_, 2) SXC_J(L_, 3) SXC_J(L_, 4)
  static_assert(kJMaxLAux == 4 && kJMaxLPrim == 3, "one case per (L, l)");
  SXC_JL(0) SXC_JL(1) SXC_JL(2) SXC_JL(3) SXC_JL(4) SXC_JL(5) SXC_JL(6)
#undef SXC_JL
#undef SXC_J
}

template <bool Rhs, int Lo, int Hi>
__global__ __launch_bounds__(64) void jmeet_kernel(const JItem* __restrict__ items, JView J,
                                                   const double* __restrict__ in, double* __restrict__ out) {
  const JItem it = items[blockIdx.x];
  jmeet<Rhs, Lo, Hi>(it, J, in, out);
}

// 2 pi^(5/2) / a coef (2a)^(-(l + s) / 2): what the Hermite coefficients of order s of an auxiliary
// primitive share.
__device__ inline double aux_scale(double a, double coef, int l, int s) {
  double f = 34.986836655249725693 / a * coef;  // 2 pi^(5/2)
  for (int k = 0; k < (l + s) / 2; ++k) f *= 0.5 / a;
  return s & 1 ? -f : f;
}

// Auxiliary functions between their Cartesian coefficients and the primitives' Hermite ones, one
// thread per primitive and Hermite index.
// U[a][tau nu phi] = (-1)^(tau + nu + phi) 2 pi^(5/2) / a coef sum_c cc_c E E E (input of step 4)
__global__ __launch_bounds__(256) void jaux_in_kernel(JView J, int naux, const int* __restrict__ prim_shell,
                                                      const DevShell* __restrict__ aux,
                                                      const double* __restrict__ prim_coef,
                                                      const int* __restrict__ cart_off, const double* __restrict__ cc,
                                                      double* __restrict__ U) {
  const int id = blockIdx.x * 256 + threadIdx.x, a = id / kJMaxHs, i = id - a * kJMaxHs;
  if (a >= naux) return;
  const int sh = prim_shell[a], l = aux[sh].l, nc = aux[sh].ncart;
  if (i >= hcount_c(l)) return;
  const int t = kHerm.t[i], u = kHerm.u[i], v = kHerm.v[i], s = t + u + v;
  double sum = 0.0;
  if (((l - s) & 1) == 0)
    for (int c = 0; c < nc; ++c) {
      const int ax = kCart.x[l][c], ay = kCart.y[l][c], az = kCart.z[l][c];
      if (t <= ax && u <= ay && v <= az)
        sum += cc[cart_off[sh] + c] * (kAux.c[ax][t] * kAux.c[ay][u] * kAux.c[az][v]);
    }
  U[J.aherm0[l] + (int64_t)(a - J.aux0[l]) * hcount_c(l) + i] =
      aux_scale(J.aux[4 * (int64_t)a + 3], prim_coef[a], l, s) * sum;
}

// bc[shell][c] = sum over the shell's primitives of the same coefficients times W (output of step 2),
// one thread per Cartesian function
__global__ __launch_bounds__(64) void jaux_out_kernel(JView J, const DevShell* __restrict__ aux, int nshell,
                                                      const int* __restrict__ shell_prim,
                                                      const double* __restrict__ prim_coef,
                                                      const int* __restrict__ cart_off, const double* __restrict__ W,
                                                      double* __restrict__ bc) {
  const int sh = blockIdx.x * 4 + (threadIdx.x >> 4), c = threadIdx.x & 15;
  if (sh >= nshell || c >= aux[sh].ncart) return;
  const int l = aux[sh].l, nal = J.aux0[l + 1] - J.aux0[l];
  const int ax = kCart.x[l][c], ay = kCart.y[l][c], az = kCart.z[l][c];
  double sum = 0.0;
  for (int k = 0; k < aux[sh].nprim; ++k) {
    const int a = shell_prim[sh] + k;
    const double ea = J.aux[4 * (int64_t)a + 3];
    const double* Wa = W + J.aherm0[l] + (a - J.aux0[l]);
    for (int i = 0; i < hcount_c(l); ++i) {
      const int t = kHerm.t[i], u = kHerm.u[i], v = kHerm.v[i], s = t + u + v;
      if (((l - s) & 1) == 0 && t <= ax && u <= ay && v <= az)
        sum += aux_scale(ea, prim_coef[a], l, s) * (kAux.c[ax][t] * kAux.c[ay][u] * kAux.c[az][v]) *
               Wa[(int64_t)i * nal];
    }
  }
  bc[cart_off[sh] + c] = sum;
}

// Auxiliary AOs from Cartesian functions, b_f = sum_c M[f][c] bc_c, and back, cc_c = sum_f c_f M[f][c]; one
// thread per shell.  bad: set where a b is not finite.
__global__ __launch_bounds__(64) void aux_to_ao_kernel(const DevShell* __restrict__ aux, int nshell,
                                                       const double* __restrict__ ang,
                                                       const int* __restrict__ cart_off,
                                                       const double* __restrict__ bc, double* __restrict__ b, int* bad) {
  const int sh = blockIdx.x * 64 + threadIdx.x;
  if (sh >= nshell) return;
  const DevShell S = aux[sh];
  for (int f = 0; f < S.nfunc; ++f) {
    double v = 0.0;
    for (int c = 0; c < S.ncart; ++c) v += ang[S.ang_off + f * S.ncart + c] * bc[cart_off[sh] + c];
    b[S.ao_off + f] = v;
    if (!isfinite(v)) *bad = 1;
  }
}
__global__ __launch_bounds__(64) void aux_to_cart_kernel(const DevShell* __restrict__ aux, int nshell,
                                                         const double* __restrict__ ang,
                                                         const int* __restrict__ cart_off,
                                                         const double* __restrict__ c, double* __restrict__ cc) {
  const int sh = blockIdx.x * 64 + threadIdx.x;
  if (sh >= nshell) return;
  const DevShell S = aux[sh];
  for (int q = 0; q < S.ncart; ++q) {
    double v = 0.0;
    for (int f = 0; f < S.nfunc; ++f) v += c[S.ao_off + f] * ang[S.ang_off + f * S.ncart + q];
    cc[cart_off[sh] + q] = v;
  }
}

// The metric's two triangular solves (M = L L^T, L row-major), 64 unknowns per launch: every workgroup
// forms the block's solution from the inverse of its diagonal block (32 KB, from L2) and subtracts
// its share from 64 of the remaining right-hand sides, so a step has no wait inside.  What bounds it
// is the chain of n / 64 launches: 0.4 ms for 2 300 unknowns, against 3.2 ms for the host's two
// solves and the way there and back.
constexpr int kSB = kSolveBlock;
__global__ __launch_bounds__(256) void solve_lower_kernel(const double* __restrict__ L, int n,
                                                          const double* __restrict__ dinv, int k,
                                                          double* __restrict__ v, double* __restrict__ x) {
  __shared__ double vk[kSB], xk[kSB];
  const int t = threadIdx.x, row = t >> 2, q = t & 3, k0 = k * kSB;
  if (t < kSB) vk[t] = k0 + t < n ? v[k0 + t] : 0.0;
  const int64_t i = (int64_t)k0 + kSB + (int64_t)blockIdx.x * kSB + row;
  double l[kSB / 4];
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) l[e] = i < n ? L[i * n + k0 + q + 4 * e] : 0.0;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) s += dinv[((int64_t)k * kSB + row) * kSB + q + 4 * e] * vk[q + 4 * e];
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  if (q == 0) {
    xk[row] = s;
    if (blockIdx.x == 0 && k0 + row < n) x[k0 + row] = s;
  }
  __syncthreads();
  s = 0.0;
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) s += l[e] * xk[q + 4 * e];
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  if (q == 0 && i < n) v[i] -= s;
}
// The same for L^T, from the last block to the first; workgroup blockIdx.x updates 64 of the k0
// unknowns before the block.
__global__ __launch_bounds__(256) void solve_upper_kernel(const double* __restrict__ L, int n,
                                                          const double* __restrict__ dinv, int k,
                                                          double* __restrict__ v, double* __restrict__ x) {
  __shared__ double vk[kSB], xk[kSB], part[4][kSB];
  const int t = threadIdx.x, col = t & 63, q = t >> 6, k0 = k * kSB;
  if (t < kSB) vk[t] = k0 + t < n ? v[k0 + t] : 0.0;
  const int j = blockIdx.x * kSB + col;
  double l[kSB / 4];
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) {
    const int i = k0 + q * (kSB / 4) + e;
    l[e] = i < n && j < k0 ? L[(int64_t)i * n + j] : 0.0;
  }
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) {
    const int i = q * (kSB / 4) + e;
    s += dinv[((int64_t)k * kSB + i) * kSB + col] * vk[i];
  }
  part[q][col] = s;
  __syncthreads();
  if (t < kSB) {
    xk[t] = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    if (blockIdx.x == 0 && k0 + t < n) x[k0 + t] = xk[t];
  }
  __syncthreads();
  s = 0.0;
#pragma unroll
  for (int e = 0; e < kSB / 4; ++e) s += l[e] * xk[q * (kSB / 4) + e];
  part[q][col] = s;
  __syncthreads();
  if (t < kSB && j < k0) v[j] -= (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
}

}  // namespace

template <bool Dens>
static void launch_jpair(hipStream_t s, int cls, const JPairItem* items, int nitem, const JPair* pairs,
                         const DevShell* shells, const double* ang, const JView& Jv, const double* in, int n,
                         double* out) {
  if (nitem <= 0) return;
  if (cls == 0)
    hipLaunchKernelGGL((jpair_kernel<Dens, 0, kJPairTop>), dim3(nitem), dim3(64), 0, s, items, pairs, shells, ang, Jv,
                       in, n, out);
  else
    hipLaunchKernelGGL((jpair_kernel<Dens, kJPairTop + 1, 2 * kJMaxLPrim>), dim3(nitem), dim3(64), 0, s, items, pairs,
                       shells, ang, Jv, in, n, out);
}

void launch_jdens(hipStream_t s, int cls, const JPairItem* items, int nitem, const JPair* pairs, const DevShell* shells,
                  const double* ang, const JView& Jv, const double* P, int n, double* D) {
  launch_jpair<true>(s, cls, items, nitem, pairs, shells, ang, Jv, P, n, D);
}

void launch_jassemble(hipStream_t s, int cls, const JPairItem* items, int nitem, const JPair* pairs,
                      const DevShell* shells, const double* ang, const JView& Jv, const double* V, int n, double* J) {
  launch_jpair<false>(s, cls, items, nitem, pairs, shells, ang, Jv, V, n, J);
}

template <bool Rhs>
static void launch_jmeet(hipStream_t s, int cls, const JItem* items, int nitem, const JView& J, const double* in,
                         double* out) {
  if (nitem <= 0) return;
  if (cls == 0)
    hipLaunchKernelGGL((jmeet_kernel<Rhs, 0, kJClassTop[0]>), dim3(nitem), dim3(64), 0, s, items, J, in, out);
  else if (cls == 1)
    hipLaunchKernelGGL((jmeet_kernel<Rhs, kJClassTop[0] + 1, kJClassTop[1]>), dim3(nitem), dim3(64), 0, s, items, J,
                       in, out);
  else
    hipLaunchKernelGGL((jmeet_kernel<Rhs, kJClassTop[1] + 1, kJMaxL>), dim3(nitem), dim3(64), 0, s, items, J, in, out);
}

void launch_jrhs(hipStream_t s, int cls, const JItem* items, int nitem, const JView& J, const double* D, double* W) {
  launch_jmeet<true>(s, cls, items, nitem, J, D, W);
}

void launch_jpot(hipStream_t s, int cls, const JItem* items, int nitem, const JView& J, const double* U, double* V) {
  launch_jmeet<false>(s, cls, items, nitem, J, U, V);
}

void launch_jaux_in(hipStream_t s, const JView& J, int naux, const int* prim_shell, const DevShell* aux,
                    const double* prim_coef, const int* cart_off, const double* cc, double* U) {
  if (naux <= 0) return;
  hipLaunchKernelGGL(jaux_in_kernel, dim3((naux * kJMaxHs + 255) / 256), dim3(256), 0, s, J, naux, prim_shell, aux, prim_coef,
                     cart_off, cc, U);
}

void launch_jaux_out(hipStream_t s, const JView& J, const DevShell* aux, int nshell, const int* shell_prim,
                     const double* prim_coef, const int* cart_off, const double* W, double* bc) {
  if (nshell <= 0) return;
  hipLaunchKernelGGL(jaux_out_kernel, dim3((nshell + 3) / 4), dim3(64), 0, s, J, aux, nshell, shell_prim, prim_coef,
                     cart_off, W, bc);
}

void launch_metric_solve(hipStream_t s, const double* L, int n, const double* dinv, const DevShell* aux, int nshell,
                         const double* ang, const int* cart_off, const double* bc, double* b, double* y, double* cc,
                         int* bad) {
  if (n <= 0) return;
  const int nblk = (n + kSB - 1) / kSB;
  hipLaunchKernelGGL(aux_to_ao_kernel, dim3((nshell + 63) / 64), dim3(64), 0, s, aux, nshell, ang, cart_off, bc, b,
                     bad);
  for (int k = 0; k < nblk; ++k)
    hipLaunchKernelGGL(solve_lower_kernel, dim3(std::max(nblk - k - 1, 1)), dim3(256), 0, s, L, n, dinv, k, b, y);
  for (int k = nblk - 1; k >= 0; --k)
    hipLaunchKernelGGL(solve_upper_kernel, dim3(std::max(k, 1)), dim3(256), 0, s, L, n, dinv, k, y, b);
  hipLaunchKernelGGL(aux_to_cart_kernel, dim3((nshell + 63) / 64), dim3(64), 0, s, aux, nshell, ang, cart_off, b, cc);
}

}  // namespace sxc
