// Device code shared by the solver's material-point kernels (constitutive.hip)
// and the callers' point updates (points.hip): the cF slip systems, the 3x3
// algebra, Hooke's law, powers, and the addressing of structure-of-arrays
// planes.
#pragma once
#include "common.h"

namespace sca {
namespace {

// cF <110>{111} slip systems (crystal.f90:41-63): direction, normal.
__device__ constexpr int SLIP[NSLIP][6] = {
    {0, 1, -1, 1, 1, 1},   {-1, 0, 1, 1, 1, 1},   {1, -1, 0, 1, 1, 1},
    {0, -1, -1, -1, -1, 1}, {1, 0, 1, -1, -1, 1},  {-1, 1, 0, -1, -1, 1},
    {0, -1, 1, 1, -1, -1}, {-1, 0, -1, 1, -1, -1}, {1, 1, 0, 1, -1, -1},
    {0, 1, 1, -1, 1, -1},  {1, 0, -1, -1, 1, -1},  {-1, -1, 0, -1, 1, -1}};

// sign pattern of P_s(i,j) = d_i n_j
__device__ __forceinline__ constexpr int psg(int s, int i, int j) { return SLIP[s][i] * SLIP[s][3 + j]; }

// cF slip-slip interaction types (reacting, acting), crystal.f90:623-640
__device__ constexpr int HTYPE[NSLIP][NSLIP] = {
    {1, 2, 2, 4, 7, 5, 3, 5, 5, 4, 6, 7}, {2, 1, 2, 7, 4, 5, 6, 4, 7, 5, 3, 5},
    {2, 2, 1, 5, 5, 3, 6, 7, 4, 7, 6, 4}, {4, 7, 6, 1, 2, 2, 4, 6, 7, 3, 5, 5},
    {7, 4, 6, 2, 1, 2, 5, 3, 5, 6, 4, 7}, {5, 5, 3, 2, 2, 1, 7, 6, 4, 6, 7, 4},
    {3, 5, 5, 4, 6, 7, 1, 2, 2, 4, 7, 6}, {6, 4, 7, 5, 3, 5, 2, 1, 2, 7, 4, 6},
    {6, 7, 4, 7, 6, 4, 2, 2, 1, 5, 5, 3}, {4, 6, 7, 3, 5, 5, 4, 7, 6, 1, 2, 2},
    {5, 3, 5, 6, 4, 7, 7, 4, 6, 2, 1, 2}, {7, 6, 4, 6, 7, 4, 5, 5, 3, 2, 2, 1}};

// Structure of the table used to share work between slip systems:
// - the systems 3p, 3p+1, 3p+2 lie on the same plane (normal), p = 0..3;
// - the systems g, g+3, g+6, g+9 (g = 0, 1, 2) have direction component g
//   zero.
// The Newton systems (constitutive.hip, points.hip) need, for every entry r = 3i+j and
// every symmetric pair (m,l), the sum over s of f_s P_s(i,j) k_s(m,l) with
// k_s(m,l) = P_s(m,m) (m = l) or P_s(m,l) + P_s(l,m).  Restricted to one
// direction group its coefficient vector is zero or plus/minus one of the
// four Hadamard rows (1,1,1,1), (1,1,-1,-1), (1,-1,1,-1), (1,-1,-1,1), so
// the sums come from the four Hadamard sums of each group's f_s.
__device__ __forceinline__ constexpr int qcoef(int s, int r, int m, int l) {
  return psg(s, r / 3, r % 3) * (m == l ? psg(s, m, m) : psg(s, m, l) + psg(s, l, m));
}
// 0 when group g does not enter Q_r(m,l), else sign * (1 + Hadamard row)
__device__ __forceinline__ constexpr int qhad(int g, int r, int m, int l) {
  const int a = qcoef(g, r, m, l), b = qcoef(g + 3, r, m, l), c = qcoef(g + 6, r, m, l);
  if (a == 0) return 0;
  return a * (1 + (b * a > 0 ? (c * a > 0 ? 0 : 1) : (c * a > 0 ? 2 : 3)));
}
constexpr bool slip_structure_holds() {
  for (int p = 0; p < 4; ++p)
    for (int k = 1; k < 3; ++k)
      for (int j = 0; j < 3; ++j)
        if (SLIP[3 * p + k][3 + j] != SLIP[3 * p][3 + j]) return false;
  for (int s = 0; s < NSLIP; ++s)
    if (SLIP[s][s % 3] != 0) return false;
  const int had[4][4] = {{1, 1, 1, 1}, {1, 1, -1, -1}, {1, -1, 1, -1}, {1, -1, -1, 1}};
  for (int r = 0; r < 9; ++r)
    for (int m = 0; m < 3; ++m)
      for (int l = m; l < 3; ++l) {
        int groups = 0;
        for (int g = 0; g < 3; ++g) {
          const int code = qhad(g, r, m, l);
          for (int k = 0; k < 4; ++k) {
            const int want = code == 0 ? 0 : (code > 0 ? 1 : -1) * had[(code > 0 ? code : -code) - 1][k];
            if (qcoef(g + 3 * k, r, m, l) != want) return false;
          }
          groups += code != 0;
        }
        if (groups == 0) return false;
      }
  return true;
}
static_assert(slip_structure_holds(), "cF slip table: planes of three systems, Hadamard-structured Jacobian sums");

// ---- small dense helpers (row-major 3x3 in registers: m[3*i+j]) ----------
__device__ __forceinline__ void mm33(const double* A, const double* B, double* C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[3 * i + j] = A[3 * i] * B[j] + A[3 * i + 1] * B[3 + j] + A[3 * i + 2] * B[6 + j];
}

// Divisions without the compiler's range fix-ups, for operands far from the
// range limits (slip resistances, the 3x3 determinants of deformation
// gradients, the pivots of the Newton system, none of them near 2^+-1000):
// 1/x as the hardware reciprocal refined by two Newton steps (as the
// compiler's own division does before its fix-ups), and a / b as the rounded
// product a (1/b) corrected once by its exact remainder a - b q (Markstein):
// the correctly rounded quotient when 1/b is the correctly rounded
// reciprocal, within one rounding of it otherwise
__device__ __forceinline__ double rcp_refined(double x) {
  double r = __builtin_amdgcn_rcp(x);
#pragma unroll
  for (int k = 0; k < 2; ++k) r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
  return r;
}
__device__ __forceinline__ double div_rcp(double a, double b, double rb) {
  const double q = a * rb;
  return __builtin_fma(__builtin_fma(-q, b, a), rb, q);
}

// math_invert33 (math.f90:511-545); returns false if |det| <= 10*tiny
__device__ __forceinline__ bool inv33(const double* A, double* R, double* detOut) {
  R[0] = A[4] * A[8] - A[5] * A[7];
  R[3] = -A[3] * A[8] + A[5] * A[6];
  R[6] = A[3] * A[7] - A[4] * A[6];
  double det = A[0] * R[0] + A[1] * R[3] + A[2] * R[6];
  if (fabs(det) <= 2.2250738585072014e-308 * 10.0) return false;
  R[1] = -A[1] * A[8] + A[2] * A[7];
  R[4] = A[0] * A[8] - A[2] * A[6];
  R[7] = -A[0] * A[7] + A[1] * A[6];
  R[2] = A[1] * A[5] - A[2] * A[4];
  R[5] = -A[0] * A[5] + A[2] * A[3];
  R[8] = A[0] * A[4] - A[1] * A[3];
  const double rd = rcp_refined(det);
#pragma unroll
  for (int k = 0; k < 9; ++k) R[k] = div_rcp(R[k], det, rd);
  if (detOut) *detOut = det;
  return true;
}

__device__ __forceinline__ double det33(const double* m) {
  return m[0] * (m[4] * m[8] - m[5] * m[7]) - m[1] * (m[3] * m[8] - m[5] * m[6]) + m[2] * (m[3] * m[7] - m[4] * m[6]);
}


// x^e for x >= 0 with e = e4/4: binary powering of the integer part times
// sqrt / sqrt-sqrt for the quarter part; libm pow() when e4 < 0
__device__ __noinline__ double pow_general(double x, double e) { return pow(x, e); }
__device__ __forceinline__ double powq(double x, int e4, double e) {
  if (e4 < 0) return pow_general(x, e);
  double r = 1.0, b = x;
  int m = e4 >> 2;
  while (m) {
    if (m & 1) r *= b;
    b *= b;
    m >>= 1;
  }
  const int q = e4 & 3;
  if (q) {
    const double h = sqrt(x);
    const double f = sqrt(h);
    r *= (q == 1) ? f : (q == 2) ? h : h * f;
  }
  return r;
}
// compile-time quarter exponent E4/4 (E4 >= 0): fully unrolled
// x^(-1/4) for x in [2^-1000, 2^1000]: a start value from the hardware
// square root and reciprocal square root, then three Newton steps
// y <- y (5 - x y^4) / 4 (quadratic: full precision from any start within
// 2^-8 of the root); two correctly rounded square roots cost about three
// times as many instructions
__device__ __forceinline__ double rqrt_refined(double x) {
  double y = __builtin_amdgcn_rsq(__builtin_amdgcn_sqrt(x));
  const double mq = -0.25 * x;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double y2 = y * y;
    y = y * __builtin_fma(mq, y2 * y2, 1.25);
  }
  return y;
}

template <int E4>
__device__ __forceinline__ double powc(double x) {
  double r = 1.0, b = x;
#pragma unroll
  for (int m = E4 >> 2; m; m >>= 1) {
    if (m & 1) r *= b;
    b *= b;
  }
  constexpr int q = E4 & 3;
  if constexpr (q == 2) {
    r *= sqrt(x);
  } else if constexpr (q != 0) {
    // x^(1/4) = x y^3 and x^(3/4) = x y with y = x^(-1/4) (within 10 ulp),
    // y taken at x clamped to [2^-1000, 2^1000] and multiplied by the true x:
    // for x = 0 this gives 0, NaN propagates, and outside the range the
    // power x^(E4 >> 2) >= x^1 (E4 >= 4) underflows to 0 or overflows to inf
    // as the exact result does (E4 < 4 exponents run the runtime path)
    static_assert(E4 >= 4, "quarter exponents below 1 are not compiled in");
    const double y = rqrt_refined(fmin(fmax(x, 0x1p-1000), 0x1p1000));
    r *= (q == 1) ? x * (y * (y * y)) : x * y;
  }
  return r;
}
// exponent dispatch: E4 >= 0 compile-time, E4 == -1 runtime (mc)
template <int E4>
__device__ __forceinline__ double powe(double x, int e4rt, double e) {
  if constexpr (E4 >= 0) return powc<E4>(x);
  else return powq(x, e4rt, e);
}

// Hooke (elastic.f90:157-195) with Fi = I, cubic C66:
// E = (Fe^T Fe - I)/2, S = C66 : E (Voigt strain with engineering shear)
__device__ __forceinline__ void hooke_S(const double* Fe, double* S, const MatConst& mc) {
  double E[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      E[3 * i + j] = 0.5 * ((Fe[i] * Fe[j] + Fe[3 + i] * Fe[3 + j] + Fe[6 + i] * Fe[6 + j]) - (i == j ? 1.0 : 0.0));
  const double e11 = E[0], e22 = E[4], e33 = E[8];
  const double s11 = mc.C11 * e11 + mc.C12 * e22 + mc.C12 * e33;
  const double s22 = mc.C12 * e11 + mc.C11 * e22 + mc.C12 * e33;
  const double s33 = mc.C12 * e11 + mc.C12 * e22 + mc.C11 * e33;
  const double s23 = mc.C44 * (2.0 * E[7]);
  const double s13 = mc.C44 * (2.0 * E[6]);
  const double s12 = mc.C44 * (2.0 * E[1]);
  S[0] = s11; S[1] = s12; S[2] = s13;
  S[3] = s12; S[4] = s22; S[5] = s23;
  S[6] = s13; S[7] = s23; S[8] = s33;
}

// tau_s = Mp : P_s with Mp = S (Fi = I), for all systems: tau_s = v d_s . (S n_s),
// the three systems of a plane sharing S n (signed sums: every entry of d_s and
// n_s is 0 or +-1)
__device__ __forceinline__ void resolved_shears(const double* S, double v, double* tau) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    double u[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double t = SLIP[3 * p][3] > 0 ? S[3 * i] : -S[3 * i];
#pragma unroll
      for (int j = 1; j < 3; ++j) t = SLIP[3 * p][3 + j] > 0 ? t + S[3 * i + j] : t - S[3 * i + j];
      u[i] = t;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int s = 3 * p + k;
      double t = 0.0;
      bool first = true;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (SLIP[s][i] != 0) {
          t = first ? (SLIP[s][i] > 0 ? u[i] : -u[i]) : (SLIP[s][i] > 0 ? t + u[i] : t - u[i]);
          first = false;
        }
      tau[s] = v * t;
    }
  }
}

// Lp = v sum_s g_s d_s n_s^T, the systems of a plane summed first:
// Lp = v sum_p (sum_{s on p} g_s d_s) n_p^T (row-major 3x3 out)
__device__ __forceinline__ void slip_sum(const double* g, double v, double* L) {
  double w[4][3];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double t = 0.0;
      bool first = true;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int s = 3 * p + k;
        if (SLIP[s][i] != 0) {
          t = first ? (SLIP[s][i] > 0 ? g[s] : -g[s]) : (SLIP[s][i] > 0 ? t + g[s] : t - g[s]);
          first = false;
        }
      }
      w[p][i] = t;
    }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double t = SLIP[0][3 + j] > 0 ? w[0][i] : -w[0][i];
#pragma unroll
      for (int p = 1; p < 4; ++p) t = SLIP[3 * p][3 + j] > 0 ? t + w[p][i] : t - w[p][i];
      L[3 * i + j] = v * t;
    }
}

// Column-major plane q = i+3j of a (3,3) field <-> row-major register 3*i+j
__device__ __forceinline__ int rm(int q) { return 3 * (q % 3) + q / 3; }

__device__ __forceinline__ void load33(const double* base, int64_t N, int64_t c, double* m) {
#pragma unroll
  for (int q = 0; q < 9; ++q) m[rm(q)] = base[q * N + c];
}

// Plane addressing by a uniform plane pointer plus the lane's 32-bit byte
// offset (scalar base + vector offset): one offset register serves every
// plane, instead of a 64-bit lane address per plane.  Needs (c_end) * 8 < 2^32,
// which the launcher checks.
//
// Every plane pointer given to ld/st/load33/store33 with a Lane must be the
// same in all lanes (formed from kernel arguments and uniform indices only):
// it is read from the first active lane, which keeps the compiler from
// folding the lane offset into a 64-bit per-lane address for every plane.
// A per-lane choice between two planes is made on the loaded values
// (load33_sel), never on the pointer.
struct Lane {
  uint32_t off;  // cell index * 8
};
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
typedef __attribute__((address_space(1))) double gdouble;  // global memory
__device__ __forceinline__ double ld(const double* plane, Lane l) {
  return *reinterpret_cast<const gdouble*>(uniform_u64(reinterpret_cast<uint64_t>(plane)) + l.off);
}
__device__ __forceinline__ void st(double* plane, Lane l, double v) {
  *reinterpret_cast<gdouble*>(uniform_u64(reinterpret_cast<uint64_t>(plane)) + l.off) = v;
}
// The plane stride as a value of this place only: pointers formed from it are
// formed here (two scalar adds a plane).  From the plain N the compiler forms
// the pointers of every access once at the kernel's entry, keeps them in
// vector lanes (it has no scalar registers for 150 of them) and reads each
// back at its use: 838 lane moves among the update kernel's 7824 instructions,
// 304 among 7478 with the stride formed where it is used.
__device__ __forceinline__ int64_t stride_here(int64_t N) {
  asm volatile("" : "+s"(N));
  return N;
}
__device__ __forceinline__ void load33(const double* base, int64_t N, Lane l, double* m) {
  const int64_t n = stride_here(N);
#pragma unroll
  for (int q = 0; q < 9; ++q) m[rm(q)] = ld(base + q * n, l);
}
__device__ __forceinline__ void store33(double* base, int64_t N, Lane l, const double* m) {
  const int64_t n = stride_here(N);
#pragma unroll
  for (int q = 0; q < 9; ++q) st(base + q * n, l, m[rm(q)]);
}
// load from a plane chosen per lane (the base may differ between lanes): a
// 64-bit lane address and one unconditional load, so that the loads of all
// lanes and planes issue together instead of in divergent branches
__device__ __forceinline__ double ldv(const double* plane, Lane l) {
  return *reinterpret_cast<const gdouble*>(reinterpret_cast<uint64_t>(plane) + l.off);
}
// per-lane choice of the plane set: sel ? a : b
__device__ __forceinline__ void load33_sel(bool sel, const double* a, const double* b, int64_t N, Lane l,
                                           double* m) {
  const double* base = sel ? a : b;
  const int64_t n = stride_here(N);
#pragma unroll
  for (int q = 0; q < 9; ++q) m[rm(q)] = ldv(base + q * n, l);
}

// (C : X)(i,j) = sum_kl C(i,j,k,l) X(k,l) for the cubic stiffness
// (math_Voigt66to3333_stiffness of C11, C12, C44): C11 X_ii + C12 sum_{k!=i}
// X_kk on the diagonal, C44 (X_ij + X_ji) off it (row-major 3x3)
__device__ __forceinline__ void cubic_contract(const double* X, double* Y, const MatConst& mc) {
  const double t = X[0] + X[4] + X[8];
  const double d = mc.C11 - mc.C12;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      Y[3 * i + j] = (i == j) ? mc.C12 * t + d * X[4 * i] : mc.C44 * (X[3 * i + j] + X[3 * j + i]);
}
// Substep scratch layout (per point, planes of N doubles): F0 (9), Lp0 (9),
// Fp0 (9), state0 (24) of the current substep start, and F of the substep
// being integrated (9).  Touched only when the first full step was cut back.
constexpr int SUB_F0 = 0, SUB_LP0 = 9, SUB_FP0 = 18, SUB_ST0 = 27, SUB_FLOC = 51, SUB_PLANES = 60;

}  // namespace
}  // namespace sca
