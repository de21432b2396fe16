// line_ops.hpp -- one-dimensional operators of the predictor along a line of B
// nodes: derived tables and the line contraction.
#pragma once

#include "exa_device.hpp"

namespace exa {

template <typename T>
__device__ constexpr T tc(double v) {
  return static_cast<T>(v);
}

// Operators derived from the tables, formed in double at compile time.
//   a_l = sum_t iK1[l][t] FLCoeff[t]: luh's share of a Picard iterate;
//   b_l = sum_t iK1[l][t] w_t: the share of a right-hand side that is the
//     same for all slices;
//   the derivative d[n][l] = Kxi[n][l] / w_l (at node l, of the basis function
//     of node n) and the volume operator Kxi[l][n], split into halves.
// Both operators change sign under (n, l) -> (B-1-n, B-1-l) (the literals of
// Kxi do, exactly), so a line contraction sum_n f(n) M[n][l] works on the sums
// e(n) = f(n) + f(B-1-n) and differences o(n) = f(n) - f(B-1-n): with
// S[n][l] = (M[n][l] + M[B-1-n][l]) / 2 and A[n][l] = (M[n][l] - M[B-1-n][l]) / 2,
// P = sum_n S e and Z = sum_n A o over the lower half of n give the results
// Z + P at l and Z - P at B-1-l.  B = 6: 18 multiply-adds, 12 additions and 18
// constants instead of 36 and 36.
namespace line_tables {
#define EXA_TABLE static constexpr
#include "dg_tables.inc"
#undef EXA_TABLE
struct Halves {
  double s[10][5][5], a[10][5][5];
};
struct Folded {
  double a[10][10], b[10][10];
  Halves d, k;
};
constexpr Folded folded() {
  Folded s{};
  for (int N = 0; N < 10; ++N) {
    const int B = N + 1;
    for (int l = 0; l < B; ++l)
      for (int t = 0; t < B; ++t) {
        s.a[N][l] += exa_ik1[N][l][t] * exa_fl_coeff[N][t];
        s.b[N][l] += exa_ik1[N][l][t] * exa_gl_weights[N][t];
      }
    for (int n = 0; n < (B + 1) / 2; ++n)
      for (int l = 0; l < (B + 1) / 2; ++l) {
        const int r = B - 1 - n;  // r == n: the middle node of an odd B, all in s
        const double dn = exa_kxi[N][n][l] / exa_gl_weights[N][l], dr = exa_kxi[N][r][l] / exa_gl_weights[N][l];
        s.d.s[N][n][l] = 0.5 * (dn + dr);
        s.d.a[N][n][l] = 0.5 * (dn - dr);
        s.k.s[N][n][l] = 0.5 * (exa_kxi[N][l][n] + exa_kxi[N][l][r]);
        s.k.a[N][n][l] = 0.5 * (exa_kxi[N][l][n] - exa_kxi[N][l][r]);
      }
  }
  return s;
}
}  // namespace line_tables
static __constant__ const line_tables::Folded exa_folded = line_tables::folded();

// out(l) = sum_n f(n) M[n][l], M = the derivative or (VOLUME) Kxi[l][n].
template <int B, bool VOLUME, typename T>
__device__ __attribute__((always_inline)) inline void contract_halves(const T* f, T* out) {
  constexpr int N = B - 1, H = B / 2;
  T e[H], o[H];
#pragma unroll
  for (int n = 0; n < H; ++n) {
    e[n] = f[n] + f[B - 1 - n];
    o[n] = f[n] - f[B - 1 - n];
  }
#pragma unroll
  for (int l = 0; l < H; ++l) {
    T p = T(0), z = T(0);
#pragma unroll
    for (int n = 0; n < H; ++n) {
      p += e[n] * tc<T>(VOLUME ? exa_folded.k.s[N][n][l] : exa_folded.d.s[N][n][l]);
      z += o[n] * tc<T>(VOLUME ? exa_folded.k.a[N][n][l] : exa_folded.d.a[N][n][l]);
    }
    if constexpr (B % 2 != 0) p += f[H] * tc<T>(VOLUME ? exa_folded.k.s[N][H][l] : exa_folded.d.s[N][H][l]);
    out[l] = z + p;
    out[B - 1 - l] = z - p;
  }
  if constexpr (B % 2 != 0) {
    T z = T(0);
#pragma unroll
    for (int n = 0; n < H; ++n) z += o[n] * tc<T>(VOLUME ? exa_folded.k.a[N][n][H] : exa_folded.d.a[N][n][H]);
    out[H] = z;
  }
}

// A value every lane holds alike, moved to scalar registers.
template <typename T>
__device__ inline T wave_uniform(T v) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __builtin_bit_cast(T, (unsigned long long)hi << 32 | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(unsigned, v)));
  }
}

}  // namespace exa
