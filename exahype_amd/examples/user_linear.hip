// user_linear.hip -- user PDEs with a non-conservative product
// (exahype_amd/user_solver.hpp), built into exahype_amd/libexa_user_example.so
// beside user_euler.hip; the tests drive them through exa_grid_create_user.
#include <exahype_amd/user_solver.hpp>

namespace {

// Linear elasticity in velocity-stress form without fluxes, as the library's
// own (variables sxx, syy, szz, sxy, syz, sxz, u, v, w; parameters lambda, mu,
// rho), followed by EXTRA parameters that the equations ignore.
template <int EXTRA>
struct UserElastic {
  static constexpr int V = 9;
  static constexpr int P = 3 + EXTRA;

  template <typename T>
  __device__ static void flux(const T*, T (*F)[V]) {
    for (int d = 0; d < 3; ++d)
      for (int m = 0; m < V; ++m) F[d][m] = T(0);
  }

  template <typename T>
  __device__ static void eigenvalues(const T* Q, int, T* lambda) {
    const T cp = sqrt((Q[9] + T(2) * Q[10]) / Q[11]), cs = sqrt(Q[10] / Q[11]);
    const T l[V] = {-cp, -cs, -cs, T(0), T(0), T(0), cs, cs, cp};
    for (int m = 0; m < V; ++m) lambda[m] = l[m];
  }

  template <typename T>
  __device__ static void algebraic_source(const T*, T* S) {
    for (int m = 0; m < V; ++m) S[m] = T(0);
  }

  template <typename T>
  __device__ static void ncp(const T* Q, const T (*g)[V], T* BgradQ) {
    const T lam = Q[9], mu = Q[10], irho = T(1) / Q[11];
    const T l2m = lam + T(2) * mu;
    BgradQ[0] = -(l2m * g[0][6] + lam * g[1][7] + lam * g[2][8]);
    BgradQ[1] = -(lam * g[0][6] + l2m * g[1][7] + lam * g[2][8]);
    BgradQ[2] = -(lam * g[0][6] + lam * g[1][7] + l2m * g[2][8]);
    BgradQ[3] = -mu * (g[0][7] + g[1][6]);
    BgradQ[4] = -mu * (g[1][8] + g[2][7]);
    BgradQ[5] = -mu * (g[0][8] + g[2][6]);
    BgradQ[6] = -irho * (g[0][0] + g[1][3] + g[2][5]);
    BgradQ[7] = -irho * (g[0][3] + g[1][1] + g[2][4]);
    BgradQ[8] = -irho * (g[0][5] + g[1][4] + g[2][2]);
  }
};

// Linear acoustics with a tracer carried by a constant wind (variables
// pressure, u, v, w, tracer).  SPLIT: half of every term as a flux and half as a
// non-conservative product, which for constant coefficients are the same
// operator, so that both forms compute the same solution.
template <bool SPLIT>
struct UserWaves {
  static constexpr int V = 5;
  static constexpr int P = 0;
  static constexpr double CFL = 0.05;  // the Picard iteration ends by its residual, not its limit

  template <typename T>
  __device__ static T wind(int d) {
    return d == 0 ? T(0.5) : (d == 1 ? T(-0.25) : T(0.75));
  }

  // A_d q: density 2, bulk modulus 3
  template <typename T>
  __device__ static void apply(int d, const T* q, T* out) {
    out[0] = T(3) * q[1 + d] + wind<T>(d) * q[0];
    for (int k = 0; k < 3; ++k) out[1 + k] = wind<T>(d) * q[1 + k] + (k == d ? T(0.5) * q[0] : T(0));
    out[4] = wind<T>(d) * q[4];
  }

  template <typename T>
  __device__ static void flux(const T* Q, T (*F)[V]) {
    for (int d = 0; d < 3; ++d) {
      apply(d, Q, F[d]);
      if (SPLIT)
        for (int m = 0; m < V; ++m) F[d][m] *= T(0.5);
    }
  }

  template <typename T>
  __device__ static void eigenvalues(const T*, int d, T* lambda) {
    const T c = sqrt(T(1.5));
    for (int m = 0; m < V; ++m) lambda[m] = wind<T>(d);
    lambda[0] -= c;
    lambda[1] += c;
  }

  template <typename T>
  __device__ static void algebraic_source(const T*, T* S) {
    for (int m = 0; m < V; ++m) S[m] = T(0);
  }

  template <typename T>
  __device__ static void ncp(const T*, const T (*g)[V], T* BgradQ) {
    T a[3][V];
    for (int d = 0; d < 3; ++d) apply(d, g[d], a[d]);
    for (int m = 0; m < V; ++m) BgradQ[m] = T(0.5) * (a[0][m] + a[1][m] + a[2][m]);
  }
};

}  // namespace

// at order 1 the parameters outnumber the rows of the predictor's iterate
EXA_USER_SOLVER(exa_user_elastic_order1_many, UserElastic<7>, 1, exa::kNCP)
EXA_USER_SOLVER(exa_user_elastic_order2, UserElastic<0>, 2, exa::kNCP)
EXA_USER_SOLVER(exa_user_elastic_order4, UserElastic<0>, 4, exa::kNCP)
EXA_USER_SOLVER(exa_user_waves_order3, UserWaves<false>, 3, exa::kFlux)
EXA_USER_SOLVER(exa_user_waves_order4, UserWaves<false>, 4, exa::kFlux)
EXA_USER_SOLVER(exa_user_waves_order5, UserWaves<false>, 5, exa::kFlux)
EXA_USER_SOLVER(exa_user_waves_split_order3, UserWaves<true>, 3, exa::kFlux | exa::kNCP)
EXA_USER_SOLVER(exa_user_waves_split_order4, UserWaves<true>, 4, exa::kFlux | exa::kNCP | exa::kSource)
EXA_USER_SOLVER(exa_user_waves_split_order5, UserWaves<true>, 5, exa::kFlux | exa::kNCP)
EXA_USER_SOLVER(exa_user_waves_source_order4, UserWaves<false>, 4, exa::kFlux | exa::kSource)
