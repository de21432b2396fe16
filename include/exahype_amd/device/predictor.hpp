// predictor.hpp -- the space-time predictor kernel (Picard iteration, time
// averaging, extrapolation, volume integral) as a template over the PDE
// functor, for the library's own PDEs and for a user's __device__ PDE
// (exahype_amd/user_solver.hpp).
//
// Reference semantics (K = ExaHyPE/kernels/aderdg/generic/c/3d):
//   predictor_kernel   K/spaceTimePredictorNonlinear.cpph:42-528,661-717
//                      + K/volumeIntegralNonlinear.cpph:136-225 (fused epilogue)
#pragma once

#include "aderdg.hpp"
#include "exa_device.hpp"
#include "line_ops.hpp"

#include <cfloat>
#include <type_traits>

namespace exa {

// Picard stopping rule (spaceTimePredictorNonlinear.cpph:314-318): stop when
// sum (lQi_new - lQi)^2 < 1e-14.  In float that absolute bound lies below the
// rounding floor of the iterate (about (6e-8 |q|)^2 per entry), so the
// FP32-bulk form stops when the root-mean-square change falls below
// kPicardRelTol32 times the root-mean-square of the iterate (or below the
// reference's bound, whichever is reached first).
constexpr double kPicardTol2 = 1e-7 * 1e-7;
constexpr float kPicardRelTol32 = 1e-6f;

// S = algebraicSource(Q) - NCP(Q, gradQ) at node (z,y,x) of a time slice whose
// variables are staged in sQ[var][node] (spaceTimePredictorNonlinear.cpph:238-266).
// ONE_LINE: one variable's line entries at a time in registers (otherwise the
// reads of all variables go out together, which takes most of the registers).
template <int B, class PDE, bool USE_SOURCE, bool USE_NCP, bool ONE_LINE, typename T>
__device__ inline void source_ncp(const T* Q, const T* sQ, const T* sDu, const T invDx[3], int z, int y,
                                  int x, T* S) {
  constexpr int V = PDE::V;
  constexpr int B2 = B * B, B3 = B2 * B;
  if (USE_SOURCE) {
    PDE::algebraic_source(Q, S);
  } else {
#pragma unroll
    for (int m = 0; m < V; ++m) S[m] = T(0);
  }
  if (USE_NCP) {
    // gradQ(dir, var) = invDx * sum_n lQi(..n..) * dudx[l][n] (:170-173, 199-202, 228-231)
    T gradQ[3][V];
#pragma unroll
    for (int m = 0; m < V; ++m) {
      T gx = T(0), gy = T(0), gz = T(0);
#pragma unroll
      for (int n = 0; n < B; ++n) {
        gx += sQ[m * B3 + (z * B + y) * B + n] * sDu[x * B + n];
        gy += sQ[m * B3 + (z * B + n) * B + x] * sDu[y * B + n];
        gz += sQ[m * B3 + (n * B + y) * B + x] * sDu[z * B + n];
      }
      gradQ[0][m] = invDx[0] * gx;
      gradQ[1][m] = invDx[1] * gy;
      gradQ[2][m] = invDx[2] * gz;
      if (ONE_LINE) __builtin_amdgcn_sched_barrier(0);
    }
    T ncp[V];
    PDE::ncp(Q, gradQ, ncp);
#pragma unroll
    for (int m = 0; m < V; ++m) S[m] -= ncp[m];
  }
}

// Where the predictor keeps the Picard iterate lQi^k of a cell (B^4 V values):
// its first NQL time slices live in LDS (as many as keep the workgroup's LDS
// within 144 KB next to one slice of fluxes sF), the other NQR slices in
// registers or, when registers run out (WSQ), in a per-cell device workspace
// that each thread reads and writes only at its own nodes.  Large sizes run
// the loop over time slices rolled (ROLLED).
// A PDE without fluxes whose slices all fit LDS takes the gradients from the
// iterate itself (IN_PLACE): no staged copy, no flux rows, and no barrier
// between slices, which only read the iterate.  In double at N=4 a cell takes
// 45 KB of LDS instead of 81, so three workgroups of two wavefronts per CU
// instead of one; LDS reads of the gradients' lines bound it.  Elastic N=4 in
// double, 41^3 cells, 8 steps: predictor 4.08 -> 2.26 ms per step together
// with the closed first iteration, the whole run 51.1 -> 46.7 ms by this form
// and the boundary fluxes left out.
template <int B, int V, int D, bool USE_NCP, typename T, int LDSK = 144, bool USE_FLUX = true,
          bool USE_SOURCE = false>
struct PredictorLayout {
  static constexpr int B2 = B * B, B3 = B2 * B;
  static constexpr int NT = node_threads(B);
  static constexpr bool IS_FP64 = sizeof(T) == sizeof(double);
  static constexpr long kLdsBudget = (long)LDSK * 1024;
  // (its B V rows also take the epilogue's D: not with parameters beyond (B - 1) V)
  static constexpr bool IN_PLACE = USE_NCP && !USE_FLUX && B * V >= D &&
                                   (long)(B * V * B3 + B2 + 64) * (long)sizeof(T) <= kLdsBudget;
  // LDS: one slice of fluxes [dir][var][node] (reused for lQhi / lFhi staging)
  static constexpr int SF = IN_PLACE ? 0 : (3 * V > D ? 3 * V : D) * B3;
  static constexpr long kSliceBytes = (long)V * B3 * sizeof(T);
  static constexpr long kOther =
      (long)(SF + (USE_NCP ? (IN_PLACE ? 0 : V * B3) + B2 : 0) + 3 + 2 * (NT / kWave)) * sizeof(T);
  static constexpr long kFree = kLdsBudget - kOther;
  // Up to B = 4 a flux-only PDE's iterate fits the registers beside the next one
  // (40 of 222 in double at B = 4): its reads and writes were a fifth of the LDS
  // traffic that binds these sizes.  64,000 cells, double and float: N=3 0.96 ->
  // 0.84 ms and 0.385 -> 0.342, N=2 0.543 -> 0.477 and 0.180 -> 0.147; N=4 loses
  // a wavefront per SIMD (1.97 -> 2.62 ms) and keeps it in LDS.
  static constexpr bool IN_REGISTERS = B <= 4 && V <= 5 && USE_FLUX && !USE_NCP;
  static constexpr int NQL = kFree <= 0 || IN_REGISTERS ? 0 : (kFree / kSliceBytes >= B ? B : (int)(kFree / kSliceBytes));
  static constexpr int NQR = B - NQL;
  // Rolled slices: the large sizes and the 9-variable PDE, whose unrolled
  // slices exhaust the registers, and the float form at N=4 and N=5, where the
  // rolled loop needs fewer registers (N=5: 110 instead of 166, one more
  // wavefront per SIMD) at the cost of uniform table loads per slice
  // (measured: N=4 -2%, N=5 -4% predictor time; at N=6 the rolled form was
  // 19% slower, so N=6 stays unrolled).
  // Double forms with fluxes up to N=5: rolled where the registers that unrolled
  // slices take beside the closed first iteration (kUnrolled, fitted to the
  // compiler's counts) are more than the wavefronts that LDS allows leave them,
  // and with a non-conservative product besides, where the unrolled slices spill.
  // 13,824 cells at N=4: flux and source 832 -> 597 us; 32,768 at N=3: flux and
  // product of five variables 4170 -> 1380 us; where they fit, the unrolled
  // slices are the faster ones (five variables at N=4, 13,824 cells: 574 us, rolled 599).
  // Not without LDS for every slice, which would take a workspace (144 KB: a
  // user's solver has none).
  static constexpr int kUnrolled = 44 + (9 * B - 5) * V + 5 * (D - V) + (USE_SOURCE ? 10 * V : 0);
  static constexpr long kLdsWaves = 160 * 1024 / (kOther + NQL * kSliceBytes) * (NT / kWave);  // per CU, of 4 SIMDs
  static constexpr bool ROLLED_DOUBLE =
      IS_FP64 && (NQR == 0 || LDSK < 144) && B >= 4 && B <= 6 &&
      (!USE_FLUX ? B == 6 && V == 5 : (USE_NCP ? V >= 2 : kUnrolled > (kLdsWaves >= 6 ? 252 : 508)));
  static constexpr bool ROLLED = (B >= 7 && (IS_FP64 || B >= 8)) || V >= 9 || (!IS_FP64 && (B == 5 || B == 6)) || ROLLED_DOUBLE;
  // 8+ waves per workgroup leave 256 registers per lane, no room for slices;
  // a rolled loop cannot index registers.
  static constexpr bool WSQ = NQR > 0 && (NT >= 8 * kWave || ROLLED);
  // unroll factor of the loop over time slices
  static constexpr int UNROLL_T = ROLLED ? 1 : B;
  static constexpr bool SPLIT = ROLLED && WSQ && NQL > 0;
  static constexpr bool LINES = USE_FLUX && (B == 4 || (B == 8 && LDSK == 144 && !USE_NCP));
  static constexpr size_t ws_bytes = WSQ ? (size_t)NQR * V * B3 * sizeof(T) : 0;
};

// ---------------------------------------------------------------------------
// Space-time predictor + time averaging + extrapolation + volume integral.
//
// Per Picard iteration and time slice t, three phases separated by barriers:
//  1. node owners evaluate the fluxes of their node and stage them in LDS as
//     sF[dir][var][node];
//  2. line owners (one task = one direction, variable and grid line) contract
//     the line with Kxi in place -- every staged value is read once, Kxi comes
//     in as scalar constants;
//  3. node owners form rhs(t) from the directional contributions and fold it
//     into the next iterate through iK1 (the reference's n order), so rhs is
//     never stored for all t.
// ---------------------------------------------------------------------------
// Waves per SIMD the register allocation must leave room for: the float
// flux-only form at N=5 and N=7 accumulates its time-averaged fluxes during
// the last iteration (3V more live registers) within the four (N=5) or three
// (N=7, 64 KB layout) waves that its LDS allows anyway; the library's elastic
// PDE, whose next iterate alone takes 9 B registers or twice that, keeps the
// wavefronts that its LDS allows (uncapped, N=4 in double takes 258 registers,
// one wavefront per SIMD; in float 168 and 189 instead of 160 and 169 at N=4, 5).
// By type, because the product of another PDE of these sizes may need more and
// would spill; elsewhere no constraint.
template <int B, class PDE, int TERMS, bool EXPORT, typename T>
__host__ __device__ constexpr int predictor_min_waves() {
  if (std::is_same_v<PDE, Elastic>) return sizeof(T) == sizeof(double) ? (B <= 5 && !EXPORT ? 2 : 1) : (B <= 5 ? 3 : 2);
  return (sizeof(T) == sizeof(float) && TERMS == kFlux) ? (B == 6 ? 4 : (B == 8 ? 3 : 1)) : 1;
}

template <int B, class PDE, int TERMS, bool EXPORT, typename T, int LDSK = 144>
__global__ __launch_bounds__(node_threads(B), (predictor_min_waves<B, PDE, TERMS, EXPORT, T>())) void predictor_kernel(
    PredictorArgs a) {
  constexpr int V = PDE::V, P = PDE::P, D = V + P;
  constexpr int N = B - 1;
  constexpr int B2 = B * B, B3 = B2 * B;
  constexpr int NT = node_threads(B);
  constexpr bool USE_FLUX = (TERMS & kFlux) != 0;
  constexpr bool USE_SOURCE = (TERMS & kSource) != 0;
  constexpr bool USE_NCP = (TERMS & kNCP) != 0;
  constexpr bool USE_SRC_NCP = USE_SOURCE || USE_NCP;
  constexpr bool IS_FP64 = sizeof(T) == sizeof(double);
  constexpr int MAX_ITER = 2 * B;  // spaceTimePredictorNonlinear.cpph:85
  using L = PredictorLayout<B, V, D, USE_NCP, T, LDSK, USE_FLUX, USE_SOURCE>;
  constexpr int NQL = L::NQL, NQR = L::NQR, UNROLL_T = L::UNROLL_T;
  constexpr bool IN_PLACE = L::IN_PLACE;
  static_assert(!IN_PLACE || (NQL == B && B * V >= D), "the iterate's rows hold the epilogue's D");
  constexpr bool SPLIT = L::SPLIT;
  constexpr bool WSQ = L::WSQ;
  __shared__ T sStage[IN_PLACE ? 1 : L::SF];
  __shared__ T sQi[NQL > 0 ? NQL * V * B3 : 1];  // lQi^k slices t < NQL, [t][var][node]
  __shared__ T sQ[USE_NCP && !IN_PLACE ? V * B3 : 1];
  T* const sF = IN_PLACE ? sQi : sStage;  // IN_PLACE: the epilogue's rows, when the iterate is done
  __shared__ T sDu[USE_NCP ? B2 : 1];  // dudx[l][n]
  __shared__ T sRed[2 * (NT / kWave)];

  T* const out_lduh = static_cast<T*>(a.lduh);
  T* const out_lQhbnd = static_cast<T*>(a.lQhbnd);
  T* const out_lFhbnd = static_cast<T*>(a.lFhbnd);

  // Lanes beyond the B^3 nodes compute node 0 again and write the same values,
  // and loops over outputs run whole rounds with the index clamped (surplus
  // lanes redo the last item), so control flow stays uniform; only the in-place
  // line contraction guards its stores.  (No instantiation may spill: the build
  // rejects any kernel with scratch memory.)
  const size_t cell = (size_t)blockIdx.x + a.cell0;
  const int tid = threadIdx.x;
  const bool active = tid < B3;
  const int node = active ? tid : 0;
  const int z = node / B2, y = (node / B) % B, x = node % B;
  // LINES: a direction's flux rows are kept by coordinate along the direction
  // and then by line, each coordinate's lines turned by four places (x) or B,
  // instead of by node: node owners and line owners both touch every bank once.
  // By node the lines along x and y meet in a quarter of the banks: B = 4 in
  // double 1.04 -> 0.96 ms for 64,000 cells, B = 8 in float 1.65 -> 1.53 ms for
  // 20,000, in double 4.90 -> 4.79 ms for 15,000.  (Not at B = 8 with the 64 KB
  // budget or the non-conservative product, which have no registers for it.)
  constexpr bool LINES = L::LINES;
  auto line_place = [](int d, int n, int line) __device__ { return n * B2 + ((line + (d == 0 ? 4 : B) * n) & (B2 - 1)); };
  const int at[3] = {LINES ? line_place(0, x, z * B + y) : node, LINES ? line_place(1, y, z * B + x) : node,
                     LINES ? line_place(2, z, y * B + x) : node};
  if (a.run_if && *a.run_if == 0) return;  // whole launch
  if (a.status && a.status[cell] >= a.status_limit) {  // whole workgroup
    if (a.iters && tid == 0) a.iters[cell] = 0;
    return;
  }

  if constexpr (USE_NCP) {
    for (int i = tid; i < B2; i += NT) sDu[i] = tc<T>(exa_dudx[N][i / B][i % B]);
  }

  const int patch = a.cell_patch ? a.cell_patch[cell] : 0;
  const double* dxp = a.cell_patch ? a.dx + (size_t)patch * 3 : a.dx + cell * a.dx_stride;
  const T invDx[3] = {T(1.0) / T(dxp[0]), T(1.0) / T(dxp[1]), T(1.0) / T(dxp[2])};
  const T dt = T(a.dt[patch]);
  // the node's weights, for the volume integral; IN_PLACE has no registers to
  // keep them through the iterations and takes them again afterwards
  T wx = tc<T>(exa_gl_weights[N][x]), wy = tc<T>(exa_gl_weights[N][y]), wz = tc<T>(exa_gl_weights[N][z]);
  T w3 = wz * wy * wx;

  T q0[D];
  {
    const double* luh = a.luh + cell * (size_t)(B3 * D) + node * D;
#pragma unroll
    for (int m = 0; m < D; ++m) q0[m] = T(luh[m]);
  }

  // Picard state: the current iterate lQi^k of this node (in LDS, each thread
  // touching only its own node's entries so no barriers are needed, or in
  // registers); the next iterate qn = lQi^{k+1} is accumulated in registers
  // slice by slice (iK1 applied in the reference's n order).
  T qi_reg[(NQR > 0 && !WSQ) ? NQR : 1][V];
  T* const ws = WSQ ? static_cast<T*>(a.ws) + (size_t)blockIdx.x * (NQR * V * B3) : nullptr;
  // Register slices are only used with compile-time t (unrolled loops).  Loads
  // and stores go through separate accessors with a uniform branch on t, so no
  // pointer that may address either LDS or global memory is ever formed.
  auto qi = [&](int t, int m) __device__ -> T {
    if (t < NQL)
      return sQi[(t * V + m) * B3 + node];
    else if (WSQ)
      return ws[((t - NQL) * V + m) * B3 + node];
    else
      return qi_reg[t - NQL][m];
  };
  auto qi_set = [&](int t, int m, T v) __device__ {
    if (t < NQL)
      sQi[(t * V + m) * B3 + node] = v;
    else if (WSQ)
      ws[((t - NQL) * V + m) * B3 + node] = v;
    else
      qi_reg[t - NQL][m] = v;
  };
#pragma unroll
  for (int t = 0; t < B; ++t)
#pragma unroll
    for (int m = 0; m < V; ++m)
      qi_set(t, m, q0[m]);
  T qn[B][V];
  int iters = MAX_ITER;
  // The first Picard iteration in closed form (see below); a call that exports
  // the temporaries evaluates every slice of it.
  constexpr bool FIRST_CLOSED = !EXPORT;
  constexpr bool FLOAT_FLUX_ONLY = !IS_FP64 && USE_FLUX && !USE_SRC_NCP;  // see ACC_FH
  // accumulating the averages needs 3V more registers: only at B = 5, 6 and
  // 8, where they fit the wavefronts per SIMD that LDS allows (B = 6 and 8
  // with the register cap of predictor_min_waves: 124 and 166 registers; the
  // epilogue's B flux evaluations go, 4% of the predictor at 81^3 N=5; B = 3
  // and 4 would drop a wavefront per SIMD, B = 7 spills under the cap; in
  // double at B = 4, beside the iterate in registers, one wavefront per SIMD
  // would be left: 0.89 -> 1.18 ms for 64,000 cells)
  constexpr bool ACC_FH = FLOAT_FLUX_ONLY && (B == 5 || B == 6 || B == 8);
  T fh[3][V];
  // Float form of a PDE without fluxes (source and/or NCP only: the elastic
  // PDE): the time-averaged source term likewise accumulates during the
  // iterations, from the S each slice's phase 3 evaluates anyway, so the
  // epilogue re-evaluates no slice (V more registers; the elastic kernels keep
  // their occupancy).
  constexpr bool ACC_SH = USE_SRC_NCP && !USE_FLUX;
  T sh[V];
  __syncthreads();

  const T gd[3] = {dt * invDx[0], dt * invDx[1], dt * invDx[2]};
  // Phase 2 tasks per direction: one (variable m, line) each, NTD of them in
  // RD rounds over the workgroup.
  constexpr int NTD = B2 * V;
  constexpr int RD = (NTD + NT - 1) / NT;

  // Line contractions by the line owners, in place: per direction d, one task =
  // one (variable, line).  A task reads its whole line before writing the
  // results back to the same positions, and no other task touches them.
  // Directions run one after the other with compile-time strides; the
  // operator's entries come in as constants.  VOLUME: sum_n Kxi[l][n] F(n) of
  // the volume integral; otherwise the derivative at every node (phase 2 of a
  // time slice, :152-236: the reference's Kxi with the weight w_l of the result
  // taken out, so that phase 3 needs one factor w_t dt / dx_d per slice).
  // Ends with a barrier.
  auto contract_lines = [&]<bool VOLUME>() __device__ __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RD; ++r) {
      if (tid + r * NT < NTD) {
        const int task = tid + r * NT;
        const int m = task / B2, line = task - (task / B2) * B2;
        const int la = line / B, lb = line - (line / B) * B;
        // line starts: x-lines (z,y) stride 1, y-lines (z,x) stride B,
        // z-lines (y,x) stride B^2
        const int off0 = m * B3 + line * B, off1 = m * B3 + la * B2 + lb, off2 = m * B3 + line;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int stride = d == 0 ? 1 : (d == 1 ? B : B2);
          const int o = d * V * B3 + (LINES ? 0 : (d == 0 ? off0 : (d == 1 ? off1 : off2)));
          T f[B], out[B];
#pragma unroll
          for (int n = 0; n < B; ++n) f[n] = sF[LINES ? o + m * B3 + line_place(d, n, line) : o + n * stride];
          contract_halves<B, VOLUME>(f, out);
#pragma unroll
          for (int l = 0; l < B; ++l) sF[LINES ? o + m * B3 + line_place(d, l, line) : o + l * stride] = out[l];
        }
      }
    }
    __syncthreads();
  };

#pragma unroll 1
  for (int iter = 0; iter < MAX_ITER; ++iter) {
    T q0i[V];
    // FLCoeff[t] luh is loop invariant; keeping B V copies of it live across
    // iterations costs more registers than recomputing it per slice.
    // IN_PLACE, whose next iterate takes most of the registers: luh is read
    // again (L1, L2) and its share sum_t iK1[l][t] FLCoeff[t] luh starts the
    // sums instead.
    if constexpr (IN_PLACE) {
      const double* luh = a.luh + cell * (size_t)(B3 * D) + node * D;
      asm volatile("" : "+v"(luh));
#pragma unroll
      for (int m = 0; m < V; ++m) q0i[m] = T(luh[m]);
    } else {
#pragma unroll
      for (int m = 0; m < V; ++m) {
        q0i[m] = q0[m];
        asm volatile("" : "+v"(q0i[m]));
      }
    }
    if constexpr (ACC_FH) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int m = 0; m < V; ++m) fh[d][m] = T(0);
    }
    if constexpr (ACC_SH) {
#pragma unroll
      for (int m = 0; m < V; ++m) sh[m] = T(0);
    }
    // Rolled (large sizes): table entries come from constant memory with a
    // uniform index; unrolled: they are immediates.
    // One time slice; with SPLIT (rolled loops over slices that live partly
    // in LDS and partly in the workspace) the LDS slices and the workspace
    // slices run in two loops, so that within each loop a slice's location is
    // known and every access is a plain LDS or global one (never a generic
    // pointer that may address either).
    auto picard_slice = [&](const int t) __device__ __attribute__((always_inline)) {
      const T wt = tc<T>(exa_gl_weights[N][t]);
      T Q[D];
#pragma unroll
      for (int m = 0; m < V; ++m) Q[m] = qi(t, m);
#pragma unroll
      for (int m = V; m < D; ++m) Q[m] = q0[m];
      // phase 1 (node owners): fluxes of this time slice -> sF[dir][var][node]
      if (USE_FLUX) {
        T F[3][V];
        PDE::flux(Q, F);
        if constexpr (ACC_FH) {
          // time average of the slice fluxes of this iterate (:367-396)
#pragma unroll
          for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < V; ++m) fh[d][m] += F[d][m] * wt;
        }
        {
#pragma unroll
          for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < V; ++m) sF[(d * V + m) * B3 + at[d]] = F[d][m];
          if (EXPORT) {
            double* lFi = a.lFi + cell * (size_t)(4 * B3 * B * V) + (((size_t)t * B3 + node) * 4) * V;
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
              for (int m = 0; m < V; ++m) lFi[d * V + m] = F[d][m];
          }
        }
      }
      if (USE_NCP && !IN_PLACE) {
#pragma unroll
        for (int m = 0; m < V; ++m) sQ[m * B3 + node] = Q[m];
      }
      if (!IN_PLACE) __syncthreads();

      if (USE_FLUX) contract_lines.template operator()<false>();

      // phase 3 (node owners): rhs / w^3 = FLCoeff[t] luh - sum_d w_t dt / dx_d
      // dF_d (+ S w_t dt) (:124-141, :238-276); lQi_new(l) += rhs / w^3
      // iK1[l][t] (:292-299, n = t)
      const T fl_t = tc<T>(exa_fl_coeff[N][t]);
      T ir[V];
      const T wg[3] = {wt * gd[0], wt * gd[1], wt * gd[2]};
#pragma unroll
      for (int m = 0; m < V; ++m) {
        ir[m] = IN_PLACE ? T(0) : fl_t * q0i[m];
        if (USE_FLUX) {
          ir[m] -= wg[0] * sF[(0 * V + m) * B3 + at[0]];
          ir[m] -= wg[1] * sF[(1 * V + m) * B3 + at[1]];
          ir[m] -= wg[2] * sF[(2 * V + m) * B3 + at[2]];
        }
      }
      if (USE_SRC_NCP) {
        T S[V];
        source_ncp<B, PDE, USE_SOURCE, USE_NCP, IN_PLACE>(Q, IN_PLACE ? sQi + t * (V * B3) : sQ, sDu, invDx, z, y, x, S);
        const T us = wt * dt;
#pragma unroll
        for (int m = 0; m < V; ++m) ir[m] += us * S[m];
        if constexpr (ACC_SH) {
          // time average of the slice sources of this iterate (:367-396)
#pragma unroll
          for (int m = 0; m < V; ++m) sh[m] += S[m] * wt;
        }
        if (EXPORT) {
          double* lFi = a.lFi + cell * (size_t)(4 * B3 * B * V) + (((size_t)t * B3 + node) * 4 + 3) * V;
#pragma unroll
          for (int m = 0; m < V; ++m) lFi[m] = S[m];
        }
      }
#pragma unroll
      for (int m = 0; m < V; ++m)
#pragma unroll
        for (int l = 0; l < B; ++l) qn[l][m] += ir[m] * tc<T>(exa_ik1[N][l][t]);
      if (USE_FLUX || (USE_NCP && !IN_PLACE)) __syncthreads();  // the next slice rewrites sF / sQ
      if (IN_PLACE) __builtin_amdgcn_sched_barrier(0);  // one slice's reads at a time in registers
    };
    if (FIRST_CLOSED && iter == 0) {
      // Every slice of the initial iterate equals luh, so one evaluation
      // R = sum_d dt / dx_d dF_d - dt S serves all slices:
      // lQi^1(l) = sum_t iK1[l][t] (FLCoeff[t] luh - w_t R) = a_l luh - b_l R,
      // a_l and b_l formed in double from the tables: one slice's evaluation
      // instead of B.  In double at N=5 (64,000 cells, 4 iterations), with the
      // halved contractions: 6.1 -> 5.1 ms; N=3 1.30 -> 1.07 ms, elastic N=4
      // 5.6 -> 4.0 ms.
      T Q[D], R[V];
#pragma unroll
      for (int m = 0; m < D; ++m) Q[m] = m < V ? q0i[m < V ? m : 0] : q0[m];
      double sw = 0.0;
#pragma unroll
      for (int t = 0; t < B; ++t) sw += exa_gl_weights[N][t];
      const T sumw = tc<T>(sw);
      if constexpr (USE_FLUX) {
        T F[3][V];
        PDE::flux(Q, F);
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int m = 0; m < V; ++m) {
            sF[(d * V + m) * B3 + at[d]] = F[d][m];
            if constexpr (ACC_FH) fh[d][m] = F[d][m] * sumw;
          }
      }
      if constexpr (USE_NCP && !IN_PLACE) {
#pragma unroll
        for (int m = 0; m < V; ++m) sQ[m * B3 + node] = Q[m];
      }
      if constexpr (!IN_PLACE) __syncthreads();
      if constexpr (USE_FLUX) contract_lines.template operator()<false>();
#pragma unroll
      for (int m = 0; m < V; ++m)
        R[m] = USE_FLUX ? gd[0] * sF[(0 * V + m) * B3 + at[0]] + gd[1] * sF[(1 * V + m) * B3 + at[1]] +
                              gd[2] * sF[(2 * V + m) * B3 + at[2]]
                        : T(0);
      if constexpr (USE_SRC_NCP) {
        T S[V];
        source_ncp<B, PDE, USE_SOURCE, USE_NCP, IN_PLACE>(Q, IN_PLACE ? sQi : sQ, sDu, invDx, z, y, x, S);
#pragma unroll
        for (int m = 0; m < V; ++m) {
          R[m] -= dt * S[m];
          if constexpr (ACC_SH) sh[m] = S[m] * sumw;
        }
      }
#pragma unroll
      for (int l = 0; l < B; ++l)
#pragma unroll
        for (int m = 0; m < V; ++m)
          qn[l][m] = tc<T>(exa_folded.a[N][l]) * q0i[m] - tc<T>(exa_folded.b[N][l]) * R[m];
      if constexpr (!IN_PLACE) __syncthreads();  // the next iteration rewrites sF / sQ
    } else {
#pragma unroll
      for (int l = 0; l < B; ++l)
#pragma unroll
        for (int m = 0; m < V; ++m) qn[l][m] = IN_PLACE ? tc<T>(exa_folded.a[N][l]) * q0i[m] : T(0);
      if constexpr (SPLIT) {
#pragma unroll 1
        for (int t = 0; t < NQL; ++t) picard_slice(t);
#pragma unroll 1
        for (int t = NQL; t < B; ++t) picard_slice(t);
      } else {
#pragma unroll UNROLL_T
        for (int t = 0; t < B; ++t) picard_slice(t);
      }
    }
    // squared residual (:303) and exit test (:314-318)
    T sq = T(0), qq = T(0);
#pragma unroll
    for (int l = 0; l < B; ++l)
#pragma unroll
      for (int m = 0; m < V; ++m) {
        const T dq = qn[l][m] - qi(l, m);
        sq += dq * dq;
        if (!IS_FP64) qq += qn[l][m] * qn[l][m];
        if (IN_PLACE && m + 1 == V) __builtin_amdgcn_sched_barrier(0);  // one slice's reads at a time in registers
      }
    if (!active) {
      sq = T(0);
      qq = T(0);
    }
    bool done;
    if (IS_FP64) {
      const T sq_res = block_sum<NT>(sq, sRed);
      done = sq_res < T(kPicardTol2);
    } else {
      const T sq_res = block_sum<NT>(sq, sRed);
      const T qq_sum = block_sum<NT>(qq, sRed + NT / kWave);
      done = sq_res < T(kPicardTol2) || sq_res < kPicardRelTol32 * kPicardRelTol32 * qq_sum;
    }
    if (done || iter + 1 == MAX_ITER) {
      iters = iter + 1;
      break;  // qi still holds lQi^k, the iterate the last fluxes were taken from
    }
    if constexpr (IN_PLACE) __syncthreads();  // every gradient of the iterate is taken
#pragma unroll
    for (int l = 0; l < B; ++l)
#pragma unroll
      for (int m = 0; m < V; ++m)
        qi_set(l, m, qn[l][m]);
    if constexpr (IN_PLACE) __syncthreads();
  }
  int own = node;
  if constexpr (IN_PLACE) {
    __syncthreads();  // the residual has read the iterate
    own = threadIdx.x;
    asm volatile("" : "+v"(own));
    own = own < B3 ? own : 0;
    wx = tc<T>(exa_gl_weights[N][own % B]);
    wy = tc<T>(exa_gl_weights[N][(own / B) % B]);
    wz = tc<T>(exa_gl_weights[N][own / B2]);
    w3 = wz * wy * wx;
  }

  // ---- epilogue: time average, extrapolation, volume integral ----
  const size_t cQb = cell * (size_t)(6 * B2 * D);
  const size_t cFb = cell * (size_t)(6 * B2 * V);
  {
    // lQhi = sum_t lQi(t) w_t of the final iterate lQi^{k+1} = qn (:397-404)
    T qh[D];
#pragma unroll
    for (int m = 0; m < D; ++m) {
      T acc = T(0);
#pragma unroll
      for (int t = 0; t < B; ++t) acc += (m < V ? qn[t][m < V ? m : 0] : q0[m]) * tc<T>(exa_gl_weights[N][t]);
      qh[m] = acc;
    }
    if (EXPORT) {
      double* lQi = a.lQi + cell * (size_t)(B3 * B * D) + (size_t)node * B * D;
#pragma unroll
      for (int t = 0; t < B; ++t)
#pragma unroll
        for (int m = 0; m < D; ++m) lQi[t * D + m] = (m < V) ? qn[t][m < V ? m : 0] : q0[m];
      double* lQhi = a.lQhi + cell * (size_t)(B3 * D) + (size_t)node * D;
#pragma unroll
      for (int m = 0; m < D; ++m) lQhi[m] = qh[m];
    }
#pragma unroll
    for (int m = 0; m < D; ++m) sF[m * B3 + node] = qh[m];
  }
  __syncthreads();
  // Face extrapolation (lQhbnd / lFhbnd, :434-527) as line tasks: per
  // direction d, one task = (face node (la, lb), datum k), k fastest so that
  // the stores of a wavefront are contiguous; a task reads its normal line
  // once and forms both faces of the direction (FL and FR coefficients, as
  // immediates).  Source values: sF[k][node] for every direction, or with
  // PER_DIR the direction's own block sF[d][k][node].
  auto extrapolate = [&]<int NK, bool PER_DIR>(T* out, size_t coff) __device__ {
    constexpr int NTK = B2 * NK;
#pragma unroll
    for (int r = 0; r < (NTK + NT - 1) / NT; ++r) {
      const int task = tid + r * NT;
      if (task < NTK) {
        const int k = task % NK, line = task / NK;
        const int la = line / B, lb = line - (line / B) * B;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int stride = d == 0 ? 1 : (d == 1 ? B : B2);
          const int o = (PER_DIR ? d * V + k : k) * B3 + (d == 0 ? line * B : (d == 1 ? la * B2 + lb : line));
          T accL = T(0), accR = T(0);
#pragma unroll
          for (int l = 0; l < B; ++l) {
            const T v = sF[LINES && PER_DIR ? (d * V + k) * B3 + line_place(d, l, line) : o + l * stride];
            accL += v * tc<T>(exa_fl_coeff[N][l]);
            accR += v * tc<T>(exa_fr_coeff[N][l]);
          }
          out[coff + (size_t)(2 * d) * NTK + task] = accL;
          out[coff + (size_t)(2 * d + 1) * NTK + task] = accR;
        }
      }
    }
  };
  extrapolate.template operator()<D, false>(out_lQhbnd, cQb);
  __syncthreads();

  // Time-averaged fluxes of the last flux evaluation, i.e. of lQi^k = qi (the
  // reference computes lFi before the final lQi update, :96-122 vs :306):
  // lFhi = sum_t w_t F(lQi^k(t)), lShi likewise (:367-396).
#pragma unroll
  for (int m = 0; m < V; ++m) {
    if constexpr (!ACC_FH) {
      fh[0][m] = T(0);
      fh[1][m] = T(0);
      fh[2][m] = T(0);
    }
    if constexpr (!ACC_SH) sh[m] = T(0);
  }
  auto average_slice = [&](const int t) __device__ __attribute__((always_inline)) {
    T Q[D];
#pragma unroll
    for (int m = 0; m < V; ++m) Q[m] = qi(t, m);
#pragma unroll
    for (int m = V; m < D; ++m) Q[m] = q0[m];
    const T wt = tc<T>(exa_gl_weights[N][t]);
    if (USE_FLUX) {
      T F[3][V];
      PDE::flux(Q, F);
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int m = 0; m < V; ++m) fh[d][m] += F[d][m] * wt;
    }
    if (USE_SRC_NCP) {
      if (USE_NCP) {
#pragma unroll
        for (int m = 0; m < V; ++m) sQ[m * B3 + node] = Q[m];
      }
      if (USE_NCP) __syncthreads();
      T S[V];
      source_ncp<B, PDE, USE_SOURCE, USE_NCP, IN_PLACE>(Q, sQ, sDu, invDx, z, y, x, S);
#pragma unroll
      for (int m = 0; m < V; ++m) sh[m] += S[m] * wt;
      if (USE_NCP) __syncthreads();
    }
  };
  if constexpr (ACC_FH || ACC_SH) {
    // fh (flux-only) or sh (no flux) holds the time average of the last
    // iteration's fluxes or sources already
  } else if constexpr (SPLIT) {
#pragma unroll 1
    for (int t = 0; t < NQL; ++t) average_slice(t);
#pragma unroll 1
    for (int t = NQL; t < B; ++t) average_slice(t);
  } else {
#pragma unroll UNROLL_T
    for (int t = 0; t < B; ++t) average_slice(t);
  }
  if (EXPORT) {
    // lFhi blocks: x (z,y,x), y (z,x,y), z (y,x,z), src (z,y,x)  (:375-393)
    double* lFhi = a.lFhi + cell * (size_t)(4 * B3 * V);
#pragma unroll
    for (int m = 0; m < V; ++m) {
      lFhi[0 * B3 * V + ((z * B + y) * B + x) * V + m] = fh[0][m];
      lFhi[1 * B3 * V + ((z * B + x) * B + y) * V + m] = fh[1][m];
      lFhi[2 * B3 * V + ((y * B + x) * B + z) * V + m] = fh[2][m];
      lFhi[3 * B3 * V + ((z * B + y) * B + x) * V + m] = sh[m];
    }
  }
  if constexpr (USE_FLUX) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int m = 0; m < V; ++m) sF[(d * V + m) * B3 + at[d]] = fh[d][m];
    __syncthreads();
  }
  // lFhbnd from lFhi_{x,y,z} (:434-527)
  if (USE_FLUX) {
    extrapolate.template operator()<V, true>(out_lFhbnd, cFb);
  } else if (!a.skip_zero_fluxes) {
#pragma unroll 1
    for (int round = 0; round < (6 * B2 * V + NT - 1) / NT; ++round)
      out_lFhbnd[cFb + min(tid + round * NT, 6 * B2 * V - 1)] = T(0);
  }
  // volume integral (volumeIntegralNonlinear.cpph:136-225), time-averaged form
  if (out_lduh) {
    T acc[V];
#pragma unroll
    for (int m = 0; m < V; ++m) acc[m] = T(0);
    if constexpr (USE_FLUX) {
      // the directional contractions sum_n Kxi[l][n] lFhi_d(n) as line tasks in
      // place, then each node sums its three directions with their weights
      __syncthreads();  // the extrapolation has read sF
      contract_lines.template operator()<true>();
      const T us[3] = {wz * wy * invDx[0], wz * wx * invDx[1], wy * wx * invDx[2]};
#pragma unroll
      for (int m = 0; m < V; ++m)
        acc[m] = us[0] * sF[(0 * V + m) * B3 + at[0]] + us[1] * sF[(1 * V + m) * B3 + at[1]] +
                 us[2] * sF[(2 * V + m) * B3 + at[2]];
    }
    if (USE_SRC_NCP) {
#pragma unroll
      for (int m = 0; m < V; ++m) acc[m] += w3 * sh[m];
    }
    T* lduh = out_lduh + cell * (size_t)(B3 * V) + own * V;
#pragma unroll
    for (int m = 0; m < V; ++m) lduh[m] = acc[m];
  }
  if (a.iters && tid == 0) a.iters[cell] = iters;
}

}  // namespace exa
