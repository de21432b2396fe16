// predictor_wave.hpp -- the space-time predictor with one wavefront per time
// slice (same mathematics and outputs as predictor_kernel in predictor.hpp; no
// exports of the temporaries).
//
// Reference semantics (K = ExaHyPE/kernels/aderdg/generic/c/3d):
//   K/spaceTimePredictorNonlinear.cpph:42-528,661-717
//   + K/volumeIntegralNonlinear.cpph:136-225 (fused epilogue)
#pragma once

#include "predictor.hpp"

namespace exa {

// One workgroup per cell, one wavefront per time slice: wavefront t holds the
// iterate lQi^k(t) of all B^3 nodes in registers (nodes lane, lane + 64, ...),
// stages the fluxes of one direction in its own LDS region and contracts them
// line by line.  All of a slice's exchange between node and line owners stays
// inside the wavefront, whose LDS operations complete in order: no workgroup
// barrier.  The slices meet once per Picard iteration, when iK1 mixes them
// (one task per node and variable, in place in the regions).
//
// N=6, whose B^2 V = 245 lines fill a wavefront's four rounds to 96%, against
// predictor_kernel, whose 343 nodes and 735 lines leave a third of its six
// wavefronts idle (flux-only Euler, 30,000 cells; 6,669; 729):
//   float:  2.29 -> 1.67 ms; 0.547 -> 0.408; 0.076 -> 0.066  (LDS 69 KB either way, 14 wavefronts per CU instead of 12)
//   double: 5.89 -> 5.50 ms; 1.39 -> 1.28;   0.167 -> 0.159  (LDS 137 KB, one workgroup per CU; no workspace)
// LDS bound.  The other sizes keep predictor_kernel: their lines or nodes fill
// a wavefront badly (N=4 float 0.87 -> 1.09 ms, N=5 1.73 -> 2.54 ms for 64,000
// cells, N=7 1.66 -> 1.71 ms for 20,000; N=3 double 0.527 -> 0.60 ms for 30,000).
template <int B, class PDE>
struct WaveLayout {
  static_assert(PDE::P == 0, "the iterate's registers hold variables only");
  static constexpr int V = PDE::V;
  static constexpr int B3 = B * B * B;
  static constexpr int NT = B * kWave;
  static constexpr int C = (B3 + kWave - 1) / kWave;  // nodes per lane
  static constexpr int ROWS = B * V;                  // V rows per slice
  static constexpr int EROWS = 3 * V;                 // sums over the slices (epilogue, first iteration)
};

template <int B, class PDE, typename T>
__global__ __launch_bounds__(B* kWave, (sizeof(T) == sizeof(float) ? 3 : 2)) void predictor_wave_kernel(PredictorArgs a) {
  using L = WaveLayout<B, PDE>;
  constexpr int V = L::V;
  constexpr int N = B - 1, B2 = B * B, B3 = L::B3, NT = L::NT, C = L::C;
  constexpr bool IS_FP64 = sizeof(T) == sizeof(double);
  constexpr int MAX_ITER = 2 * B;  // spaceTimePredictorNonlinear.cpph:85
  __shared__ T sS[L::ROWS * B3];   // [slice][variable][node]
  __shared__ T sE[L::EROWS * B3];
  __shared__ T sRed[2][2 * B];

  const size_t cell = (size_t)blockIdx.x + a.cell0;
  if (a.run_if && *a.run_if == 0) return;              // whole launch
  if (a.status && a.status[cell] >= a.status_limit) {  // whole workgroup
    if (a.iters && threadIdx.x == 0) a.iters[cell] = 0;
    return;
  }
  int tid = threadIdx.x;
  const int t = __builtin_amdgcn_readfirstlane(tid / kWave);  // the wavefront's slice
  const int lane = tid & (kWave - 1);
  const int patch = a.cell_patch ? a.cell_patch[cell] : 0;
  const double* dxp = a.cell_patch ? a.dx + (size_t)patch * 3 : a.dx + cell * a.dx_stride;
  const T dt = T(a.dt[patch]);
  T gd[3];  // dt / dx_d
#pragma unroll
  for (int d = 0; d < 3; ++d) gd[d] = wave_uniform(dt * (T(1.0) / T(dxp[d])));
  const double* const luh = a.luh + cell * (size_t)(B3 * V);
  T* const sG = sS + t * (V * B3);
  // node c of this lane; surplus nodes repeat the last one and store nothing
  auto node_of = [&](int c) __device__ { return (c + 1) * kWave <= B3 || lane + c * kWave < B3 ? lane + c * kWave : B3 - 1; };
  auto owns = [&](int c) __device__ { return (c + 1) * kWave <= B3 || lane + c * kWave < B3; };

  // In-place contraction of one line along DIR with compile-time operators.
  auto contract_line = [&]<int DIR, bool VOLUME>(T* p) __device__ __attribute__((always_inline)) {
    constexpr int stride = DIR == 0 ? 1 : (DIR == 1 ? B : B2);
    T f[B];
#pragma unroll
    for (int n = 0; n < B; ++n) f[n] = p[n * stride];
    T out[B];
    contract_halves<B, VOLUME>(f, out);
#pragma unroll
    for (int l = 0; l < B; ++l) p[l * stride] = out[l];
  };
  // V rows, one task = one (variable, line): a task's first entry is B task
  // for x lines, m B^3 + la B^2 + lb for y lines (la, lb) and m B^3 + line for
  // z lines.
  constexpr int NTD = B2 * V;
  auto line_y = [](int task) __device__ {
    const int m = task / B2, line = task - m * B2;
    return m * B3 + line / B * B2 + line % B;
  };
  auto line_z = [](int task) __device__ { return task + task / B2 * (B3 - B2); };
  // by the whole workgroup
  auto contract = [&]<int DIR, bool VOLUME>(T* base) __device__ __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < (NTD + NT - 1) / NT; ++r) {
      const int task = tid + r * NT;
      if ((r + 1) * NT <= NTD || task < NTD)
        contract_line.template operator()<DIR, VOLUME>(base + (DIR == 0 ? task * B : (DIR == 1 ? line_y(task) : line_z(task))));
    }
  };
  // by one wavefront on its own slice's rows: the y and z lines' first entries
  // are kept packed, one register per round
  constexpr int RW = (NTD + kWave - 1) / kWave;
  static_assert(V * B3 < 65536, "line offsets are packed in 16 bits");
  unsigned lines[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int task = lane + r * kWave;
    lines[r] = (unsigned)line_y(task) | (unsigned)line_z(task) << 16;
  }
  auto contract_slice = [&]<int DIR>() __device__ __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int task = lane + r * kWave;
      unsigned pk = lines[r];
      asm volatile("" : "+v"(pk));  // unpacked where it is used
      if ((r + 1) * kWave <= NTD || task < NTD)
        contract_line.template operator()<DIR, false>(sG + (DIR == 0 ? task * B : (DIR == 1 ? (int)(pk & 0xffff) : (int)(pk >> 16))));
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  T qi[C][V];           // lQi^k(t)
  int iters = MAX_ITER;

  // First iteration: every slice of the initial iterate equals luh, so one
  // evaluation R = dt sum_d dF_d/dx_d of luh serves all slices:
  // lQi^1(l) = a_l luh - b_l R.
  for (int n = tid; n < B3; n += NT) {
    T Q[V], F[3][V];
#pragma unroll
    for (int m = 0; m < V; ++m) Q[m] = T(luh[(size_t)n * V + m]);
    PDE::flux(Q, F);
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int m = 0; m < V; ++m) sE[(d * V + m) * B3 + n] = F[d][m];
  }
  __syncthreads();
  contract.template operator()<0, false>(sE);
  contract.template operator()<1, false>(sE + V * B3);
  contract.template operator()<2, false>(sE + 2 * V * B3);
  __syncthreads();
  T qn[C][V];  // lQi^{k+1}(t)
  {
    const T al = tc<T>(exa_folded.a[N][t]), bl = tc<T>(exa_folded.b[N][t]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int n = node_of(c);
#pragma unroll
      for (int m = 0; m < V; ++m) {
        const T q = T(luh[(size_t)n * V + m]);
        const T R = gd[0] * sE[m * B3 + n] + gd[1] * sE[(V + m) * B3 + n] + gd[2] * sE[(2 * V + m) * B3 + n];
        qi[c][m] = q;
        qn[c][m] = al * q - bl * R;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

#pragma unroll 1
  for (int iter = 0;; ++iter) {
    // squared residual (:303) and exit test (:314-318)
    T sq = T(0), qq = T(0);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      T s = T(0), u = T(0);
#pragma unroll
      for (int m = 0; m < V; ++m) {
        const T dq = qn[c][m] - qi[c][m];
        s += dq * dq;
        if (!IS_FP64) u += qn[c][m] * qn[c][m];
      }
      sq += owns(c) ? s : T(0);
      if (!IS_FP64) qq += owns(c) ? u : T(0);
    }
    sq = wave_sum(sq);
    if (!IS_FP64) qq = wave_sum(qq);
    T* const red = sRed[iter & 1];
    red[t] = sq;
    if (!IS_FP64) red[B + t] = qq;
    __syncthreads();
    T sq_res = red[0], qq_sum = IS_FP64 ? T(0) : red[B];
#pragma unroll
    for (int w = 1; w < B; ++w) {
      sq_res += red[w];
      if (!IS_FP64) qq_sum += red[B + w];
    }
    bool done = sq_res < T(kPicardTol2);
    if constexpr (!IS_FP64) done = done || sq_res < kPicardRelTol32 * kPicardRelTol32 * qq_sum;
    if (done || iter + 1 == MAX_ITER) {
      iters = iter + 1;
      break;  // qi still holds lQi^k, the iterate the last fluxes were taken from
    }
    if (iter == 0 && t == 0) {  // luh, for the mixing of the slices below
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (owns(c)) {
#pragma unroll
          for (int m = 0; m < V; ++m) sE[m * B3 + node_of(c)] = qi[c][m];
        }
    }
    T rr[C][V];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int m = 0; m < V; ++m) qi[c][m] = qn[c][m];
    // dt sum_d dF_d/dx_d of the slice, one direction at a time
    auto direction = [&]<int DIR>() __device__ __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        T Q[V], F[3][V];
#pragma unroll
        for (int m = 0; m < V; ++m) Q[m] = qi[c][m];
#pragma unroll
        for (int m = 0; m < V; ++m) asm volatile("" : "+v"(Q[m]));
        PDE::flux(Q, F);
        if (owns(c)) {
#pragma unroll
          for (int m = 0; m < V; ++m) sG[m * B3 + node_of(c)] = F[DIR][m];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      wave_lds_sync();
      contract_slice.template operator()<DIR>();
      wave_lds_sync();
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int m = 0; m < V; ++m) {
          const T v = gd[DIR] * sG[m * B3 + node_of(c)];
          rr[c][m] = DIR == 0 ? v : rr[c][m] + v;
          if (m + 1 == V) __builtin_amdgcn_sched_barrier(0);
        }
      wave_lds_sync();
    };
    direction.template operator()<0>();
    direction.template operator()<1>();
    direction.template operator()<2>();
    {
      const T wt = tc<T>(exa_gl_weights[N][t]);
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (owns(c)) {
#pragma unroll
          for (int m = 0; m < V; ++m) sG[m * B3 + node_of(c)] = wt * rr[c][m];
        }
    }
    __syncthreads();
    // lQi^{k+1}(l) = a_l luh - sum_t iK1[l][t] w_t R(t) of every node and
    // variable, in place
#pragma unroll
    for (int r = 0; r < (V * B3 + NT - 1) / NT; ++r) {
      const int e = tid + r * NT;
      if ((r + 1) * NT <= V * B3 || e < V * B3) {
        T v[B];
#pragma unroll
        for (int s = 0; s < B; ++s) v[s] = sS[s * (V * B3) + e];
        const T q = sE[e];
#pragma unroll
        for (int l = 0; l < B; ++l) {
          T acc = tc<T>(exa_folded.a[N][l]) * q;
#pragma unroll
          for (int s = 0; s < B; ++s) acc -= v[s] * tc<T>(exa_ik1[N][l][s]);
          sS[l * (V * B3) + e] = acc;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int m = 0; m < V; ++m) qn[c][m] = sG[m * B3 + node_of(c)];
    }
  }

  // ---- epilogue: time average, extrapolation, volume integral ----
  asm volatile("" : "+v"(tid));  // its index arithmetic stays here: nothing of it is held across the iterations
  const size_t cb = cell * (size_t)(6 * B2 * V);
  T* const out_lduh = static_cast<T*>(a.lduh);
  T* const out_lQhbnd = static_cast<T*>(a.lQhbnd);
  T* const out_lFhbnd = static_cast<T*>(a.lFhbnd);
  const T wt = tc<T>(exa_gl_weights[N][t]);
  // the slices' V rows added up into V rows of sE
  auto add_slices = [&](T* to) __device__ __attribute__((always_inline)) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < (V * B3 + NT - 1) / NT; ++r) {
      const int e = tid + r * NT;
      if ((r + 1) * NT <= V * B3 || e < V * B3) {
        T v = sS[e];
#pragma unroll
        for (int s = 1; s < B; ++s) v += sS[s * (V * B3) + e];
        to[e] = v;
      }
    }
    __syncthreads();
  };
  // Face extrapolation (lQhbnd / lFhbnd, :434-527) of NK rows at base along
  // DIR: one task = (face node, datum k), k fastest; both faces of DIR.
  auto extrapolate = [&]<int DIR, int NK>(const T* base, T* out, size_t coff) __device__ __attribute__((always_inline)) {
    constexpr int NTK = B2 * NK;
    constexpr int stride = DIR == 0 ? 1 : (DIR == 1 ? B : B2);
#pragma unroll
    for (int r = 0; r < (NTK + NT - 1) / NT; ++r) {
      const int task = tid + r * NT;
      if ((r + 1) * NT <= NTK || task < NTK) {
        const int k = task % NK, line = task / NK;
        const int la = line / B, lb = line - (line / B) * B;
        const T* const p = base + k * B3 + (DIR == 0 ? line * B : (DIR == 1 ? la * B2 + lb : line));
        T accL = T(0), accR = T(0);
#pragma unroll
        for (int l = 0; l < B; ++l) {
          const T v = p[l * stride];
          accL += v * tc<T>(exa_fl_coeff[N][l]);
          accR += v * tc<T>(exa_fr_coeff[N][l]);
        }
        out[coff + (size_t)(2 * DIR) * NTK + task] = accL;
        out[coff + (size_t)(2 * DIR + 1) * NTK + task] = accR;
      }
    }
  };
  // lQhi = sum_t lQi(t) w_t of the final iterate lQi^{k+1} = qn (:397-404)
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (owns(c)) {
#pragma unroll
      for (int m = 0; m < V; ++m) sG[m * B3 + node_of(c)] = wt * qn[c][m];
    }
  add_slices(sE);
  extrapolate.template operator()<0, V>(sE, out_lQhbnd, cb);
  extrapolate.template operator()<1, V>(sE, out_lQhbnd, cb);
  extrapolate.template operator()<2, V>(sE, out_lQhbnd, cb);
  // Time-averaged fluxes of the last evaluation, i.e. of lQi^k = qi (:96-122
  // vs :306, :367-396): lFhi_d = sum_t w_t F_d(lQi^k(t)).
  auto average = [&]<int DIR>() __device__ __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      T Q[V], F[3][V];
#pragma unroll
      for (int m = 0; m < V; ++m) Q[m] = qi[c][m];
      PDE::flux(Q, F);
      if (owns(c)) {
#pragma unroll
        for (int m = 0; m < V; ++m) sG[m * B3 + node_of(c)] = wt * F[DIR][m];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    add_slices(sE + DIR * V * B3);
  };
  average.template operator()<0>();
  average.template operator()<1>();
  average.template operator()<2>();
  extrapolate.template operator()<0, V>(sE, out_lFhbnd, cb);
  extrapolate.template operator()<1, V>(sE + V * B3, out_lFhbnd, cb);
  extrapolate.template operator()<2, V>(sE + 2 * V * B3, out_lFhbnd, cb);
  if (a.iters && tid == 0) a.iters[cell] = iters;
  if (!out_lduh) return;
  // volume integral (volumeIntegralNonlinear.cpph:136-225): the directional
  // contractions sum_n Kxi[l][n] lFhi_d(n) in place, then per node
  __syncthreads();
  contract.template operator()<0, true>(sE);
  contract.template operator()<1, true>(sE + V * B3);
  contract.template operator()<2, true>(sE + 2 * V * B3);
  __syncthreads();
  for (int n = tid; n < B3; n += NT) {
    const T wx = tc<T>(exa_gl_weights[N][n % B]), wy = tc<T>(exa_gl_weights[N][(n / B) % B]),
            wz = tc<T>(exa_gl_weights[N][n / B2]);
    const T us[3] = {wz * wy * (T(1.0) / T(dxp[0])), wz * wx * (T(1.0) / T(dxp[1])), wy * wx * (T(1.0) / T(dxp[2]))};
    T* const lduh = out_lduh + cell * (size_t)(B3 * V) + (size_t)n * V;
#pragma unroll
    for (int m = 0; m < V; ++m)
      lduh[m] = us[0] * sE[m * B3 + n] + us[1] * sE[(V + m) * B3 + n] + us[2] * sE[(2 * V + m) * B3 + n];
  }
}

}  // namespace exa
