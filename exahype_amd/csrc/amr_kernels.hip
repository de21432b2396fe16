// amr_kernels.hip -- ADER-DG AMR transfer operators on gfx950, FP64: face and
// volume unknowns prolongation (coarse -> fine) and restriction (fine ->
// coarse, accumulated), over one or more levels.
//
// Reference semantics (K = ExaHyPE/kernels/aderdg/generic/c/3d):
//   K/amrRoutines.cpph:23-143   faceUnknownsProlongation (+ single level)
//   K/amrRoutines.cpph:145-260  faceUnknownsRestriction
//   K/amrRoutines.cpph:285-384  volumeUnknownsProlongation
//   K/amrRoutines.cpph:386-491  volumeUnknownsRestriction
//
// One wavefront per transfer.  A level is the tensor product of three (two for
// faces) 1-D operators; it runs as NDIM passes over the block in LDS, each
// contracting every grid line of every value in place (one lane per line, the
// operator of the pass in scalar registers), instead of the reference's
// B^NDIM-term sum per node (the same linear map; the sums round in another
// order).  The 1-D operator of direction d at a level is fineGridProjector1d[j_d]
// (prolongation: out_m = sum_n in_n P[j][n][m]) or w_n P[j][m][n] / (3 w_m)
// (restriction), j_d the subinterval digit of that level.  Restriction adds the
// restricted blocks of a destination's transfers, in list order, to the
// destination block.
//
// Bound: HBM (a prolongation writes every fine block once).  With one workgroup
// per transfer, one thread per node and a B-term sum per node and pass, the
// wavefronts waited for LDS and for the transfer's own chain of loads (item,
// claim, block) behind workgroup barriers; a wavefront per transfer has no
// barrier in a prolongation, reads each value once per pass, and keeps 16 or
// more transfers per CU in flight.  183,141 transfers of 6^3 x 5 values: the
// prolongation 1.11 -> 0.55 ms (2.9 TB/s), the restriction 1.40 -> 0.68 ms (2.4
// TB/s; its next block is loaded while the last is restricted).
#include "amr.hpp"
#include "exa_device.hpp"

namespace exa {

namespace amr_tables {
#define EXA_TABLE static constexpr
#include "dg_tables.inc"
#undef EXA_TABLE
constexpr int kMaxB = 6;
struct Operators {  // [order][restriction][subinterval][n][m]
  double m[kMaxB][2][3][kMaxB][kMaxB];
};
constexpr Operators operators() {
  Operators o{};
  for (int N = 0; N < kMaxB; ++N)
    for (int j = 0; j < 3; ++j)
      for (int n = 0; n <= N; ++n)
        for (int m = 0; m <= N; ++m) {
          o.m[N][0][j][n][m] = exa_fine_proj[N][j][n][m];
          o.m[N][1][j][n][m] = exa_gl_weights[N][n] * exa_fine_proj[N][j][m][n] / exa_gl_weights[N][m] / 3.0;
        }
  return o;
}
}  // namespace amr_tables
static __constant__ const amr_tables::Operators amr_operators = amr_tables::operators();

// A workgroup barrier for LDS data only: global loads in flight stay in flight.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The workgroup's index in a list dealt so that each of the 8 XCDs (workgroups
// go to them in turn) takes one contiguous run: the children of a coarse block
// (adjacent in the list) then read it through the same L2.  A bijection on
// [0, gridDim).
__device__ inline long xcd_run_index() {
  const long g = gridDim.x, b = blockIdx.x, q = g / 8, r = g % 8, xcd = b % 8, idx = b / 8;
  return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

// Is the item's every index in range?
template <int NDIM>
__device__ inline bool item_ok(const AmrArgs& a, const int* item) {
  bool ok = item[0] >= 0 && item[0] < a.dst_blocks && item[1] >= 0 && item[1] < a.src_blocks;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) ok = ok && item[2 + d] >= 0 && item[2 + d] < a.ndigits;
  return ok;
}

// Takes the destination block's bit; true: this caller is the first.
__device__ inline bool claim(const AmrArgs& a, long db) {
  const unsigned bit = 1u << (db & 31);
  return (atomicOr(a.claimed + (db >> 5), bit) & bit) == 0;
}

// One wavefront applies the item's operators to the block s ([node][value], LDS)
// in place.  nv: values per node.
template <int B, int NDIM, bool RESTRICT>
__device__ inline void transfer(const AmrArgs& a, const int* item, double* s, int nv, int lane) {
  constexpr int N = B - 1;
  const int ntasks = (NDIM == 3 ? B * B : B) * nv;
  int sig = 1;  // prolongation decodes from the top digit, restriction from the bottom
  if (!RESTRICT)
    for (int l = 1; l < a.level_delta; ++l) sig *= 3;
  for (int l = 0; l < a.level_delta; ++l) {
#pragma unroll
    for (int d = 0; d < NDIM; ++d) {
      const int stride = d == 0 ? 1 : (d == 1 ? B : B * B);
      const double(*M)[amr_tables::kMaxB] = amr_operators.m[N][RESTRICT ? 1 : 0][(item[2 + d] / sig) % 3];
      wave_lds_sync();  // the block, or the previous pass, complete
      for (int task = lane; task < ntasks; task += kWave) {
        const int line = task / nv, v = task - line * nv;  // value fastest: neighbouring lanes, neighbouring entries
        const int node = d == 0 ? line * B : (d == 1 ? line / B * (B * B) + line % B : line);
        double* const p = s + node * nv + v;
        double f[B];
#pragma unroll
        for (int n = 0; n < B; ++n) f[n] = p[n * stride * nv];
#pragma unroll
        for (int m = 0; m < B; ++m) {
          double acc = 0.0;
#pragma unroll
          for (int n = 0; n < B; ++n) acc += f[n] * M[n][m];
          p[m * stride * nv] = acc;
        }
      }
    }
    sig = RESTRICT ? sig * 3 : sig / 3;
  }
  wave_lds_sync();
}

// NV: values per node at compile time (the block's loads then go out together),
// 0: a.nv.
template <int B, int NDIM, int NV>
__global__ __launch_bounds__(256) void amr_prolong_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  extern __shared__ double smem[];
  const int nv = NV ? NV : a.nv, n = NN * nv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const long k = xcd_run_index() * (blockDim.x / kWave) + wave;
  if (k >= a.nitems) return;
  const int* const item = a.items + 5 * k;
  if (!item_ok<NDIM>(a, item)) {  // the item is skipped and reported
    if (lane == 0) atomicOr(a.error, 1);
    return;
  }
  // claim the destination block: a second transfer naming it writes nothing
  int first = 0;
  if (lane == 0) first = claim(a, item[0]);
  double* const s = smem + (size_t)wave * n;
  const double* const src = a.src + (size_t)item[1] * a.src_block;
#pragma unroll(NV ? (NN * NV + kWave - 1) / kWave : 1)
  for (int e = lane; e < n; e += kWave) s[e] = src[e];
  transfer<B, NDIM, false>(a, item, s, nv, lane);
  if (__builtin_amdgcn_readfirstlane(first) == 0) {
    if (lane == 0) atomicOr(a.error, 1);
    return;
  }
  double* const dst = a.dst + (size_t)item[0] * a.dst_block;
#pragma unroll(NV ? (NN * NV + kWave - 1) / kWave : 1)
  for (int e = lane; e < n; e += kWave) dst[e] = s[e];
}

// One workgroup per destination: its wavefronts restrict as many transfers at
// a time, whose results all threads then add in list order (as successive
// single calls add).
template <int B, int NDIM, int NV>
__global__ __launch_bounds__(256) void amr_restrict_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  constexpr int R = NV ? (NN * NV + kWave - 1) / kWave : 1;  // a block's entries per lane
  extern __shared__ double smem[];
  __shared__ int taken;
  const int nv = NV ? NV : a.nv, n = NN * nv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int W = blockDim.x / kWave;
  const long k = xcd_run_index();
  const long i0 = a.ptr[k], i1 = a.ptr[k + 1];
  if (i0 < 0 || i1 < i0 || i1 > a.nitems) {  // a malformed range: nothing is read
    if (threadIdx.x == 0) atomicOr(a.error, 1);
    return;
  }
  // the destination of the range: that of its first item in range
  long db = -1;
  for (long it = i0; it < i1 && db < 0; ++it)
    if (item_ok<NDIM>(a, a.items + 5 * it)) db = a.items[5 * it];
  if (db < 0) {
    if (i1 > i0 && threadIdx.x == 0) atomicOr(a.error, 1);
    return;
  }
  auto usable = [&](long it) __device__ {
    return it < i1 && item_ok<NDIM>(a, a.items + 5 * it) && a.items[5 * it] == db;
  };
  // claim the destination block: a second workgroup naming it writes nothing
  if (threadIdx.x == 0) taken = !claim(a, db);
  double* const s = smem + (size_t)wave * n;
  // The destination block: a thread's own entries, in registers (NV: always
  // four wavefronts) or in LDS behind the transfers' blocks.
  constexpr int RA = NV ? (NN * NV + 255) / 256 : 1;
  double acc[RA];
  double* const sAcc = smem + (size_t)W * n;
  double* const dst = a.dst + (size_t)db * a.dst_block;
  if constexpr (NV != 0) {
#pragma unroll
    for (int r = 0; r < RA; ++r) acc[r] = (int)threadIdx.x + r * 256 < n ? dst[threadIdx.x + r * 256] : 0.0;
  } else {
    for (int e = threadIdx.x; e < n; e += blockDim.x) sAcc[e] = dst[e];
  }
  // With NV the next transfer's block is loaded while this one is restricted.
  double next[R];
  auto fetch = [&](long it) __device__ {
    if constexpr (NV != 0) {
      if (!usable(it)) return;
      const double* const src = a.src + (size_t)a.items[5 * it + 1] * a.src_block;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (lane + r * kWave < n) next[r] = src[lane + r * kWave];
    }
  };
  fetch(i0 + wave);
  for (long it0 = i0; it0 < i1; it0 += W) {
    const long it = it0 + wave;
    if (usable(it)) {
      if constexpr (NV != 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (lane + r * kWave < n) s[lane + r * kWave] = next[r];
      } else {
        const double* const src = a.src + (size_t)a.items[5 * it + 1] * a.src_block;
        for (int e = lane; e < n; e += kWave) s[e] = src[e];
      }
    } else if (it < i1 && lane == 0) {
      atomicOr(a.error, 1);  // the item is skipped and reported
    }
    fetch(it + W);
    if (usable(it)) transfer<B, NDIM, true>(a, a.items + 5 * it, s, nv, lane);
    lds_barrier();
    for (int w = 0; w < W; ++w) {
      if (!usable(it0 + w)) continue;
      if constexpr (NV != 0) {
#pragma unroll
        for (int r = 0; r < RA; ++r)
          if ((int)threadIdx.x + r * 256 < n) acc[r] += smem[(size_t)w * n + threadIdx.x + r * 256];
      } else {
        for (int e = threadIdx.x; e < n; e += blockDim.x) sAcc[e] += smem[(size_t)w * n + e];
      }
    }
    lds_barrier();  // the blocks are free for the next transfers
  }
  if (taken) {
    if (threadIdx.x == 0) atomicOr(a.error, 1);
    return;
  }
  if constexpr (NV != 0) {
#pragma unroll
    for (int r = 0; r < RA; ++r)
      if ((int)threadIdx.x + r * 256 < n) dst[threadIdx.x + r * 256] = acc[r];
  } else {
    for (int e = threadIdx.x; e < n; e += blockDim.x) dst[e] = sAcc[e];
  }
}

template <int NDIM, bool RESTRICT>
static hipError_t launch_amr_b(const AmrArgs& a, long ngroups, hipStream_t s) {
  auto go = [&]<int B>() -> hipError_t {
    constexpr int NN = NDIM == 3 ? B * B * B : B * B;
    const size_t block = sizeof(double) * (size_t)NN * a.nv;
    // blocks of up to 64 KiB with a second buffer (and the destination) beside them
    if ((RESTRICT ? 3 : 2) * block + sizeof(double) * NDIM * B * B > 64 * 1024) return hipErrorNotSupported;
    // wavefronts per workgroup: four where their blocks fit 64 KiB (5 values
    // per node: always)
    const bool five = a.nv == 5;
    const int extra = RESTRICT && !five ? 1 : 0;  // the destination block
    int W = 4;
    while (W > 1 && (W + extra) * block + 64 > 64 * 1024) W /= 2;
    const size_t lds = (W + extra) * block;
    const dim3 grid((unsigned)(RESTRICT ? ngroups : (ngroups + W - 1) / W)), threads(W * kWave);
    auto launch = [&]<int NV>() {
      if constexpr (RESTRICT)
        hipLaunchKernelGGL((amr_restrict_kernel<B, NDIM, NV>), grid, threads, lds, s, a);
      else
        hipLaunchKernelGGL((amr_prolong_kernel<B, NDIM, NV>), grid, threads, lds, s, a);
      return hipGetLastError();
    };
    if (five) return launch.template operator()<5>();
    return launch.template operator()<0>();
  };
  switch (a.order) {
    case 1: return go.template operator()<2>();
    case 2: return go.template operator()<3>();
    case 3: return go.template operator()<4>();
    case 4: return go.template operator()<5>();
    case 5: return go.template operator()<6>();
    default: return hipErrorNotSupported;
  }
}

hipError_t launch_amr(const AmrArgs& a, int ndim, bool restrict_, long ngroups, hipStream_t s) {
  if (ngroups <= 0) return hipSuccess;
  if (a.nv < 1 || a.level_delta < 1 || a.level_delta > kAmrMaxLevelDelta) return hipErrorInvalidValue;
  if (ndim == 3) return restrict_ ? launch_amr_b<3, true>(a, ngroups, s) : launch_amr_b<3, false>(a, ngroups, s);
  if (ndim == 2) return restrict_ ? launch_amr_b<2, true>(a, ngroups, s) : launch_amr_b<2, false>(a, ngroups, s);
  return hipErrorInvalidValue;
}

}  // namespace exa
