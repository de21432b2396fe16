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
// A level is the tensor product of three (two for faces) 1-D operators; it runs
// as NDIM passes over the block in LDS, instead of the reference's B^NDIM-term
// sum per node (the same linear map; the sums round in another order).  The 1-D
// operator of direction d at a level is fineGridProjector1d[j_d] (prolongation:
// out_m = sum_n in_n P[j][n][m]) or w_n P[j][m][n] / (3 w_m) (restriction), j_d
// the subinterval digit of that level.  Restriction adds the restricted blocks
// of a destination's transfers, in list order, to the destination block.
//
// Forms (launch_amr_b says which is taken where, and what they measured):
//   by wavefronts: one per transfer, four to a workgroup; a lane contracts whole
//     grid lines in place with the pass's operator in scalar registers.  A
//     prolongation has no workgroup barrier; a restriction's four wavefronts
//     take four transfers of one destination at a time and meet twice, before
//     their results are added and after.  For long lists: 16 or more transfers
//     per CU are in flight;
//   by workgroup: the lines of one transfer over up to four wavefronts, all
//     levels' operators staged in LDS with the block;
//   by value: one thread per value of the block, which stays in a register.
// Bound: the chain item, block, passes, store of a transfer, in short lists and
// in long ones, where three to four wavefronts per SIMD spend more than half of
// their time waiting (the LDS is busy in 45% of the cycles of a prolongation, VALU
// instructions are active in 30%; a third of the LDS cycles are bank conflicts).
// 183,141 transfers of 6^3 x 5 values by wavefronts: the prolongation 0.55 ms
// (2.9 TB/s), the restriction 0.68 ms (2.4 TB/s; its next block is loaded while
// the last is restricted); with a thread per node and B-term sums per node and
// pass 1.11 and 1.40.
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

constexpr int kAmrWaves = 4;  // wavefronts, and transfers at a time, of a workgroup

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

// task / nv by a float product: exact, as the quotient (a line, below 36) is far
// smaller than 2^24 / nv (an integer division costs a pass of few values more
// than its arithmetic).
struct ByValues {
  int nv;
  float inv;
  __device__ explicit ByValues(int n) : nv(n), inv(1.0f / (float)n) {}
  __device__ int operator()(int task) const { return (int)(((float)task + 0.5f) * inv); }
};

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
template <int B, int NDIM, bool RESTRICT, int NV>
__device__ inline void transfer(const AmrArgs& a, const int* item, double* s, int nv, int lane) {
  constexpr int N = B - 1;
  const ByValues by_values(nv);
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
        const int line = NV ? task / nv : by_values(task);
        const int v = task - line * nv;  // value fastest: neighbouring lanes, neighbouring entries
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

// A block of n values between device memory and LDS, by `lanes` lanes with eight loads
// each in flight.
__device__ inline void copy_block(double* to, const double* from, int n, int lane, int lanes) {
  constexpr int U = 8;
  for (int e0 = lane; e0 < n; e0 += U * lanes) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = e0 + u * lanes < n ? from[e0 + u * lanes] : 0.0;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + u * lanes < n) to[e0 + u * lanes] = v[u];
  }
}

// NV: values per node at compile time (the block's loads then go out together),
// 0: a.nv.
template <int B, int NDIM, int NV>
__global__ __launch_bounds__(kAmrWaves* kWave) void amr_prolong_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  extern __shared__ double smem[];
  const int nv = NV ? NV : a.nv, n = NN * nv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const long k = xcd_run_index() * kAmrWaves + wave;
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
  if constexpr (NV != 0) {
#pragma unroll
    for (int r = 0; r < (NN * NV + kWave - 1) / kWave; ++r)
      if (lane + r * kWave < n) s[lane + r * kWave] = src[lane + r * kWave];
  } else {
    copy_block(s, src, n, lane, kWave);
  }
  transfer<B, NDIM, false, NV>(a, item, s, nv, lane);
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
__global__ __launch_bounds__(kAmrWaves* kWave) void amr_restrict_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  constexpr int R = NV ? (NN * NV + kWave - 1) / kWave : 1;  // a block's entries per lane
  extern __shared__ double smem[];
  __shared__ int taken;
  const int nv = NV ? NV : a.nv, n = NN * nv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  constexpr int W = kAmrWaves;
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
  // The destination block: a thread's own entries, in registers (NV) or in LDS
  // behind the transfers' blocks.
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
        copy_block(s, src, n, lane, kWave);
      }
    } else if (it < i1 && lane == 0) {
      atomicOr(a.error, 1);  // the item is skipped and reported
    }
    fetch(it + W);
    if (usable(it)) transfer<B, NDIM, true, NV>(a, a.items + 5 * it, s, nv, lane);
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

// The passes of one transfer by a workgroup: the operators of all levels are in
// LDS (sM, [pass in order][n][m]).
template <int B, int NDIM>
__device__ inline void transfer_team(int passes, double* s, const double* sM, int nv) {
  const int ntasks = (NDIM == 3 ? B * B : B) * nv;
  const ByValues by_values(nv);
  int d = 0;
  for (int l = 0; l < passes; ++l) {
    const int stride = d == 0 ? 1 : (d == 1 ? B : B * B);
    const double* const M = sM + l * (B * B);
    lds_barrier();  // the block, or the previous pass, complete
    for (int task = threadIdx.x; task < ntasks; task += blockDim.x) {
      const int line = by_values(task), v = task - line * nv;
      const int node = d == 0 ? line * B : (d == 1 ? line / B * (B * B) + line % B : line);
      double* const p = s + node * nv + v;
      double f[B];
#pragma unroll
      for (int n = 0; n < B; ++n) f[n] = p[n * stride * nv];
#pragma unroll
      for (int m = 0; m < B; ++m) {
        double acc = 0.0;
#pragma unroll
        for (int n = 0; n < B; ++n) acc += f[n] * M[n * B + m];
        p[m * stride * nv] = acc;
      }
    }
    d = d + 1 == NDIM ? 0 : d + 1;
  }
  lds_barrier();
}

// The item's operators into sM, in the order of the passes.
template <int B, int NDIM, bool RESTRICT>
__device__ inline void stage_operators(const AmrArgs& a, const int* item, double* sM) {
  const int i0 = item[2], i1 = item[3], i2 = NDIM == 3 ? item[4] : 0;
  for (int e = threadIdx.x; e < a.level_delta * NDIM * B * B; e += blockDim.x) {
    const int pass = e / (B * B), r = e - pass * (B * B), l = pass / NDIM, d = pass - l * NDIM;
    int digit = d == 0 ? i0 : (d == 1 ? i1 : i2);  // prolongation decodes from the top digit, restriction from the bottom
    for (int k = RESTRICT ? l : a.level_delta - 1 - l; k > 0; --k) digit /= 3;
    sM[e] = amr_operators.m[B - 1][RESTRICT ? 1 : 0][digit % 3][r / B][r % B];
  }
}

// One workgroup per transfer.
template <int B, int NDIM>
__global__ __launch_bounds__(256) void amr_prolong_team_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  extern __shared__ double smem[];
  __shared__ int taken;
  const int n = NN * a.nv;
  const int* const item = a.items + 5 * xcd_run_index();
  if (!item_ok<NDIM>(a, item)) {  // the item is skipped and reported
    if (threadIdx.x == 0) atomicOr(a.error, 1);
    return;
  }
  // claim the destination block: a second transfer naming it writes nothing
  if (threadIdx.x == 0) taken = !claim(a, item[0]);
  double* const sM = smem + n;
  stage_operators<B, NDIM, false>(a, item, sM);
  copy_block(smem, a.src + (size_t)item[1] * a.src_block, n, threadIdx.x, blockDim.x);
  transfer_team<B, NDIM>(a.level_delta * NDIM, smem, sM, a.nv);
  if (taken) {
    if (threadIdx.x == 0) atomicOr(a.error, 1);
    return;
  }
  copy_block(a.dst + (size_t)item[0] * a.dst_block, smem, n, threadIdx.x, blockDim.x);
}

// A block of at most 1024 values: one thread per value, which it keeps in a
// register between the passes.
template <int B, int NDIM>
__global__ __launch_bounds__(1024) void amr_prolong_value_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  extern __shared__ double smem[];
  __shared__ int taken;
  const int n = NN * a.nv, e = threadIdx.x;
  const bool active = e < n;
  const int* const item = a.items + 5 * xcd_run_index();
  if (!item_ok<NDIM>(a, item)) {  // the item is skipped and reported
    if (e == 0) atomicOr(a.error, 1);
    return;
  }
  double* const s = smem;
  double* const sM = smem + n;
  double x = active ? a.src[(size_t)item[1] * a.src_block + e] : 0.0;
  // claim the destination block: a second transfer naming it writes nothing
  if (e == 0) taken = !claim(a, item[0]);
  stage_operators<B, NDIM, false>(a, item, sM);
  const int node = active ? ByValues(a.nv)(e) : 0;
  const int c[3] = {node % B, (node / B) % B, node / (B * B)};
  int d = 0;
  for (int l = 0; l < a.level_delta * NDIM; ++l) {
    const int stride = (d == 0 ? 1 : (d == 1 ? B : B * B)) * a.nv;
    const int m = d == 0 ? c[0] : (d == 1 ? c[1] : c[2]);
    if (active) s[e] = x;
    lds_barrier();  // the block complete
    const double* const p = s + (active ? e - m * stride : 0);
    const double* const M = sM + l * (B * B) + m;
    x = 0.0;
#pragma unroll
    for (int k = 0; k < B; ++k) x += p[k * stride] * M[k * B];
    lds_barrier();  // the block read
    d = d + 1 == NDIM ? 0 : d + 1;
  }
  if (taken) {
    if (e == 0) atomicOr(a.error, 1);
    return;
  }
  if (active) a.dst[(size_t)item[0] * a.dst_block + e] = x;
}

// One workgroup per destination, one transfer at a time; the next one's block is
// loaded meanwhile.  Every thread loads and adds the same entries of a block, at
// most a third of 64 KiB over 256 threads (or B with a thread per line).
constexpr int kTeamEntries = (64 * 1024 / 3 / 8 + 255) / 256;
static_assert(kTeamEntries >= amr_tables::kMaxB);
template <int B, int NDIM>
__global__ __launch_bounds__(256) void amr_restrict_team_kernel(AmrArgs a) {
  constexpr int NN = NDIM == 3 ? B * B * B : B * B;
  extern __shared__ double smem[];
  __shared__ int taken;
  const int n = NN * a.nv, tid = threadIdx.x, nt = blockDim.x;
  const long k = xcd_run_index();
  const long i0 = a.ptr[k], i1 = a.ptr[k + 1];
  if (i0 < 0 || i1 < i0 || i1 > a.nitems) {  // a malformed range: nothing is read
    if (tid == 0) atomicOr(a.error, 1);
    return;
  }
  // the destination of the range: that of its first item in range
  long db = -1;
  for (long it = i0; it < i1 && db < 0; ++it)
    if (item_ok<NDIM>(a, a.items + 5 * it)) db = a.items[5 * it];
  if (db < 0) {
    if (i1 > i0 && tid == 0) atomicOr(a.error, 1);
    return;
  }
  auto usable = [&](long it) __device__ {
    return it < i1 && item_ok<NDIM>(a, a.items + 5 * it) && a.items[5 * it] == db;
  };
  // claim the destination block: a second workgroup naming it writes nothing
  if (tid == 0) taken = !claim(a, db);
  double* const sM = smem + n;
  double* const dst = a.dst + (size_t)db * a.dst_block;
  double acc[kTeamEntries], next[kTeamEntries];
  auto fetch = [&](const double* from, double* v) __device__ __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kTeamEntries; ++r) v[r] = tid + r * nt < n ? from[tid + r * nt] : 0.0;
  };
  fetch(dst, acc);
  if (usable(i0)) fetch(a.src + (size_t)a.items[5 * i0 + 1] * a.src_block, next);
  for (long it = i0; it < i1; ++it) {
    const bool ok = usable(it);
    if (ok) {
#pragma unroll
      for (int r = 0; r < kTeamEntries; ++r)
        if (tid + r * nt < n) smem[tid + r * nt] = next[r];
      stage_operators<B, NDIM, true>(a, a.items + 5 * it, sM);
    } else if (tid == 0) {
      atomicOr(a.error, 1);  // the item is skipped and reported
    }
    if (usable(it + 1)) fetch(a.src + (size_t)a.items[5 * (it + 1) + 1] * a.src_block, next);
    if (!ok) continue;
    transfer_team<B, NDIM>(a.level_delta * NDIM, smem, sM, a.nv);
#pragma unroll
    for (int r = 0; r < kTeamEntries; ++r)
      if (tid + r * nt < n) acc[r] += smem[tid + r * nt];
  }
  __syncthreads();  // taken
  if (taken) {
    if (tid == 0) atomicOr(a.error, 1);
    return;
  }
#pragma unroll
  for (int r = 0; r < kTeamEntries; ++r)
    if (tid + r * nt < n) dst[tid + r * nt] = acc[r];
}

template <int NDIM, bool RESTRICT>
static hipError_t launch_amr_b(const AmrArgs& a, long ngroups, hipStream_t s) {
  auto go = [&]<int B>() -> hipError_t {
    constexpr int NN = NDIM == 3 ? B * B * B : B * B;
    const size_t block = sizeof(double) * (size_t)NN * a.nv;
    // blocks of up to 64 KiB with a second buffer (and the destination) beside them
    if ((RESTRICT ? 3 : 2) * block + sizeof(double) * NDIM * B * B > 64 * 1024) return hipErrorNotSupported;
    // Which form (see the top of the file), by the values of a block and the length
    // of the list; us of a prolongation by wavefronts against the form taken:
    //   up to 256 values: a thread per value (4^3 x 1, 1080 transfers 12.5 -> 11.3,
    //     6000 over three levels 24.4 -> 19.6; no slower up to 32,400);
    //   up to 512 while the list is short (6^3 x 2, 27 transfers 8.5 -> 6.0; 4050:
    //     22.2 and 21.6; 32,400: 79 and 110), up to 1024 while it fills the CUs
    //     hardly more than once (6^3 x 4, 108: 11.6 -> 8.1; 4050: 1.4 times slower);
    //   above, a workgroup per transfer for short lists (5^3 x 12, 27 transfers 1.31
    //     times faster, 1080 1.07, 32,400 0.97) and where 64 KiB do not hold four
    //     transfers' blocks: 6^3 x 12, 32,400 transfers 366 -> 260, the restriction
    //     757 -> 396 (before wavefronts took a transfer each: 592 and 1212).
    const int values = NN * a.nv, lines = values / B;
    const bool five = a.nv == 5;
    const size_t lds = (kAmrWaves + (RESTRICT && !five ? 1 : 0)) * block;  // a restriction's destination besides
    const size_t lds_one = block + sizeof(double) * a.level_delta * NDIM * B * B;
    const bool four = lds + 64 <= 64 * 1024;
    const dim3 one_each((unsigned)ngroups), by_lines(lines >= 256 ? 256 : round_up(lines, kWave));
    if constexpr (RESTRICT) {
      if (!four) {
        hipLaunchKernelGGL((amr_restrict_team_kernel<B, NDIM>), one_each, by_lines, lds_one, s, a);
        return hipGetLastError();
      }
    } else {
      if (values <= 256 || (values <= 512 && a.nitems <= 2048) || (values <= 1024 && a.nitems <= 1152)) {
        hipLaunchKernelGGL((amr_prolong_value_kernel<B, NDIM>), one_each, dim3(round_up(values, kWave)), lds_one, s, a);
        return hipGetLastError();
      }
      if (!four || a.nitems <= 512) {
        hipLaunchKernelGGL((amr_prolong_team_kernel<B, NDIM>), one_each, by_lines, lds_one, s, a);
        return hipGetLastError();
      }
    }
    const dim3 grid((unsigned)(RESTRICT ? ngroups : (ngroups + kAmrWaves - 1) / kAmrWaves)), threads(kAmrWaves * kWave);
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
