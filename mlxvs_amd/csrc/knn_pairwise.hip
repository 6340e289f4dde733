// cuVS's other distances (PairwiseMetric, knn_kernels.h) for batches of
// queries: a query per lane.
//
// The scan of topk_merge.hip gives a workgroup one query, so every query
// reads every row (100,000 x 128 rows, 1,000 queries: 51 GB through L2, which
// set its 2.97 ms for L1).  Here a lane holds its query's values in registers
// and its wavefront walks its split's rows, so a row is read once for 64
// queries.  Each 16 lanes hold a whole row, DQ / 16 values a lane, and the
// arithmetic takes a value from lane n of the 16 as a DPP operand (row
// broadcast): an L1 value costs its subtraction and its addition and nothing
// else, no lane sums to meet, no LDS, no barrier; rows arrive four ahead.
// (Rows through scalar loads instead: the compiler gathered them in front of
// their use and waited for each.)  Bound: VALU, 0.65 ms of L1's two operations
// a value for that case; measured 0.80 ms (2.97 before).
//
// A lane keeps the best T rows of its query (a sorted stream list, as the
// fused kernels), and all splits of a query share a bound on its k-th best
// (SharedBound).  With k > T the queries whose lists may have been too short are
// searched again by the scan (launch_pairwise_scan under the merge's flags).
// Segments: one per split (part [nq][nsplit][T]).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "knn_kernels.h"
#include "topk_common.h"

namespace mlxvs::kern {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// (Canberra's divisions, the logarithms and the powers spill when a row's
// values are in flight together: those stay with the scan)
constexpr bool lanes_metric(int m) {
  return m == kPwL1 || m == kPwLinf || m == kPwCorrelation || m == kPwHellinger ||
         m == kPwBrayCurtis || m == kPwHamming || m == kPwRusselRao;
}

template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// The same terms, precision and finish as MetricChunkScorer's; the sums are
// eight partial ones met in pairs as there (here each of every eighth value).
template <int MET>
struct LaneMetric {
  static constexpr int NA = MET == kPwCorrelation ? 3 : MET == kPwBrayCurtis ? 2 : 1;
  float A[NA][8];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int t = 0; t < NA; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) A[t][e] = 0.0f;
  }
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int t = 0; t < NA; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(A[t][e]));
  }
  __device__ __forceinline__ void add(int e, float a, float b) {
    if constexpr (MET == kPwL1) {
      A[0][e] += fabsf(a - b);
    } else if constexpr (MET == kPwLinf) {
      A[0][e] = fmaxf(A[0][e], fabsf(a - b));
    } else if constexpr (MET == kPwCorrelation) {
      A[0][e] += a * b;
      A[1][e] += b;
      A[2][e] += b * b;
    } else if constexpr (MET == kPwHellinger) {
      A[0][e] += a * sqrtf(b);  // (a: the query value's square root)
    } else if constexpr (MET == kPwBrayCurtis) {
      A[0][e] += fabsf(a - b);
      A[1][e] += fabsf(a + b);
    } else if constexpr (MET == kPwHamming) {
      A[0][e] += a != b ? 1.0f : 0.0f;
    } else {
      A[0][e] += a * b;
    }
  }
  __device__ __forceinline__ float total(int t) const {
    const float(&x)[8] = A[t];
    if (MET == kPwLinf)
      return fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                   fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
    return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  }
  __device__ __forceinline__ float finish(float fd, float qs, float qss) const {
    if constexpr (MET == kPwL1 || MET == kPwLinf) return total(0);
    else if constexpr (MET == kPwCorrelation) {
      const float ab = total(0), sb = total(1), sbb = total(2);
      return 1.0f - (fd * ab - qs * sb) / sqrtf((fd * qss - qs * qs) * (fd * sbb - sb * sb));
    } else if constexpr (MET == kPwHellinger) return sqrtf(fmaxf(1.0f - total(0), 0.0f));
    else if constexpr (MET == kPwBrayCurtis) return total(0) / total(1);
    else if constexpr (MET == kPwHamming) return total(0) / fd;
    else return (fd - total(0)) / fd;
  }
};

template <int DQ, int MET, int T>
__global__ __launch_bounds__(256, 2) void pairwise_lanes_kernel(PairwiseArgs a) {
  static_assert(DQ % 32 == 0, "chunks of 32 values");
  constexpr int PER = DQ / 16;  // row values a lane holds
  const int lane = threadIdx.x & 63;
  const int waves = blockDim.x >> 6;
  const int wv = threadIdx.x >> 6;
  const int split = blockIdx.x % a.nsplit;
  const int64_t q = ((int64_t)(blockIdx.x / a.nsplit) * waves + wv) * 64 + lane;
  const bool qvalid = q < a.nq;
  // the split's rows r0, r0 + row_step, ..: every nsplit-th row, so that rows
  // side by side -- a dataset in the order of its groups -- do not meet in one
  // split's list (100k x 128 rows in groups of 200, 1,000 queries, k = 50: with
  // splits of neighbouring rows every query was flagged and the call took 38.9
  // ms); neighbouring rows past 2^31 bytes of them
  const int64_t row_step = a.strided ? a.nsplit : 1;
  const int64_t r0 = min(a.n, a.strided ? (int64_t)split : (int64_t)split * a.rows_per_split);
  const int64_t span = a.strided ? a.n - r0 : min(a.n - r0, a.rows_per_split);  // rows to the last's end
  const int nrows = (int)((span + row_step - 1) / row_step);

  float qv[DQ];
  {
    const float* qr = a.queries + (qvalid ? q : 0) * DQ;
#pragma unroll
    for (int v = 0; v < DQ / 4; ++v) {
      typedef float floatx4 __attribute__((ext_vector_type(4)));
      const floatx4 x = *(const floatx4*)(qr + 4 * v);
#pragma unroll
      for (int u = 0; u < 4; ++u) qv[4 * v + u] = x[u];
    }
  }
  float qs = 0.0f, qss = 0.0f;
  if constexpr (MET == kPwCorrelation) {
#pragma unroll
    for (int c = 0; c < DQ; ++c) {  // (zeros past d add nothing)
      qs += qv[c];
      qss += qv[c] * qv[c];
    }
  }
  if constexpr (MET == kPwHellinger) {
#pragma unroll
    for (int c = 0; c < DQ; ++c) qv[c] = sqrtf(qv[c]);
  }
  const float fd = (float)a.d;

  uint32_t K[T], I[T];
#pragma unroll
  for (int i = 0; i < T; ++i) K[i] = I[i] = 0;
  // a row's key must reach this (all ones: a lane without a query)
  uint32_t need = qvalid ? 1u : 0xffffffffu;
  constexpr int S = bound_slots<T>();
  const bool share = a.mslots > 0;
  uint32_t* gk = a.gkey + (qvalid ? q : 0) * S;
  const int myslot = share ? split % a.mslots : 0;
  uint32_t published = 0;
  const uint32_t* fw = a.allow ? a.allow + (qvalid ? q : 0) * a.allow_stride : nullptr;

  // lane n of 16 holds values 64 v + 4 n .. + 3 of a row (the last 32 of an odd
  // count: 64 v + 2 n, + 1); rows past the split read zero
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.base + r0 * DQ), (short)0, (int)(span * DQ * 4), 0x00020000);
  const uint32_t step = (uint32_t)row_step * (DQ * 4);
  constexpr int V4 = DQ / 64, V2 = DQ % 64 / 32;
  constexpr int AHEAD = 4;
  uint32_t x[AHEAD][PER];
  auto load = [&](int r, uint32_t (&y)[PER]) {
    const uint32_t off = (uint32_t)r * step;
#pragma unroll
    for (int v = 0; v < V4; ++v) {
      const u32x4 t = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 256 * v + 16 * (lane & 15), 0, 0));
#pragma unroll
      for (int u = 0; u < 4; ++u) y[4 * v + u] = t[u];
    }
    if constexpr (V2 != 0) {
      const u32x2 t = __builtin_bit_cast(
          u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off + 256 * V4 + 8 * (lane & 15), 0, 0));
      y[4 * V4] = t[0];
      y[4 * V4 + 1] = t[1];
    }
  };
  LaneMetric<MET> m;
  auto value = [&](uint32_t v, auto n) {  // v of lane n of the 16
    return __uint_as_float(
        (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + decltype(n)::value, 0xf, 0xf, true));
  };
  // the key of row r, whose values y holds; then row r + AHEAD's into y
  auto row_key = [&](int r, uint32_t (&y)[PER]) {
    m.clear();
    each<16>([&](auto n) {
      constexpr int N = decltype(n)::value;
#pragma unroll
      for (int v = 0; v < V4; ++v)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          m.add((4 * N + u) & 7, qv[64 * v + 4 * N + u], value(y[4 * v + u], n));
      if constexpr (V2 != 0) {
        m.add((2 * N) & 7, qv[64 * V4 + 2 * N], value(y[4 * V4], n));
        m.add((2 * N + 1) & 7, qv[64 * V4 + 2 * N + 1], value(y[4 * V4 + 1], n));
      }
    });
    // (the sums stay here: sunk past the branches below, their operands would
    // be moved out of the row's lanes one by one first)
    m.pin();
    __builtin_amdgcn_sched_barrier(0);  // (a row at a time, its load three rows ahead of its use)
    load(r + AHEAD, y);
    __builtin_amdgcn_sched_barrier(0);
    return key_nz(-m.finish(fd, qs, qss));
  };
  // nothing else may be outstanding in the loop: a query value's load would
  // make every iteration wait for its own rows too
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_sched_barrier(0);
  if (nrows > 0) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) load(u, x[u]);
  }
  // four rows' keys, then one vote for the four
  for (int r = 0; r < nrows; r += AHEAD) {
    uint32_t key[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) key[u] = row_key(r + u, x[u]);
    if (fw) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int64_t j = r0 + min(r + u, nrows - 1) * row_step;
        if (!((fw[j >> 5] >> (j & 31)) & 1u)) key[u] = 0u;
      }
    }
    if (r + AHEAD > nrows) {
#pragma unroll
      for (int u = 1; u < AHEAD; ++u)
        if (r + u >= nrows) key[u] = 0u;
    }
    // the shared bound: after 8, 16 and every 32 rows
    if (share && r > 0 && ((r & 31) == 0 || r == 8 || r == 16)) {
      SharedBound<S> seen;
      seen.clear();
      seen.load(gk, a.mslots);
      need = max(need, qvalid ? seen.bound() : 0xffffffffu);
    }
    const uint32_t best = max(max(key[0], key[1]), max(key[2], key[3]));
    if (__builtin_amdgcn_ballot_w64(best >= need) != 0) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const bool pass = key[u] >= need;
        if (__builtin_amdgcn_ballot_w64(pass) == 0) continue;
        stream_insert<T>(K, I, pass ? key[u] : 0u, (uint32_t)(r0 + (r + u) * row_step));
        // (a later row needs a larger key than the last: equal ones lose)
        need = max(need, qvalid && K[T - 1] ? K[T - 1] + 1u : need);
      }
      if (share && qvalid) {
        const uint32_t kp = list_key(K, a.pubj);
        if (kp > published) {
          published = kp;
          __hip_atomic_fetch_max(gk + myslot, kp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
  }
  if (qvalid) {
    uint64_t* dst = a.part + (q * a.nsplit + split) * T;
#pragma unroll
    for (int i = 0; i < T; ++i) dst[i] = stream_rank(K[i], I[i]);
  }
}

template <int DQ, int MET>
hipError_t lanes_inst(const PairwiseArgs& a, int T, dim3 grid, dim3 block, hipStream_t s) {
  if (T == 10)
    hipLaunchKernelGGL((pairwise_lanes_kernel<DQ, MET, 10>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((pairwise_lanes_kernel<DQ, MET, 16>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <int MET>
hipError_t lanes_dq(const PairwiseArgs& a, int T, dim3 grid, dim3 block, hipStream_t s) {
  switch (a.ld) {
    case 32: return lanes_inst<32, MET>(a, T, grid, block, s);
    case 64: return lanes_inst<64, MET>(a, T, grid, block, s);
    case 96: return lanes_inst<96, MET>(a, T, grid, block, s);
    case 128: return lanes_inst<128, MET>(a, T, grid, block, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool pairwise_lanes_supported(int metric, int ld) {
  return lanes_metric(metric) && ld % 32 == 0 && ld >= 32 && ld <= 128;
}

hipError_t launch_pairwise_lanes(const PairwiseArgs& a, int T, hipStream_t s) {
  if (a.nq <= 0) return hipSuccess;
  if (!pairwise_lanes_supported(a.metric, a.ld) || (T != 10 && T != 16) || a.nsplit < 1 ||
      a.rows_per_split < 1 || (int64_t)a.nsplit * a.rows_per_split < a.n || a.d > a.ld ||
      (uintptr_t)a.base % 16 != 0 || (uintptr_t)a.queries % 16 != 0 || !a.part || !a.gkey ||
      (a.strided ? a.n + 8 * (int64_t)a.nsplit : a.rows_per_split + 8) * a.ld * 4 >=
          (int64_t(1) << 31) ||
      (a.allow && a.allow_stride != 0 && a.allow_stride < (a.n + 31) / 32))
    return hipErrorInvalidValue;
  const int64_t groups = (a.nq + 63) / 64;
  const int waves = (int)(groups < 4 ? groups : 4);
  const int64_t blocks = (groups + waves - 1) / waves * a.nsplit;
  if (blocks >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(64 * waves);
  switch (a.metric) {
    case kPwL1: return lanes_dq<kPwL1>(a, T, grid, block, s);
    case kPwLinf: return lanes_dq<kPwLinf>(a, T, grid, block, s);
    case kPwCorrelation: return lanes_dq<kPwCorrelation>(a, T, grid, block, s);
    case kPwHellinger: return lanes_dq<kPwHellinger>(a, T, grid, block, s);
    case kPwBrayCurtis: return lanes_dq<kPwBrayCurtis>(a, T, grid, block, s);
    case kPwHamming: return lanes_dq<kPwHamming>(a, T, grid, block, s);
    case kPwRusselRao: return lanes_dq<kPwRusselRao>(a, T, grid, block, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace mlxvs::kern
