// Deep rows (longer than 256 values) for at most 32 queries: HBM-bound, the
// four wavefronts of a workgroup taking the four 32-row blocks of each 128-row
// tile against the same 32 queries.
//
// Each tile is a K loop over 128-byte chunks of its rows and of the queries
// (32 fp32 or 64 binary16 values), staged in LDS by direct loads in three
// stages: two chunks of rows are in flight while one is multiplied, and the
// wait before the barrier leaves the newest chunk's loads outstanding.  What
// the rows' stream needs is bytes in flight: with one chunk ahead (two stages
// that also held 128 query rows) 500k x 768 fp32 rows, 24 queries, took 314 us,
// 4.9 TB/s; three stages 294 us, 5.2 TB/s.
//
// The rows' squared norms are summed here, from the fragments that the products
// read (eight partial sums a row, as row_norms_kernel): a pass of their own
// read every row a second time (the same rows, L2, k = 10, 32 queries 595 -> 328
// us a call).
//
// Segments 8 split + 2 w + h (part [nq][8 nsplit][T]), no shared bound.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "knn_kernels.h"
#include "lds_stage.h"
#include "topk_common.h"

namespace mlxvs::kern {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr int kChunkBytes = 128;
constexpr int kChunkDwords = kChunkBytes / 4;
constexpr int kRows = kDeepRows;
constexpr int kQueries = 32;
constexpr int kStages = 3;
constexpr int kLoadsA = kRows / 32;      // LDS-direct loads a wavefront and chunk: 8 rows each
constexpr int kLoads = kLoadsA + 1;      // and 8 of the queries
constexpr int kKeep = kLoads * (kStages - 2);
static_assert(kKeep < 16, "vmcnt's low bits");

// FILT: with a prefilter (FusedArgs::allow), lists of 16.  COS: cosine by
// factors (FusedArgs::qnorm).
template <int T, bool L2, bool F16, bool FILT, bool COS>
__global__ __launch_bounds__(256, 2) void deep_rs_kernel(FusedArgs a) {
  constexpr int esize = F16 ? 2 : 4;
  // separately named stages, so that loads into one are not taken to alias
  // the reads of another
  __shared__ __align__(16) uint32_t tA0[kRows * kChunkDwords], tA1[kRows * kChunkDwords],
      tA2[kRows * kChunkDwords];
  __shared__ __align__(16) uint32_t tQ0[kQueries * kChunkDwords], tQ1[kQueries * kChunkDwords],
      tQ2[kQueries * kChunkDwords];
  constexpr bool NORM = L2 || COS;
  __shared__ __align__(16) float tnorm[NORM ? kRows : 4];  // a wavefront's 32 rows each

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, col = lane & 31;
  const int split = blockIdx.x;
  const int q = col;
  const bool qvalid = q < a.nq;
  const int rowb = a.ld * esize;
  const int NC = rowb / kChunkBytes;
  const int64_t r0 = (int64_t)split * a.rows_per_split;
  const int64_t r1 = min(a.n, r0 + a.rows_per_split);
  const int nrows = r1 > r0 ? (int)(r1 - r0) : 0;
  const int ntiles = (nrows + kRows - 1) / kRows;
  const int nsteps = ntiles * NC;

  // buffer resources per chunk in scalar registers (base at the chunk, range =
  // the bytes left: rows past the split and queries past nq read zero)
  const char* sbase = (const char*)a.base + r0 * rowb;
  const int srows_bytes = nrows * rowb;
  const char* qbase = (const char*)a.queries;
  const int qrows_bytes = min(kQueries, a.nq) * rowb;
  // load j of wavefront w: rows 32 j + 8 w .. + 7, lane l row l / 8 and slot l %
  // 8; vector v of row r sits at slot v ^ swz(r) (deep_kernel)
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  auto swz = [](int r) { return (r & 7) ^ ((r >> 3) & 1); };
  const int lrow = 8 * wave + (lane >> 3);
  const uint32_t voff = (uint32_t)(lrow * rowb + 16 * ((lane & 7) ^ swz(lrow)));
  int pc = 0, pt = 0;  // chunk and tile of the next fetch
  auto issue_loads = [&](uint32_t* dA, uint32_t* dQ) {
    const int cdone = pc * kChunkBytes;
    const int tc = pt * (kRows * rowb) + cdone;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(sbase + tc), (short)0, max(srows_bytes - tc, 0), 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(qbase + cdone), (short)0, max(qrows_bytes - cdone, 0), 0x00020000);
#pragma unroll
    for (int j = 0; j < kLoadsA; ++j)
      load16_to_lds(ra, dA + (4 * j + wv) * 256, voff + (uint32_t)(32 * j * rowb));
    load16_to_lds(rq, dQ + wv * 256, voff);
    if (++pc == NC) {
      pc = 0;
      ++pt;
    }
  };

  uint32_t K[T], I[T];
#pragma unroll
  for (int i = 0; i < T; ++i) K[i] = I[i] = 0;
  // (+inf for a lane without a query: nothing passes)
  float thr = qvalid ? score_of_key(0u) : INFINITY;
  const uint32_t* fw = FILT ? a.allow + (int64_t)(qvalid ? q : 0) * a.allow_stride : nullptr;
  // COS: the lane's query's inverse norm
  const float qinv = (COS && qvalid) ? 1.0f / fmaxf(sqrtf(a.qnorm[q]), 1e-30f) : 0.0f;

  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // NORM: the lane's half of row col's squares
  int c = 0, t = 0;
  auto step = [&](const uint32_t* cA, const uint32_t* cQ, uint32_t* nA, uint32_t* nQ) {
    // every wavefront's loads of this chunk have landed (the next chunk's may
    // be under way), and every wavefront has left the chunk before
    __builtin_amdgcn_s_waitcnt(0x0F70 | kKeep);
    __syncthreads();
    issue_loads(nA, nQ);
    __builtin_amdgcn_sched_barrier(0);
    const bool last = c + 1 == NC;
    const uint32_t* qrow = cQ + col * kChunkDwords;
    const uint32_t* arow = cA + (32 * wave + col) * kChunkDwords;
    const int sw = swz(col);
    typedef typename std::conditional<F16, halfx8, floatx4>::type fragv;
    fragv bq[2], av[2];
    auto fetch = [&](int v, int b) {
      const int slot = F16 ? 4 * ((2 * v + h) ^ sw) : 4 * ((4 * h + v) ^ sw);
      bq[b] = *(const fragv*)(qrow + slot);
      av[b] = *(const fragv*)(arow + slot);
    };
    fetch(0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (v + 1 < 4) fetch(v + 1, (v + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (F16) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[v & 1], bq[v & 1], acc, 0, 0, 0);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[v & 1][u], bq[v & 1][u], acc, 0, 0, 0);
      }
      if constexpr (NORM) {
        constexpr int E = F16 ? 8 : 4;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float x = (float)av[v & 1][e];
          ss[e & 3] = __builtin_fmaf(x, x, ss[e & 3]);
        }
      }
    }
    if (last) {
      const int lim0 = nrows - t * kRows - 32 * wave;
      const uint32_t id0 = (uint32_t)(r0 + (int64_t)t * kRows + 32 * wave);
      uint32_t am = 0xffffffffu;
      if constexpr (FILT) am = qvalid && lim0 > 0 ? allowed_positions(fw[id0 >> 5], h) : 0u;
      if constexpr (NORM) {
        // row col's norm, into the lanes of the score layout through LDS (the
        // wavefront's own words: no barrier)
        float nn = (ss[0] + ss[1]) + (ss[2] + ss[3]);
        nn += __shfl_xor(nn, 32);
        // (L2: -|b|^2 / 2, +0 for a zero row; COS: the inverse norm)
        const float v = COS ? 1.0f / fmaxf(sqrtf(nn), 1e-30f) : nn > 0.0f ? -0.5f * nn : 0.0f;
        if (h == 0) {
          tnorm[32 * wave + col] = v;
          if (L2 && a.norm_out && col < lim0) a.norm_out[id0 + col] = v;
        }
        ss[0] = ss[1] = ss[2] = ss[3] = 0.0f;
      }
      float sc[16];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        floatx4 hn = {};
        if constexpr (NORM) hn = *(const floatx4*)&tnorm[32 * wave + 8 * j + 4 * h];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float x = acc[4 * j + u];
          // COS: 1 / max(|b|, 1e-30) (reference src/knn.cpp:30-33; a zero row
          // scales a zero dot product); L2: the half score, one rounding
          sc[4 * j + u] = COS ? (x * hn[u]) * qinv : L2 ? x + hn[u] : x;
        }
      }
      select_block<T, L2>(K, I, thr, sc, h, id0, lim0, am);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
    if (++c == NC) {
      c = 0;
      ++t;
    }
  };
  if (nsteps > 0) {
    issue_loads(tA0, tQ0);
    issue_loads(tA1, tQ1);
  }
  for (int s = 0; s < nsteps; s += 3) {
    step(tA0, tQ0, tA2, tQ2);
    if (s + 1 < nsteps) step(tA1, tQ1, tA0, tQ0);
    if (s + 2 < nsteps) step(tA2, tQ2, tA1, tQ1);
  }
  // the fetches past the last chunk land before the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0F70);

  if (qvalid) {
    uint64_t* dst = a.part + ((int64_t)q * (8 * a.nsplit) + 8 * split + 2 * wave + h) * T;
#pragma unroll
    for (int i = 0; i < T; ++i) dst[i] = stream_rank(K[i], I[i]);
  }
}

template <int T, bool F16>
hipError_t rs_inst(const FusedArgs& a, hipStream_t s) {
  const dim3 grid(a.nsplit);
  if constexpr (T == 16) {
    if (a.allow) {  // a prefilter: lists of 16 only
      if (a.metric == kL2)
        hipLaunchKernelGGL((deep_rs_kernel<T, true, F16, true, false>), grid, dim3(256), 0, s, a);
      else
        hipLaunchKernelGGL((deep_rs_kernel<T, false, F16, true, false>), grid, dim3(256), 0, s, a);
      return hipGetLastError();
    }
  }
  if (a.allow) return hipErrorInvalidValue;
  if (a.metric == kCosine) {
    if constexpr (F16) {
      return hipErrorInvalidValue;  // cosine by factors: fp32 rows only
    } else {
      if (!a.qnorm) return hipErrorInvalidValue;
      hipLaunchKernelGGL((deep_rs_kernel<T, false, F16, false, true>), grid, dim3(256), 0, s, a);
      return hipGetLastError();
    }
  }
  if (a.metric == kL2)
    hipLaunchKernelGGL((deep_rs_kernel<T, true, F16, false, false>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((deep_rs_kernel<T, false, F16, false, false>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_deep_rs(const FusedArgs& a, bool f16, hipStream_t s) {
  if (!deep_supported(a.ld, a.T, f16) || a.nq > kQueries || a.nqb != 1 || a.mslots != 0)
    return hipErrorInvalidValue;
  switch (a.T) {
    case 4: return f16 ? rs_inst<4, true>(a, s) : rs_inst<4, false>(a, s);
    case 8: return f16 ? rs_inst<8, true>(a, s) : rs_inst<8, false>(a, s);
    case 10: return f16 ? rs_inst<10, true>(a, s) : rs_inst<10, false>(a, s);
    case 16: return f16 ? rs_inst<16, true>(a, s) : rs_inst<16, false>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace mlxvs::kern
