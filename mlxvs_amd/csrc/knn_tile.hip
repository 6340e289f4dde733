// Deep rows (too long for a query to stay in registers) in batches, on
// v_mfma_f32_32x32x16_f16: binary16 rows, or float32 rows as two binary16
// pieces (SplitState, knn_kernels.h).
//
// A workgroup of eight wavefronts owns 256 queries and walks the 256-row tiles
// of its split; for each tile it runs a K loop over 128-byte chunks of the
// tile's rows and of its queries (64 binary16 values, or 32 values' two
// pieces), staged in LDS by direct loads, one chunk ahead in the other of two
// stages.  Wavefront w multiplies rows 128 (w % 2) .. + 127 with queries 64
// (w / 2) .. + 63: four by two 32 x 32 blocks, so six fragments read from LDS
// feed eight products, and a workgroup fetches 512 rows for 256 x 256 scores.
// Lists of 16 (two of them a lane beside 128 accumulators would spill) take
// all 256 rows with 32 queries a wavefront: nine fragments for eight.
//
// With pieces a chunk's fragments feed lo x hi, hi x lo and hi x hi (three
// products of a chunk that costs two to fetch and to read).
//
// What bounds it: at these rates the card lowers its clock (1.82 GHz of 2.4 with
// pieces, 1.73 on binary16 rows), and the MFMA is busy 67% and 62% of the time,
// so what counts is the work and the waits beside the products.  Tried at 1M x 1536 x 10,000,
// binary16 / float32 rows: deep_kernel's 128 x 128 (five fragments for four
// products) 35.2 / 227 ms (on the float32 MFMA); 256 x 128 with four
// wavefronts, two workgroups a CU, 64-byte chunks and three stages 37.1 / 108;
// 256 x 256, 64-byte chunks, four stages 32.4 / 82; this form 28.6 / 79: 1.07
// and 1.16 PFLOP/s of products, where a large library matrix product reaches
// 1.2 on this card.
//
// After the last chunk of a tile a lane filters its scores -- two queries of
// 64 rows each, or one of 128 -- into their lists: segments 4 split + 2 (w %
// 2) + h, or 2 split + h.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "knn_kernels.h"
#include "lds_stage.h"
#include "topk_common.h"

namespace mlxvs::kern {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr int kTR = kTileKernelRows;
constexpr int kQB = kTileQueries;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kChunkBytes = 128;
constexpr int kChunkDwords = kChunkBytes / 4;
constexpr int kVecs = kChunkBytes / 16;           // 16-byte vectors of a row's chunk
constexpr int kRowsPerLoad = 1024 / kChunkBytes;  // rows of one load instruction
constexpr int kLoadsA = kTR / kRowsPerLoad / kWaves;
constexpr int kLoadsQ = kQB / kRowsPerLoad / kWaves;
static_assert(kTilePieceRun * 4 == kChunkBytes, "a chunk is a run of hi and a run of lo pieces");

// Vector v of row r sits at slot v ^ swz(r): the sixteen rows whose 16-byte
// reads the LDS serves together then cover all its banks.
__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Queries (of 32) and 32-row blocks per wavefront.
template <int T>
constexpr int tile_nc() { return T > 10 ? 1 : 2; }
template <int T>
constexpr int tile_nb() { return 8 / tile_nc<T>(); }

template <int T, bool L2, bool PIECES, bool FILT>
__global__ __launch_bounds__(kThreads, 1) void tile_kernel(FusedArgs a) {
  uint32_t sflags = 0;
  if (a.split) {
    sflags = a.split->flags;
    if ((split_route(*a.split) == 0) != (a.route == 0)) return;
  }
  // separately named stages, so that loads into one are not taken to alias
  // the reads of another
  __shared__ __align__(16) uint32_t tA0[kTR * kChunkDwords], tA1[kTR * kChunkDwords];
  __shared__ __align__(16) uint32_t tQ0[kQB * kChunkDwords], tQ1[kQB * kChunkDwords];
  __shared__ __align__(16) float tnorm[L2 ? 2 * kTR : 4];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, col = lane & 31;
  constexpr int NC2 = tile_nc<T>(), NB = tile_nb<T>();
  // the wavefront's first row of a tile, and query of the block
  const int row_w = NC2 == 2 ? 128 * (wave & 1) : 0;
  const int q_w = NC2 == 2 ? 64 * (wave >> 1) : 32 * wave;
  int split, qb;
  tile_of_workgroup(blockIdx.x, a.nsplit, a.nqb, a.xcd_major, split, qb);
  const int qb0 = qb * kQB;
  const bool wave_on = qb0 + q_w < a.nq;
  const int rowb = a.ld * (PIECES ? 4 : 2);
  const int NC = rowb / kChunkBytes;
  const int64_t r0 = (int64_t)split * a.rows_per_split;
  const int64_t r1 = min(a.n, r0 + a.rows_per_split);
  const int nrows = r1 > r0 ? (int)(r1 - r0) : 0;
  const int ntiles = (nrows + kTR - 1) / kTR;
  const int nsteps = ntiles * NC;

  // buffer resources are built per chunk in scalar registers (base at the
  // chunk, range = the bytes left: rows past the split read zero)
  const char* sbase = (const char*)a.base + r0 * rowb;
  const int srows_bytes = nrows * rowb;
  const char* qbase = (const char*)a.queries + (int64_t)qb0 * rowb;
  const int qrows_bytes = min(kQB, a.nq - qb0) * rowb;
  const __amdgpu_buffer_rsrc_t rn = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(L2 ? a.bnorm + r0 : (const float*)a.base), (short)0, L2 ? nrows * 4 : 0, 0x00020000);

  // Load j of wavefront w fills rows 8 (8 j + w) .. + 7 of a stage: lane l row
  // l / 8 of them, slot l % 8.
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int lrow = kRowsPerLoad * wave + lane / kVecs;
  const uint32_t voff = (uint32_t)(lrow * rowb + 16 * ((lane % kVecs) ^ swz(lrow)));
  int pc = 0, pt = 0;  // chunk and tile of the next fetch
  auto issue_loads = [&](uint32_t* dA, uint32_t* dQ) {
    const int cdone = pc * kChunkBytes;
    const int tc = pt * (kTR * rowb) + cdone;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(sbase + tc), (short)0, max(srows_bytes - tc, 0), 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(qbase + cdone), (short)0, max(qrows_bytes - cdone, 0), 0x00020000);
    if (L2 && pc == 0 && wv < 4)
      load4_to_lds(rn, tnorm + kTR * (pt & 1) + 64 * wv, (uint32_t)(pt * kTR + tid) * 4u);
#pragma unroll
    for (int j = 0; j < kLoadsA; ++j)
      load16_to_lds(ra, dA + (kWaves * j + wv) * 256, voff + (uint32_t)(kRowsPerLoad * kWaves * j * rowb));
#pragma unroll
    for (int j = 0; j < kLoadsQ; ++j)
      load16_to_lds(rq, dQ + (kWaves * j + wv) * 256, voff + (uint32_t)(kRowsPerLoad * kWaves * j * rowb));
    if (++pc == NC) {
      pc = 0;
      ++pt;
    }
  };

  // the lane's two queries: lists, filters, shared bounds
  constexpr int S = bound_slots<T>();
  const bool share = a.mslots > 0;
  const int seg = NC2 == 2 ? 4 * split + 2 * (wave & 1) + h : 2 * split + h;
  const int myslot = share ? seg % a.mslots : 0;
  int q[NC2];
  bool qvalid[NC2];
  uint32_t K[NC2][T], I[NC2][T];
  float thr[NC2];
#pragma unroll
  for (int c = 0; c < NC2; ++c) {
    q[c] = qb0 + q_w + 32 * c + col;
    qvalid[c] = q[c] < a.nq;
#pragma unroll
    for (int i = 0; i < T; ++i) K[c][i] = I[c][i] = 0;
    // (+inf for a lane without a query: nothing passes)
    thr[c] = qvalid[c] ? score_of_key(0u) : INFINITY;
  }

  floatx16 acc[NB][NC2];

  const bool blow = sflags & kSplitBaseLow, qlow = sflags & kSplitQueryLow;
  const bool lowlow = PIECES && split_low_low(sflags);
  const bool seeds_first = a.ld <= kMaxFusedDimF32;
  int cc = 0, t = 0;
  auto step = [&](const uint32_t* cA, const uint32_t* cQ, uint32_t* nA, uint32_t* nQ) {
    // every wavefront's loads of this chunk have landed, and every wavefront
    // has left the one before
    dma_barrier();
    issue_loads(nA, nQ);
    __builtin_amdgcn_sched_barrier(0);
    const bool last = cc + 1 == NC;
    if (wave_on) {
      // L2: the sums start at the rows' -|b|^2 / 2 up to 256 values, where the
      // float32 route's do too, and take it at their end above.  Whichever keeps
      // them smaller on the way rounds less: values of one sign 0.53 units (rms,
      // of 2^-24 of the sum of magnitudes) against 0.98 at 200 dims; values of
      // both signs 1.40 against 0.56 at 384, and 3.0 against 0.73 at 1,536
      if (cc == 0) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            floatx4 hn = {};
            if (L2 && seeds_first)
              hn = *(const floatx4*)&tnorm[kTR * (t & 1) + row_w + 32 * b + 8 * j + 4 * h];
#pragma unroll
            for (int c = 0; c < NC2; ++c)
#pragma unroll
              for (int u = 0; u < 4; ++u) acc[b][c][4 * j + u] = hn[u];
          }
      }
      const int sw = swz(col);
      const uint32_t* arow = cA + (row_w + col) * kChunkDwords;
      const uint32_t* qrow = cQ + (q_w + col) * kChunkDwords;
      typedef halfx8 rowfrags[4];
      typedef halfx8 queryfrags[NC2];
      auto rows4 = [&](rowfrags& x, int g, int v) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
          x[b] = *(const halfx8*)(arow + (4 * g + b) * 32 * kChunkDwords + 4 * (v ^ sw));
      };
      auto queries = [&](queryfrags& y, int v) {
#pragma unroll
        for (int c = 0; c < NC2; ++c)
          y[c] = *(const halfx8*)(qrow + c * 32 * kChunkDwords + 4 * (v ^ sw));
      };
      auto mult = [&](int g, const rowfrags& x, const queryfrags& y) {
#pragma unroll
        for (int c = 0; c < NC2; ++c)
#pragma unroll
          for (int b = 0; b < 4; ++b)
            acc[4 * g + b][c] =
                __builtin_amdgcn_mfma_f32_32x32x16_f16(x[b], y[c], acc[4 * g + b][c], 0, 0, 0);
      };
      if constexpr (PIECES) {
        constexpr int LV = kVecs / 2;  // the lo pieces' first vector
#pragma unroll
        for (int k = 0; k < kVecs / 4; ++k) {
          queryfrags yh, yl;
          queries(yl, LV + 2 * k + h);
          queries(yh, 2 * k + h);
#pragma unroll
          for (int g = 0; g < NB / 4; ++g) {
            // the small products first
            rowfrags xh, xl;
            rows4(xh, g, 2 * k + h);
            if (qlow) mult(g, xh, yl);
            if (blow) {
              rows4(xl, g, LV + 2 * k + h);
              mult(g, xl, yh);
            }
            mult(g, xh, yh);
          }
          if (lowlow) {  // (short values, rare: the products that keep their sums exact)
            queries(yl, LV + 2 * k + h);
#pragma unroll
            for (int g = 0; g < NB / 4; ++g) {
              rowfrags xl;
              rows4(xl, g, LV + 2 * k + h);
              mult(g, xl, yl);
            }
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < kVecs / 2; ++k) {
          queryfrags y;
          queries(y, 2 * k + h);
#pragma unroll
          for (int g = 0; g < NB / 4; ++g) {
            rowfrags x;
            rows4(x, g, 2 * k + h);
            mult(g, x, y);
          }
        }
      }
      if (last) {
        const int lim0 = nrows - t * kTR - row_w;
        const uint32_t id0 = (uint32_t)(r0 + (int64_t)t * kTR + row_w);
#pragma unroll
        for (int c = 0; c < NC2; ++c) {
          uint32_t* gk = a.gkey + (int64_t)(qvalid[c] ? q[c] : 0) * S;
          SharedBound<S> seen;
          seen.clear();
          if (share) {
            seen.load(gk, a.mslots);
            thr[c] = fmaxf(thr[c], filter_of<L2>(score_of_key(seen.bound())));
          }
          bool inserted = false;
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            // the prefilter's word of the block's rows (rows past the split:
            // none allowed, and no word read past the filter)
            uint32_t am = 0xffffffffu;
            if constexpr (FILT) {
              am = 0u;
              if (qvalid[c] && lim0 > 32 * b)
                am = allowed_positions(
                    a.allow[(int64_t)q[c] * a.allow_stride + ((id0 + 32 * b) >> 5)], h);
            }
            float sc[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              // L2 half scores q.b + (-|b|^2 / 2), one rounding (deep_kernel)
              floatx4 hn = {};
              if (L2 && !seeds_first)
                hn = *(const floatx4*)&tnorm[kTR * (t & 1) + row_w + 32 * b + 8 * j + 4 * h];
#pragma unroll
              for (int u = 0; u < 4; ++u)
                sc[4 * j + u] = L2 ? acc[b][c][4 * j + u] + hn[u] : acc[b][c][4 * j + u];
            }
            inserted |= select_block<T, L2>(K[c], I[c], thr[c], sc, h, id0 + 32 * b,
                                            lim0 - 32 * b, am);
          }
          if (share && qvalid[c] && inserted) {
            const uint32_t kp = list_key(K[c], a.pubj);
            if (kp > seen.slot(myslot))
              __hip_atomic_fetch_max(gk + myslot, kp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (++cc == NC) {
      cc = 0;
      ++t;
    }
  };
  if (nsteps > 0) issue_loads(tA0, tQ0);
  for (int s = 0; s < nsteps; s += 2) {
    step(tA0, tQ0, tA1, tQ1);
    if (s + 1 < nsteps) step(tA1, tQ1, tA0, tQ0);
  }
  // the fetches past the last chunk land before the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0F70);

#pragma unroll
  for (int c = 0; c < NC2; ++c)
    if (qvalid[c]) {
      uint64_t* dst = a.part + ((int64_t)q[c] * (2 * NC2 * a.nsplit) + seg) * T;
#pragma unroll
      for (int i = 0; i < T; ++i) dst[i] = stream_rank(K[c][i], I[c][i]);
    }
}

template <int T, bool PIECES>
int tile_occupancy() {
  int blocks = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &blocks, tile_kernel<T, true, PIECES, false>, kThreads, 0);
  return e == hipSuccess && blocks > 0 ? blocks : 1;
}

template <int T, bool PIECES>
hipError_t tile_inst(const FusedArgs& a, hipStream_t s) {
  const dim3 grid(a.nsplit * a.nqb);
  if constexpr (T == 16) {
    if (a.allow) {  // a prefilter: lists of 16 only
      if (a.metric == kL2)
        hipLaunchKernelGGL((tile_kernel<T, true, PIECES, true>), grid, dim3(kThreads), 0, s, a);
      else
        hipLaunchKernelGGL((tile_kernel<T, false, PIECES, true>), grid, dim3(kThreads), 0, s, a);
      return hipGetLastError();
    }
  }
  if (a.allow) return hipErrorInvalidValue;
  if (a.metric == kL2)
    hipLaunchKernelGGL((tile_kernel<T, true, PIECES, false>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((tile_kernel<T, false, PIECES, false>), grid, dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace

bool tile_supported(int ld, int T, bool pieces) {
  // (a tile's norms are fetched with its first chunk into one of two slots:
  // at least two chunks a tile)
  const int rowb = ld * (pieces ? 4 : 2);
  return (T == 10 || T == 16) && rowb % kChunkBytes == 0 && rowb >= 2 * kChunkBytes &&
         (int64_t)kTR * rowb < (int64_t(1) << 28);
}

int tile_blocks_per_cu(int T, bool pieces) {
  if (T == 10) return pieces ? tile_occupancy<10, true>() : tile_occupancy<10, false>();
  return pieces ? tile_occupancy<16, true>() : tile_occupancy<16, false>();
}

int tile_segments(int T) { return T == 10 ? 2 * tile_nc<10>() : 2 * tile_nc<16>(); }

hipError_t launch_tile(const FusedArgs& a, bool pieces, hipStream_t s) {
  if (!tile_supported(a.ld, a.T, pieces) || (pieces && !a.split)) return hipErrorInvalidValue;
  if (a.T == 10) return pieces ? tile_inst<10, true>(a, s) : tile_inst<10, false>(a, s);
  return pieces ? tile_inst<16, true>(a, s) : tile_inst<16, false>(a, s);
}

}  // namespace mlxvs::kern
