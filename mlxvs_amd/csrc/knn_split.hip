// Float32 rows as two binary16 pieces (SplitState, knn_kernels.h): the pass
// that makes them, for the kernels that multiply them on the fp16 MFMA.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "knn_kernels.h"
#include "topk_common.h"

namespace mlxvs::kern {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSampleThreads = 1024;
constexpr int kSamplePer = 8;
// The sample's largest value is scaled to [2^11, 2^12): binary16 ends at
// 2^16, so values up to 16 times larger still fit, and its spacing below
// 2^-13 is 2^-24, so a value down to 2^-2 keeps 23 bits and smaller ones have an
// error of up to 2^-25 (split_route: where that is too much).
constexpr int kSampleExp = 11;
// Samples whose largest value lies outside 2^-40 .. 2^40 take the float32
// route: with both scales in 2^-28 .. 2^52 their product and its inverse, and
// the seeds -|b|^2 / 2 sbase squery (below d 2^112, as sbase |b| < 2^16 sqrt(d)
// and squery / sbase <= 2^80), stay inside float32.
constexpr int kMaxSampleExp = 40;
// Unit rows: their values are at most 1 (and a rounding), scaled to 2^15.
constexpr float kUnitScale = 32768.0f;

// The sample: up to 8,192 values of the base rows and of the queries, 64
// neighbouring columns of each of 128 rows spread over all of them (the
// columns by a multiplicative hash).  One workgroup, 16 coalesced loads a lane in
// flight together (values scattered one by one took it 50 us, not 5).
__global__ __launch_bounds__(kSampleThreads) void split_init_kernel(SplitInitArgs a) {
  constexpr int W = kSampleThreads / 64;
  __shared__ float wmax[2][W], wspread[2][W], wsquare[2][W];
  __shared__ int wunit[2][W], wzero[2][W];
  __shared__ uint32_t wflags[W];
  const int tid = threadIdx.x, wave = tid >> 6;
  float m[2] = {0.0f, 0.0f};
  int unit[2] = {0, 0}, zeros[2] = {0, 0};
  // what the sample's bits show already (values of more than 11 and 16 bits,
  // values that two pieces do not hold, fractions): set here, the workgroups of
  // the pass need not all report it at once
  uint32_t shown = 0;
  float v[2][kSamplePer];
  // (one branch on the type around all loads, which stay in flight together)
  auto fetch = [&](auto zero) {
    using E = decltype(zero);
    E raw[2][kSamplePer];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const E* x = (const E*)(side ? a.queries : a.base);
      const int64_t n = side ? a.nq : a.n;
#pragma unroll
      for (int i = 0; i < kSamplePer; ++i) {
        const uint32_t j = (uint32_t)(i * W + wave);
        const int64_t r = (int64_t)j * n / (kSamplePer * W);
        const uint32_t c = ((j * 2654435761u >> 8) + (tid & 63)) % (uint32_t)a.d;
        raw[side][i] = x[r * a.ld + c];
      }
    }
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int i = 0; i < kSamplePer; ++i) v[side][i] = (float)raw[side][i];
  };
  if (a.f16)
    fetch((_Float16)0.0f);
  else
    fetch(0.0f);
#pragma unroll
  for (int side = 0; side < 2; ++side)
#pragma unroll
    for (int i = 0; i < kSamplePer; ++i) {
      const float x = v[side][i];
      const uint32_t bits = __float_as_uint(x);
      m[side] = fmaxf(m[side], fabsf(x));
      zeros[side] += __popcll(__builtin_amdgcn_ballot_w64(x == 0.0f));
      if (a.unit) {
        if (a.factors && (bits & 0x7fffu)) shown |= kSplitOver9;
        // x = odd 2^low, |x| = man 2^(exponent - 150)
        const uint32_t ex = bits >> 23 & 0xffu;
        const uint32_t man = (bits & 0x7fffffu) | (ex ? 0x800000u : 0u);
        if (man) unit[side] = min(unit[side], (int)max(ex, 1u) - 150 + __builtin_ctz(man));
        continue;
      }
      const float f = __builtin_amdgcn_frexp_mantf(x);  // (+-[1/2, 1))
      if (bits & 0x1fffu) shown |= side ? kSplitQueryLow : kSplitBaseLow;
      if (bits & 0xffu) shown |= side ? kSplitQueryLong : kSplitBaseLong;
      const float rest = f - (float)(_Float16)f;
      if (rest - (float)(_Float16)rest != 0.0f) shown |= kSplitCut;
      if (__float_as_uint(__builtin_amdgcn_fractf(x)) & 0x7fffffffu) shown |= kSplitFrac;
    }
  // Each row's (sum |x|)^2 / (64 sum x^2): 16 rows' sums over the wavefront, lane
  // l % 16 ending with row l % 16 (base rows, then queries)
  float s1[2 * kSamplePer], s2[2 * kSamplePer];
#pragma unroll
  for (int i = 0; i < 2 * kSamplePer; ++i) {
    s1[i] = fabsf(v[i / kSamplePer][i % kSamplePer]);
    s2[i] = s1[i] * s1[i];
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bool up = tid >> b & 1;
#pragma unroll
    for (int i = 0; i < kSamplePer >> b; ++i) {
      const float a1 = up ? s1[2 * i + 1] : s1[2 * i], b1 = up ? s1[2 * i] : s1[2 * i + 1];
      const float a2 = up ? s2[2 * i + 1] : s2[2 * i], b2 = up ? s2[2 * i] : s2[2 * i + 1];
      s1[i] = a1 + __shfl_xor(b1, 1 << b);
      s2[i] = a2 + __shfl_xor(b2, 1 << b);
    }
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    s1[0] += __shfl_xor(s1[0], o);
    s2[0] += __shfl_xor(s2[0], o);
  }
  // (squares past float32's ends: taken as spread evenly)
  const float sq = s1[0] * s1[0];
  float spread = s1[0] == 0.0f ? 0.0f : sq >= 0x1p-100f && sq < 0x1p120f ? sq / (64.0f * s2[0]) : 1.0f;
  float square = s2[0];  // the largest row's
#pragma unroll
  for (int o = 1; o < kSamplePer; o <<= 1) {
    spread += __shfl_xor(spread, o);
    square = fmaxf(square, __shfl_xor(square, o));
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    m[0] = fmaxf(m[0], __shfl_xor(m[0], o));
    m[1] = fmaxf(m[1], __shfl_xor(m[1], o));
    unit[0] = min(unit[0], __shfl_xor(unit[0], o));
    unit[1] = min(unit[1], __shfl_xor(unit[1], o));
    shown |= __shfl_xor(shown, o);
  }
  static_assert(kSamplePer == 8, "lane 8: the first query row's");
  if ((tid & 63) == 0 || (tid & 63) == 8) {
    wspread[tid >> 3 & 1][wave] = spread;
    wsquare[tid >> 3 & 1][wave] = square;
  }
  if ((tid & 63) == 0) {
    for (int side = 0; side < 2; ++side) {
      wmax[side][wave] = m[side];
      wunit[side][wave] = unit[side];
      wzero[side][wave] = zeros[side];
    }
    wflags[wave] = shown;
  }
  __syncthreads();
  // the first wavefront: lane 16 side + w takes wavefront w's of that side (lanes
  // from 32 on repeat them), then lane 0 writes the state
  if (tid >= 64) return;
  static_assert(W == 16, "sixteen lanes a side");
  const int side = tid >> 4 & 1, w = tid & 15;
  float x = wmax[side][w], part = wspread[side][w], sq2 = wsquare[side][w];
  int u = wunit[side][w], z = wzero[side][w];
  uint32_t flags = wflags[w];
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    x = fmaxf(x, __shfl_xor(x, o));
    part += __shfl_xor(part, o);
    sq2 = fmaxf(sq2, __shfl_xor(sq2, o));
    u = min(u, __shfl_xor(u, o));
    z += __shfl_xor(z, o);
    flags |= __shfl_xor(flags, o);
  }
  const float sp = part / (float)(kSamplePer * W);
  const float held = 1.0f - (float)z / (float)(kSamplePer * kSampleThreads);
  const float fix = a.factors ? ldexpf(1.0f, min(-u, 100)) : 1.0f;
  // (a row's sum of squares past 2^24, in these units and with a rounding: what
  // the pass would find)
  if (a.factors && !(sq2 * fix * fix < 0x1p25f)) flags |= kSplitFrac;
  float sc = a.unit ? kUnitScale : 1.0f;
  // both sides past 2^26: every value an integer, no sum exact
  const uint32_t large = !a.unit && x >= 0x1p26f;
  if (!a.unit && x != 0.0f) {  // (a sample of zeros: the pass over all rows decides)
    int e = kMaxSampleExp + 1;
    if (x < INFINITY) (void)frexpf(x, &e);  // x = f 2^e, f in [1/2, 1)
    if (e < -kMaxSampleExp || e > kMaxSampleExp)
      flags |= kSplitRows32;
    else
      sc = ldexpf(1.0f, kSampleExp + 1 - e);
  }
  flags |= __shfl_xor(flags, 16);
  const float sp_q = __shfl_xor(sp, 16), held_q = __shfl_xor(held, 16);
  const float sc_q = __shfl_xor(sc, 16), fix_q = __shfl_xor(fix, 16);
  const uint32_t large_q = __shfl_xor(large, 16);
  if (tid != 0) return;
  if (a.d < (a.l2 ? kSplitShortL2 : kSplitShortDot) ||
      split_few_terms(a.d, a.l2, (float)a.d * sp * sp_q * kSplitNormalSpread, held * held_q))
    flags |= kSplitShort;
  if (a.unit) flags |= a.factors ? kSplitFactors : kSplitFrac;
  if (large && large_q) flags |= kSplitFrac;
  const float cap = split_cap(a.d);
  SplitState st;
  st.flags = flags;
  st.sbase = sc;
  st.squery = sc_q;
  st.inv = 1.0f / (sc * sc_q);  // powers of two: exact
  // (the largest values, sums and losses that dense rows reach: only rows past
  // them are reported)
  st.cap = cap;
  st.room = (float)a.d * cap;
  st.fix[0] = fix;
  st.fix[1] = fix_q;
  for (int i = 0; i < 2; ++i) {
    st.lost[i] = 0x1p-25f;
    st.top[i] = 0x1p12f;
    st.least[i] = 0.75f * (float)a.d * cap;
  }
  *a.st = st;
}

// 256 rows per workgroup, a 32-value slab at a time through LDS: fetched with
// coalesced loads (VEC: 16 bytes a lane; else a value a lane), summed row by
// row in the order of row_norms_kernel (the norms are those), and turned into
// pieces eight values a thread, 64 contiguous bytes a row and piece.  HBM
// bound: each row is read once and written once (4 bytes a value both ways).
// Workgroups [0, na) take the base rows, [na, na + nb) the queries, the rest
// the shared bounds.
template <bool F16, bool VEC>
__global__ __launch_bounds__(256) void split_rows_kernel(SplitRowsArgs ab, SplitRowsArgs aq,
                                                         BoundsInit bi, uint32_t na, uint32_t nb) {
  constexpr int SS = 36;  // LDS row stride (floats), as row_norms_kernel
  __shared__ __align__(16) float sh[256 * SS];
  if (blockIdx.x >= na + nb) {
    init_bounds(bi, blockIdx.x - na - nb);
    return;
  }
  const SplitRowsArgs& a = blockIdx.x < na ? ab : aq;
  const int tid = threadIdx.x;
  const int64_t row0 = (int64_t)(blockIdx.x < na ? blockIdx.x : blockIdx.x - na) * 256;
  // Once the rows are known to take the float32 route their pieces are not
  // made, and only the norms are left to do (an outlier halfway through
  // 500k x 768 rows, 700 queries: 5.15 -> 5.09 ms a call, float32 alone 4.69).
  // (one thread's view for the whole workgroup, behind the loop's first barrier)
  __shared__ bool s_rows32;
  if (threadIdx.x == 0) {
    const uint32_t known =
        __hip_atomic_load(&a.st->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_rows32 = (known & kSplitRows32) ||
               ((known & kSplitShort) && (known & (kSplitBaseLow | kSplitQueryLow)));
  }
  const float scale = a.query ? a.st->squery : a.st->sbase;
  const float seed_scale = a.st->sbase * a.st->squery;
  const float cap = a.st->cap;
  const float fix = a.st->fix[a.query];
  // (the values' own bits are looked at while the state does not show what they
  // would)
  const bool factors = a.st->flags & kSplitFactors;
  const uint32_t shown = kSplitFrac | (factors ? kSplitOver9 : 0u);
  const bool look = (a.st->flags & shown) != shown;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  constexpr int EPV = F16 ? 8 : 4;
  constexpr int VPR = 32 / EPV;
  float pv[VEC ? VPR : 32][VEC ? EPV : 1];
  auto load_slab = [&](int c0) {
    if constexpr (VEC) {
#pragma unroll
      for (int j = 0; j < VPR; ++j) {
        const int e = tid + 256 * j;
        const int r = e / VPR, c = (e % VPR) * EPV;
        const int64_t row = row0 + r;
        if (row < a.n && c0 + c < a.d) {
          if constexpr (F16) {
            const halfx8 hv = *(const halfx8*)((const _Float16*)a.x + row * a.ld + c0 + c);
#pragma unroll
            for (int u = 0; u < 8; ++u) pv[j][u] = (float)hv[u];
          } else {
            const floatx4 f = *(const floatx4*)((const float*)a.x + row * a.ld + c0 + c);
#pragma unroll
            for (int u = 0; u < 4; ++u) pv[j][u] = f[u];
          }
        } else {
#pragma unroll
          for (int u = 0; u < EPV; ++u) pv[j][u] = 0.0f;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const int e = tid + 256 * j;
        const int r = e >> 5, c = c0 + (e & 31);
        const int64_t row = row0 + r;
        float v = 0.0f;
        if (row < a.n && c < a.d)
          v = F16 ? (float)((const _Float16*)a.x)[row * a.ld + c]
                  : ((const float*)a.x)[row * a.ld + c];
        pv[j][0] = v;
      }
    }
  };
  // pieces: thread t converts values 8 (t % 4) .. + 7 of rows t / 4 + 64 j
  // (rows' errors past rounding and what they are held against, SplitState;
  // L2: both squared)
  float lost[4] = {0, 0, 0, 0}, mass[4] = {0, 0, 0, 0}, top = 0.0f;
  // (what the flags need is gathered as ORs of bits, one operation a value:
  // with compares and selects instead the pass was bound by them, 500k x 768
  // cosine, 2,000 queries 5.25 ms a call against 5.10)
  uint32_t lowbits = 0;   // of the lo pieces, two a word
  uint32_t cutbits = 0;   // of what the pieces leave out: bit 30 (2 and above) only if
                          // a value is past binary16's range or not finite
  uint32_t fracbits = 0;  // of the values' fractions
  uint32_t rawbits = 0;   // of the values (unit rows)
  bool rows32_seen = false;
  load_slab(0);
  for (int c0 = 0; c0 < a.out_ld; c0 += 32) {
    if constexpr (VEC) {
#pragma unroll
      for (int j = 0; j < VPR; ++j) {
        const int e = tid + 256 * j;
        const int r = e / VPR, c = (e % VPR) * EPV;
#pragma unroll
        for (int u = 0; u < EPV; u += 4)
          *(floatx4*)&sh[r * SS + c + u] = floatx4{pv[j][u], pv[j][u + 1], pv[j][u + 2], pv[j][u + 3]};
      }
    } else {
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const int e = tid + 256 * j;
        sh[(e >> 5) * SS + (e & 31)] = pv[j][0];
      }
    }
    if (c0 + 32 < a.out_ld) load_slab(c0 + 32);
    __syncthreads();
    const bool rows32 = s_rows32;
    if (rows32 && !a.norm && !a.seed) return;
    if (a.norm || a.seed) {
#pragma unroll
      for (int j4 = 0; j4 < 32; j4 += 4) {
        const floatx4 v = *(const floatx4*)&sh[tid * SS + j4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (c0 + j4 + u < a.d) acc[(j4 + u) & 7] += v[u] * v[u];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = (tid >> 2) + 64 * j, c = 8 * (tid & 3);
      const int64_t row = row0 + r;
      if (rows32 || row >= a.n || c0 + c >= a.out_ld) continue;
      float x[8];
      *(floatx4*)&x[0] = *(const floatx4*)&sh[r * SS + c];
      *(floatx4*)&x[4] = *(const floatx4*)&sh[r * SS + c + 4];
      if (look && !a.unit_norms) {
#pragma unroll
        for (int u = 0; u < 8; ++u) fracbits |= __float_as_uint(__builtin_amdgcn_fractf(x[u]));
      } else if (look) {
        // (in units of the side's, SplitState::fix)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          fracbits |= __float_as_uint(__builtin_amdgcn_fractf(x[u] * fix));
          rawbits |= __float_as_uint(x[u]);
        }
        const float nn = a.unit_norms[row];
        if (!(nn * fix * fix < 0x1p24f)) fracbits = 1u;  // (the sums may pass 2^24)
      }
      if (a.unit_norms) {
        const float nn = a.unit_norms[row];
        const float nrm = sqrtf(nn);
        const float den = nrm > 1e-30f ? nrm : 1e-30f;
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = x[u] / den;
      }
      halfx8 hi, lo;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float xs = x[u] * scale, ax = fabsf(xs);
        const _Float16 hv = (_Float16)xs;
        const float rest = xs - (float)hv;  // exact
        const _Float16 lv = (_Float16)rest;
        hi[u] = hv;
        lo[u] = lv;
        float err = fabsf(rest - (float)lv);  // exact
        if (scale < 1.0f && xs == 0.0f && x[u] != 0.0f) err = 0x1p-25f;  // (underflow)
        cutbits |= __float_as_uint(err);
        // (from 2^-2 on at most a last bit)
        if (!(ax < 0.25f)) err = 0.0f;
        if (a.l2) {
          lost[j] = __builtin_fmaf(err, err, lost[j]);
          mass[j] = __builtin_fmaf(xs, xs, mass[j]);
        } else {
          lost[j] += err;
          mass[j] += fminf(ax, cap);
          top = fmaxf(top, ax);
        }
      }
      {
        const u32x4 lw = __builtin_bit_cast(u32x4, lo);
        lowbits |= (lw[0] | lw[1]) | (lw[2] | lw[3]);
      }
      // (interleaved: a run of hi pieces, then their lo pieces)
      constexpr int R = kTilePieceRun;
      const int cc = c0 + c;
      uint16_t* dh = a.lo ? a.hi + row * a.out_ld + cc
                          : a.hi + row * 2 * a.out_ld + cc / R * (2 * R) + cc % R;
      uint16_t* dl = a.lo ? a.lo + row * a.out_ld + cc : dh + R;
      *(u32x4*)dh = __builtin_bit_cast(u32x4, hi);
      *(u32x4*)dl = __builtin_bit_cast(u32x4, lo);
    }
    __syncthreads();
  }
  // each row's four threads' sums (a row past the end: zeros)
  float worst = 0.0f, least = INFINITY;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float l = lost[j], m = mass[j];
    l += __shfl_xor(l, 1);
    m += __shfl_xor(m, 1);
    l += __shfl_xor(l, 2);
    m += __shfl_xor(m, 2);
    if (a.l2) {
      if (l > 0x1p-50f * m) rows32_seen = true;
    } else {
      worst = fmaxf(worst, l);
      if (m > 0.0f || l > 0.0f) least = fminf(least, m);
    }
  }
  if ((a.norm || a.seed) && row0 + tid < a.n) {
    const float s01 = acc[0] + acc[1], s23 = acc[2] + acc[3];
    const float s45 = acc[4] + acc[5], s67 = acc[6] + acc[7];
    const float nn = (s01 + s23) + (s45 + s67);
    // (squared norms near the ends of float32: their sums are not the
    // scaled ones)
    if (!(nn < 0x1p100f) || (nn > 0.0f && nn < 0x1p-100f)) rows32_seen = true;
    const float half = nn > 0.0f ? -0.5f * nn : 0.0f;  // (+0, as row_norms_kernel)
    if (a.norm) a.norm[row0 + tid] = a.half_neg ? half : nn;
    if (a.seed) a.seed[row0 + tid] = half * seed_scale;
  }
  // One report a workgroup, and only of what the state does not show yet: the
  // workgroups of a small call end together, and their atomics on one line
  // would serialise (a wavefront's own values each: 76,775 x 78 rows, inner
  // product, 125 us of preparation against 64).  (A lo piece's sign does not
  // count; more than five bits of one: a value of more than 16.)
  auto any_of = [](bool b) { return __builtin_amdgcn_ballot_w64(b) != 0; };
  const uint32_t any =
      (any_of(lowbits & 0x7fff7fffu) ? (a.query ? kSplitQueryLow : kSplitBaseLow) : 0u) |
      (any_of(lowbits & 0x003f003fu) ? (a.query ? kSplitQueryLong : kSplitBaseLong) : 0u) |
      (any_of(rows32_seen || (cutbits & 0x40000000u)) ? kSplitRows32 : 0u) |
      (any_of(fracbits & 0x7fffffffu) ? kSplitFrac : 0u) |
      (any_of(rawbits & 0x7fffu) ? kSplitOver9 : 0u) | (any_of(cutbits) ? kSplitCut : 0u) |
      (any_of(worst > 0.0f) ? (a.query ? kSplitQueryLoss : kSplitBaseLoss) : 0u);
  __shared__ uint32_t rflags[4];
  __shared__ float red[3][4];
  if (!a.l2) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      worst = fmaxf(worst, __shfl_xor(worst, o));
      least = fminf(least, __shfl_xor(least, o));
      top = fmaxf(top, __shfl_xor(top, o));
    }
  }
  if ((tid & 63) == 0) {
    rflags[tid >> 6] = any;
    red[0][tid >> 6] = worst;
    red[1][tid >> 6] = top;
    red[2][tid >> 6] = least;
  }
  __syncthreads();
  if (tid != 0) return;
  SplitState* st = a.st;
  auto word = [](const void* p) {
    return __hip_atomic_load((const unsigned*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const uint32_t all = (rflags[0] | rflags[1]) | (rflags[2] | rflags[3]);
  if (all & ~word(&st->flags))
    __hip_atomic_fetch_or(&st->flags, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (a.l2) return;
  // (not negative: their bits order as they do)
  const unsigned w = __float_as_uint(fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3])));
  const unsigned t = __float_as_uint(fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3])));
  const unsigned l = __float_as_uint(fminf(fminf(red[2][0], red[2][1]), fminf(red[2][2], red[2][3])));
  if (w > word(&st->lost[a.query]))
    __hip_atomic_fetch_max((unsigned*)&st->lost[a.query], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (t > word(&st->top[a.query]))
    __hip_atomic_fetch_max((unsigned*)&st->top[a.query], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (l < word(&st->least[a.query]))
    __hip_atomic_fetch_min((unsigned*)&st->least[a.query], l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

hipError_t launch_split_init(const SplitInitArgs& a, hipStream_t s) {
  if (a.n < 1 || a.nq < 1 || a.d < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(split_init_kernel, dim3(1), dim3(kSampleThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_split_rows(const SplitRowsArgs& base, const SplitRowsArgs& queries,
                             const BoundsInit& bi, hipStream_t s) {
  if (base.n < 1 || queries.n < 1 || base.f16 != queries.f16) return hipErrorInvalidValue;
  bool vec = true;
  for (const SplitRowsArgs* a : {&base, &queries}) {
    if (a->out_ld % (a->lo ? 8 : kTilePieceRun) != 0 || a->out_ld < a->d) return hipErrorInvalidValue;
    const int esize = a->f16 ? 2 : 4;
    vec = vec && (uintptr_t)a->x % 16 == 0 && ((int64_t)a->ld * esize) % 16 == 0 &&
          (a->d * esize) % 16 == 0;
  }
  const unsigned na = (unsigned)((base.n + 255) / 256), nb = (unsigned)((queries.n + 255) / 256);
  const dim3 grid(na + nb + bounds_blocks(bi));
  if (base.f16) {
    if (vec) hipLaunchKernelGGL((split_rows_kernel<true, true>), grid, dim3(256), 0, s, base, queries, bi, na, nb);
    else hipLaunchKernelGGL((split_rows_kernel<true, false>), grid, dim3(256), 0, s, base, queries, bi, na, nb);
  } else {
    if (vec) hipLaunchKernelGGL((split_rows_kernel<false, true>), grid, dim3(256), 0, s, base, queries, bi, na, nb);
    else hipLaunchKernelGGL((split_rows_kernel<false, false>), grid, dim3(256), 0, s, base, queries, bi, na, nb);
  }
  return hipGetLastError();
}

}  // namespace mlxvs::kern
