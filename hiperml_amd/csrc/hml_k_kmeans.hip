// hml_k_kmeans.hip -- k-means nearest-centroid assignment on gfx950.
//
// Replaces the reference's assign kernels hmlKmeansAssignCtrdSmem /
// SmemUnroll / Gmem (include/hml_kmeans_kernel_template.h:18-88, 90-316,
// 323-367), which give each thread one row and loop over every centroid
// with scalar FMAs.  Their result is defined by that arithmetic: per
// centroid k ascending, dist = sum over dims ascending of delta*delta
// (delta = x - c, one rounding per step), first k strictly below the
// running minimum (from FLT_MAX).  Same result here, different machine:
//
//  1. Screening on the 16-bit matrix cores.  |x - c|^2 = |x|^2 - 2 a_k with
//     a_k = x.c_k - |c_k|^2 / 2, and x.c_k for 32 rows against 32 centroids
//     is a product of fp16 terms x = xh + xl, c = ch + cl (round to nearest,
//     22 bits together): three v_mfma_f32_32x32x16_f16 per 16 dims (cl.xh,
//     ch.xl, ch.xh), the accumulator starting at -|c|^2 / 2.  Rows and
//     centroids are taken relative to a point amid the centroids (when the
//     origin is not amid them) and scaled by one power of two that brings them
//     to about 1, both from a sample of 8; what then leaves the range of fp16
//     is compared exactly.  FP32 MFMAs would take 5 times as long for the same
//     dims; their rms error against 64 bits is 0.97e-7 (32 dims, clustered
//     rows), that of the terms 1.17e-7 (64 dims, |x| >> |c|: 1.5e-7 and
//     0.8e-7).  Two bf16 terms, 16 bits together, are off by up to
//     2^-15 |x||c|.
//  2. A bound on how far the reference's float distance can be from
//     |x|^2 - 2 a~_k (the screened value).  With u = 2^-24, X = |x|, C >=
//     |c_k|, q = X C + C^2 / 2 (which bounds the partial sums of a_k), KS =
//     D / 16 rounded up, all moved and scaled, a~_k is off by at most u times
//       2 q                 moving the values, a rounding each
//       12 X C + 4 (X + C)  the terms: a residual is at most 2^-11 of the
//                           value and rounds at 2^-22 of it or, below fp16's
//                           normal range, at 2^-25; xl.cl (2^-22) is left out
//       96 KS q             the accumulation of 48 KS products, 2 u of the
//                           partial sums' bound each
//       (4 KS + 1) C^2      the norm: 8 KS + 2 roundings of C^2 / 2
//       30 q                the index kept in the low 4 bits of a~_k
//     and the reference's distance by (D + 3) u of itself (D additions, the
//     square twice the difference's rounding).  If k is the reference's
//     argmin and j has the largest a~, then a~_k >= a~_j - M, and with X C <=
//     (X^2 + C^2) / 2, X + C <= (X^2 + C^2) / 2 + 1
//       M = (D + 4) u d + u ((96 KS + 48) X^2 + (200 KS + 82) C^2 + 8)
//     d bounding the distance of j: (1 + 2^-9) ||x|^2 - 2 a~_j| + 3 2^-11 X^2 +
//     2^-20 max |c| + 2^-31 (its error is below 2^-10 X^2 + 2^-20 (X + max |c|),
//     and 2^-20 X below 2^-11 X^2 + 2^-31).  Neither j nor k is then farther
//     from x than sqrt(d), so C^2 = (X + sqrt(d))^2 <= 2 (X^2 + d) will do where
//     that is less than max |c|^2: a few far centroids do not widen the margin
//     of the others' rows.  Only centroids with a~_k >= max a~ - M can be the
//     exact argmin.
//  3. Each lane keeps the two largest a~ of its even and of its odd centroid
//     tiles.  If a row's second largest value lies below the limit its
//     argmin is known (the usual case: no distance is computed).  Otherwise
//     the trackers' centroids above the limit or, when a value that no tracker
//     names could be above it, all centroids above it (found by screening the
//     tile again) are compared by the reference's own arithmetic.  A wave
//     gathers such (row, centroid) pairs over its lanes and compares 64 at a
//     time, a lane each; the smallest (distance, index) of a row is the
//     reference's "first strict minimum".  Each lane on its own candidates in
//     turn waited for memory once per candidate of the busiest lane: 0/1
//     features, 2^20 rows 32 x 64, 135 us, now 61.
//
// What bounds it: for few centroids the row stream (2^24 rows, 32 dims x 16
// clusters: 0.39 ms, 5.6 TB/s), for many the matrix cores and the three vector
// instructions per (row, centroid) of the trackers.  Where rows have no
// clusters, more have pairs to compare.  2^24 rows, ms, clustered / uniform: 32
// x 64 0.45 / 0.49 (FP32 products 1.04 clustered), 64 x 64 0.93 / 1.00 (1.75),
// 32 x 256 1.08 / 1.13 (3.08), 16 x 256 0.80 / 0.80; 2^23 rows 64 x 256 0.99 /
// 1.03 (3.11).  64 rows per wave halve the LDS reads per row but held 2-3 waves
// per SIMD: 2-15% slower.  Four trackers per lane make the second screening
// rarer and cost registers: up to 10% slower.
//
// Centroids live in LDS as fp16 terms in MFMA operand order (a fragment is
// one conflict-free 16-byte read per lane) beside their norms, staged once
// per workgroup when they fit, else chunk by chunk per row step with the
// workgroup's waves in lockstep.  Every wave streams its rows 32 at a time
// straight into its own LDS area (buffer_load ... lds), the next tile's load
// in flight while this one is screened.
#include <float.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "hml_internal.h"
#include "hml_kdev.h"

namespace hml {
namespace {

constexpr uint32_t kNone = 0xffffffffu;

// s_waitcnt immediates (gfx9 encoding): vmcnt(0) lgkmcnt(0), and lgkmcnt(0)
constexpr int kWaitAll = 0x0070;
constexpr int kWaitLgkm0 = 0xC07F;

struct KmParams {
  const float *rows;
  const float *ctrds;
  uint32_t *assign;
  int64_t nrows;
  int64_t steps;  // row steps of kKmWaves wave tiles per workgroup (uniform)
  int32_t D, K;
  int32_t KC;     // centroids per LDS chunk (screened: a multiple of 32)
  int32_t xfloats;  // screened: floats of one wave's row tile in LDS
};

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool FUSED>
__device__ __forceinline__ float exact_step(float dist, float x, float c) {
  const float delta = x - c;
  if (FUSED) return __builtin_fmaf(delta, delta, dist);
  {
#pragma clang fp contract(off)
    const float sq = delta * delta;
    return dist + sq;
  }
}

// Reference distance of row xr to centroid cr, both in global memory at any
// 4-byte alignment; 16 dims of each are loaded before their arithmetic.
struct __attribute__((packed, aligned(4))) KmQuad {
  float v[4];
};
template <bool FUSED, int KS>
__device__ __forceinline__ float exact_dist(const float *__restrict__ xr,
                                            const float *__restrict__ cr, int D) {
  float dist = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    KmQuad xv[4], cv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (16 * s + 4 * j + 4 <= D) {
        xv[j] = *reinterpret_cast<const KmQuad *>(xr + 16 * s + 4 * j);
        cv[j] = *reinterpret_cast<const KmQuad *>(cr + 16 * s + 4 * j);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (16 * s + 4 * j + 4 <= D) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dist = exact_step<FUSED>(dist, xv[j].v[e], cv[j].v[e]);
      }
  }
  for (int d = D & ~3; d < D; ++d) dist = exact_step<FUSED>(dist, xr[d], cr[d]);
  return dist;
}

// Largest of the lanes' values (none negative), the same in every lane:
// rotations within rows of 16 lanes, then the four rows.
__device__ __forceinline__ float wave_max(float x) {
#define KM_ROR(n) \
  __builtin_fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + n, 0xf, 0xf, true)))
  x = KM_ROR(1);
  x = KM_ROR(2);
  x = KM_ROR(4);
  x = KM_ROR(8);
#undef KM_ROR
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < 64; i += 16)
    m = __builtin_fmaxf(m, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i)));
  return m;
}

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

// hi / lo fp16 terms of 8 floats (round to nearest; the residual is exact)
__device__ __forceinline__ void split8(const float (&v)[8], h8 &hi, h8 &lo) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const h2 h = __builtin_convertvector(f2{v[j], v[j + 1]}, h2);
    hi[j] = h[0];
    hi[j + 1] = h[1];
    const h2 l = __builtin_convertvector(f2{v[j] - (float)h[0], v[j + 1] - (float)h[1]}, h2);
    lo[j] = l[0];
    lo[j + 1] = l[1];
  }
}

// Scaled squared norms at or above kKmNormMax (and NaN) take a centroid out
// of the screen; rows that could still choose it (|x|^2 or the best screened
// distance not below kKmRowMax), or whose distances could overflow
// (kKmDistMax, unscaled), are refined over every centroid.
constexpr float kKmNormMax = 0x1p30f;
constexpr float kKmRowMax = 0x1p26f;
constexpr float kKmDistMax = 0x1p118f;
// screen value of an excluded or padding centroid
constexpr float kKmExcluded = -1e38f;
constexpr float kKmSampleMax = 0x1p60f;
// LDS before the centroids: the sample (later the pairs to compare), the
// point, the rows' best keys and the pairs' rows
constexpr int kKmHeadBytes = (2 * kKmWaves + 1) * 256 + kKmWaves * 64;

// KS = k-steps of 16 dims, MULTI = the centroids take several LDS chunks,
// VEC = dims a multiple of 4.  ROOMY: LDS holds one workgroup per CU, two
// waves per SIMD, which may use 256 registers (64 dims need 150 to 180; capped
// at 128, several chunks spilled 19 and took 37 us instead of 33 for 32768 rows
// 64 x 512, one chunk spills 1 to 8).
template <int KS, bool MULTI, bool VEC, bool FUSED, bool ROOMY = MULTI>
__global__ __launch_bounds__(64 * kKmWaves, ROOMY ? 2 : 4) void k_kmeans_screen(KmParams p) {
  constexpr int NQ = KS * 2;  // 1 KB DMA loads per row tile (at most)
  extern __shared__ f4 km_lds4[];
  char *lds = reinterpret_cast<char *>(km_lds4);
  float *smp = reinterpret_cast<float *>(lds), *mus = smp + 64 * kKmWaves;
  h8 *cf = reinterpret_cast<h8 *>(lds + kKmHeadBytes);  // centroid fragments
  float *nrm = reinterpret_cast<float *>(lds + kKmHeadBytes + (size_t)p.KC * KS * 64);  // -|c|^2 / 2
  // max as a median with infinity (in a register the compiler does not see
  // through), without the canonicalising moves fmaxf needs for unknown
  // inputs; a result that a NaN could have entered is never used
  float inf;
  asm("s_mov_b32 %0, 0x7f800000" : "=s"(inf));
  auto vmax = [&](float a, float b) { return __builtin_amdgcn_fmed3f(a, b, inf); };
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int D = p.D, K = p.K;
  float *xs = nrm + p.KC + w * p.xfloats;  // this wave's row tile
  // this wave's pairs to compare (the sample's row, once that is used) and
  // the best of each of its rows
  int *pair_k = reinterpret_cast<int *>(smp + 64 * w);
  unsigned long long *best = reinterpret_cast<unsigned long long *>(lds + (kKmWaves + 1) * 256) + 32 * w;
  uint8_t *pair_r = reinterpret_cast<uint8_t *>(lds + (2 * kKmWaves + 1) * 256) + 64 * w;
  const int h = lane >> 5, r = lane & 31;
  const int nchunks = MULTI ? (K + p.KC - 1) / p.KC : 1;
  // The point that rows and centroids are moved by, and the scale, a power of
  // two, from a sample of centroids, one per wave: per dim a middle value (a
  // median of medians) and, over the dims, the largest distance from it but
  // for one extreme in each group of three.  Centroids that lie about the
  // origin, no dim's middle farther from it than that, stay (moving each row
  // costs LDS reads, and the middle of 8 is off by as much), and where they are
  // of a size of 1/2 to 64 nothing is scaled either.  The sample is
  // exchanged through LDS (smp, a row of 64 dims each): the loads start here,
  // the exchange shares the barrier that staging the centroids begins with.
  // Every wave then writes the same -point x scale to mus.
  const float mine = lane < D ? p.ctrds[(int64_t)((uint64_t)w * (uint32_t)K / kKmWaves) * D + lane] : 0.f;
  float sc = 1.f;
  bool moved = false;  // or scaled
  auto set_scale = [&]() {
    static_assert(kKmWaves == 8, "groups of a sample of 8");
    float v[kKmWaves];
#pragma unroll
    for (int i = 0; i < kKmWaves; ++i) v[i] = smp[64 * i + lane];
    auto med = [](float a, float b, float c) { return __builtin_amdgcn_fmed3f(a, b, c); };
    float mid = med(med(v[0], v[1], v[2]), med(v[3], v[4], v[5]), 0.5f * v[6] + 0.5f * v[7]);
    float far = 0.f;
#pragma unroll
    for (int i = 0; i < kKmWaves; ++i) {
      v[i] = __builtin_fabsf(v[i] - mid);
      far = __builtin_fmaxf(far, v[i]);
    }
    const float dev = __builtin_fmaxf(__builtin_fmaxf(med(v[0], v[1], v[2]), med(v[3], v[4], v[5])),
                                      __builtin_fminf(v[6], v[7]));
    const float at = wave_max(__builtin_fabsf(mid));
    float big = wave_max(dev);
    const bool off = at > big;
    if (!off) mid = 0.f;
    // without any spread all of the sample's, else the point's own size
    if (!(big > 0.f)) big = wave_max(far);
    if (!(big > 0.f)) big = at;
    int ex = min(max((int)(__float_as_uint(big) >> 23) - 127, -60), 60);
    moved = off || ex < -1 || ex > 5;
    if (!moved) ex = 0;
    sc = __uint_as_float((uint32_t)(127 - ex) << 23);
    mus[lane] = -mid * sc;
    wave_lds_sync();
  };
  // margin factors, see the error terms at the top of the file (2^-7 for the
  // second order and the margin's own roundings)
  constexpr float kU = 0x1p-24f * (1.0f + 0x1p-7f);
  constexpr float kMx = (96 * KS + 48) * kU, kMc = (200 * KS + 82) * kU;
  const float md = (float)(D + 4) * kU;

  // Stages centroids c0 .. c0 + KC - 1 (zeros past K) and returns the
  // largest |c|^2 among those in the screen.  Lanes l and l ^ 32 hold the two
  // halves of a centroid's dims, in the fragment layout itself: (tile of 32,
  // k-step, hi / lo, lane, 8 dims).
  auto stage = [&](int c0) -> float {
    float v[KS][8];
    auto load = [&](int i) {  // the 8 KS dims of thread item i
      const int k = 32 * (i >> 6) + r;
      const float *c = p.ctrds + (int64_t)(c0 + k) * D + 8 * h;
      const int n = i < p.KC * 2 && c0 + k < K ? D - 8 * h : 0;  // floats at c
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          // 16 bytes at a time: element loads are 64 lines each, 10 us per
          // chunk of 350 centroids of 64 dims
          KmQuad q = {};
          if (16 * s + j + 4 <= n)
            q = *reinterpret_cast<const KmQuad *>(c + 16 * s + j);
          else if (!VEC)
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (16 * s + j + e < n) q.v[e] = c[16 * s + j + e];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[s][j + e] = q.v[e];
        }
    };
    if (!MULTI) load(threadIdx.x);
    __syncthreads();  // every wave is done with the previous chunk, or has its sample in LDS
    if (!MULTI) set_scale();
    for (int i = threadIdx.x; i < p.KC * 2; i += 64 * kKmWaves) {
      const int t = i >> 6, k = 32 * t + r;
      if (MULTI || i != (int)threadIdx.x) load(i);
      float s2 = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          v[s][j] = __builtin_fmaf(v[s][j], sc, mus[16 * s + 8 * h + j]);  // zero past D
          s2 = __builtin_fmaf(v[s][j], v[s][j], s2);
        }
      s2 += __shfl_xor(s2, 32);
      const bool in = c0 + k < K && s2 < kKmNormMax;
      if (h == 0) nrm[k] = in ? -0.5f * s2 : kKmExcluded;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (!in) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[s][j] = 0.f;
        }
        h8 hi, lo;
        split8(v[s], hi, lo);
        cf[(t * KS + s) * 128 + lane] = hi;
        cf[(t * KS + s) * 128 + 64 + lane] = lo;
      }
    }
    __syncthreads();
    float mx = 0.f;  // the largest |c|^2 in the screen
    for (int k = lane; k < p.KC; k += 64) {
      const float n2 = nrm[k];
      mx = n2 > 0.5f * kKmExcluded ? __builtin_fmaxf(mx, -2.0f * n2) : mx;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, off));
    return mx;
  };

  // The wave's 32 rows are one contiguous block of memory, DMAed flat
  // into the wave's LDS tile.  With D a multiple of 4, row x's 16-byte chunk
  // c goes to chunk x nc + (c + x nc / 16) % nc (nc = D / 4), which spreads
  // 8 consecutive rows' reads of one chunk over distinct banks; otherwise
  // the block is stored as it is and read float by float.
  const int nc = D >> 2;
  const int nchunk16 = 8 * D;  // 16-byte chunks of the tile
  uint32_t aoff[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int pos = 64 * q + lane;
    int src = pos;
    if (VEC) {
      const int x = pos / nc, sl = pos - x * nc;
      int c = sl - ((x * nc) >> 4) % nc;
      if (c < 0) c += nc;
      src = x * nc + c;
    }
    aoff[q] = pos < nchunk16 ? (uint32_t)src * 16u : kOOB;
  }
  // LDS offsets (floats) of this lane's chunks: dims 16 s + 8 h + 4 j .. +3
  // of row r
  int xo[VEC ? 2 * KS : 1];
  if (VEC) {
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      int c = 4 * (i >> 1) + 2 * h + (i & 1);
      if (c >= nc) c = 0;  // past the row: masked
      xo[i] = 4 * (r * nc + (c + ((r * nc) >> 4)) % nc);
    }
  } else {
    xo[0] = r * D + 8 * h;
  }

  const int64_t wstep = (int64_t)gridDim.x * kKmWaves;
  int64_t tile = (int64_t)blockIdx.x * kKmWaves + w;
  // rows of a tile into the wave's LDS area (its earlier reads are done)
  auto load_rows = [&](int64_t tl) {
    const int64_t row0 = tl * 32;
    if (row0 >= p.nrows) return;
    const float *base = p.rows + row0 * D;
    if (row0 + 32 <= p.nrows) {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(base, 32 * D * 4);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if (64 * q < nchunk16) buf_load_lds16<kBufNT>(rs, xs + 256 * q, aoff[q], 0);
    } else {
      const int n = (int)(p.nrows - row0) * D;
      for (int i = lane; i < n; i += 64) {
        int o = i;
        if (VEC) {
          const int x = i / D, d = i - x * D;
          o = 4 * (x * nc + ((d >> 2) + ((x * nc) >> 4)) % nc) + (d & 3);
        }
        xs[o] = base[i];
      }
    }
  };

  load_rows(tile);
  float cmax2 = 0.f;  // largest |c|^2 so far
  smp[64 * w + lane] = __builtin_fabsf(mine) < kKmSampleMax ? mine : 0.f;
  if (!MULTI) {
    cmax2 = stage(0);
  } else {
    __syncthreads();
    set_scale();
  }
  // absolute terms of M (8 u, and underflow: in the screen and, D 2^-149
  // unscaled, in the reference) and the largest row in range
  const float m0 = __builtin_fmaf((float)D * 0x1p-148f * sc, sc, 8 * kU);
  const float rmax = __builtin_fminf(kKmRowMax, kKmDistMax * sc * sc);

  // the row steps; rows that stay as they are have a loop of their own
  auto steps = [&](auto move) {
    for (int64_t st = 0; st < p.steps; ++st, tile += wstep) {
      const int64_t row0 = tile * 32;
      const bool live = row0 < p.nrows;  // wave-uniform
      if (!MULTI && !live) break;        // later steps only go further

      h8 xh[KS], xl[KS];
      float xx = 0.f;
      if (!MULTI || live) {
        __builtin_amdgcn_s_waitcnt(kWaitAll);  // the tile is in LDS
        __builtin_amdgcn_sched_barrier(0);
        wave_lds_sync();
        float v[KS][8];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          if (VEC) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const f4 q = *reinterpret_cast<const f4 *>(xs + xo[2 * s + j]);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[s][4 * j + e] = q[e];
            }
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[s][j] = xs[xo[0] + 16 * s + j];
          }
        }
        wave_lds_sync();
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);  // the reads above are done
        __builtin_amdgcn_sched_barrier(0);
        load_rows(tile + wstep);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(move)::value) {
#pragma unroll
          for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const f4 q = *reinterpret_cast<const f4 *>(mus + 16 * s + 8 * h + 4 * j);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[s][4 * j + e] = __builtin_fmaf(v[s][4 * j + e], sc, q[e]);
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (s == KS - 1) v[s][j] = 16 * s + 8 * h + j < D ? v[s][j] : 0.f;
            xx = __builtin_fmaf(v[s][j], v[s][j], xx);
          }
          split8(v[s], xh[s], xl[s]);
        }
        xx += __shfl_xor(xx, 32);
      }

      // lane (h, r), entry i: x.c - |c|^2 / 2 for row r and centroid
      // 32 tl + 8 (i / 4) + 4 h + i % 4 of the chunk
      auto screen_tile = [&](int tl) -> f16v {
        f16v acc;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f4 q = *reinterpret_cast<const f4 *>(nrm + 32 * tl + 8 * i + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * i + e] = q[e];
        }
        const h8 *f = cf + tl * KS * 128 + lane;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const h8 ch = f[s * 128], cl = f[s * 128 + 64];
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(cl, xh[s], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ch, xl[s], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ch, xh[s], acc, 0, 0, 0);
        }
        return acc;
      };

      // The two largest screen values of each lane's even (g = 0) and odd
      // centroid tiles.  The entry's index in its tile sits in the low 4 bits
      // of the value; bk holds the first centroid of the largest's tile.
      float m1[2], m2[2];
      int bk[2] = {0, 0};
#pragma unroll
      for (int g = 0; g < 2; ++g) m1[g] = m2[g] = 2.f * kKmExcluded;
      for (int c = 0; c < nchunks; ++c) {
        if (MULTI) {
          const float cm = stage(c * p.KC);
          cmax2 = __builtin_fmaxf(cmax2, cm);
          if (!live) continue;
        }
        const int k0 = c * p.KC;
        const int ntl = (min(p.KC, K - k0) + 31) >> 5;
        for (int tl = 0; tl < ntl; tl += 2) {
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            if (tl + g >= ntl) break;  // wave-uniform
            const f16v acc = screen_tile(tl + g);
            const float was = m1[g];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float v = __uint_as_float((__float_as_uint(acc[i]) & ~15u) | (uint32_t)i);
              m2[g] = __builtin_amdgcn_fmed3f(m1[g], m2[g], v);
              m1[g] = vmax(m1[g], v);
            }
            bk[g] = m1[g] != was ? k0 + 32 * (tl + g) : bk[g];
          }
        }
      }

      const float d0 = __builtin_fmaf(0x1p-20f, __builtin_amdgcn_sqrtf(cmax2), 0x1p-31f);  // absolute part of d
      // The row's unique candidate, or a comparison of the trackers' largest
      // values (need) or of every centroid above the limit (full).
      float lim = 0.f;
      uint32_t ans = 0;
      int kc[2] = {0, 0};
      bool need = false, full = false;
      if (!MULTI || live) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const int id = (int)(__float_as_uint(m1[g]) & 15u);
          kc[g] = bk[g] + 8 * (id >> 2) + (id & 3) + 4 * h;
        }
        const bool odd = m1[1] > m1[0];
        const float a1 = odd ? m1[1] : m1[0];  // this lane's largest, its other tracker's
        const float a2 = odd ? m1[0] : m1[1];
        const float rest = vmax(m2[0], m2[1]);
        const int k = odd ? kc[1] : kc[0];
        const float o1 = __shfl_xor(a1, 32), o2 = __shfl_xor(a2, 32), orest = __shfl_xor(rest, 32);
        const int ok = __shfl_xor(k, 32);
        const float s1 = vmax(a1, o1);
        const float unnamed = vmax(rest, orest);  // every value that no tracker names is below
        const float s2 = vmax(vmax(unnamed, o1 < a1 ? o1 : a1), vmax(a2, o2));
        const float t = xx - 2.f * s1;
        const float d = __builtin_fmaf(1.0f + 0x1p-9f, __builtin_fabsf(t), __builtin_fmaf(3 * 0x1p-11f, xx, d0));
        const float C2 = __builtin_fminf(cmax2, 2.f * (xx + d));
        const float M = __builtin_fmaf(kMx, xx, __builtin_fmaf(kMc, C2, __builtin_fmaf(md, d, m0)));
        // small enough that no distance overflows and excluded centroids are
        // farther (false for NaN)
        const bool range = xx < rmax && t < rmax;
        ans = (uint32_t)(o1 > a1 ? ok : k);
        need = row0 + r < p.nrows && !(range && s1 - s2 > M);
        full = need && !(range && s1 - unnamed > M);
        lim = range ? s1 - M : -__builtin_inff();
      }
      const bool any_need = __any(need), any_full = __any(full);

      // Reference distances of the candidates: (row, centroid) pairs gathered
      // over the wave, 64 at a time, a lane each.  The smallest (distance,
      // index) of a row is the reference's first strict minimum.
      int npair = 0;  // wave-uniform
      auto compare = [&]() {
        wave_lds_sync();
        if (lane < npair) {
          const int k = pair_k[lane], rr = pair_r[lane];
          const float dist = exact_dist<FUSED, KS>(p.rows + (row0 + rr) * D, p.ctrds + (int64_t)k * D, D);
          if (dist < FLT_MAX)
            atomicMin(best + rr, (unsigned long long)__float_as_uint(dist) << 32 | (uint32_t)k);
        }
        wave_lds_sync();
        npair = 0;
      };
      // the set bits of cand, each a centroid of the lane's row
      auto gather = [&](uint32_t cand, auto centroid) {
        while (const unsigned long long who = __ballot(cand != 0)) {
          const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0));
          if (cand && npair + rank < 64) {
            pair_k[npair + rank] = centroid(__builtin_ctz(cand));
            pair_r[npair + rank] = (uint8_t)r;
            cand &= cand - 1;
          }
          npair = min(64, npair + (int)__popcll(who));
          if (npair == 64) compare();
        }
      };
      if (any_need) {
        if (h == 0) best[r] = ~0ull;
        wave_lds_sync();
        if (!any_full)
          gather(need ? (m1[0] >= lim ? 1u : 0u) | (m1[1] >= lim ? 2u : 0u) : 0u,
                 [&](int b) { return kc[b]; });
      }
      if (MULTI ? (bool)__syncthreads_or(any_full) : any_full) {
#pragma unroll 1
        for (int c = 0; c < nchunks; ++c) {
          if (MULTI) {
            stage(c * p.KC);
            if (!any_full) continue;
          }
          const int k0 = c * p.KC;
          const int ntl = (min(p.KC, K - k0) + 31) >> 5;
#pragma unroll 1
          for (int tl = 0; tl < ntl; ++tl) {
            const f16v acc = screen_tile(tl);
            const int k = k0 + 32 * tl + 4 * h;
            uint32_t cand = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i)
              cand |= !(acc[i] < lim) && k + 8 * (i >> 2) + (i & 3) < K ? 1u << i : 0u;
            gather(need ? cand : 0u, [&](int b) { return k + 8 * (b >> 2) + (b & 3); });
          }
        }
      }
      if (any_need) {
        if (npair) compare();
        const unsigned long long key = best[r];
        if (need) ans = key == ~0ull ? (uint32_t)K : (uint32_t)key;
      }
      if ((!MULTI || live) && h == 0 && row0 + r < p.nrows) p.assign[row0 + r] = ans;
    }
  };
  // (both loops in 128 registers spill 8 where rows are read float by float
  // for 64 dims: 2^23 rows 62 x 55 749 us, one loop 506)
  constexpr bool kOneLoop = KS == 4 && !VEC && !ROOMY;
  if (moved || kOneLoop)
    steps(std::true_type());
  else
    steps(std::integral_constant<bool, kOneLoop>());
}

typedef void (*KmKernel)(KmParams);

// ---------------------------------------------------------------------------
// Direct form, for narrow rows: each lane takes one row (64 rows per wave)
// and runs the reference's loop itself -- per centroid ascending, per dim
// ascending, one subtraction and one fused (or separately rounded)
// multiply-add -- with the centroids staged in LDS (row stride 4 ceil(D/4),
// zero padded) and read by all lanes at once (broadcast 16-byte reads).
// The wave's 64 x D block of rows is contiguous: it is loaded with
// coalesced 16-byte loads (the next step's while this step computes),
// split into rows in the wave's LDS area (odd row stride: conflict-free)
// and read back one row per lane.  When the centroids exceed one LDS chunk
// the workgroup's waves step through the chunks in lockstep.
// ---------------------------------------------------------------------------
template <int D, bool FUSED>
__global__ __launch_bounds__(64 * kKmDirectWaves) void k_kmeans_direct(KmParams p) {
  constexpr int DS = (D + 3) / 4 * 4;   // staged floats per centroid
  constexpr int XS = D | 1;             // LDS row stride of the row block
  constexpr int NP = (16 * D + 63) / 64;  // 16-byte pieces per lane per block
  extern __shared__ f4 kmd_lds4[];
  float *cs = reinterpret_cast<float *>(kmd_lds4);  // KC x DS
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float *xs = cs + p.KC * DS + w * 64 * XS;  // this wave's 64 rows
  const int K = p.K;
  const int nchunks = (K + p.KC - 1) / p.KC;
  auto stage = [&](int c0) {
    __syncthreads();
    for (int idx = threadIdx.x; idx < p.KC * DS; idx += blockDim.x) {
      const int k = idx / DS, d = idx - k * DS;
      cs[idx] = (c0 + k < K && d < D) ? p.ctrds[(int64_t)(c0 + k) * D + d] : 0.f;
    }
    __syncthreads();
  };
  if (nchunks == 1) stage(0);
  auto row0_of = [&](int64_t st) {
    return ((st * gridDim.x + blockIdx.x) * kKmDirectWaves + w) * 64;
  };
  // piece f = lane + 64 i of the block: floats 4f .. 4f+3 (past the end of
  // the array: zero; a piece that crosses it element by element)
  auto load_block = [&](int64_t st, f4 (&dst)[NP]) {
    const int64_t row0 = row0_of(st);
    const int64_t left = row0 < p.nrows ? (p.nrows - row0) * D * 4 : 0;
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(p.rows + (row0 < p.nrows ? row0 : 0) * D, left < kRsrcMax ? (int32_t)left : kRsrcMax);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t o = 16 * (int64_t)(lane + 64 * i);
      if (lane + 64 * i >= 16 * D || o >= left) {
        dst[i] = f4{0.f, 0.f, 0.f, 0.f};
      } else if (o + 16 <= left) {
        dst[i] = buf_load4<kBufNT>(rs, (uint32_t)o, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[i][e] = buf_load1(rs, o + 4 * e < left ? (uint32_t)(o + 4 * e) : kOOB, 0);
      }
    }
  };
  f4 pnext[NP];
  load_block(0, pnext);
  for (int64_t st = 0; st < p.steps; ++st) {
    const int64_t row0 = row0_of(st);
    const bool live = row0 < p.nrows;  // wave-uniform
    if (nchunks == 1 && !live) break;
    float x[DS];
    if (live) {
      // split the block into rows: element 4f + e is row (4f+e)/D, dim (4f+e)%D
#pragma unroll
      for (int i = 0; i < NP; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int idx = 4 * (lane + 64 * i) + e;
          if (idx < 64 * D) xs[(idx / D) * XS + idx % D] = pnext[i][e];
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int d = 0; d < DS; ++d) x[d] = d < D ? xs[lane * XS + d] : 0.f;
      wave_lds_sync();  // the next step's split may overwrite the area
    }
    if (st + 1 < p.steps) load_block(st + 1, pnext);
    const bool rin = row0 + lane < p.nrows;
    float best = FLT_MAX;
    uint32_t bk = kNone;
    for (int c = 0; c < nchunks; ++c) {
      if (nchunks > 1) stage(c * p.KC);
      if (!live) continue;
      const int kc = min(p.KC, K - c * p.KC);
      for (int k = 0; k < kc; ++k) {
        const float *cr = cs + k * DS;
        float dist = 0.f;
#pragma unroll
        for (int j = 0; j < DS / 4; ++j) {
          const f4 cv = *reinterpret_cast<const f4 *>(cr + 4 * j);
#pragma unroll
          for (int e = 0; e < 4; ++e) dist = exact_step<FUSED>(dist, x[4 * j + e], cv[e]);
        }
        if (dist < best) {
          best = dist;
          bk = (uint32_t)(c * p.KC + k);
        }
      }
    }
    if (live && rin) p.assign[row0 + lane] = bk == kNone ? (uint32_t)K : bk;
  }
}

template <int D>
KmKernel kmd_pick(bool fused) {
  return fused ? k_kmeans_direct<D, true> : k_kmeans_direct<D, false>;
}

template <int... Ds>
KmKernel kmd_find(int d, bool fused, std::integer_sequence<int, Ds...>) {
  KmKernel out = nullptr;
  ((d == Ds + 1 ? (out = kmd_pick<Ds + 1>(fused), 0) : 0), ...);
  return out;
}

KmKernel kmd_kernel(int d, bool fused) {
  return kmd_find(d, fused, std::make_integer_sequence<int, kKmDirectMaxDims>{});
}

template <int KS, bool FUSED>
KmKernel kms_pick(bool multi, bool vec, bool roomy) {
  if constexpr (KS == 4)
    if (!multi && roomy)
      return vec ? k_kmeans_screen<KS, false, true, FUSED, true> : k_kmeans_screen<KS, false, false, FUSED, true>;
  if (multi) return vec ? k_kmeans_screen<KS, true, true, FUSED> : k_kmeans_screen<KS, true, false, FUSED>;
  return vec ? k_kmeans_screen<KS, false, true, FUSED> : k_kmeans_screen<KS, false, false, FUSED>;
}

KmKernel kms_kernel(int ks, bool multi, bool vec, bool roomy, bool fused) {
  switch (ks) {
    case 1: return fused ? kms_pick<1, true>(multi, vec, roomy) : kms_pick<1, false>(multi, vec, roomy);
    case 2: return fused ? kms_pick<2, true>(multi, vec, roomy) : kms_pick<2, false>(multi, vec, roomy);
    case 3: return fused ? kms_pick<3, true>(multi, vec, roomy) : kms_pick<3, false>(multi, vec, roomy);
    default: return fused ? kms_pick<4, true>(multi, vec, roomy) : kms_pick<4, false>(multi, vec, roomy);
  }
}

int cu_count() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    return 256;
  return n;
}

}  // namespace

KmeansPlan plan_kmeans(int64_t nrows, int D, int K, int mode) {
  KmeansPlan pl;
  // The direct kernel's time grows with dims x clusters from the row stream
  // up, the screened one's starts at the cost of splitting the rows and
  // barely grows.  Measured on MI355X over 2^21 clustered rows (screened /
  // direct, us; uniform rows within 2): 5 x 24 32.8 / 29.1, 5 x 32 32.1 / 36.2,
  // 8 x 24 33.4 / 29.9, 8 x 32 33.3 / 37.3, 16 x 12 34.5 / 33.5, 16 x 16 34.5 /
  // 38.1, 24 x 8 44.7 / 39.0, 24 x 10 45.1 / 44.1, 24 x 12 45.5 / 48.7, 32 x 8
  // 49.6 / 48.4, 32 x 12 49.1 / 59.1; 4 x 8 31.9 / 11.9 and 16 x 128 64 / 221
  // far from the line.  They cross near 140 for the shortest rows, between 200
  // and 300 for most.
  pl.direct = (mode == 2 && D <= kKmDirectMaxDims) ||
              (mode == 0 && D <= kKmDirectMaxDims && (int64_t)K * D < kKmDirectWork);
  if (pl.direct) {
    // one row per lane; centroids in chunks of at most kKmDirectLdsBytes,
    // plus each wave's 64-row area
    pl.ni = D;
    const int64_t ds = (D + 3) / 4 * 4;
    const int64_t rows_f = (int64_t)kKmDirectWaves * 64 * (D | 1);
    int64_t kc = (int64_t)(kKmDirectLdsBytes / 4) / ds;
    if (kc > K) kc = K;
    pl.KC = (int)kc;
    pl.lds = (size_t)(kc * ds + rows_f) * 4;
    pl.tiles = (nrows + 63) / 64;  // 64-row wave blocks
    return pl;
  }
  pl.ni = (D + 15) / 16;
  const int64_t kpad = ((int64_t)K + 31) / 32 * 32;
  // LDS: the sample of centroids, per centroid 64 ni bytes of fp16 terms and
  // its norm, each wave's row tile in whole 1 KB loads, 256 bytes that reads past the last tile's
  // last row may touch, and 256 for the workgroup vote
  pl.xfloats = (D + 7) / 8 * 256;
  const int64_t rows_b = (int64_t)kKmWaves * pl.xfloats * 4 + 256 + kKmHeadBytes;
  const int64_t room = (int64_t)kKmLdsBytes - 256 - rows_b;
  pl.KC = (int)std::min<int64_t>(kpad, room / (64 * pl.ni + 4) / 32 * 32);
  pl.lds = (size_t)(pl.KC * (64 * pl.ni + 4) + rows_b);
  pl.tiles = (nrows + 31) / 32;
  return pl;
}

hipError_t launch_kmeans_assign(const KmeansPlan &pl, uint32_t *assign, const float *rows,
                                int64_t nrows, int D, const float *ctrds, int K, bool fused,
                                hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  if (pl.direct ? pl.KC < 1 : pl.KC < 32) return hipErrorInvalidValue;
  KmKernel fn = pl.direct ? kmd_kernel(pl.ni, fused)
                          : kms_kernel(pl.ni, pl.KC < K, D % 4 == 0, 2 * pl.lds > kKmLdsBytes, fused);
  if (!fn) return hipErrorInvalidValue;
  const int waves = pl.direct ? kKmDirectWaves : kKmWaves;
  hipError_t e;
  if (pl.lds > 65536) {
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds);
    if (e != hipSuccess) return e;
  }
  int per_cu = 0;
  e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(fn),
                                                   64 * waves, pl.lds);
  if (e != hipSuccess) return e;
  if (per_cu < 1) per_cu = 1;
  const int64_t wgs_needed = (pl.tiles + waves - 1) / waves;
  int64_t grid = (int64_t)per_cu * cu_count();
  if (grid > wgs_needed) grid = wgs_needed;
  KmParams p;
  p.rows = rows;
  p.ctrds = ctrds;
  p.assign = assign;
  p.nrows = nrows;
  p.steps = (pl.tiles + grid * waves - 1) / (grid * waves);
  p.D = D;
  p.K = K;
  p.KC = pl.KC;
  p.xfloats = pl.xfloats;
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(64 * waves), pl.lds, st, p);
  return hipGetLastError();
}

}  // namespace hml
