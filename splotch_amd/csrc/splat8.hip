// Wave-per-block splat (8 x 8 pixel blocks) with heaviest-first scheduling.
//
// A work unit is one 8x8 pixel block of a reference tile (blocks aligned to
// the tile origin); its particle list holds exactly the particles whose
// footprint box (splotch_host.cc:462-472, tile frame) overlaps the block, in
// render order.  One wave owns one unit: lane = pixel.  Per batch of 64
// particles, lane l tabulates particle l's 8 column ranges + Gaussian column
// factors and 8 row factors (splotch_host.cc:596-607) into the wave's LDS
// slice; then the wave walks the batch in order and every lane updates its
// pixel exactly as render_new does, so each pixel sees the reference's
// summation / compositing order and rounding.
//
// Scheduling: units are issued heaviest first (work items sorted by list
// length, descending).  In the ordered mode the per-pixel chain is serial, so a
// long list is the critical path; units with at least `split` entries are
// issued as three items, one per colour channel (the channels' chains are
// independent), which cuts the serial work per lane to about a third.
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

#include "device_util.hpp"
#include "workspace.hpp"

namespace splhip {
namespace {

__device__ __forceinline__ int64_t gtid() {
  return static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
}
__device__ __forceinline__ int64_t gstride() {
  return static_cast<int64_t>(gridDim.x) * blockDim.x;
}

// exptable op with the x86 conversion semantics folded in: p = arg*expfac;
// p >= 2^31 or NaN -> INT_MIN -> 1; p in [2^20, 2^31) -> 0; p <= -1 -> negative
// index -> 1; otherwise the table product at trunc(p).
__device__ __forceinline__ float xop(const float *tab, float arg, float expfac) {
  const float p = arg * expfac;
  if (p < 1048576.f) {
    if (p > -1.f) {
      const int i = static_cast<int>(p);
      return tab[i >> 10] * tab[1024 + (i & 1023)];
    }
    return 1.f;
  }
  return (p < 2147483648.f) ? 0.f : 1.f;
}

// xop in two steps, so that several lookups can be in flight: xop_reads
// reads the two table entries for p = arg * expfac (at an in-range index in
// every case), xop_value gives xop's result from them.
__device__ __forceinline__ void xop_reads(const float *tab, float p, float &t1, float &t2) {
  const bool ok = (p < 1048576.f) && (p > -1.f);
  const int i = static_cast<int>(ok ? p : 0.f);
  t1 = tab[i >> 10];
  t2 = tab[1024 + (i & 1023)];
}
__device__ __forceinline__ float xop_value(float p, float t1, float t2) {
  const bool hi_ok = p < 1048576.f;
  const bool ok = hi_ok && (p > -1.f);
  return ok ? t1 * t2 : ((hi_ok || !(p < 2147483648.f)) ? 1.f : 0.f);
}

__device__ __forceinline__ float xexpm1(const float *tab, float arg, float expfac, float tl) {
  if (fabsf(arg) < tl) return arg;
  return xop(tab, arg, expfac) - 1.f;
}

// Branch-free xexpm1 (same results as xop/xexpm1): the table is always read
// at an in-range index so that several lookups can be in flight at once.
__device__ __forceinline__ float xexpm1_bf(const float *tab, float arg, float expfac, float tl) {
  const float p = arg * expfac;
  const bool hi_ok = p < 1048576.f;
  const bool ok = hi_ok && (p > -1.f);
  const int i = static_cast<int>(ok ? p : 0.f);
  const float prod = tab[i >> 10] * tab[1024 + (i & 1023)];
  const float opv = ok ? prod : ((hi_ok || !(p < 2147483648.f)) ? 1.f : 0.f);
  return (fabsf(arg) < tl) ? arg : opv - 1.f;
}

// Absorption range of the fast table path: att * a * expfac stays in [0, 2^20)
// for att in [0, 1] (expfac = 2^20 / -20).  A fast particle also has finite
// q_c (e_c / (e_c + gray_absorption) is not when gray_absorption <= 0 meets
// e_c = -gray_absorption): the fast paths apply it outside the footprint as
// l + ((l - q) * m1) * 0, which must be l.
constexpr float kFastA = -19.5f;

__device__ __forceinline__ bool finite3(float x, float y, float z) {
  const float inf = __builtin_inff();
  return fabsf(x) < inf && fabsf(y) < inf && fabsf(z) < inf;
}

// exptable::expm1 (splotchutils.h:203-214) split in two for pipelining:
// xexp_index gives the table index for p = arg*expfac (0 where the table does
// not apply), and xexpm1_finish combines the two table values t1, t2 fetched
// at that index with the out-of-range and Taylor cases.
__device__ __forceinline__ float xexpm1_finish(float arg, float p, float t1, float t2, float tl) {
  const bool hi_ok = p < 1048576.f;
  const bool ok = hi_ok && (p > -1.f);
  const float opv = ok ? t1 * t2 : ((hi_ok || !(p < 2147483648.f)) ? 1.f : 0.f);
  return (fabsf(arg) < tl) ? arg : opv - 1.f;
}

// Table entries of the fast path, where p = arg * expfac lies in [0, 2^20):
// i4 = trunc(arg * 4 expfac) = 4 trunc(p) + (0..3) (scaling by 4 is exact), so
// the byte offsets of tab1[trunc(p) >> 10] and tab2[trunc(p) & 1023] are two
// masks of i4.
__device__ __forceinline__ void xtab_fast(const float *tab, float arg, float expfac4, float &t1,
                                          float &t2) {
  const uint32_t i4 = static_cast<uint32_t>(static_cast<int>(arg * expfac4));
  const char *b = reinterpret_cast<const char *>(tab);
  t1 = *reinterpret_cast<const float *>(b + ((i4 >> 10) & 0xffcu));
  t2 = *reinterpret_cast<const float *>(b + 4096 + (i4 & 0xffcu));
}

__device__ __forceinline__ int xexp_index(float p) {
  const bool ok = (p < 1048576.f) && (p > -1.f);
  return static_cast<int>(ok ? p : 0.f);
}

// v of the lane j of every group of four lanes (a DPP operand of the
// instruction that uses it, at no instruction of its own).
template <int J>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), J * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_of(float v, int j) {  // j: constant after unrolling
  switch (j & 3) {
    case 0: return quad_lane<0>(v);
    case 1: return quad_lane<1>(v);
    case 2: return quad_lane<2>(v);
    default: return quad_lane<3>(v);
  }
}
__device__ __forceinline__ float4 quad_of(const float4 &v, int j) {
  return make_float4(quad_of(v.x, j), quad_of(v.y, j), quad_of(v.z, j), quad_of(v.w, j));
}
// x where bit 8 (j & 3) of the pixel's coverage word m is set (byte j: particle
// j of four, shifted down by the pixel's row), else +0: the bit, sign-extended,
// masks x's bits.
__device__ __forceinline__ float covered(float x, uint32_t m, int j) {
  const uint32_t all =
      static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(m), 8 * (j & 3), 1));
  return __uint_as_float(__float_as_uint(x) & all);
}

constexpr int kColPad = 68;  // bytes per column of coverage (a word per four particles)

// One fast chunk of the ordered walk (all particles of the chunk have every
// a_c in [kFastA, 0] and finite q_c) for channel class CH: J particles from
// slot k0, their constants in cst; bit j of TB set: particle k0 + j takes the
// Taylor branch at every pixel of its footprint in the block, so its update
// is l += ((l - q) * a) * att (att replaced by +0 outside the footprint) with
// no table work.
//
// The walk issues VALU work most of the time and keeps the CU's LDS busy half
// of it, and waits on the LDS's returns where 16 waves do not hide them (at
// 2.4 GHz a linear or broadcast b32 read of a wave takes its CU 2.5 clocks, a
// b128 one 4.3, whether or not the lanes share addresses; a random table lookup
// 6).  So the constants of four particles are read once, lane l those of
// particle l % 4, and reach the operations as quad-permuted DPP operands (2
// VALU clocks more per use), and four particles' coverage of a column is one
// word: 52 -> 44 LDS clocks per particle in the expm1 branch, 16 -> 8 in the
// Taylor branch.
template <int CH, int J, uint32_t TB>
__device__ __forceinline__ void fast_chunk(int k0, int cx, int cy, const uint8_t (*col)[kColPad],
                                           const float (*pre2)[kPad],
                                           const float (*pre1)[kPad], const float *tab,
                                           const float4 *cst, float expfac4, float tl,
                                           float &l0, float &l1, float &l2) {
  constexpr bool C0 = (CH == 3 || CH == 0), C1 = (CH == 3 || CH == 1), C2 = (CH == 3 || CH == 2);
  // constants and coverage of four particles, or where a chunk has fewer, of one
  // (by lane from the four's: 100k additive particles at 512^2, hip_ppw 1, nothing
  // staged, 2.15 ms; so 1.39)
  constexpr bool kQuads = J >= 4;
  constexpr int JQ = kQuads ? J / 4 : J;
  float at[J], m2[J], g0[J], g1[J], g2[J], u0[J], w0[J], u1[J], w1[J], u2[J], w2[J];
  float4 ca[JQ], cq[JQ];
  uint32_t cov[JQ];
  bool tay[J];
  // slots past the batch hold finite values of earlier batches (or
  // zeros) and are masked; table offsets are masked into the tables
#pragma unroll
  for (int q = 0; q < JQ; ++q) {
    const int k = kQuads ? k0 + 4 * q : k0 + q, kl = kQuads ? k + (cy & 3) : k;
    ca[q] = cst[2 * kl];
    cq[q] = cst[2 * kl + 1];
    cov[q] = (kQuads ? *reinterpret_cast<const uint32_t *>(&col[cx][k]) : col[cx][k]) >> cy;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k = k0 + j;
    at[j] = covered(pre1[cy][k] * pre2[cx][k], kQuads ? cov[j / 4] : cov[j], kQuads ? j : 0);
  }
  auto con = [&](const float4 (&v)[JQ], int j) { return kQuads ? quad_of(v[j / 4], j) : v[j]; };
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if ((TB >> j) & 1u) {
      m2[j] = at[j];
      continue;
    }
    const float4 a4 = con(ca, j);
    tay[j] = (a4.w * at[j]) < tl;
    m2[j] = tay[j] ? at[j] : 1.f;
    if (C0) { g0[j] = at[j] * a4.x; xtab_fast(tab, g0[j], expfac4, u0[j], w0[j]); }
    if (C1) { g1[j] = at[j] * a4.y; xtab_fast(tab, g1[j], expfac4, u1[j], w1[j]); }
    if (C2) { g2[j] = at[j] * a4.z; xtab_fast(tab, g2[j], expfac4, u2[j], w2[j]); }
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const float4 a4 = con(ca, j), q4 = con(cq, j);
    if ((TB >> j) & 1u) {
      if (C0) l0 = l0 + ((l0 - q4.x) * a4.x) * m2[j];
      if (C1) l1 = l1 + ((l1 - q4.y) * a4.y) * m2[j];
      if (C2) l2 = l2 + ((l2 - q4.z) * a4.z) * m2[j];
      continue;
    }
    // the table product is formed before the select: written inside
    // it, the compiler may move the table reads into a branch that
    // waits for every LDS read in flight
    if (C0) {
      const float ex = u0[j] * w0[j] - 1.f;
      const float em = (fabsf(g0[j]) < tl) ? g0[j] : ex;
      const float m1 = tay[j] ? a4.x : em;
      l0 = l0 + ((l0 - q4.x) * m1) * m2[j];
    }
    if (C1) {
      const float ex = u1[j] * w1[j] - 1.f;
      const float em = (fabsf(g1[j]) < tl) ? g1[j] : ex;
      const float m1 = tay[j] ? a4.y : em;
      l1 = l1 + ((l1 - q4.y) * m1) * m2[j];
    }
    if (C2) {
      const float ex = u2[j] * w2[j] - 1.f;
      const float em = (fabsf(g2[j]) < tl) ? g2[j] : ex;
      const float m1 = tay[j] ? a4.z : em;
      l2 = l2 + ((l2 - q4.z) * m1) * m2[j];
    }
  }
}

// Chunked walk of one batch for one channel class CH (0..2 one channel, 3 all):
// for J particles at a time, phase 1 issues every LDS read of the chunk (column
// masks, Gaussian factors, then the exp-table entries of each fragment) and
// phase 2 applies the J updates in list order.  No loaded value is carried
// across chunks, so the LDS latency is paid twice per chunk, not per particle.
// The code is branch-free: loads past the batch end read slots whose column
// masks are 0 (phase A clears them), and a pixel outside a footprint adds +0.
// The accumulators start at +0 and a sum of floats is -0 only if both terms
// are -0, so they never hold -0 and l + 0 == l bit for bit: the result equals
// the reference's skip.
template <int ADD, int CH, int J>
__device__ __forceinline__ void walk_chunks(int nb, int cx, int cy, const uint8_t (*col)[kColPad],
                                            const float (*pre2)[kPad], const float (*pre1)[kPad],
                                            const float *tab, float va0, float va1, float va2,
                                            float vq0, float vq1, float vq2, float vmax,
                                            const float4 *cst, uint64_t fastmask,
                                            uint64_t taymask, float expfac, float tl,
                                            float &l0, float &l1,
                                            float &l2) {
  constexpr bool C0 = (CH == 3 || CH == 0), C1 = (CH == 3 || CH == 1), C2 = (CH == 3 || CH == 2);
  static_assert(64 % J == 0, "chunks tile a batch: slot k0 + j < 64");
  const float expfac4 = 4.f * expfac;  // exact
  for (int k0 = 0; k0 < nb; k0 += J) {
    if (!ADD) {
      // Fast chunk: every particle of the chunk has all absorptions a_c in
      // [kFastA, 0], so arg = att*a_c (att in [0, 1]) gives p = arg*expfac in
      // [0, 2^20): the table index is trunc(p) with no range cases.  The
      // update is written l += ((l - q) * m1) * m2 with
      //   Taylor branch: m1 = a, m2 = att;  expm1 branch: m1 = em, m2 = 1
      //   (x * 1 == x);  outside the footprint: m2 = 0 (l + +-0 == l, as l is
      //   never -0),
      // which is render_new's update bit for bit (splotch_host.cc:648-658).
      // The particles' constants come from LDS (cst: (a0, a1, a2, max |a|),
      // (q0, q1, q2, 0)) as vector operands.
      const int cnt = min(J, nb - k0);
      const uint64_t need = ((1ull << cnt) - 1ull) << k0;
      if ((fastmask & need) == need) {
        // bit j: particle k0 + j takes the Taylor branch at every pixel of
        // its footprint in the block (wave-uniform): no table work for it.
        // Three-channel chunks of 4 have a straight-line body per pattern.
        const uint32_t tb = static_cast<uint32_t>(taymask >> k0);
        if (CH == 3 && J == 4) {
          switch (tb & 15u) {
#define SPLHIP_FAST(T) case T: fast_chunk<CH, J, T>(k0, cx, cy, col, pre2, pre1, tab, cst, expfac4, tl, l0, l1, l2); break;
            SPLHIP_FAST(0) SPLHIP_FAST(1) SPLHIP_FAST(2) SPLHIP_FAST(3)
            SPLHIP_FAST(4) SPLHIP_FAST(5) SPLHIP_FAST(6) SPLHIP_FAST(7)
            SPLHIP_FAST(8) SPLHIP_FAST(9) SPLHIP_FAST(10) SPLHIP_FAST(11)
            SPLHIP_FAST(12) SPLHIP_FAST(13) SPLHIP_FAST(14) SPLHIP_FAST(15)
#undef SPLHIP_FAST
          }
        } else {
          fast_chunk<CH, J, 0u>(k0, cx, cy, col, pre2, pre1, tab, cst, expfac4, tl, l0, l1, l2);
        }
        continue;
      }
    } else {
      // Additive: constants and coverage as in the fast chunks (cst: (a0, a1,
      // a2, 0)); slots past the batch (stale or uninitialised values) are read
      // at their own offsets and their products masked, as their coverage is 0.
      constexpr bool kQuads = J >= 4;
      constexpr int JQ = kQuads ? J / 4 : J;
      float at[J];
      float4 ca[JQ];
      uint32_t cov[JQ];
#pragma unroll
      for (int q = 0; q < JQ; ++q) {
        const int k = kQuads ? k0 + 4 * q : k0 + q;
        ca[q] = cst[kQuads ? k + (cy & 3) : k];
        cov[q] = (kQuads ? *reinterpret_cast<const uint32_t *>(&col[cx][k]) : col[cx][k]) >> cy;
      }
#pragma unroll
      for (int j = 0; j < J; ++j) at[j] = pre1[cy][k0 + j] * pre2[cx][k0 + j];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const float4 a4 = kQuads ? quad_of(ca[j / 4], j) : ca[j];
        const uint32_t m = kQuads ? cov[j / 4] : cov[j];
        if (C0) l0 = l0 + covered(a4.x * at[j], m, kQuads ? j : 0);
        if (C1) l1 = l1 + covered(a4.y * at[j], m, kQuads ? j : 0);
        if (C2) l2 = l2 + covered(a4.z * at[j], m, kQuads ? j : 0);
      }
      continue;
    }
    // ordered, with a particle in the chunk that is not fast
    float att[J], g0[J], g1[J], g2[J], p0[J], p1[J], p2[J];
    float u0[J], w0[J], u1[J], w1[J], u2[J], w2[J];
    uint32_t msk[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = min(k0 + j, nb - 1);  // uniform; out-of-batch slots masked below
      const uint32_t mk = col[cx][k];
      msk[j] = (k0 + j < nb) ? mk : 0u;
      att[j] = pre1[cy][k] * pre2[cx][k];
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = min(k0 + j, nb - 1);
      if (C0) { g0[j] = att[j] * lane_f(va0, k); p0[j] = g0[j] * expfac; const int i = xexp_index(p0[j]); u0[j] = tab[i >> 10]; w0[j] = tab[1024 + (i & 1023)]; }
      if (C1) { g1[j] = att[j] * lane_f(va1, k); p1[j] = g1[j] * expfac; const int i = xexp_index(p1[j]); u1[j] = tab[i >> 10]; w1[j] = tab[1024 + (i & 1023)]; }
      if (C2) { g2[j] = att[j] * lane_f(va2, k); p2[j] = g2[j] * expfac; const int i = xexp_index(p2[j]); u2[j] = tab[i >> 10]; w2[j] = tab[1024 + (i & 1023)]; }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = min(k0 + j, nb - 1);
      const bool in = (msk[j] >> cy) & 1u;
      const float at = att[j];
      const bool tay = (lane_f(vmax, k) * at) < tl;
      if (C0) {
        const float em = xexpm1_finish(g0[j], p0[j], u0[j], w0[j], tl);
        const float d = l0 - lane_f(vq0, k);
        const float ta = (d * lane_f(va0, k)) * at, te = em * d;
        l0 = l0 + (in ? (tay ? ta : te) : 0.f);
      }
      if (C1) {
        const float em = xexpm1_finish(g1[j], p1[j], u1[j], w1[j], tl);
        const float d = l1 - lane_f(vq1, k);
        const float ta = (d * lane_f(va1, k)) * at, te = em * d;
        l1 = l1 + (in ? (tay ? ta : te) : 0.f);
      }
      if (C2) {
        const float em = xexpm1_finish(g2[j], p2[j], u2[j], w2[j], tl);
        const float d = l2 - lane_f(vq2, k);
        const float ta = (d * lane_f(va2, k)) * at, te = em * d;
        l2 = l2 + (in ? (tay ? ta : te) : 0.f);
      }
    }
  }
}

// Software-pipelined walk of one batch for one channel class CH (0..2 one
// channel, 3 all).  Iteration k updates particle k with table values fetched in
// iteration k-1, computes particle k+1's attenuation and issues its table
// reads, and loads particle k+2's column mask and Gaussian factors, so that the
// only serial dependency per step is the pixel's own update.
template <int ADD, int CH>
__device__ __forceinline__ void walk_batch(int nb, int cx, int cy, const uint32_t (*cmask)[kPad],
                                           const float (*pre2)[kPad], const float (*pre1)[kPad],
                                           const float *tab, float va0, float va1, float va2,
                                           float vq0, float vq1, float vq2, float vmax,
                                           float expfac, float tl, float &l0, float &l1,
                                           float &l2) {
  constexpr bool C0 = (CH == 3 || CH == 0), C1 = (CH == 3 || CH == 1), C2 = (CH == 3 || CH == 2);
  // stage inputs
  uint32_t m_n = cmask[cx][0];                               // mask of k (current)
  float att_n = pre1[cy][0] * pre2[cx][0];                    // att of k
  uint32_t m_nn = 0;
  float p1_nn = 0.f, p2_nn = 0.f;
  if (nb > 1) {
    m_nn = cmask[cx][1];
    p1_nn = pre1[cy][1];
    p2_nn = pre2[cx][1];
  }
  float arg0 = 0.f, arg1 = 0.f, arg2 = 0.f, pp0 = 0.f, pp1 = 0.f, pp2 = 0.f;
  float t10 = 0.f, t20 = 0.f, t11 = 0.f, t21 = 0.f, t12 = 0.f, t22 = 0.f;
  if (!ADD) {
    const float e_ = expfac;
    if (C0) { arg0 = att_n * lane_f(va0, 0); pp0 = arg0 * e_; const int i = xexp_index(pp0); t10 = tab[i >> 10]; t20 = tab[1024 + (i & 1023)]; }
    if (C1) { arg1 = att_n * lane_f(va1, 0); pp1 = arg1 * e_; const int i = xexp_index(pp1); t11 = tab[i >> 10]; t21 = tab[1024 + (i & 1023)]; }
    if (C2) { arg2 = att_n * lane_f(va2, 0); pp2 = arg2 * e_; const int i = xexp_index(pp2); t12 = tab[i >> 10]; t22 = tab[1024 + (i & 1023)]; }
  }
  for (int k = 0; k < nb; ++k) {
    // current particle k: values computed / fetched in the previous step
    const uint32_t m = m_n;
    const float att = att_n;
    const float carg0 = arg0, carg1 = arg1, carg2 = arg2;
    const float cp0 = pp0, cp1 = pp1, cp2 = pp2;
    const float c10 = t10, c20 = t20, c11 = t11, c21 = t21, c12 = t12, c22 = t22;
    // particle k+1: attenuation from the prefetched factors, issue its table reads
    if (k + 1 < nb) {
      m_n = m_nn;
      att_n = p1_nn * p2_nn;
      if (!ADD) {
        if (C0) { arg0 = att_n * lane_f(va0, k + 1); pp0 = arg0 * expfac; const int i = xexp_index(pp0); t10 = tab[i >> 10]; t20 = tab[1024 + (i & 1023)]; }
        if (C1) { arg1 = att_n * lane_f(va1, k + 1); pp1 = arg1 * expfac; const int i = xexp_index(pp1); t11 = tab[i >> 10]; t21 = tab[1024 + (i & 1023)]; }
        if (C2) { arg2 = att_n * lane_f(va2, k + 1); pp2 = arg2 * expfac; const int i = xexp_index(pp2); t12 = tab[i >> 10]; t22 = tab[1024 + (i & 1023)]; }
      }
      // particle k+2: prefetch column mask and factors
      if (k + 2 < nb) {
        m_nn = cmask[cx][k + 2];
        p1_nn = pre1[cy][k + 2];
        p2_nn = pre2[cx][k + 2];
      }
    }
    // update of particle k (splotch_host.cc:615 / 648-658)
    const bool in = (m >> cy) & 1u;
    if (ADD) {
      if (C0) l0 = in ? l0 + lane_f(va0, k) * att : l0;
      if (C1) l1 = in ? l1 + lane_f(va1, k) * att : l1;
      if (C2) l2 = in ? l2 + lane_f(va2, k) * att : l2;
    } else {
      const bool tay = (lane_f(vmax, k) * att) < tl;
      if (C0) {
        const float em = xexpm1_finish(carg0, cp0, c10, c20, tl);
        const float d = l0 - lane_f(vq0, k);
        const float t = tay ? (d * lane_f(va0, k)) * att : em * d;
        l0 = in ? l0 + t : l0;
      }
      if (C1) {
        const float em = xexpm1_finish(carg1, cp1, c11, c21, tl);
        const float d = l1 - lane_f(vq1, k);
        const float t = tay ? (d * lane_f(va1, k)) * att : em * d;
        l1 = in ? l1 + t : l1;
      }
      if (C2) {
        const float em = xexpm1_finish(carg2, cp2, c12, c22, tl);
        const float d = l2 - lane_f(vq2, k);
        const float t = tay ? (d * lane_f(va2, k)) * att : em * d;
        l2 = in ? l2 + t : l2;
      }
    }
  }
}

// Phase A of a batch, lane = particle (splotch_host.cc:462-476 + 596-607, tile
// frame): the lane's particle (record R) tabulates, for the block's 8
// columns, its row range (BITS: bit r set when block row byo + r lies in the
// column's [lo, hi); else lo | hi << 16) and Gaussian column factor, and for
// the 8 rows its Gaussian row factor, into column `lane` of the wave's LDS
// slices.  att_bound: the largest row factor times the largest column factor
// (+inf if one is NaN); float multiplication being monotone, every pixel's
// att = pre1 * pre2 is at most it, and vmax * att at most vmax * att_bound.
template <bool BITS, class Col>
__device__ __forceinline__ void tabulate(const SplatArgs &a, const Rec &R, int lane, int x0s,
                                        int y0s, int w, int h, int bxo, int byo,
                                        const float *s_tab, Col col,
                                        float (*pre2)[kPad], float (*pre1)[kPad],
                                        float expfac, float &att_bound) {
  const float rfacr = R.r * a.rfac;
  const float posx = R.x - static_cast<float>(x0s), posy = R.y - static_cast<float>(y0s);
  const int bx0 = max(cvt_i32(posx - rfacr + 1), 0), bx1 = min(cvt_i32(posx + rfacr + 1), w);
  const int by0 = max(cvt_i32(posy - rfacr + 1), 0), by1 = min(cvt_i32(posy + rfacr + 1), h);
  const float radsq = rfacr * rfacr;
  const float sigma = a.h2sigma * R.r;
  const float stp = -1.f / (sigma * sigma);
  // branch-free: every column and row is computed (outside the box the
  // values are discarded, e.g. the square root of a negative number), the
  // table reads of all 16 lookups are issued before any of them is used,
  // and the LDS stores follow
  uint32_t lohi[8];
  bool cin[8], rin[8];
  float pc[8], pr[8], t1[16], t2[16];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int x = bxo + c;
    cin[c] = x >= bx0 && x < bx1;
    const float dxsq = (static_cast<float>(x) - posx) * (static_cast<float>(x) - posx);
    const float dy = sqrtf(radsq - dxsq);
    const int lo = max(by0, cvt_i32(posy - dy + 1));
    const int hi = min(by1, cvt_i32(posy + dy + 1));
    uint32_t lh;
    if (BITS) {
      const int r0 = min(max(lo - byo, 0), 8), r1 = min(max(hi - byo, 0), 8);
      lh = (r1 > r0) ? (((1u << r1) - 1u) & ~((1u << r0) - 1u)) : 0u;
    } else {
      lh = static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
    }
    lohi[c] = (cin[c] && hi > lo) ? lh : 0u;
    pc[c] = (stp * dxsq) * expfac;
    xop_reads(s_tab, pc[c], t1[c], t2[c]);
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int y = byo + r;
    rin[r] = y >= by0 && y < by1;
    const float dyf = static_cast<float>(y) - posy;
    pr[r] = (stp * dyf * dyf) * expfac;
    xop_reads(s_tab, pr[r], t1[8 + r], t2[8 + r]);
  }
  // every read is used here, so that none is moved into a branch of the
  // selects below
#pragma unroll
  for (int k = 0; k < 16; ++k) asm volatile("" : "+v"(t1[k]), "+v"(t2[k]));
  float b2 = 0.f, b1 = 0.f;
  bool nan = false;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float p2 = cin[c] ? xop_value(pc[c], t1[c], t2[c]) : 0.f;
    b2 = fmaxf(b2, p2);
    nan |= p2 != p2;
    col[c][lane] = lohi[c];
    pre2[c][lane] = p2;
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float p1 = rin[r] ? xop_value(pr[r], t1[8 + r], t2[8 + r]) : 0.f;
    b1 = fmaxf(b1, p1);
    nan |= p1 != p1;
    pre1[r][lane] = p1;
  }
  att_bound = nan ? __builtin_inff() : b1 * b2;
}

// The lane's particle R over the block at (bxo, byo) of the tile (tile frame):
// tabulate's column masks (bit r: row byo + r of the column lies in the
// footprint) ...
__device__ __forceinline__ void column_masks(const SplatArgs &a, const Rec &R, int x0s, int y0s,
                                             int w, int h, int bxo, int byo, uint32_t (&cm)[8]) {
  const float rfacr = R.r * a.rfac;
  const float posx = R.x - static_cast<float>(x0s), posy = R.y - static_cast<float>(y0s);
  const int bx0 = max(cvt_i32(posx - rfacr + 1), 0), bx1 = min(cvt_i32(posx + rfacr + 1), w);
  const int by0 = max(cvt_i32(posy - rfacr + 1), 0), by1 = min(cvt_i32(posy + rfacr + 1), h);
  const float radsq = rfacr * rfacr;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int x = bxo + c;
    const float dxsq = (static_cast<float>(x) - posx) * (static_cast<float>(x) - posx);
    const float dy = sqrtf(radsq - dxsq);
    const int lo = max(by0, cvt_i32(posy - dy + 1));
    const int hi = min(by1, cvt_i32(posy + dy + 1));
    const int r0 = min(max(lo - byo, 0), 8), r1 = min(max(hi - byo, 0), 8);
    // hi > lo first: a column outside the disc has hi = INT_MIN (NaN root)
    cm[c] = (x >= bx0 && x < bx1 && hi > lo && r1 > r0)
                ? (((1u << r1) - 1u) & ~((1u << r0) - 1u)) : 0u;
  }
}

// ... and its Gaussian column and row factors (splotch_host.cc:596-607), for
// every column and row of the block: outside the footprint they are not used.
__device__ __forceinline__ void block_factors(const SplatArgs &a, const Rec &R, int lane, int x0s,
                                              int y0s, int bxo, int byo, const float *s_tab,
                                              float (*pre2)[kPad], float (*pre1)[kPad],
                                              float expfac) {
  const float posx = R.x - static_cast<float>(x0s), posy = R.y - static_cast<float>(y0s);
  const float sigma = a.h2sigma * R.r;
  const float stp = -1.f / (sigma * sigma);
  float p[16], t1[16], t2[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float dx = static_cast<float>(bxo + k) - posx, dy = static_cast<float>(byo + k) - posy;
    p[k] = (stp * (dx * dx)) * expfac;
    p[8 + k] = (stp * dy * dy) * expfac;
    xop_reads(s_tab, p[k], t1[k], t2[k]);
    xop_reads(s_tab, p[8 + k], t1[8 + k], t2[8 + k]);
  }
  // every read is used here, so that none is moved into a branch of the
  // selects below
#pragma unroll
  for (int k = 0; k < 16; ++k) asm volatile("" : "+v"(t1[k]), "+v"(t2[k]));
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    pre2[k][lane] = xop_value(p[k], t1[k], t2[k]);
    pre1[k][lane] = xop_value(p[8 + k], t1[8 + k], t2[8 + k]);
  }
}

// Work items of a launch: items[0, n), or with device counts (dc: the pass's
// item total and long-list total) the items after the first min(dc[1], cap)
// (those go to the producer/consumer kernel).
__device__ __forceinline__ uint32_t splat_items(const uint32_t *&items, uint32_t n,
                                                const ItemCounts &dc) {
  if (!dc.items) return n;
  const uint32_t tot = *dc.items, nh = min(min(*dc.heavy, dc.heavy_cap), tot);
  items += nh;
  return tot - nh;
}

// The wave's LDS of the 8x8 splat.  col: per column and particle the row bits
// (a byte each in variant 4, whose chunks read four particles' at once; row
// stride kColPad) or, in variants 1 and 2, the row range.
template <int ADD, int VAR>
struct SplatLds {
  typename std::conditional<VAR == 4, uint8_t, uint32_t>::type
      __attribute__((aligned(16))) col[8][VAR == 4 ? kColPad : kPad];
  float pre2[8][kPad], pre1[8][kPad];
  // per-particle constants: ordered (a0, a1, a2, max |a|), (q0, q1, q2, 0);
  // additive (a0, a1, a2, 0)
  float4 cst[64 * (ADD ? 1 : 2)];
};

// Cleared once per wave: the ordered fast chunks read every slot of a chunk,
// also past a short batch (masked there), and start from finite values.
template <int ADD, int VAR>
__device__ __forceinline__ void clear_slots(SplatLds<ADD, VAR> &L, int lane) {
  if (ADD) return;
  for (int i = lane; i < static_cast<int>(sizeof(L.col) / 4); i += 64)
    reinterpret_cast<uint32_t *>(L.col)[i] = 0u;
  for (int i = lane; i < 8 * kPad; i += 64) {
    (&L.pre2[0][0])[i] = 0.f;
    (&L.pre1[0][0])[i] = 0.f;
  }
  L.cst[2 * lane] = make_float4(0.f, 0.f, 0.f, 0.f);
  L.cst[2 * lane + 1] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Applies list entries [e0, e1) to the lane's pixel (lx, ly) of the unit, in
// list order, for channel chan (3: all).  PPW (variant 4): particles per chunk
// of the walk (1, 2, 4 or 8; 0: 8 for one channel, 8 additive / 4 ordered for
// all three).
template <int ADD, int VAR, int PPW>
__device__ __forceinline__ void walk_list(const SplatArgs &a, const UnitGeom &ug, uint32_t e0,
                                          uint32_t e1, int chan, int lane, const float *s_tab,
                                          SplatLds<ADD, VAR> &L, float &l0, float &l1, float &l2) {
  constexpr int J1 = PPW ? PPW : 8, J3 = PPW ? PPW : (ADD ? 8 : 4);
  const int bxo = ug.gx * 8, byo = ug.gy * 8;  // tile frame
  const int cx = lane >> 3, cy = lane & 7;
  const int ly = byo + cy;
  auto *col = L.col;
  float(*pre2)[kPad] = L.pre2;
  float(*pre1)[kPad] = L.pre1;
  float4 *wcst = L.cst;
  const float expfac = a.expfac, tl = a.taylorlimit;
  // The records of a batch are gathered one batch ahead and their slots two
  // ahead, so that the walk of a batch covers the latency of the next gather.
  Rec rn{};
  uint32_t sn = 0;
  if (e0 + lane < e1) rn = a.recs[a.ent[e0 + lane]];
  if (e0 + 64u + lane < e1) sn = a.ent[e0 + 64u + lane];
  for (uint32_t base = e0; base < e1; base += 64) {
    const int nb = static_cast<int>(uniform(min<uint32_t>(64u, e1 - base)));
    const Rec R = rn;
    if (base + 64u + lane < e1) rn = a.recs[sn];
    if (base + 128u + lane < e1) sn = a.ent[base + 128u + lane];
    // Phase A: lane = particle (splotch_host.cc:462-476 + 596-607, tile frame)
    float va0 = 0.f, va1 = 0.f, va2 = 0.f, vq0 = 0.f, vq1 = 0.f, vq2 = 0.f, vmax = 0.f;
    bool vfast = false, vtay = false;
    if (lane < nb) {
      float ab;
      tabulate<VAR >= 3>(a, R, lane, ug.x0s, ug.y0s, ug.w, ug.h, bxo, byo, s_tab, col, pre2, pre1,
                         expfac, ab);
      va0 = -R.e0;
      va1 = -R.e1;
      va2 = -R.e2;
      if (!ADD) {
        const float g = ug.grayabsorb;
        vq0 = R.e0 / (R.e0 + g);
        vq1 = R.e1 / (R.e1 + g);
        vq2 = R.e2 / (R.e2 + g);
        vmax = fmaxf(fabsf(va0), fmaxf(fabsf(va1), fabsf(va2)));
        vfast = va0 >= kFastA && va0 <= 0.f && va1 >= kFastA && va1 <= 0.f && va2 >= kFastA &&
                va2 <= 0.f && finite3(vq0, vq1, vq2);
        // Taylor particle: vmax * att < tl at every pixel of the block
        // (splotch_host.cc:648), shown by the bound on att
        vtay = vfast && (vmax * ab) < tl;
        // only the fast chunks read these, also for masked slots past the
        // batch, so a particle that is not fast (possibly a non-finite a or
        // q) leaves zeros, which a masked slot applies as l + 0
        const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
        wcst[2 * lane] = vfast ? make_float4(va0, va1, va2, vmax) : z4;
        wcst[2 * lane + 1] = vfast ? make_float4(vq0, vq1, vq2, 0.f) : z4;
      } else {
        wcst[lane] = make_float4(va0, va1, va2, 0.f);
      }
    } else {
      // a slot past a short batch: no pixel in its footprint
#pragma unroll
      for (int c = 0; c < 8; ++c) col[c][lane] = 0u;
    }
    wave_sync();
    const uint64_t fastmask = __ballot(vfast), taymask = __ballot(vtay);
    // Phase B: lane = pixel, particles in list order.
    if constexpr (VAR == 4) {
      switch (chan) {
        case 0: walk_chunks<ADD, 0, J1>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, wcst, fastmask, taymask, expfac, tl, l0, l1, l2); break;
        case 1: walk_chunks<ADD, 1, J1>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, wcst, fastmask, taymask, expfac, tl, l0, l1, l2); break;
        case 2: walk_chunks<ADD, 2, J1>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, wcst, fastmask, taymask, expfac, tl, l0, l1, l2); break;
        default: walk_chunks<ADD, 3, J3>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, wcst, fastmask, taymask, expfac, tl, l0, l1, l2); break;
      }
      wave_sync();
      continue;
    }
    if constexpr (VAR == 3) {
      switch (chan) {
        case 0: walk_batch<ADD, 0>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, expfac, tl, l0, l1, l2); break;
        case 1: walk_batch<ADD, 1>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, expfac, tl, l0, l1, l2); break;
        case 2: walk_batch<ADD, 2>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, expfac, tl, l0, l1, l2); break;
        default: walk_batch<ADD, 3>(nb, cx, cy, col, pre2, pre1, s_tab, va0, va1, va2, vq0, vq1, vq2, vmax, expfac, tl, l0, l1, l2); break;
      }
      wave_sync();
      continue;
    }
    if constexpr (VAR == 1) {
      for (int k = 0; k < nb; ++k) {
        const uint32_t lohi = col[cx][k];
        if (ly >= static_cast<int>(lohi & 0xffffu) && ly < static_cast<int>(lohi >> 16)) {
          const float att = pre1[cy][k] * pre2[cx][k];
          if (ADD) {
            if (chan == 3 || chan == 0) l0 += lane_f(va0, k) * att;
            if (chan == 3 || chan == 1) l1 += lane_f(va1, k) * att;
            if (chan == 3 || chan == 2) l2 += lane_f(va2, k) * att;
          } else {
            const float a0 = lane_f(va0, k), a1 = lane_f(va1, k), a2 = lane_f(va2, k);
            const float q0 = lane_f(vq0, k), q1 = lane_f(vq1, k), q2 = lane_f(vq2, k);
            if ((lane_f(vmax, k) * att) < tl) {
              if (chan == 3 || chan == 0) l0 += ((l0 - q0) * a0) * att;
              if (chan == 3 || chan == 1) l1 += ((l1 - q1) * a1) * att;
              if (chan == 3 || chan == 2) l2 += ((l2 - q2) * a2) * att;
            } else {
              if (chan == 3 || chan == 0) l0 += xexpm1(s_tab, att * a0, expfac, tl) * (l0 - q0);
              if (chan == 3 || chan == 1) l1 += xexpm1(s_tab, att * a1, expfac, tl) * (l1 - q1);
              if (chan == 3 || chan == 2) l2 += xexpm1(s_tab, att * a2, expfac, tl) * (l2 - q2);
            }
          }
        }
      }
      wave_sync();
      continue;
    }
    // 4 particles per step: the table reads of a step are issued together and
    // only the update chain is serial.
    for (int k0 = 0; k0 < nb; k0 += 4) {
      float att[4];
      bool in[4];
      int kk[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kk[j] = min(k0 + j, nb - 1);
        const uint32_t lohi = col[cx][kk[j]];
        in[j] = (k0 + j < nb) && ly >= static_cast<int>(lohi & 0xffffu) &&
                ly < static_cast<int>(lohi >> 16);
        att[j] = pre1[cy][kk[j]] * pre2[cx][kk[j]];
      }
      if (ADD) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a0 = lane_f(va0, kk[j]), a1 = lane_f(va1, kk[j]), a2 = lane_f(va2, kk[j]);
          if (chan == 3 || chan == 0) l0 = in[j] ? l0 + a0 * att[j] : l0;
          if (chan == 3 || chan == 1) l1 = in[j] ? l1 + a1 * att[j] : l1;
          if (chan == 3 || chan == 2) l2 = in[j] ? l2 + a2 * att[j] : l2;
        }
      } else {
        float em0[4], em1[4], em2[4];
        bool tay[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = kk[j];
          tay[j] = (lane_f(vmax, k) * att[j]) < tl;
          if (chan == 3 || chan == 0) em0[j] = xexpm1_bf(s_tab, att[j] * lane_f(va0, k), expfac, tl);
          if (chan == 3 || chan == 1) em1[j] = xexpm1_bf(s_tab, att[j] * lane_f(va1, k), expfac, tl);
          if (chan == 3 || chan == 2) em2[j] = xexpm1_bf(s_tab, att[j] * lane_f(va2, k), expfac, tl);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = kk[j];
          const float at = att[j];
          if (chan == 3 || chan == 0) {
            const float a0 = lane_f(va0, k), q0 = lane_f(vq0, k);
            const float t = tay[j] ? ((l0 - q0) * a0) * at : em0[j] * (l0 - q0);
            l0 = in[j] ? l0 + t : l0;
          }
          if (chan == 3 || chan == 1) {
            const float a1 = lane_f(va1, k), q1 = lane_f(vq1, k);
            const float t = tay[j] ? ((l1 - q1) * a1) * at : em1[j] * (l1 - q1);
            l1 = in[j] ? l1 + t : l1;
          }
          if (chan == 3 || chan == 2) {
            const float a2 = lane_f(va2, k), q2 = lane_f(vq2, k);
            const float t = tay[j] ? ((l2 - q2) * a2) * at : em2[j] * (l2 - q2);
            l2 = in[j] ? l2 + t : l2;
          }
        }
      }
    }
    wave_sync();
  }
}

// Four workgroups per CU (their LDS, 35 KB each, and at most 128 VGPRs a lane):
// the walk waits on LDS returns, and 16 waves hide more of them than the 12
// that 142 VGPRs allow (64 views with 137M ordered and 124M additive entries:
// 31.9 -> 30.6 ms; 32.1 with constants and coverage read per particle).  Ordered
// chunks of 8 (hip_ppw 8) hold 181 VGPRs: two (1M particles at 1024^2, nothing
// staged: 6.4 ms; 7.9 with 128 VGPRs and the rest in scratch).
template <int ADD, int PPW>
constexpr int splat_waves() {
  return !ADD && PPW == 8 ? 2 : 4;
}
template <int ADD, int VAR, int PPW>
__global__ __launch_bounds__(256, (splat_waves<ADD, PPW>())) void k_splat8(
    SplatArgs a, const uint32_t *items, uint32_t nitems_, ItemCounts dc, uint32_t nsplit_) {
  const uint32_t nreal = splat_items(items, nitems_, dc);
  // the first nsplit items are long lists served as three one-channel items
  const uint32_t nsplit = min(dc.nsplit ? *dc.nsplit : nsplit_, nreal);
  const uint32_t nitems = nreal + 2u * nsplit;
  __shared__ float s_tab[2048];
  __shared__ SplatLds<ADD, VAR> s_wave[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // a workgroup past the items (a grid sized for a capacity) leaves at once
  if (blockIdx.x * 4u >= nitems) return;
  for (int i = tid; i < 2048; i += 256) s_tab[i] = a.exptab[i];
  __syncthreads();
  const uint32_t it = blockIdx.x * 4u + wave;
  if (it >= nitems) return;
  const uint64_t t_start = a.trace ? __builtin_amdgcn_s_memrealtime() : 0;
  // wave-uniform values are moved to scalar registers so that loop bounds and
  // channel selection compile to scalar branches
  const uint32_t item = it < 3u * nsplit ? (uniform(items[it / 3u]) & ~3u) | (it % 3u)
                                          : uniform(items[it - 2u * nsplit]);
  const uint32_t u = item >> 2;
  // 3: all channels (variant 1 looks at it per particle)
  const int chan = static_cast<int>(VAR == 1 ? uniform(item & 3u) : item & 3u);
  const UnitGeom ug = unit_geom_uniform(a, u);
  const int lx = ug.gx * 8 + (lane >> 3), ly = ug.gy * 8 + (lane & 7);
  clear_slots(s_wave[wave], lane);

  float l0 = 0.f, l1 = 0.f, l2 = 0.f;
  const bool pix_in = lx < ug.w && ly < ug.h;
  if (ug.accumulate == 2 && pix_in) {  // a later chunk: continue the chain
    const float *d = ug.pic + (static_cast<int64_t>(ug.x0s + lx) * ug.yres + (ug.y0s + ly)) * 3;
    l0 = d[0];
    l1 = d[1];
    l2 = d[2];
  }
  const uint32_t e0 = uniform(a.bin_off[u]), e1 = uniform(a.bin_off[u + 1]);
  // long lists are near the critical path: let their waves issue ahead of the
  // rest (priority 2; the producer/consumer workgroups, the critical path, run at 3)
  if (e1 - e0 >= a.prio_len) __builtin_amdgcn_s_setprio(2);
  walk_list<ADD, VAR, PPW>(a, ug, e0, e1, chan, lane, s_tab, s_wave[wave], l0, l1, l2);
  if (a.trace && lane == 0) {
    uint64_t *tr = a.trace + 4 * static_cast<uint64_t>(it);
    tr[0] = t_start;
    tr[1] = __builtin_amdgcn_s_memrealtime();
    tr[2] = static_cast<uint64_t>(e1 - e0) | (static_cast<uint64_t>(chan) << 32);
    tr[3] = static_cast<uint64_t>(__smid());
  }
  if (pix_in) {
    float *d = ug.pic + (static_cast<int64_t>(ug.x0s + lx) * ug.yres + (ug.y0s + ly)) * 3;
    const bool add = ug.accumulate == 1;
    if (chan == 3 || chan == 0) d[0] = add ? d[0] + l0 : l0;
    if (chan == 3 || chan == 1) d[1] = add ? d[1] + l1 : l1;
    if (chan == 3 || chan == 2) d[2] = add ? d[2] + l2 : l2;
  }
}

// ---------------------------------------------------------------------------
// Long ordered lists in segments.
//
// A pixel's chain l <- l + (l - q) m1 m2 contracts: what it held before is
// scaled by exp(-optical depth), and once that falls below the rounding of the
// sums, two chains through the same entries soon hold the same bits, whatever
// they started from.  A list is therefore cut into segments that are walked at
// once, each from 0 a warm-up stretch before its first entry, and the kept
// states then prove the result: where the state a segment had at its first
// entry equals, bit for bit in all 64 pixels, the state the segment before it
// ended with, the segment walked exactly what the serial chain walks.  Where
// they differ, k_seg_join walks on serially from the true state until it meets
// a kept state of the segment.  So the result is the serial chain's in every
// case; the sampled optical depths only decide where it is cut and how often a
// stretch is walked twice.  (The 16M-particle frames: of 1885 to 4292 segments
// 1 to 4 % differ, for 2.5 steps of 1024 entries each; with 24 optical depths
// at the least covered pixel.  20, 30 and 36 are 0 to 8 % slower.)
//
// The walk is the 8x8 splat's, bound by LDS returns as that is; sampling,
// windows and cuts take 0.15 to 0.3 ms before it.

// Flags cleared; the units of at least 2 * seglen entries collected, with a
// chunk (candidate, first of 8 samples) per wave of k_seg_sample.
constexpr uint32_t kSegChunk = 8;

__global__ __launch_bounds__(256) void k_seg_cand(SplatArgs a, uint32_t nunits, SegArgs g) {
  for (int64_t i = gtid(); i < nunits; i += gstride()) {
    const uint32_t u = static_cast<uint32_t>(i);
    g.flag[u] = 0u;
    const uint32_t len = a.bin_off[u + 1] - a.bin_off[u];
    if (len < 2u * g.seglen) continue;
    const UnitGeom G = unit_geom(a, u);
    if (G.gx * 8 >= G.w || G.gy * 8 >= G.h) continue;
    const uint32_t ns = len / kSegSample, nc = (ns + kSegChunk - 1u) / kSegChunk;
    const uint32_t k = atomicAdd(&g.cnt[SC_CAND], 1u);
    const uint32_t b = atomicAdd(&g.cnt[SC_SAMPLE], ns), c0 = atomicAdd(&g.cnt[SC_CHUNK], nc);
    g.cand[k] = SegCand{u, b, 0u};
    for (uint32_t c = 0; c < nc; ++c) {
      g.chunk[2 * (c0 + c)] = k;
      g.chunk[2 * (c0 + c) + 1] = c * kSegChunk;
    }
  }
}

// A wave per chunk of samples: each pixel's absorption per channel over the
// sample's batch (the additive walk of the records sums -a_c * att).
__global__ __launch_bounds__(256) void k_seg_sample(SplatArgs a, SegArgs g) {
  __shared__ float s_tab[2048];
  __shared__ SplatLds<1, 4> s_wave[4];
  const uint32_t nc = uniform(g.cnt[SC_CHUNK]);
  if (blockIdx.x * 4u >= nc) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < 2048; i += 256) s_tab[i] = a.exptab[i];
  __syncthreads();
  const uint32_t ci = blockIdx.x * 4u + wave;
  if (ci >= nc) return;
  const uint32_t k = uniform(g.chunk[2 * ci]), s0 = uniform(g.chunk[2 * ci + 1]);
  const uint32_t u = uniform(g.cand[k].unit);
  const UnitGeom ug = unit_geom_uniform(a, u);
  const uint32_t b0 = uniform(a.bin_off[u]), len = uniform(a.bin_off[u + 1]) - b0;
  const uint32_t s1 = min(s0 + kSegChunk, len / kSegSample);
  const bool pix_in = ug.gx * 8 + (lane >> 3) < ug.w && ug.gy * 8 + (lane & 7) < ug.h;
  uint32_t on = 0u;
  float *out = g.sample + (static_cast<uint64_t>(uniform(g.cand[k].samples)) + s0) * 192u;
  for (uint32_t i = s0; i < s1; ++i, out += 192) {
    const uint32_t at = b0 + i * kSegSample + (kSegSample - 64u) / 2u;
    float l0 = 0.f, l1 = 0.f, l2 = 0.f;
    walk_list<1, 4, 0>(a, ug, at, at + 64u, 3, lane, s_tab, s_wave[wave], l0, l1, l2);
    out[lane] = -l0;
    out[64 + lane] = -l1;
    out[128 + lane] = -l2;
    if (pix_in) on |= (l0 != 0.f ? 1u : 0u) | (l1 != 0.f ? 2u : 0u) | (l2 != 0.f ? 4u : 0u);
  }
  on = (__any(on & 1u) ? 1u : 0u) | (__any(on & 2u) ? 2u : 0u) | (__any(on & 4u) ? 4u : 0u);
  if (lane == 0 && on) atomicOr(&g.cand[k].on, on);
}

// Warm-up: the optical depth at the least covered pixel of the block, by the
// samples, in the channels the list absorbs in.  (exp(-17) is the rounding of a
// sum; the rest is for the bits to meet, and for the samples' error.)
constexpr float kSegDepth = 24.f;
constexpr uint32_t kSegCuts = 2048;  // per list at most

// A wave per chunk of samples, lane = pixel: per sample the shortest window of
// samples up to it that holds kSegDepth in every pixel (0: none of kSegWarm).
__global__ __launch_bounds__(256) void k_seg_win(SplatArgs a, SegArgs g) {
  const uint32_t nc = uniform(g.cnt[SC_CHUNK]);
  const int lane = threadIdx.x & 63;
  const uint32_t ci = uniform(blockIdx.x * 4u + (threadIdx.x >> 6));
  if (ci >= nc) return;
  const uint32_t k = uniform(g.chunk[2 * ci]), s0 = uniform(g.chunk[2 * ci + 1]);
  const uint32_t u = uniform(g.cand[k].unit), on = uniform(g.cand[k].on);
  const UnitGeom ug = unit_geom_uniform(a, u);
  const uint32_t ns = (uniform(a.bin_off[u + 1]) - uniform(a.bin_off[u])) / kSegSample;
  const uint32_t base = uniform(g.cand[k].samples);
  const float *sm = g.sample + static_cast<uint64_t>(base) * 192u + lane;
  const bool pix_in = ug.gx * 8 + (lane >> 3) < ug.w && ug.gy * 8 + (lane & 7) < ug.h;
  constexpr float kNeed = kSegDepth * 64.f / kSegSample;
  const float n0 = (pix_in && (on & 1u)) ? kNeed : 0.f, n1 = (pix_in && (on & 2u)) ? kNeed : 0.f,
              n2 = (pix_in && (on & 4u)) ? kNeed : 0.f;
  for (uint32_t i = s0; i < min(s0 + kSegChunk, ns); ++i) {
    float d0 = 0.f, d1 = 0.f, d2 = 0.f;
    uint32_t w = 0, found = 0;
    const uint32_t most = min(i + 1u, kSegWarm);
    while (on && !found && w < most) {
      const float *q = sm + static_cast<uint64_t>(i - w) * 192u;
      d0 += q[0];
      d1 += q[64];
      d2 += q[128];
      ++w;
      if (__all(d0 >= n0 && d1 >= n1 && d2 >= n2)) found = w;
    }
    if (lane == 0) g.win[base + i] = found;
  }
}

// A wave per candidate: a cut is made seglen entries after the last one as soon
// as the samples before it hold a warm-up.  Segments that would take much
// longer than the others are walked by channel, three waves each (about half
// the time, at 1.5 times the work); a list with a still longer one keeps its
// other path.
__global__ __launch_bounds__(64) void k_seg_cut(SplatArgs a, SegArgs g) {
  __shared__ uint32_t s_cut[kSegCuts], s_warm[kSegCuts];
  if (blockIdx.x >= g.cnt[SC_CAND]) return;
  const int lane = threadIdx.x;
  const uint32_t u = uniform(g.cand[blockIdx.x].unit);
  const uint32_t b0 = uniform(a.bin_off[u]), len = uniform(a.bin_off[u + 1]) - b0;
  const uint32_t ns = len / kSegSample;
  const uint32_t *win = g.win + uniform(g.cand[blockIdx.x].samples);
  const uint32_t smin = g.seglen / kSegSample;
  uint32_t cut = 0, n = 0, longest = 0, extra = 0;
  for (uint32_t base = 0; base < ns; base += 64u) {
    const uint32_t w = base + lane < ns ? win[base + lane] : 0u;
    uint64_t can = __ballot(w != 0u);
    while (can) {
      const int j = __ffsll(static_cast<long long>(can)) - 1;
      can &= can - 1u;
      const uint32_t hi = base + j + 1u;  // samples before the cut
      if (hi - cut < smin || ns - hi < smin / 2u || n >= kSegCuts) continue;
      const uint32_t wj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w), j));
      if (lane == 0) {
        s_cut[n] = hi;
        s_warm[n] = wj;
      }
      const uint32_t walk = hi - cut + extra;
      longest = max(longest, walk);
      extra = wj;
      cut = hi;
      ++n;
    }
  }
  longest = max(longest, ns - cut + extra);
  if (n == 0 || longest > g.longest) return;
  if (lane == 0) {
    uint32_t m = 0, slots = 0, e = 0, x = 0;  // walks (three per long segment), kept states
    for (uint32_t k = 0; k <= n; ++k) {
      const uint32_t hi = k < n ? s_cut[k] : ns;
      m += hi - e + x > g.split ? 3u : 1u;
      slots += 1u + ((k < n ? hi * kSegSample : len) - e * kSegSample + kSegCheck - 1u) / kSegCheck;
      e = hi;
      x = k < n ? s_warm[k] : 0u;
    }
    uint32_t first = atomicAdd(&g.cnt[SC_SEG], m), slot = atomicAdd(&g.cnt[SC_SLOT], slots);
    const uint32_t li = atomicAdd(&g.cnt[SC_LIST], 1u);
    g.lists[li] = SegList{u, first, m};
    g.flag[u] = 1u;
    e = x = 0;
    for (uint32_t k = 0; k <= n; ++k) {
      const uint32_t hi = k < n ? s_cut[k] : ns;
      Seg S{li, b0 + e * kSegSample, k < n ? b0 + hi * kSegSample : b0 + len, x * kSegSample, slot, 3u};
      if (hi - e + x > g.split)
        for (uint32_t c = 0; c < 3u; ++c) {
          S.chan = c;
          g.segs[first++] = S;
        }
      else
        g.segs[first++] = S;
      slot += 1u + (S.e1 - S.e0 + kSegCheck - 1u) / kSegCheck;
      e = hi;
      x = k < n ? s_warm[k] : 0u;
    }
  }
}

__device__ __forceinline__ void keep_state(float *st, int lane, uint32_t chan, float l0, float l1,
                                           float l2) {
  if (chan == 3u || chan == 0u) st[lane] = l0;
  if (chan == 3u || chan == 1u) st[64 + lane] = l1;
  if (chan == 3u || chan == 2u) st[128 + lane] = l2;
}
// One wave per segment.  Kept states: slot 0 at its first entry, slot j after j
// * kSegCheck entries, the last after its last entry.
__global__ __launch_bounds__(256, 4) void k_seg_walk(SplatArgs a, SegArgs g, uint32_t nseg,
                                                     float *states) {
  __shared__ float s_tab[2048];
  __shared__ SplatLds<0, 4> s_wave[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < 2048; i += 256) s_tab[i] = a.exptab[i];
  __syncthreads();
  const uint32_t si = blockIdx.x * 4u + wave;
  if (si >= nseg) return;
  const Seg *S = g.segs + si;
  const uint32_t li = uniform(S->list), e0 = uniform(S->e0), e1 = uniform(S->e1);
  const uint32_t warm = uniform(S->warm), u = uniform(g.lists[li].unit), chan = uniform(S->chan);
  const UnitGeom ug = unit_geom_uniform(a, u);
  clear_slots(s_wave[wave], lane);
  __builtin_amdgcn_s_setprio(2);
  float l0 = 0.f, l1 = 0.f, l2 = 0.f;
  float *st = states + static_cast<uint64_t>(uniform(S->slot)) * 192u;
  uint32_t pos = e0 - warm, next = e0;
  if (warm == 0) {  // the list's first
    const int lx = ug.gx * 8 + (lane >> 3), ly = ug.gy * 8 + (lane & 7);
    if (ug.accumulate == 2 && lx < ug.w && ly < ug.h) {  // a later chunk: continue the chain
      const float *d = ug.pic + (static_cast<int64_t>(ug.x0s + lx) * ug.yres + (ug.y0s + ly)) * 3;
      l0 = d[0];
      l1 = d[1];
      l2 = d[2];
    }
    if (a.trace && lane == 0 && (chan == 3u || chan == 0u))
      a.trace[4 * static_cast<uint64_t>(li)] = __builtin_amdgcn_s_memrealtime();
    next = e0 + kSegCheck;
    st += 192;
  }
  while (pos < e1) {
    next = min(next, e1);
    walk_list<0, 4, 0>(a, ug, pos, next, static_cast<int>(chan), lane, s_tab, s_wave[wave], l0, l1,
                       l2);
    keep_state(st, lane, chan, l0, l1, l2);
    st += 192;
    pos = next;
    next = pos + kSegCheck;
  }
}

// Three waves per list, one a channel: the segments' states joined, then the block's
// pixels.  A channel walks a segment again until it meets a kept state, at about 100
// ns per entry (one wave for all channels: 200), so where the samples do not represent
// the lists at all a pass ends at worst 100 ns per entry of its longest cut list
// after its other work, twice a producer/consumer workgroup's 48.  (Absorption in the
// sampled batch of 64 in 2048 only: four such lists of 1M in 273M entries 65 ms
// without segments, 93 here, 105 with one wave; 23 of 1.2M in 229M 53, 122 and 140;
// 1296 of 160k 39, 40 and 32.  Handing such lists to those workgroups after all
// measured 101, 95 and 39, and a launch of them that finds none delays a batch by 8 %,
// as each waits for a whole CU.)
__global__ __launch_bounds__(64) void k_seg_join(SplatArgs a, SegArgs g, const float *states) {
  __shared__ float s_tab[2048];
  __shared__ SplatLds<0, 4> s_wave;
  const int lane = threadIdx.x, c = static_cast<int>(blockIdx.x % 3u);
  for (int i = lane; i < 2048; i += 64) s_tab[i] = a.exptab[i];
  __syncthreads();
  const SegList &L = g.lists[blockIdx.x / 3u];
  const uint32_t u = uniform(L.unit), n = uniform(L.n), first = uniform(L.first);
  const UnitGeom ug = unit_geom_uniform(a, u);
  clear_slots(s_wave, lane);
  float l[3] = {0.f, 0.f, 0.f};
  auto chain = [&]() -> float & { return c == 0 ? l[0] : c == 1 ? l[1] : l[2]; };
  uint64_t code = 4;  // the trace's channel code
  for (uint32_t k = 0; k < n; ++k) {
    const Seg *S = g.segs + first + k;
    const uint32_t chan = uniform(S->chan);
    if (chan != 3u) code |= 1u;
    if (chan == 1u || chan == 2u) continue;  // (walks of the segment before)
    const uint32_t e0 = uniform(S->e0), e1 = uniform(S->e1);
    const float *st = states + static_cast<uint64_t>(uniform(S->slot)) * 192u + 64 * c + lane;
    const float *end = st + 192u * ((e1 - e0 + kSegCheck - 1u) / kSegCheck);
    // the wave's state is the kept one in all bits
    auto is_state = [&]() {
      return __all(__float_as_uint(*st) == __float_as_uint(chain())) != 0;
    };
    bool met = k == 0 || is_state();
    for (uint32_t pos = e0; !met && pos < e1;) {
      const uint32_t next = min(pos + kSegCheck, e1);
      walk_list<0, 4, 0>(a, ug, pos, next, c, lane, s_tab, s_wave, l[0], l[1], l[2]);
      pos = next;
      st += 192;
      met = is_state();
    }
    if (met) chain() = *end;
  }
  if (a.trace && c == 0 && lane == 0) {
    uint64_t *tr = a.trace + 4 * static_cast<uint64_t>(blockIdx.x / 3u);
    tr[1] = __builtin_amdgcn_s_memrealtime();
    tr[2] = static_cast<uint64_t>(a.bin_off[u + 1] - a.bin_off[u]) | (code << 32);
    tr[3] = static_cast<uint64_t>(__smid());
  }
  const int lx = ug.gx * 8 + (lane >> 3), ly = ug.gy * 8 + (lane & 7);
  if (lx < ug.w && ly < ug.h) {
    float *d = ug.pic + (static_cast<int64_t>(ug.x0s + lx) * ug.yres + (ug.y0s + ly)) * 3 + c;
    *d = ug.accumulate == 1 ? *d + chain() : chain();
  }
}

// ---------------------------------------------------------------------------
// Long lists: producer / consumer workgroups, one per 8x8 block, all three
// colour channels.
//
// A block whose list holds thousands to hundreds of thousands of particles is
// near the critical path of the frame: its pixels' update chains are serial.
// Such a block gets a 768-thread workgroup.  Wave 0 is the consumer: lane =
// pixel, and per particle it only applies, per channel c,
//     l_c += ((l_c - q_c) * m1_c) * m2     (ordered)     l_c += t_c   (additive)
// with operands that reproduce render_new's update bit for bit
// (splotch_host.cc:615, 648-658):
//   Taylor branch   m1 = a,  m2 = att           -> ((l - q) * a) * att
//   expm1 branch    m1 = expm1(att * a), m2 = 1 -> (l - q) * em      (x*1 == x)
//   additive        t = a * att
//   outside         m1 = m2 = t = 0             -> l + (+-0) == l
// (l starts at +0 and a float sum is -0 only if both terms are -0, so l is
// never -0 and adding a zero leaves it unchanged, as the reference's skip.
// For finite records l - q stays finite, so (l - q) * 0 is a zero.)
// Waves 1..11 run a pipeline ahead of the consumer: particle set-up three
// steps ahead (tile-frame position, box, Gaussian width, emission /
// absorption; splotch_host.cc:462-476, 591-632), the separable column / row
// tables two steps ahead (splotch_host.cc:596-607), and the operands one step
// ahead, with lane = pixel and each producer wave on its own four particles
// of the step: the producers do the table work of the lane-per-pixel kernel
// once for all three channels, the consumer four operations per channel.
// The consumer runs at a higher wave priority than the producers, which
// share its SIMD.
// Records reach the set-up through LDS in super-batches that wave 1 loads
// about five steps before their use, so the gather latency stays off the
// critical path.  Three waves per SIMD hide most of the LDS latency of the
// stages; a workgroup occupies its CU (LDS and registers).
constexpr int kPW = 11;                // producer waves (three waves per SIMD)
constexpr int kPB = 4;                 // particles per producer wave and step
constexpr int kB = kPW * kPB;          // particles per step
constexpr int kQ = 4;                  // operand stage: particles per group of LDS reads
static_assert(kPB % kQ == 0, "groups tile a producer's particles");
constexpr int kPThreads = 64 * (kPW + 1);
constexpr int kPProd = 64 * kPW;       // producer lanes
constexpr int kSB = 5;                 // steps per record super-batch
constexpr int kSR = kSB * kB;          // records per super-batch
constexpr int kSRL = (kSR + 63) / 64;  // records per wave-1 lane and super-batch
static_assert(kSB >= 5, "a super-batch is stored four steps before its first use");
constexpr int kSRP = kSRL * 64;        // staging row: whole wave stores (tail unused)
static_assert(kB <= 64, "fast-particle mask is 64 bits");

struct PcPart {
  float posx, posy, radsq, stp;
  int bx0, bx1, by0, by1;
};

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int ADD>
__global__ __launch_bounds__(kPThreads) void k_splat_pc(SplatArgs a, const uint32_t *items,
                                                        uint32_t npc, ItemCounts dc) {
  // device counts: *dc.npc items from *dc.first on; the rest of the grid
  // (sized for a capacity) has no work (uniform per workgroup, before any
  // barrier)
  if (dc.npc && blockIdx.x >= *dc.npc) return;
  // One LDS block with the exp table at address 0, so that a table entry's
  // address is its byte offset (no base to add per lookup).
  struct Lds {
    float tab[2048];
    float4 op[2][kB][64];   // consumer operands (m1_0, m1_1, m1_2, m2) / (t0, t1, t2, 0)
    float4 ca[4][kB];       // (a0, a1, a2, max |a|)
    float4 cq[4][kB];       // (q0, q1, q2, 0)
    Rec rec[2][kSRP];       // staged records, two super-batches
    PcPart part[2][kB];
    uint64_t fast[4];       // bit k: particle k has every a_c in [kFastA, 0]
    uint32_t cm[2][kB][8];  // column row-masks
    float p2[2][kB][8];     // column factors
    float p1[2][kB][8];     // row factors
  };
  __shared__ Lds L;
  float(&s_tab)[2048] = L.tab;
  Rec(&s_rec)[2][kSRP] = L.rec;
  PcPart(&s_part)[2][kB] = L.part;
  float4(&s_ca)[4][kB] = L.ca;
  float4(&s_cq)[4][kB] = L.cq;
  uint64_t(&s_fast)[4] = L.fast;
  uint32_t(&s_cm)[2][kB][8] = L.cm;
  float(&s_p2)[2][kB][8] = L.p2;
  float(&s_p1)[2][kB][8] = L.p1;
  float4(&s_op)[2][kB][64] = L.op;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = static_cast<int>(uniform(static_cast<uint32_t>(tid >> 6)));
  const bool producer = wave >= 1;
  // table task rank: waves 4 and 8 share SIMD 0 with the consumer (waves go
  // to the SIMDs in turn) and take the last, cheaper row tasks
  const int trank = (wave & 3) == 0 ? 8 + (wave >> 2) : wave - 1 - (wave >> 2);
  const int ptid = trank * 64 + lane;
  for (int i = tid; i < 2048; i += kPThreads) s_tab[i] = a.exptab[i];
  const uint32_t it = blockIdx.x + (dc.first ? uniform(*dc.first) : 0u);
  const uint64_t t_start = a.trace ? __builtin_amdgcn_s_memrealtime() : 0;
  const uint32_t u = uniform(items[it]) >> 2;
  const UnitGeom ug = unit_geom_uniform(a, u);
  const int gy = ug.gy, gx = ug.gx, x0s = ug.x0s, y0s = ug.y0s, w = ug.w, h = ug.h;
  const int bxo = gx * 8, byo = gy * 8;
  const uint32_t e0 = uniform(a.bin_off[u]), e1 = uniform(a.bin_off[u + 1]);
  const int n = static_cast<int>(e1 - e0);
  const int nbat = (n + kB - 1) / kB;
  const float expfac = a.expfac, tl = a.taylorlimit;
  const float expfac4 = 4.f * expfac;  // exact
  const int cx = lane >> 3, cy = lane & 7;  // producers and consumer: lane = pixel
  if (producer) __builtin_amdgcn_s_setprio(2);
  else __builtin_amdgcn_s_setprio(3);

  auto count = [&](int b) { return min(kB, n - b * kB); };
  // particle set-up of batch b (wave 1, lane = particle).  Lanes past the
  // batch (and batches past the list) use clamped records, which the
  // operand stage masks.
  auto setup = [&](int b, const Rec &R) {
    const float rfacr = R.r * a.rfac;
    const float posx = R.x - static_cast<float>(x0s), posy = R.y - static_cast<float>(y0s);
    PcPart P;
    P.posx = posx;
    P.posy = posy;
    P.bx0 = max(cvt_i32(posx - rfacr + 1), 0);
    P.bx1 = min(cvt_i32(posx + rfacr + 1), w);
    P.by0 = max(cvt_i32(posy - rfacr + 1), 0);
    P.by1 = min(cvt_i32(posy + rfacr + 1), h);
    P.radsq = rfacr * rfacr;
    const float sigma = a.h2sigma * R.r;
    P.stp = -1.f / (sigma * sigma);
    const float a0 = -R.e0, a1 = -R.e1, a2 = -R.e2;
    float q0 = 0.f, q1 = 0.f, q2 = 0.f, mx = 0.f;
    bool fast = false;
    if (!ADD) {
      const float g = ug.grayabsorb;
      q0 = R.e0 / (R.e0 + g);
      q1 = R.e1 / (R.e1 + g);
      q2 = R.e2 / (R.e2 + g);
      mx = fmaxf(fabsf(a0), fmaxf(fabsf(a1), fabsf(a2)));
      fast = a0 >= kFastA && a0 <= 0.f && a1 >= kFastA && a1 <= 0.f && a2 >= kFastA &&
             a2 <= 0.f && finite3(q0, q1, q2);
    }
    const uint64_t fb = __ballot(fast);
    if (lane < kB) {
      s_part[b & 1][lane] = P;
      s_ca[b & 3][lane] = make_float4(a0, a1, a2, mx);
      s_cq[b & 3][lane] = make_float4(q0, q1, q2, 0.f);
    }
    if (lane == 0) s_fast[b & 3] = fb;  // bits past the batch are not read
  };
  // Column ranges / factors and row factors of batch b into slot b & 1: task
  // (particle k, j) is column j (j < 8) or row j - 8.  Unrolled over a lane's
  // tasks with every LDS read issued before the arithmetic that uses it.
  auto tables = [&](int b) {
    const int ts = b & 1, cnt = count(b);
    const PcPart(&part)[kB] = s_part[b & 1];
    constexpr int NT = (kB * 16 + kPProd - 1) / kPProd;
    PcPart P[NT];
    int kt[NT], jt[NT];
    bool vt[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      // tasks [0, 8 kB) are columns, [8 kB, 16 kB) rows, so a wave runs
      // one kind (the column path is the longer one)
      const int t = ptid + i * kPProd;
      const bool row = t >= kB * 8;
      const int tr = row ? t - kB * 8 : t;
      vt[i] = t < kB * 16 && (tr >> 3) < cnt;
      kt[i] = vt[i] ? tr >> 3 : 0;
      jt[i] = vt[i] ? (tr & 7) + (row ? 8 : 0) : 0;
      P[i] = part[kt[i]];
    }
    float arg[NT], dd[NT];
    bool on[NT];
    uint32_t mk[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int j = jt[i];
      mk[i] = 0;
      if (j < 8) {
        const int x = bxo + j;
        on[i] = x >= P[i].bx0 && x < P[i].bx1;
        const float dxsq = (static_cast<float>(x) - P[i].posx) * (static_cast<float>(x) - P[i].posx);
        const float dy = sqrtf(P[i].radsq - dxsq);
        const int lo = max(P[i].by0, cvt_i32(P[i].posy - dy + 1));
        const int hi = min(P[i].by1, cvt_i32(P[i].posy + dy + 1));
        const int r0 = min(max(lo - byo, 0), 8), r1 = min(max(hi - byo, 0), 8);
        if (on[i] && hi > lo && r1 > r0) mk[i] = ((1u << r1) - 1u) & ~((1u << r0) - 1u);
        arg[i] = P[i].stp * dxsq;
      } else {
        const int y = byo + (j - 8);
        on[i] = y >= P[i].by0 && y < P[i].by1;
        const float dyf = static_cast<float>(y) - P[i].posy;
        arg[i] = P[i].stp * dyf * dyf;
      }
      dd[i] = on[i] ? xop(s_tab, arg[i], expfac) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      if (!vt[i]) continue;
      const int k = kt[i], j = jt[i];
      if (j < 8) {
        s_cm[ts][k][j] = mk[i];
        s_p2[ts][k][j] = dd[i];
      } else {
        s_p1[ts][k][j - 8] = dd[i];
      }
    }
  };
  // Consumer operands of batch b: producer wave pw covers particles
  // [pw * kPB, pw * kPB + kPB) of the batch, lane = pixel, in groups of kQ
  // with every LDS read of a group issued first.  Particles past the batch
  // get zero operands.
  // FAST: every particle of the group has all a_c in [kFastA, 0], so the
  // exp-table index is trunc(p) with p in [0, 2^20).
  auto operands_group = [&](int b, int kb, auto fast_tag) {  // particles [kb, kb + kQ)
    constexpr bool FAST = decltype(fast_tag)::value;
    const int ts = b & 1, cs = b & 3, cnt = count(b);
    uint32_t mk[kQ];
    float p1[kQ], p2[kQ];
    float4 ca[kQ];
#pragma unroll
    for (int j = 0; j < kQ; ++j) {
      const int k = kb + j;
      mk[j] = s_cm[ts][k][cx];
      p1[j] = s_p1[ts][k][cy];
      p2[j] = s_p2[ts][k][cx];
      ca[j] = s_ca[cs][k];
    }
    float4 op[kQ];
    if (ADD) {
#pragma unroll
      for (int j = 0; j < kQ; ++j) {
        const float at = p1[j] * p2[j];
        const bool in = (kb + j < cnt) && ((mk[j] >> cy) & 1u);
        op[j] = in ? make_float4(ca[j].x * at, ca[j].y * at, ca[j].z * at, 0.f)
                   : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < kQ; ++j) s_op[ts][kb + j][lane] = op[j];
      return;
    }
    float at[kQ];
    bool in[kQ], tay[kQ];
    uint32_t tb = 0;  // bit j: every pixel of particle j takes the Taylor branch or is outside
#pragma unroll
    for (int j = 0; j < kQ; ++j) {
      at[j] = p1[j] * p2[j];
      in[j] = (kb + j < cnt) && ((mk[j] >> cy) & 1u);
      tay[j] = (ca[j].w * at[j]) < tl;
      if (__ballot(tay[j] || !in[j]) == ~0ull) tb |= 1u << j;
    }
    // One straight-line body per pattern: the all-Taylor particles skip the
    // exp-table work, the others' table reads are all issued before their
    // arithmetic.  op = (a_c, att) for a Taylor pixel, (expm1(att a_c), 1)
    // otherwise, zero outside.
    auto body = [&](auto tb_tag) {
      constexpr uint32_t TB = decltype(tb_tag)::value;
      float g0[kQ], g1[kQ], g2[kQ], pg0[kQ], pg1[kQ], pg2[kQ];
      float u0[kQ], w0[kQ], u1[kQ], w1[kQ], u2[kQ], w2[kQ];
#pragma unroll
      for (int j = 0; j < kQ; ++j) {
        if ((TB >> j) & 1u) continue;
        g0[j] = at[j] * ca[j].x;
        g1[j] = at[j] * ca[j].y;
        g2[j] = at[j] * ca[j].z;
        if (FAST) {
          xtab_fast(s_tab, g0[j], expfac4, u0[j], w0[j]);
          xtab_fast(s_tab, g1[j], expfac4, u1[j], w1[j]);
          xtab_fast(s_tab, g2[j], expfac4, u2[j], w2[j]);
        } else {
          pg0[j] = g0[j] * expfac;
          pg1[j] = g1[j] * expfac;
          pg2[j] = g2[j] * expfac;
          const int i0 = xexp_index(pg0[j]), i1 = xexp_index(pg1[j]), i2 = xexp_index(pg2[j]);
          u0[j] = s_tab[i0 >> 10];
          w0[j] = s_tab[1024 + (i0 & 1023)];
          u1[j] = s_tab[i1 >> 10];
          w1[j] = s_tab[1024 + (i1 & 1023)];
          u2[j] = s_tab[i2 >> 10];
          w2[j] = s_tab[1024 + (i2 & 1023)];
        }
      }
#pragma unroll
      for (int j = 0; j < kQ; ++j) {
        if ((TB >> j) & 1u) {
          op[j] = in[j] ? make_float4(ca[j].x, ca[j].y, ca[j].z, at[j])
                        : make_float4(0.f, 0.f, 0.f, 0.f);
          continue;
        }
        float em0, em1, em2;
        if (FAST) {
          em0 = (fabsf(g0[j]) < tl) ? g0[j] : u0[j] * w0[j] - 1.f;
          em1 = (fabsf(g1[j]) < tl) ? g1[j] : u1[j] * w1[j] - 1.f;
          em2 = (fabsf(g2[j]) < tl) ? g2[j] : u2[j] * w2[j] - 1.f;
        } else {
          em0 = xexpm1_finish(g0[j], pg0[j], u0[j], w0[j], tl);
          em1 = xexpm1_finish(g1[j], pg1[j], u1[j], w1[j], tl);
          em2 = xexpm1_finish(g2[j], pg2[j], u2[j], w2[j], tl);
        }
        op[j] = in[j] ? make_float4(tay[j] ? ca[j].x : em0, tay[j] ? ca[j].y : em1,
                                    tay[j] ? ca[j].z : em2, tay[j] ? at[j] : 1.f)
                      : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < kQ; ++j) s_op[ts][kb + j][lane] = op[j];
    };
    static_assert(kQ == 4, "one body per pattern of four particles");
    switch (uniform(tb)) {
#define SPLHIP_PCT(T) case T: body(std::integral_constant<uint32_t, T>{}); break;
      SPLHIP_PCT(0) SPLHIP_PCT(1) SPLHIP_PCT(2) SPLHIP_PCT(3)
      SPLHIP_PCT(4) SPLHIP_PCT(5) SPLHIP_PCT(6) SPLHIP_PCT(7)
      SPLHIP_PCT(8) SPLHIP_PCT(9) SPLHIP_PCT(10) SPLHIP_PCT(11)
      SPLHIP_PCT(12) SPLHIP_PCT(13) SPLHIP_PCT(14) SPLHIP_PCT(15)
#undef SPLHIP_PCT
    }
  };
  auto operands = [&](int b, int pw) {
    const uint64_t f64 = s_fast[b & 3];
    const uint64_t fb = (static_cast<uint64_t>(uniform(static_cast<uint32_t>(f64 >> 32))) << 32) |
                        uniform(static_cast<uint32_t>(f64));
#pragma unroll
    for (int g = 0; g < kPB; g += kQ) {
      const int kb = pw * kPB + g;
      const uint64_t want = ((uint64_t(1) << kQ) - 1u) << kb;
      if (!ADD && (fb & want) == want)
        operands_group(b, kb, std::true_type{});
      else
        operands_group(b, kb, std::false_type{});
    }
  };

  // Records through LDS: wave 1 holds the next super-batch's records and the
  // one after that's list indices in registers (positions clamped to the list
  // end), and stores a super-batch into its half of s_rec four steps before
  // its first set-up.
  auto entry = [&](int J, int r) { return a.ent[e0 + min(J * kSR + r * 64 + lane, n - 1)]; };
  // records as two 4-float halves in native vector registers (the arrays
  // must stay in registers: struct copies would keep them in memory)
  typedef float v4f __attribute__((ext_vector_type(4)));
  v4f RA[kSRL], RB[kSRL];
  uint32_t I[kSRL];
  auto load_recs = [&]() {
#pragma unroll
    for (int r = 0; r < kSRL; ++r) {
      const v4f *src = reinterpret_cast<const v4f *>(a.recs + I[r]);
      RA[r] = src[0];
      RB[r] = src[1];
    }
  };
  auto store_recs = [&](int slot) {
#pragma unroll
    for (int r = 0; r < kSRL; ++r) {
      v4f *dst = reinterpret_cast<v4f *>(&s_rec[slot][r * 64 + lane]);
      dst[0] = RA[r];
      dst[1] = RB[r];
    }
  };
  if (wave == 1) {
#pragma unroll
    for (int r = 0; r < kSRL; ++r) I[r] = entry(0, r);
    load_recs();
    store_recs(0);
#pragma unroll
    for (int r = 0; r < kSRL; ++r) I[r] = entry(1, r);
    load_recs();
#pragma unroll
    for (int r = 0; r < kSRL; ++r) I[r] = entry(2, r);
  }

  float l0 = 0.f, l1 = 0.f, l2 = 0.f;  // consumer: pixel lane
  const int hlx = bxo + cx, hly = byo + cy;
  const bool hpix = hlx < min(bxo + 8, w) && hly < min(byo + 8, h);
  float *hdst = ug.pic + (static_cast<int64_t>(x0s + hlx) * ug.yres + (y0s + hly)) * 3;
  if (!producer && ug.accumulate == 2 && hpix) {  // a later chunk: continue the chains
    l0 = hdst[0];
    l1 = hdst[1];
    l2 = hdst[2];
  }
  __syncthreads();  // s_tab, s_rec[0]
  for (int s = -3; s < nbat; ++s) {
    if (producer) {
      if (wave == 1) {
        const int b = s + 3;
        setup(b, s_rec[(b / kSB) & 1][(b % kSB) * kB + min(lane, kB - 1)]);
        if ((s + 4) % kSB == 0 && s + 4 > 0) {  // super-batch J starts next step
          const int J = (s + 4) / kSB;
          store_recs(J & 1);
          load_recs();
#pragma unroll
          for (int r = 0; r < kSRL; ++r) I[r] = entry(J + 2, r);
        }
      }
      if (s + 2 >= 0 && s + 2 < nbat) tables(s + 2);
      if (s + 1 >= 0 && s + 1 < nbat) operands(s + 1, wave - 1);
    } else if (s >= 0) {
      const float4(*op)[64] = s_op[s & 1];
      const float4 *cq = s_cq[s & 3];
      const int cnt = count(s);
      constexpr int C = 4;  // particles per group of reads
      static_assert(kB % C == 0, "groups tile the batch");
#pragma unroll
      for (int k0 = 0; k0 < kB; k0 += C) {
        if (k0 >= cnt) break;
        float4 m[C], q[C];
#pragma unroll
        for (int j = 0; j < C; ++j) {
          m[j] = op[k0 + j][lane];
          if (!ADD) q[j] = cq[k0 + j];
        }
#pragma unroll
        for (int j = 0; j < C; ++j) {
          if (ADD) {
            l0 = l0 + m[j].x;
            l1 = l1 + m[j].y;
            l2 = l2 + m[j].z;
          } else {
            l0 = l0 + ((l0 - q[j].x) * m[j].x) * m[j].w;
            l1 = l1 + ((l1 - q[j].y) * m[j].y) * m[j].w;
            l2 = l2 + ((l2 - q[j].z) * m[j].z) * m[j].w;
          }
        }
      }
    }
    lds_barrier();
  }
  if (a.trace && tid == 0) {
    uint64_t *tr = a.trace + 4 * static_cast<uint64_t>(it);
    tr[0] = t_start;
    tr[1] = __builtin_amdgcn_s_memrealtime();
    tr[2] = static_cast<uint64_t>(n) | (uint64_t(3) << 32);
    tr[3] = static_cast<uint64_t>(__smid());
  }
  if (!producer && hpix) {
    const bool add = ug.accumulate == 1;
    hdst[0] = add ? hdst[0] + l0 : l0;
    hdst[1] = add ? hdst[1] + l1 : l1;
    hdst[2] = add ? hdst[2] + l2 : l2;
  }
}

// ---------------------------------------------------------------------------
// Staged long lists.  A long list's pixel chains are serial, and in a
// lane-per-pixel wave (or a producer/consumer workgroup) the per-particle
// table work, not the chain, sets their pace.  The staged path moves that
// work off the chain and drops what a pixel's chain does not need: for every
// pixel only the entries whose footprint covers it, in list order.
//   k_stage_rows  (every CU) per batch of 64 entries: each pixel's coverage as
//                 a 64-bit mask, and each column's longest count of covering
//                 entries ("rows"), whose scan places the operands
//   k_stage_ops   (every CU) writes the rows' operands to HBM
//   k_stage_chain one wave per list, channel and pixel column streams them back
//                 and applies only the chain's own operations
//                 (splotch_host.cc:615, 648-658):
//     additive  l_c = l_c + t_c                 t_c = a_c * att
//     ordered   l_c = l_c + ((l_c - q_c) * m1_c) * m2
//               Taylor branch m1 = a, m2 = att; expm1 branch m1 =
//               expm1(att a), m2 = 1 (x * 1 == x)
// A pixel with fewer rows than its column gets t = +0, or q = m1 = m2 = 0, in
// the rest (l + +-0 == l: l starts at +0 and a float sum is -0 only if both
// terms are -0; l stays finite where every q_c of the pass is finite, and
// ordered lists are staged only then), so every pixel sees the reference's
// sums and compositing, rounded as it rounds them.
//
// Why rows: a long list of small particles covers a pixel with few of its
// entries (1M particles at 800^2: 17-40 %), and both the chains' length and
// the operands' HBM traffic shrink with the coverage.
//
// Layout: a stream per list and pixel column (8 pixels); its rows in groups
// of 4 per batch, group g of plane c being 8 float4 (lane = pixel row,
// components = the 4 rows) at ops + (c * stride + g) * 8, planes t_c
// (additive) or m1_0..2, m2, q_0..2 (ordered).  Streams lie list after list,
// column after column: group offsets gofs from the scan of the counts rows[],
// both indexed 8 (batches of the lists before) + h * nb + b for batch b of
// column h of a list of nb batches.  A list of n entries has at most
// stage_groups(n) groups per column.
__host__ __device__ constexpr uint32_t stage_groups(uint32_t len) {
  return (len + 31u) / 32u * 8u;
}
template <int ADD>
__host__ __device__ constexpr uint32_t stage_planes() {
  return ADD ? 3u : 7u;
}

// List offsets of the staged items (one workgroup): cbase (groups per column
// at most) and cbat (batches of 64 entries), exclusive, totals at [n]; and the
// counts of rows[] of lists [0, n1) and [n1, n).
__global__ __launch_bounds__(256) void k_stage_base(SplatArgs a, const uint32_t *items,
                                                    uint32_t n, uint32_t n1, uint32_t *cbase,
                                                    uint32_t *cbat, uint32_t *nrows,
                                                    const uint32_t *dn) {
  if (dn) n = min(n, *dn);
  __shared__ uint32_t s_g[256], s_b[256];
  __shared__ uint32_t s_carry[2];
  const int tid = threadIdx.x;
  if (tid == 0) s_carry[0] = s_carry[1] = 0;
  __syncthreads();
  for (uint32_t i0 = 0; i0 < n; i0 += 256) {
    const uint32_t i = i0 + tid;
    uint32_t len = 0;
    if (i < n) {
      const uint32_t u = items[i] >> 2;
      len = a.bin_off[u + 1] - a.bin_off[u];
    }
    const uint32_t g = stage_groups(len), b = (len + 63) / 64;
    s_g[tid] = g;
    s_b[tid] = b;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {  // inclusive scan (Hillis-Steele)
      const uint32_t vg = tid >= d ? s_g[tid - d] : 0u, vb = tid >= d ? s_b[tid - d] : 0u;
      __syncthreads();
      s_g[tid] += vg;
      s_b[tid] += vb;
      __syncthreads();
    }
    if (i < n) {
      cbase[i] = s_carry[0] + s_g[tid] - g;
      cbat[i] = s_carry[1] + s_b[tid] - b;
    }
    __syncthreads();
    if (tid == 0) {
      s_carry[0] += s_g[255];
      s_carry[1] += s_b[255];
    }
    __syncthreads();
  }
  if (tid == 0) {
    cbase[n] = s_carry[0];
    cbat[n] = s_carry[1];
    n1 = min(n1, n);
    const uint32_t b1 = n1 < n ? cbat[n1] : s_carry[1];
    nrows[0] = 8u * b1;
    nrows[1] = 8u * (s_carry[1] - b1);
  }
}

// A wave's run of consecutive batches of staged lists [i0, i1) (their batches
// split evenly over the launch's waves): visit(i, b, gb) for batch b of list
// i, the gb-th batch of all staged lists (all wave-uniform).
template <class F>
__device__ __forceinline__ void staged_batches(uint32_t i0, uint32_t i1, const uint32_t *cbat,
                                               uint32_t w, uint32_t nw, F &&visit) {
  const uint32_t first = uniform(cbat[i0]), total = uniform(cbat[i1]) - first;
  const uint32_t span = (total + nw - 1) / nw;
  uint32_t gb = first + w * span;
  const uint32_t gend = first + min(total, w * span + span);
  if (gb >= gend) return;
  // the staged item holding batch gb: cbat[lo] <= gb < cbat[lo + 1]
  uint32_t lo = i0, hi = i1;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (uniform(cbat[mid]) <= gb) lo = mid;
    else hi = mid;
  }
  uint32_t i = lo, b = gb - uniform(cbat[lo]);
  for (; gb < gend; ++gb, ++b) {
    while (gb >= uniform(cbat[i + 1])) {  // next list (uniform)
      ++i;
      b = 0;
    }
    visit(i, b, gb);
  }
}

// Pixel coverage of the batches of staged lists [i0, i1): lane = entry builds
// the 8 column masks of its footprint (tabulate's rule), lane = pixel gathers
// its bit of the 64 entries.  masks[64 gb + pixel]; rows as described above,
// counted from list i0 on.
__global__ __launch_bounds__(256) void k_stage_rows(SplatArgs a, const uint32_t *items,
                                                    uint32_t i0, uint32_t i1,
                                                    const uint32_t *cbat, uint64_t *masks,
                                                    uint32_t *rows, const uint32_t *dn) {
  if (dn) i1 = min(i1, *dn);
  if (i1 <= i0) return;  // the whole grid (device count)
  __builtin_amdgcn_s_setprio(3);
  // byte [column][entry]: bit r = row r of the block (16-byte rows, padded)
  __shared__ __align__(16) uint8_t s_cb[4][8][80];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cx = lane >> 3, cy = lane & 7;
  uint8_t(*cb)[80] = s_cb[wave];
  staged_batches(i0, i1, cbat, blockIdx.x * 4u + static_cast<uint32_t>(wave), gridDim.x * 4u,
                 [&](uint32_t i, uint32_t b, uint32_t gb) {
    const uint32_t u = uniform(items[i]) >> 2;
    const UnitGeom ug = unit_geom_uniform(a, u);
    const uint32_t e0 = uniform(a.bin_off[u]), e1 = uniform(a.bin_off[u + 1]);
    const uint32_t base = e0 + 64u * b;
    const int bxo = ug.gx * 8, byo = ug.gy * 8;
    uint32_t cm[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (base + lane < e1) {
      const Rec R = a.recs[a.ent[base + lane]];
      column_masks(a, R, ug.x0s, ug.y0s, ug.w, ug.h, bxo, byo, cm);
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) cb[c][lane] = static_cast<uint8_t>(cm[c]);
    wave_sync();
    // bit cy of the column's 64 bytes: four bytes at a time, their bits 0
    // gathered by a multiplication (bytes 0..3 to bits 24..27)
    uint32_t m[2] = {0, 0};
    const uint4 *src = reinterpret_cast<const uint4 *>(&cb[cx][0]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint4 v = src[q];
      const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t t = (w4[k] >> cy) & 0x01010101u;
        m[q >> 1] |= ((t * 0x01020408u) >> 24) << (16 * (q & 1) + 4 * k);
      }
    }
    wave_sync();
    masks[static_cast<size_t>(gb) * 64u + lane] =
        static_cast<uint64_t>(m[0]) | (static_cast<uint64_t>(m[1]) << 32);
    int n = __popc(m[0]) + __popc(m[1]);
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) n = max(n, __shfl_xor(n, d, 64));
    const uint32_t nb = (e1 - e0 + 63u) / 64u;
    if (cy == 0)
      rows[(uniform(cbat[i]) - uniform(cbat[i0])) * 8u + static_cast<uint32_t>(cx) * nb + b] =
          static_cast<uint32_t>(n + 3) >> 2;
  });
}

// Operands of staged lists [i0, i1): per batch lane = entry tabulates the
// block's Gaussian factors and the entry's constants, then lane = pixel walks
// its own covering entries (the bits of its mask), four rows at a time.
// Bound by its LDS gathers (three or four per row, plus six table lookups for
// an ordered one); only covering entries are computed and written.
template <int ADD>
__global__ __launch_bounds__(256) void k_stage_ops(SplatArgs a, const uint32_t *items,
                                                   uint32_t i0, uint32_t i1,
                                                   const uint32_t *cbase, const uint32_t *cbat,
                                                   const uint64_t *masks, const uint32_t *rows,
                                                   const uint32_t *gofs, float4 *ops,
                                                   uint64_t stride, const uint32_t *dn) {
  if (dn) i1 = min(i1, *dn);
  if (i1 <= i0) return;  // the whole grid (device count)
  // the chains wait for these operands: issue ahead of the 8x8 splat's waves
  __builtin_amdgcn_s_setprio(3);
  __shared__ float s_tab[2048];
  __shared__ float s_pre2[4][8][kPad];
  __shared__ float s_pre1[4][8][kPad];
  __shared__ float4 s_a[4][64];  // (a0, a1, a2, max |a|)
  __shared__ float4 s_q[4][ADD ? 1 : 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < 2048; i += 256) s_tab[i] = a.exptab[i];
  __syncthreads();
  float(*pre2)[kPad] = s_pre2[wave];
  float(*pre1)[kPad] = s_pre1[wave];
  float4 *ca = s_a[wave], *cq = s_q[wave];
  const float expfac = a.expfac, tl = a.taylorlimit;
  const int cx = lane >> 3, cy = lane & 7;
  float4 *phase = ops + static_cast<size_t>(uniform(cbase[i0])) * 64u;
  staged_batches(i0, i1, cbat, blockIdx.x * 4u + static_cast<uint32_t>(wave), gridDim.x * 4u,
                 [&](uint32_t i, uint32_t b, uint32_t gb) {
    const uint32_t u = uniform(items[i]) >> 2;
    const UnitGeom ug = unit_geom_uniform(a, u);
    const uint32_t e0 = uniform(a.bin_off[u]), e1 = uniform(a.bin_off[u + 1]);
    const uint32_t base = e0 + 64u * b, nb = (e1 - e0 + 63u) / 64u;
    uint64_t M = masks[static_cast<size_t>(gb) * 64u + lane];
    const uint32_t ri = (uniform(cbat[i]) - uniform(cbat[i0])) * 8u +
                        static_cast<uint32_t>(cx) * nb + b;
    const uint32_t ng = rows[ri];  // of the lane's column
    float4 *dst = phase + static_cast<size_t>(gofs[ri]) * 8u + cy;
    if (base + lane < e1) {
      const Rec R = a.recs[a.ent[base + lane]];
      block_factors(a, R, lane, ug.x0s, ug.y0s, ug.gx * 8, ug.gy * 8, s_tab, pre2, pre1, expfac);
      const float a0 = -R.e0, a1 = -R.e1, a2 = -R.e2;
      ca[lane] = make_float4(a0, a1, a2, fmaxf(fabsf(a0), fmaxf(fabsf(a1), fabsf(a2))));
      if (!ADD) {
        const float gray = ug.grayabsorb;
        cq[lane] = make_float4(R.e0 / (R.e0 + gray), R.e1 / (R.e1 + gray), R.e2 / (R.e2 + gray),
                               0.f);
      }
    }
    wave_sync();
    for (uint32_t j = 0; __ballot(M != 0) != 0; ++j) {
      float o[stage_planes<ADD>()][4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool in = M != 0;
        const int k = in ? __builtin_ctzll(M) : 0;  // slot 0 holds an entry of the batch
        M &= M - 1;
        const float at = pre1[cy][k] * pre2[cx][k];
        const float4 c = ca[k];
        if (ADD) {
          o[0][r] = in ? c.x * at : 0.f;
          o[1][r] = in ? c.y * at : 0.f;
          o[2][r] = in ? c.z * at : 0.f;
        } else {
          const float4 q = cq[k];
          const bool tay = (c.w * at) < tl;
          const float em0 = xexpm1_bf(s_tab, at * c.x, expfac, tl);
          const float em1 = xexpm1_bf(s_tab, at * c.y, expfac, tl);
          const float em2 = xexpm1_bf(s_tab, at * c.z, expfac, tl);
          o[0][r] = in ? (tay ? c.x : em0) : 0.f;
          o[1][r] = in ? (tay ? c.y : em1) : 0.f;
          o[2][r] = in ? (tay ? c.z : em2) : 0.f;
          o[stage_planes<ADD>() - 4][r] = in ? (tay ? at : 1.f) : 0.f;
          o[stage_planes<ADD>() - 3][r] = in ? q.x : 0.f;
          o[stage_planes<ADD>() - 2][r] = in ? q.y : 0.f;
          o[stage_planes<ADD>() - 1][r] = in ? q.z : 0.f;
        }
      }
      if (j < ng) {
#pragma unroll
        for (uint32_t c = 0; c < stage_planes<ADD>(); ++c)
          dst[(c * stride + j) * 8u] = make_float4(o[c][0], o[c][1], o[c][2], o[c][3]);
      }
    }
    wave_sync();
  });
}

// The chains of the staged lists.  A wave applies channel c of list i to
// pixel column h: workgroup (3 i + c) 8 + h.  One load brings 8 consecutive
// groups of a plane (32 rows, lane = group part * 8 + pixel, 1 KB) straight
// into a ring of kRing slots in LDS, so the loads in flight hold no registers;
// lanes [0, 8) run the chains and read the 8 parts of a slot one step ahead.
// A chain's wave is bound by its own issue: a dependent operation every 4.2
// clocks and about as much per other instruction (18 per 32 rows additive, 35
// ordered).  With the loads in registers, the copies at the end of each round
// waited for every load in flight (500k ordered at 512^2, longest list 79.7k
// entries: 15.3 -> 9.8 ns per entry).
// slots of the ring (ordered: one each of m1_c, m2 and q_c)
template <int ADD> constexpr int chain_ring() { return ADD ? 32 : 10; }
static_assert(2 * chain_ring<1>() * 8 <= static_cast<int>(kStagePad) &&
                  2 * chain_ring<0>() * 8 <= static_cast<int>(kStagePad),
              "the chains' loads past a stream stay inside the operands");

// LDS byte address of a shared object.
__device__ __forceinline__ uint32_t lds_address(const void *p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (const __attribute__((address_space(3))) void *)p));
}

// 16 bytes per lane from base + off into LDS at byte address lds + 16 lane.
// Completion counts in vmcnt; the caller waits for it.
__device__ __forceinline__ void load_lds16(uint32_t lds, const void *base, uint32_t off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}

template <int ADD>
__global__ __launch_bounds__(64) void k_stage_chain(
    SplatArgs a, const uint32_t *items, uint32_t i0, const uint32_t *cbase, const uint32_t *cbat,
    const uint32_t *rows, const uint32_t *gofs, const float4 *ops, uint64_t stride,
    const uint32_t *dn) {
  constexpr int kS = 8;  // groups per load
  constexpr int kRing = chain_ring<ADD>();
  constexpr int kPl = ADD ? 1 : 3;  // planes per slot
  static_assert(kPl * (kRing - 2) < 64, "vmcnt holds the loads in flight");
  typedef float v4f __attribute__((ext_vector_type(4)));
  __shared__ v4f ring[kRing][kPl][64];
  const uint32_t i = i0 + blockIdx.x / 24u;
  if (dn && i >= *dn) return;  // past the device count (uniform per workgroup)
  const uint32_t r3 = blockIdx.x % 24u;
  const int c = static_cast<int>(r3 >> 3), h = static_cast<int>(r3 & 7u);
  const int lane = threadIdx.x, pl = lane & 7;
  const uint64_t t_start = a.trace ? __builtin_amdgcn_s_memrealtime() : 0;
  __builtin_amdgcn_s_setprio(3);
  const uint32_t u = uniform(items[i]) >> 2;
  const UnitGeom ug = unit_geom_uniform(a, u);
  const uint32_t len = uniform(a.bin_off[u + 1]) - uniform(a.bin_off[u]);
  // the stream: its first group and number of groups (the list is not empty)
  const uint32_t nb = (len + 63u) / 64u;
  const uint32_t r0 = (uniform(cbat[i]) - uniform(cbat[i0])) * 8u + static_cast<uint32_t>(h) * nb;
  const uint32_t g0 = uniform(gofs[r0]);
  const uint32_t G = uniform(gofs[r0 + nb - 1u]) + uniform(rows[r0 + nb - 1u]) - g0;
  const int lx = ug.gx * 8 + h, ly = ug.gy * 8 + pl;
  const bool pix_in = lane < 8 && lx < min(ug.gx * 8 + 8, ug.w) && ly < min(ug.gy * 8 + 8, ug.h);
  float *d = ug.pic + (static_cast<int64_t>(ug.x0s + lx) * ug.yres + (ug.y0s + ly)) * 3 + c;
  float l = 0.f;
  if (ug.accumulate == 2 && pix_in) l = *d;  // a later chunk: continue the chain
  // l is in its register before the operand loads are issued
  asm volatile("" : "+v"(l));
  // A load: a wave-uniform base per plane, advanced by the scalar unit.  Loads
  // run up to 2 kRing steps past the stream's end (kStagePad groups of slack
  // behind the planes; never applied).
  const char *pm = reinterpret_cast<const char *>(
      ops + (static_cast<size_t>(uniform(cbase[i0])) * 8u + g0) * 8u);
  const char *pw = pm + 3u * stride * 128u, *pq = pw + static_cast<uint64_t>(c + 1) * stride * 128u;
  pm += static_cast<uint64_t>(c) * stride * 128u;
  const uint32_t vo = static_cast<uint32_t>(lane) * 16u;
  const uint32_t lds = lds_address(&ring[0][0][0]);
  auto refill = [&](int r) {  // slot r: the next load
    const uint32_t at = lds + static_cast<uint32_t>(r * kPl) * 1024u;
    load_lds16(at, pm, vo);
    pm += 1024;
    if (!ADD) {
      load_lds16(at + 1024u, pw, vo);
      load_lds16(at + 2048u, pq, vo);
      pw += 1024;
      pq += 1024;
    }
  };
  struct Step {  // one load's 32 rows: m1_c (or t_c), m2 and q_c
    v4f m[kS], w[ADD ? 1 : kS], q[ADD ? 1 : kS];
  };
  auto read = [&](int r) {  // slot r, once its loads have landed
    // loads complete in order, and behind slot r's at least those of kRing - 2
    // other slots have been issued
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kPl * (kRing - 2)) : "memory");
    Step st;
#pragma unroll
    for (int k = 0; k < kS; ++k) {
      st.m[k] = ring[r][0][pl + k * 8];
      if (!ADD) {
        st.w[k] = ring[r][kPl - 2][pl + k * 8];
        st.q[k] = ring[r][kPl - 1][pl + k * 8];
      }
    }
    asm volatile("" ::: "memory");
    return st;
  };
  auto apply = [&](const Step &st, int k) {  // load part k: rows 4k .. 4k + 3
    if (ADD) {
      l = l + st.m[k].x;
      l = l + st.m[k].y;
      l = l + st.m[k].z;
      l = l + st.m[k].w;
    } else {
      l = l + ((l - st.q[k].x) * st.m[k].x) * st.w[k].x;
      l = l + ((l - st.q[k].y) * st.m[k].y) * st.w[k].y;
      l = l + ((l - st.q[k].z) * st.m[k].z) * st.w[k].z;
      l = l + ((l - st.q[k].w) * st.m[k].w) * st.w[k].w;
    }
  };
#pragma unroll
  for (int r = 0; r < kRing; ++r) refill(r);  // issued in the order they are consumed
  Step cur = read(0);
  // Software pipeline: step r starts the reads of slot r + 1, then applies the
  // rows of slot r (read a step earlier: one wait for all of them, as they
  // return in order), and then refills slot r.  Whole rounds first (every
  // group applies: one straight-line block per round), then the last,
  // partial round.
  auto round = [&](uint32_t g, bool whole) {
#pragma unroll
    for (int r = 0; r < kRing; ++r) {
      const uint32_t gr = g + static_cast<uint32_t>(r * kS);
      if (!whole && gr >= G) break;
      Step nxt = read((r + 1) % kRing);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" : "+v"(l) : "v"(ADD ? cur.m[kS - 1].w : cur.q[ADD ? 0 : kS - 1].w));
#pragma unroll
      for (int k = 0; k < kS; ++k)
        if (whole || gr + static_cast<uint32_t>(k) < G) apply(cur, k);
      cur = nxt;
      // the sums stay ahead of the refill of their slot
      asm volatile("" : "+v"(l) : : "memory");
      __builtin_amdgcn_sched_barrier(0);
      refill(r);
    }
  };
  uint32_t g = 0;
  for (; g + kRing * kS <= G; g += kRing * kS) round(g, true);
  if (g < G) round(g, false);
  // no load is in flight into the LDS of an ended workgroup
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (a.trace && c == 0 && h == 0 && lane == 0) {
    uint64_t *tr = a.trace + 4 * static_cast<uint64_t>(i);
    tr[0] = t_start;
    tr[1] = __builtin_amdgcn_s_memrealtime();
    tr[2] = static_cast<uint64_t>(len) | (uint64_t(3) << 32);
    tr[3] = static_cast<uint64_t>(__smid());
  }
  if (pix_in) *d = ug.accumulate == 1 ? *d + l : l;
}

// Work items per unit: none for units outside their tile; none for empty units
// when accumulating; one producer/consumer item for lists of at least
// heavy_len; otherwise three (one per channel) for long ordered lists, else one.
// (need_empty: the job's pass writes its whole image, so empty blocks are
// written too.)
// The list length from which a unit goes to the producer/consumer kernel:
// none when the pass has a particle with a non-finite q_c.
__device__ __forceinline__ uint32_t heavy_len_of(const SplatArgs &a) {
  return (a.qbad && *a.qbad) ? 0xffffffffu : a.heavy_len;
}

// The list length from which a unit is staged: none when the pass has a
// particle with a non-finite q_c (a staged ordered list applies zero operands
// outside the footprints, as the producer/consumer kernel does).
__device__ __forceinline__ uint32_t stage_len_of(const SplatArgs &a) {
  return (a.qbad && *a.qbad) ? 0xffffffffu : a.stage_len;
}

// Long lists (one item each, sorted first): staged lists, then the
// producer/consumer kernel's.
__device__ __forceinline__ uint32_t long_len_of(const SplatArgs &a) {
  return min(heavy_len_of(a), stage_len_of(a));
}

__device__ __forceinline__ uint32_t unit_items(const SplatArgs &a, uint32_t u, int ordered,
                                               uint32_t split, uint32_t &len) {
  len = a.bin_off[u + 1] - a.bin_off[u];
  const UnitGeom g = unit_geom(a, u);
  if (g.gx * 8 >= g.w || g.gy * 8 >= g.h) return 0;
  if (a.seg && a.seg[u]) return 0;  // walked in segments
  if (len == 0) return g.need_empty ? 1u : 0u;
  if (len >= long_len_of(a)) return 1u;  // staged, or one producer/consumer workgroup
  return (len >= (ordered ? split : 2 * split)) ? 3u : 1u;
}

__global__ __launch_bounds__(256) void k_items_count(SplatArgs a, uint32_t nunits, int ordered,
                                                     uint32_t split, uint32_t *cnt,
                                                     uint32_t *heavy_cnt, uint32_t *stage_cnt,
                                                     uint32_t *stage_grp, uint32_t *lmax) {
  // the block's counts in LDS, then one atomic per count (thousands of long
  // lists would queue up on the same few words)
  __shared__ uint32_t s_cnt[kStageLevels], s_grp[kStageLevels], s_heavy, s_lmax;
  const int tid = threadIdx.x;
  if (tid < kStageLevels) s_cnt[tid] = s_grp[tid] = 0;
  if (tid == 0) s_heavy = s_lmax = 0;
  __syncthreads();
  for (int64_t u = gtid(); u < nunits; u += gstride()) {
    uint32_t len;
    const uint32_t k = unit_items(a, static_cast<uint32_t>(u), ordered, split, len);
    cnt[u] = k;
    if (k == 0) continue;
    if (len >= heavy_len_of(a)) atomicAdd(&s_heavy, k);
    const uint32_t sl = stage_len_of(a);
    if (len >= sl) {  // counts per level of sl
      int j = 0;
      while (j < kStageLevels - 1 && static_cast<uint64_t>(len) >= stage_level(sl, j + 1)) ++j;
      atomicAdd(&s_cnt[j], 1u);
      atomicAdd(&s_grp[j], stage_groups(len));
    }
    atomicMax(&s_lmax, len);
  }
  __syncthreads();
  if (tid == 0) {
    if (heavy_cnt && s_heavy) atomicAdd(heavy_cnt, s_heavy);
    if (lmax && s_lmax) atomicMax(lmax, s_lmax);
    // lists whose top level is j, to lists from level j on
    for (int j = kStageLevels - 2; j >= 0; --j) {
      s_cnt[j] += s_cnt[j + 1];
      s_grp[j] += s_grp[j + 1];
    }
  }
  __syncthreads();
  if (stage_cnt && tid < kStageLevels && s_cnt[tid]) {
    atomicAdd(stage_cnt + tid, s_cnt[tid]);
    atomicAdd(stage_grp + tid, s_grp[tid]);
  }
}

// Sort key of a list: the long lists (one item each) first, then by length in
// quarter octaves, longest first.  8 bits are one radix pass; the splats only
// need the order of scheduling, not the exact lengths.
__device__ __forceinline__ uint32_t item_key(uint32_t len, uint32_t long_len) {
  uint32_t q = 0;
  if (len > 0) {
    const uint32_t e = 31u - static_cast<uint32_t>(__clz(static_cast<int>(len)));
    q = 4u * e + ((e >= 2u ? len >> (e - 2u) : len << (2u - e)) & 3u);
  }
  return (len >= long_len ? 0u : 128u) + 127u - q;
}

__global__ __launch_bounds__(256) void k_items_emit(SplatArgs a, uint32_t nunits, int ordered,
                                                    uint32_t split, const uint32_t *off,
                                                    uint32_t *keys, uint32_t *vals) {
  for (int64_t u = gtid(); u < nunits; u += gstride()) {
    uint32_t len;
    const uint32_t k = unit_items(a, static_cast<uint32_t>(u), ordered, split, len);
    const uint32_t o = off[u];
    for (uint32_t c = 0; c < k; ++c) {
      keys[o + c] = item_key(len, long_len_of(a));
      vals[o + c] = (static_cast<uint32_t>(u) << 2) | (k == 3 ? c : 3u);
    }
  }
}

unsigned grid_for(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g < 1) g = 1;
  if (g > (1 << 20)) g = 1 << 20;
  return static_cast<unsigned>(g);
}

}  // namespace

void launch_items_count(const uint32_t *bin_off, uint32_t nunits, const SplatArgs &a,
                        int ordered, uint32_t split, uint32_t *cnt, uint32_t *heavy_cnt,
                        hipStream_t s, uint32_t *stage_cnt, uint32_t *stage_grp,
                        uint32_t *lmax) {
  if (nunits == 0) return;
  SplatArgs b = a;
  b.bin_off = bin_off;
  k_items_count<<<grid_for(nunits), 256, 0, s>>>(b, nunits, ordered, split, cnt, heavy_cnt,
                                                 stage_cnt, stage_grp, lmax);
  hip_check(hipGetLastError(), "k_items_count launch");
}

void launch_items_emit(const uint32_t *bin_off, uint32_t nunits, const SplatArgs &a, int ordered,
                       uint32_t split, const uint32_t *off, uint32_t *keys, uint32_t *vals,
                       hipStream_t s) {
  if (nunits == 0) return;
  SplatArgs b = a;
  b.bin_off = bin_off;
  k_items_emit<<<grid_for(nunits), 256, 0, s>>>(b, nunits, ordered, split, off, keys, vals);
  hip_check(hipGetLastError(), "k_items_emit launch");
}

// A candidate has 2 seglen entries or more, a segment more than seglen / 2 or
// it is its list's last, and the lists have etot entries or fewer.
void seg_caps(uint64_t etot, uint32_t seglen, SegArgs &g) {
  g.seglen = seglen;
  // a pass takes about 0.07 ns per entry, a lone wave's walk up to 200 ns (ListRates;
  // by channel half): longer walks would outlast it (64 views, 160M and 169M entries: 33.9
  // and 34.6 ms; 42.9 and 42.0 with 123k and 205k entries whatever the pass)
  g.split = static_cast<uint32_t>(etot / 2700u / kSegSample);
  g.longest = static_cast<uint32_t>(etot / 1500u / kSegSample);
  g.candcap = static_cast<uint32_t>(etot / (2u * seglen)) + 1u;
  g.samplecap = static_cast<uint32_t>(etot / kSegSample) + 1u;
  g.chunkcap = g.samplecap / kSegChunk + g.candcap;
  g.segcap = 3u * (static_cast<uint32_t>(etot / (seglen / 2u)) + g.candcap);
}

void launch_seg_pick(uint32_t nunits, const SegArgs &g, const SplatArgs &a, hipStream_t s) {
  if (nunits == 0) return;
  k_seg_cand<<<grid_for(nunits), 256, 0, s>>>(a, nunits, g);
  hip_check(hipGetLastError(), "k_seg_cand launch");
  k_seg_sample<<<(g.chunkcap + 3u) / 4u, 256, 0, s>>>(a, g);
  hip_check(hipGetLastError(), "k_seg_sample launch");
  k_seg_win<<<(g.chunkcap + 3u) / 4u, 256, 0, s>>>(a, g);
  hip_check(hipGetLastError(), "k_seg_win launch");
  k_seg_cut<<<g.candcap, 64, 0, s>>>(a, g);
  hip_check(hipGetLastError(), "k_seg_cut launch");
}

void launch_seg_walk(const SegArgs &g, uint32_t nseg, float *states, const SplatArgs &a,
                     hipStream_t s) {
  if (nseg == 0) return;
  k_seg_walk<<<(nseg + 3u) / 4u, 256, 0, s>>>(a, g, nseg, states);
  hip_check(hipGetLastError(), "k_seg_walk launch");
}

void launch_seg_join(const SegArgs &g, uint32_t nlists, const float *states, const SplatArgs &a,
                     hipStream_t s) {
  if (nlists == 0) return;
  k_seg_join<<<3u * nlists, 64, 0, s>>>(a, g, states);
  hip_check(hipGetLastError(), "k_seg_join launch");
}

uint64_t stage_stride(uint64_t groups) { return 8u * groups + kStagePad; }

uint64_t stage_floats(bool additive, uint64_t groups) {
  return (additive ? stage_planes<1>() : stage_planes<0>()) * stage_stride(groups) * 32u;
}

uint64_t stage_groups_in(bool additive, uint64_t bytes) {
  return (bytes / (128u * (additive ? stage_planes<1>() : stage_planes<0>())) - kStagePad) / 8u;
}

uint64_t stage_batches(uint64_t groups, uint32_t n) { return groups / 16u + n; }

void launch_stage_base(const uint32_t *items, uint32_t n, uint32_t n1, uint32_t *cbase,
                       uint32_t *cbat, uint32_t *nrows, const SplatArgs &a, hipStream_t s,
                       const uint32_t *dn) {
  if (n == 0) return;
  k_stage_base<<<1, 256, 0, s>>>(a, items, n, n1, cbase, cbat, nrows, dn);
  hip_check(hipGetLastError(), "k_stage_base launch");
}

// Workgroups of kernel k (256 threads) resident at once on the current device.
unsigned resident_grid(const void *k, int slot) {
  static unsigned cache[3][16] = {};
  int dev = 0;
  hip_check(hipGetDevice(&dev), "get device");
  unsigned &r = cache[slot][dev & 15];
  if (!r) {
    int cus = 0, per = 0;
    hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "CU count");
    hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, 256, 0), "occupancy");
    r = static_cast<unsigned>(std::max(1, cus * per));
  }
  return r;
}

// Grid of a kernel that walks the staged batches (at most `batches`): a wave
// per batch up to one round of resident workgroups (a second round would queue
// behind the 8x8 splat's workgroups, and the chains wait for all of them).
static unsigned stage_grid(const void *k, int slot, uint64_t batches) {
  return std::max(1u, static_cast<unsigned>(
                          std::min<uint64_t>(resident_grid(k, slot), (batches + 3) / 4)));
}

void launch_stage_rows(const uint32_t *items, uint32_t i0, uint32_t i1, uint64_t batches,
                       const uint32_t *cbat, uint64_t *masks, uint32_t *rows, const SplatArgs &a,
                       hipStream_t s, const uint32_t *dn) {
  if (i1 <= i0) return;
  const unsigned grid = stage_grid(reinterpret_cast<const void *>(k_stage_rows), 2, batches);
  k_stage_rows<<<grid, 256, 0, s>>>(a, items, i0, i1, cbat, masks, rows, dn);
  hip_check(hipGetLastError(), "k_stage_rows launch");
}

void launch_stage_ops(bool additive, const uint32_t *items, uint32_t i0, uint32_t i1,
                      uint64_t batches, const uint32_t *cbase, const uint32_t *cbat,
                      const uint64_t *masks, const uint32_t *rows, const uint32_t *gofs,
                      float4 *ops, uint64_t stride, const SplatArgs &a, hipStream_t s,
                      const uint32_t *dn) {
  if (i1 <= i0) return;
  const void *k = additive ? reinterpret_cast<const void *>(k_stage_ops<1>)
                           : reinterpret_cast<const void *>(k_stage_ops<0>);
  const unsigned grid = stage_grid(k, additive ? 1 : 0, batches);
  if (additive)
    k_stage_ops<1><<<grid, 256, 0, s>>>(a, items, i0, i1, cbase, cbat, masks, rows, gofs, ops,
                                        stride, dn);
  else
    k_stage_ops<0><<<grid, 256, 0, s>>>(a, items, i0, i1, cbase, cbat, masks, rows, gofs, ops,
                                        stride, dn);
  hip_check(hipGetLastError(), "k_stage_ops launch");
}

void launch_stage_chain(bool additive, const uint32_t *items, uint32_t i0, uint32_t i1,
                        const uint32_t *cbase, const uint32_t *cbat, const uint32_t *rows,
                        const uint32_t *gofs, const float4 *ops, uint64_t stride,
                        const SplatArgs &a, hipStream_t s, const uint32_t *dn) {
  if (i1 <= i0) return;
  const unsigned grid = 24u * (i1 - i0);  // channels x pixel columns
  if (additive)
    k_stage_chain<1><<<grid, 64, 0, s>>>(a, items, i0, cbase, cbat, rows, gofs, ops, stride, dn);
  else
    k_stage_chain<0><<<grid, 64, 0, s>>>(a, items, i0, cbase, cbat, rows, gofs, ops, stride, dn);
  hip_check(hipGetLastError(), "k_stage_chain launch");
}

__global__ __launch_bounds__(64) void k_partition(PartitionArgs a, uint32_t *out) {
  __shared__ uint32_t s_cnt[kStageLevels], s_grp[kStageLevels];  // (read at once)
  if (threadIdx.x < kStageLevels) {
    s_cnt[threadIdx.x] = a.stage_cnt[threadIdx.x];
    s_grp[threadIdx.x] = a.stage_grp[threadIdx.x];
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const uint32_t nh = *a.heavy_cnt;
  const ListCounts c{s_cnt, s_grp, a.len0, nh, a.heavy_max, a.heavy_len, *a.lmax, *a.etot};
  uint32_t ns = 0, staged = 0;
  float longest = static_cast<float>(c.lmax);
  if (a.len0 != 0xffffffffu)
    for (int j = stage_rule(c, a.mode); j >= 0 && j < kStageLevels; ++j)
      if (s_cnt[j] <= a.ns_cap && s_grp[j] <= a.groups_cap) {
        ns = s_cnt[j];
        staged = s_grp[j];
        if (ns) longest = static_cast<float>(stage_level(a.len0, j));
        break;
      }
  const uint32_t npc = (a.heavy_max == 0 || nh <= ns) ? 0u : min(nh - ns, a.heavy_max);
  if (npc && npc == nh - ns) longest = fminf(longest, static_cast<float>(a.heavy_len));
  const uint32_t nlong = a.len0 <= a.heavy_len ? s_cnt[0] : nh;
  out[0] = ns;
  out[1] = npc;
  out[2] = ns + npc;
  out[3] = split_lists(c, nlong, ns + npc, staged, longest, a.additive, a.split);
}

void launch_partition(const PartitionArgs &pa, uint32_t *out, hipStream_t s) {
  k_partition<<<1, 64, 0, s>>>(pa, out);
  hip_check(hipGetLastError(), "k_partition launch");
}

void launch_splat_pc(bool additive, const uint32_t *items, uint32_t npc, const SplatArgs &a,
                     hipStream_t s, const ItemCounts &dc) {
  if (npc == 0) return;
  if (additive) k_splat_pc<1><<<npc, kPThreads, 0, s>>>(a, items, npc, dc);
  else k_splat_pc<0><<<npc, kPThreads, 0, s>>>(a, items, npc, dc);
  hip_check(hipGetLastError(), "k_splat_pc launch");
}

void launch_splat8(bool additive, int variant, const uint32_t *items, uint32_t nitems,
                   const SplatArgs &a, hipStream_t s, const ItemCounts &dc, int ppw,
                   uint32_t nsplit, bool beside) {
  if (nitems == 0) return;
  // device counts: nitems, a capacity of three items per unit, also bounds
  // the items with the long lists served by channel
  if (dc.items) nsplit = 0;
  const unsigned grid = static_cast<unsigned>((uint64_t(nitems) + 2u * uint64_t(nsplit) + 3) / 4);
  // Beside producer/consumer workgroups a small grid would fit whole on the CUs that
  // they leave, four workgroups each, and stay there when the others are free: three
  // (by LDS) leave some for those (1296 lists of 100k ordered entries, 192 of them in
  // such workgroups: 27.9 ms with four, 24.9 with three; grids of tens of thousands
  // are 3 % slower with three).
  const unsigned spread = beside && grid <= 2048u ? 6144u : 0u;
#define SPLAT8(ADDV, VARV, PPWV) \
  k_splat8<ADDV, VARV, PPWV><<<grid, 256, spread, s>>>(a, items, nitems, dc, nsplit)
  if (variant == 4) {
    switch (ppw) {
      case 1: if (additive) SPLAT8(1, 4, 1); else SPLAT8(0, 4, 1); break;
      case 2: if (additive) SPLAT8(1, 4, 2); else SPLAT8(0, 4, 2); break;
      case 4: if (additive) SPLAT8(1, 4, 4); else SPLAT8(0, 4, 4); break;
      case 8: if (additive) SPLAT8(1, 4, 8); else SPLAT8(0, 4, 8); break;
      default: if (additive) SPLAT8(1, 4, 0); else SPLAT8(0, 4, 0); break;
    }
  } else if (variant == 3) {
    if (additive) SPLAT8(1, 3, 0); else SPLAT8(0, 3, 0);
  } else if (variant == 2) {
    if (additive) SPLAT8(1, 2, 0); else SPLAT8(0, 2, 0);
  } else {
    if (additive) SPLAT8(1, 1, 0); else SPLAT8(0, 1, 0);
  }
#undef SPLAT8
  hip_check(hipGetLastError(), "k_splat8 launch");
}

}  // namespace splhip
