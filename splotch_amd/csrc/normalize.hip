// particle_normalize on the GPU (splotch/scenemaker.cc:40-296, host branch):
// per particle the optional log10 / asinh of intensity and colour, per type
// the min / max of intensity, colour and smoothing length, then the clamp of
// Normalizer::normAndClamp (splotch/splotchutils.h:138-171).  Two passes over
// the SoA fields (transform + reduce, then clamp), both HBM-bound.
//
// The per-type extremes are kept as order-preserving 32-bit keys (sign-
// flipped float bits) so they reduce with integer atomics: per thread in
// registers, per wave by shuffles, per block in LDS, then one atomic per
// block and value.  The per-type switches are staged in LDS (a lane-indexed
// kernel argument would be copied to private memory).  NaN
// never enters (std::min / std::max never take it); of +0 and -0 the minimum
// takes -0 and the maximum +0 (the reference keeps whichever its thread order
// meets first).
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

#include "workspace.hpp"

namespace splhip {
namespace {

__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float fdekey(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// log10 of a float, rounded from the double result.
__device__ __forceinline__ float log10_f(float v) {
  return static_cast<float>(log10(static_cast<double>(v)));
}

// my_asinh (splotchutils.cc:31-32): log(v + sqrt(1 + v v)) in double.
__device__ __forceinline__ float asinh_f(float v) {
  const double d = static_cast<double>(v);
  return static_cast<float>(log(d + sqrt(1. + d * d)));
}

// Slots of a type's keys: colour min / max, intensity min / max, size min / max.
enum { K_CMIN, K_CMAX, K_IMIN, K_IMAX, K_RMIN, K_RMAX, K_N };

__global__ __launch_bounds__(256) void k_norm_init(uint32_t *keys, int nt) {
  const int i = threadIdx.x;
  if (i < nt * K_N) keys[i] = (i % 2 == 0) ? fkey(1e37f) : fkey(-1e37f);
}

__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#pragma unroll
  for (int d = 32; d; d >>= 1)
    v = min(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), d, 64)));
  return v;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
  for (int d = 32; d; d >>= 1)
    v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), d, 64)));
  return v;
}

// W consecutive values at p + m, of n: one 16-byte vector (4 type bytes) where
// W = 4 (aligned fields) and four are left; those past the end are not touched.
template <int W, class T, class V>
__device__ __forceinline__ void load_w(const T *p, int64_t m, int64_t n, T (&v)[W]) {
  if constexpr (W == 4) {
    if (m + 4 <= n) {
      const V w = *reinterpret_cast<const V *>(p + m);
      v[0] = w.x;
      v[1] = w.y;
      v[2] = w.z;
      v[3] = w.w;
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < W; ++j)
    if (m + j < n) v[j] = p[m + j];
}
template <int W>
__device__ __forceinline__ void store_w(float *p, int64_t m, int64_t n, const float (&v)[W]) {
  if constexpr (W == 4) {
    if (m + 4 <= n) {
      *reinterpret_cast<float4 *>(p + m) = make_float4(v[0], v[1], v[2], v[3]);
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < W; ++j)
    if (m + j < n) p[m + j] = v[j];
}

// Loads per thread, field and step (all issued before the first is used): two
// vectors of four particles, or four single particles.
template <int W> constexpr int loads() { return W == 4 ? 2 : 4; }

// Pass 1: transforms in place and reduces the extremes of NT types.  Both
// passes are bound by HBM (13 B, then 17 B per particle); a thread takes four
// consecutive particles per 16-byte load.  16M particles of two types: 122 ->
// 97 us without logs (4.9 TB/s), against a float per load and four loads in flight
// per thread and field.
// GEN: some type has a log10, an asinh or a vector colour, VEC: some type has a
// vector colour (else that code, and its registers, are left out).
template <int NT, int W, bool GEN, bool VEC, int kT>
__global__ __launch_bounds__(kT) void k_norm_reduce(NormArgs a, uint32_t *keys) {
  __shared__ int32_t s_flags[NT][4];
  if (threadIdx.x < NT * 4) s_flags[threadIdx.x / 4][threadIdx.x % 4] =
      a.flags[threadIdx.x / 4][threadIdx.x % 4];
  __syncthreads();
  uint32_t k[NT][K_N];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < K_N; ++q) k[t][q] = (q % 2 == 0) ? 0xffffffffu : 0u;
  constexpr int kV = loads<W>();
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kT * W;
  for (int64_t m0 = (static_cast<int64_t>(blockIdx.x) * kT + threadIdx.x) * W; m0 < a.n;
       m0 += kV * stride) {
    uint8_t tv[kV][W] = {};
    float Iv[kV][W], ev[kV][W], rv[kV][W], gv[VEC ? kV : 1][W], bv[VEC ? kV : 1][W];
#pragma unroll
    for (int q = 0; q < kV; ++q) {
      const int64_t m = m0 + q * stride;
      if (m < a.n) {
        if (VEC) {
          load_w<W, float, float4>(a.eg, m, a.n, gv[VEC ? q : 0]);
          load_w<W, float, float4>(a.eb, m, a.n, bv[VEC ? q : 0]);
        }
        if (a.type) load_w<W, uint8_t, uchar4>(a.type, m, a.n, tv[q]);
        load_w<W, float, float4>(a.I, m, a.n, Iv[q]);
        load_w<W, float, float4>(a.er, m, a.n, ev[q]);
        load_w<W, float, float4>(a.r, m, a.n, rv[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < kV; ++q) {
      const int64_t mq = m0 + q * stride;
      bool put_I = false, put_e = false, put_v = false;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const int64_t m = mq + j;
        const int t = m < a.n ? tv[q][j] : NT;
        if (t >= NT) continue;  // past the end, or a type beyond ptypes (not rendered)
        const int f_il = GEN ? s_flags[t][0] : 0, f_cl = GEN ? s_flags[t][1] : 0,
                  f_ca = GEN ? s_flags[t][2] : 0, f_cv = VEC ? s_flags[t][3] : 0;
        // extremes of this particle (min keys start high, max keys low)
        uint32_t cmin = 0xffffffffu, cmax = 0u, imin = 0xffffffffu, imax = 0u;
        const float r = rv[q][j];
        if (r == r) {
          const uint32_t kr = fkey(r);
#pragma unroll
          for (int u = 0; u < NT; ++u)
            if (u == t) {
              k[u][K_RMIN] = min(k[u][K_RMIN], kr);
              k[u][K_RMAX] = max(k[u][K_RMAX], kr);
            }
        }
        float I = Iv[q][j];
        bool icol = true;
        if (f_il) {
          if (I > 0) {
            I = log10_f(I);
          } else {
            I = -38.f;
            icol = false;
          }
          Iv[q][j] = I;
          put_I = true;
        }
        if (icol && I == I) imin = imax = fkey(I);
        float e = ev[q][j];
        bool ccol = true;
        if (f_cl) {
          if (e > 0) {
            e = log10_f(e);
          } else {
            e = -38.f;
            ccol = false;
          }
        } else if (f_ca) {
          e = asinh_f(e);
        }
        if (f_cl || f_ca) {
          ev[q][j] = e;
          put_e = true;
        }
        if (ccol && e == e) cmin = cmax = fkey(e);
        if (f_cv) {
          float &g = gv[VEC ? q : 0][j], &b = bv[VEC ? q : 0][j];
          if (f_cl) {
            g = log10_f(g);
            b = log10_f(b);
          }
          if (f_ca) {
            g = asinh_f(g);
            b = asinh_f(b);
          }
          put_v |= f_cl || f_ca;
          if (g == g) {
            cmin = min(cmin, fkey(g));
            cmax = max(cmax, fkey(g));
          }
          if (b == b) {
            cmin = min(cmin, fkey(b));
            cmax = max(cmax, fkey(b));
          }
        }
#pragma unroll
        for (int u = 0; u < NT; ++u)
          if (u == t) {
            k[u][K_CMIN] = min(k[u][K_CMIN], cmin);
            k[u][K_CMAX] = max(k[u][K_CMAX], cmax);
            k[u][K_IMIN] = min(k[u][K_IMIN], imin);
            k[u][K_IMAX] = max(k[u][K_IMAX], imax);
          }
      }
      // unchanged particles of the four get their own value back
      if (put_I) store_w<W>(a.I, mq, a.n, Iv[q]);
      if (put_e) store_w<W>(a.er, mq, a.n, ev[q]);
      if (put_v) {
        store_w<W>(a.eg, mq, a.n, gv[VEC ? q : 0]);
        store_w<W>(a.eb, mq, a.n, bv[VEC ? q : 0]);
      }
    }
  }
  // per wave by shuffles, per block through LDS, then one atomic per block
  // and value (thousands of atomics on a few addresses would serialize)
  __shared__ uint32_t s_k[kT / 64][NT * K_N];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < K_N; ++q) {
      const uint32_t v = (q % 2 == 0) ? wave_min(k[t][q]) : wave_max(k[t][q]);
      if (lane == 0) s_k[wave][t * K_N + q] = v;
    }
  __syncthreads();
  const int i = threadIdx.x;
  if (i < NT * K_N) {
    const bool is_min = (i % K_N) % 2 == 0;
    uint32_t v = s_k[0][i];
    for (int w = 1; w < kT / 64; ++w) v = is_min ? min(v, s_k[w][i]) : max(v, s_k[w][i]);
    if (is_min) {
      if (v != 0xffffffffu) atomicMin(&keys[i], v);
    } else {
      if (v != 0u) atomicMax(&keys[i], v);
    }
  }
}

// The range a type's values are clamped to (after the parameter overrides).
struct Range {
  float minv, maxv;
  __device__ __forceinline__ void clamp(float &v) const {
    if (maxv == minv) {
      v = 1.f;
    } else {
      const float lo = (v < maxv) ? v : maxv;   // std::min(maxv, v)
      const float hi = (minv < lo) ? lo : minv; // std::max(minv, lo)
      v = (hi - minv) / (maxv - minv);
    }
  }
};

// Pass 2: normAndClamp of intensity (unless NO_I_NORM) and colour; the
// block first stages every type's two ranges and vector flag in LDS.
template <int W, bool GEN, bool VEC, int kT>
__global__ __launch_bounds__(kT) void k_norm_clamp(NormArgs a, const uint32_t *keys) {
  __shared__ Range s_int[kMaxTypes], s_col[kMaxTypes];
  __shared__ int32_t s_vec[kMaxTypes];
  const int i = threadIdx.x;
  if (i < a.ntypes) {
    Range I, C;
    I.minv = a.ovr_set[i][0] ? a.ovr[i][0] : fdekey(keys[i * K_N + K_IMIN]);
    I.maxv = a.ovr_set[i][1] ? a.ovr[i][1] : fdekey(keys[i * K_N + K_IMAX]);
    C.minv = a.ovr_set[i][2] ? a.ovr[i][2] : fdekey(keys[i * K_N + K_CMIN]);
    C.maxv = a.ovr_set[i][3] ? a.ovr[i][3] : fdekey(keys[i * K_N + K_CMAX]);
    s_int[i] = I;
    s_col[i] = C;
    s_vec[i] = a.flags[i][3];
  }
  __syncthreads();
  constexpr int kV = loads<W>();
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kT * W;
  for (int64_t m0 = (static_cast<int64_t>(blockIdx.x) * kT + threadIdx.x) * W; m0 < a.n;
       m0 += kV * stride) {
    uint8_t tv[kV][W] = {};
    float Iv[kV][W], ev[kV][W], gv[VEC ? kV : 1][W], bv[VEC ? kV : 1][W];
#pragma unroll
    for (int q = 0; q < kV; ++q) {  // loads first
      const int64_t m = m0 + q * stride;
      if (m < a.n) {
        if (VEC) {
          load_w<W, float, float4>(a.eg, m, a.n, gv[VEC ? q : 0]);
          load_w<W, float, float4>(a.eb, m, a.n, bv[VEC ? q : 0]);
        }
        if (a.type) load_w<W, uint8_t, uchar4>(a.type, m, a.n, tv[q]);
        load_w<W, float, float4>(a.I, m, a.n, Iv[q]);
        load_w<W, float, float4>(a.er, m, a.n, ev[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < kV; ++q) {
      const int64_t mq = m0 + q * stride;
      bool put = false, put_v = false;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const int64_t m = mq + j;
        const int t = m < a.n ? tv[q][j] : kMaxTypes;
        if (t >= a.ntypes) continue;
        put = true;
        if (a.norm_int) s_int[t].clamp(Iv[q][j]);
        const Range C = s_col[t];
        C.clamp(ev[q][j]);
        if (VEC && s_vec[t]) {
          put_v = true;
          C.clamp(gv[VEC ? q : 0][j]);
          C.clamp(bv[VEC ? q : 0][j]);
        }
      }
      if (put) {
        if (a.norm_int) store_w<W>(a.I, mq, a.n, Iv[q]);
        store_w<W>(a.er, mq, a.n, ev[q]);
      }
      if (put_v) {
        store_w<W>(a.eg, mq, a.n, gv[VEC ? q : 0]);
        store_w<W>(a.eb, mq, a.n, bv[VEC ? q : 0]);
      }
    }
  }
}

template <int W, bool GEN, bool VEC, int kT>
void launch_passes(const NormArgs &a, uint32_t *keys, hipStream_t s) {
  const unsigned grid = static_cast<unsigned>(
      std::min<int64_t>((a.n + W * kT - 1) / (W * kT), 1024));
#define SPLHIP_NORM(N) \
  case N: k_norm_reduce<N, W, GEN, VEC, kT><<<grid, kT, 0, s>>>(a, keys); break;
  switch (a.ntypes) {
    SPLHIP_NORM(1) SPLHIP_NORM(2) SPLHIP_NORM(3) SPLHIP_NORM(4)
    SPLHIP_NORM(5) SPLHIP_NORM(6) SPLHIP_NORM(7) SPLHIP_NORM(8)
  }
#undef SPLHIP_NORM
  hip_check(hipGetLastError(), "k_norm_reduce launch");
  k_norm_clamp<W, GEN, VEC, kT><<<grid, kT, 0, s>>>(a, keys);
  hip_check(hipGetLastError(), "k_norm_clamp launch");
}

}  // namespace

void launch_normalize(const NormArgs &a, uint32_t *keys, hipStream_t s) {
  k_norm_init<<<1, 256, 0, s>>>(keys, a.ntypes);
  hip_check(hipGetLastError(), "k_norm_init launch");
  if (a.n <= 0) return;
  auto at = [](const void *p, uintptr_t m) { return reinterpret_cast<uintptr_t>(p) % m == 0; };
  NormArgs b = a;
  bool gen = false;
  b.vector = 0;
  for (int t = 0; t < a.ntypes; ++t) {
    gen = gen || a.flags[t][0] || a.flags[t][1] || a.flags[t][2] || a.flags[t][3];
    b.vector |= a.flags[t][3];
  }
  // four particles per load where the fields are aligned and there are enough
  // to fill the GPU that way; else one (20k particles with logs: 14.8 us with
  // one, 16.3 with four, whose logarithms a thread takes in turn)
  const bool vec = a.n >= (1 << 19) && at(a.I, 16) && at(a.er, 16) && at(a.r, 16) &&
                   at(a.type, 4) && (!b.vector || (at(a.eg, 16) && at(a.eb, 16)));
  // Logs and vector colours hold the passes at 3 waves per SIMD, where workgroups
  // of 512 threads fit a CU once, two waves per SIMD, and those of 256 three times
  // (16M particles, logs, fields not aligned: 204 us with 512, 144 with 256; 4M
  // aligned, four types in random order: 118 and 85); small fields have a workgroup
  // per CU at most, and fewer of them end in fewer atomics (600k, two types: 30 us
  // with 512, 37 with 256).
  auto go = [&](auto w) {
    constexpr int W = decltype(w)::value;
    const bool small = a.n < (b.vector ? 1 << 21 : 1 << 20);
    if (b.vector && small) launch_passes<W, true, true, 512>(b, keys, s);
    else if (b.vector) launch_passes<W, true, true, 256>(b, keys, s);
    else if (gen && small) launch_passes<W, true, false, 512>(b, keys, s);
    else if (gen) launch_passes<W, true, false, 256>(b, keys, s);
    else launch_passes<W, false, false, 512>(b, keys, s);
  };
  if (vec) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 1>{});
}

}  // namespace splhip
