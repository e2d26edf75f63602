// Post-processing and 8-bit output of a rendered frame on the GPU: the
// master's epilogue of splotch.cc:272-310 fused into one pass over the image.
//
//   a_eq_e:        c = -xexp.expm1(c)                     splotch.cc:275-284
//   colour_adjust: c = float(contrast * pow(double(c), gamma) + brightness),
//                  only when gamma != 1, brightness != 0 or contrast != 1
//                                                         splotchutils.cc:230-250
//   add_colorbar:  bar k (the k-th type with a scalar palette) covers rows
//                  yres-1-10k-y, y < 10, with the palette colour at
//                  ix / double(xres)                      splotchutils.cc:35-56
//   Colour8:       byte = max(0, min(255, int(c * 256))), x86 truncation
//                                                         ls_image.h:65-75
//
// The float image is read once; the bytes go out either in the image's own
// x-major order (LS_Image's pixel[ix][iy]) or as the body of the TGA file
// LS_Image::write_TGA writes (rows iy ascending, pixels ix ascending, B G R;
// ls_image.cc:178-202), which is a transpose of the image: that form is
// staged through LDS in pixel tiles so both the float reads and the byte
// writes are contiguous.
#include "kernels.hpp"

#include <algorithm>

#include "workspace.hpp"

namespace splhip {
namespace {

// The value of channel c of pixel (ix, iy) after the float steps.
__device__ __forceinline__ float post_value(const PostArgs &a, float v, int ix, int iy, int c) {
  if (a.a_eq_e) v = -xexp_expm1(a.exptab, v, a.expfac, a.taylorlimit);
  if (a.adjust) {
    const double d = static_cast<double>(v);
    // pow(x, 1) is x for every x (C99 F.9.4.4), so gamma 1 skips the call
    const double pw = a.gamma == 1.0 ? d : pow(d, a.gamma);
    v = static_cast<float>(a.contrast * pw + a.brightness);
  }
  if (a.nbars > 0) {
    const int k = (a.yres - 1 - iy) / 10;
    if (k < a.nbars) {
      const int t = a.bar_type[k];
      float r, g, b;
      palette_val(a.pal_x + static_cast<int64_t>(t) * a.pal_stride,
                  a.pal_rgb + static_cast<int64_t>(t) * a.pal_stride * 3, a.pal_n[t],
                  static_cast<double>(ix) / static_cast<double>(a.xres), r, g, b);
      v = c == 0 ? r : c == 1 ? g : b;
    }
  }
  return v;
}

// max(0, min(255, int(c * 256))) with x86 truncation: below 0 (and NaN) it
// gives 0, and past the int range INT_MIN, so 0.
__device__ __forceinline__ uint8_t colour8(float v) {
  const float f = fmaxf(v * 256.f, 0.f);
  const int i = f < 2147483648.f ? static_cast<int>(f) : 0;
  return static_cast<uint8_t>(min(255, i));
}

// -xexp_expm1 of four values with the table in LDS, branch-free: the eight
// reads (at an in-range index in every case) are issued before any is used.
// With p = v expfac: p >= 2^31 or NaN converts to INT_MIN on x86 and gives exp
// 1, p in [2^20, 2^31) gives 0, p <= -1 gives 1.
__device__ __forceinline__ void tone4(const float *tab, float expfac, float tl, float (&v)[4]) {
  float p[4], t1[4], t2[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[q] = v[q] * expfac;
    const bool ok = p[q] < 1048576.f && p[q] > -1.f;
    const int k = static_cast<int>(ok ? p[q] : 0.f);
    t1[q] = tab[k >> 10];
    t2[q] = tab[1024 + (k & 1023)];
  }
  // every read is used here, so that none is moved into a branch below
#pragma unroll
  for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(t1[q]), "+v"(t2[q]));
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool lo = p[q] < 1048576.f, ok = lo && p[q] > -1.f;
    const float op = ok ? t1[q] * t2[q] : (lo || !(p[q] < 2147483648.f)) ? 1.f : 0.f;
    v[q] = -(fabsf(v[q]) < tl ? v[q] : op - 1.f);
  }
}

// A frame without colour_adjust and colorbars (kPostEq with, kPostPlain without
// a_eq_e) is handled four values at a time; kPostGeneral takes post_value's
// steps one by one.
enum PostKind { kPostEq, kPostPlain, kPostGeneral };

__device__ __forceinline__ void stage_table(float4 *s_tab, const float *exptab) {
  for (int i = threadIdx.x; i < 512; i += blockDim.x)
    s_tab[i] = reinterpret_cast<const float4 *>(exptab)[i];
  __syncthreads();
}

// Bytes in the image's order (or only the float image).
__global__ __launch_bounds__(256) void k_post_xmajor(PostArgs a) {
  // 3 xres yres < 2^31 (checked by the caller)
  const uint32_t yres = static_cast<uint32_t>(a.yres);
  const uint32_t n = static_cast<uint32_t>(a.xres) * yres * 3;
  for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
    const uint32_t p = e / 3;
    const int c = static_cast<int>(e - p * 3);
    const uint32_t ix = p / yres, iy = p - ix * yres;
    const float v = post_value(a, a.pic[e], static_cast<int>(ix), static_cast<int>(iy), c);
    if (a.out) a.out[e] = v;
    if (a.rgb8) a.rgb8[e] = colour8(v);
  }
}

// The same where a value does not depend on its pixel: four consecutive values
// per thread and step (vec_in: 16-byte aligned images, vec_out: 4-byte aligned
// bytes).  2048^2: 40.1 us a value at a time, each table lookup behind a branch.
template <PostKind KIND>
__global__ __launch_bounds__(256) void k_post_stream(PostArgs a) {
  __shared__ float4 s_tab[KIND == kPostEq ? 512 : 1];
  if (KIND == kPostEq) stage_table(s_tab, a.exptab);
  const uint32_t n = static_cast<uint32_t>(a.xres) * static_cast<uint32_t>(a.yres) * 3;
  for (uint32_t e = (blockIdx.x * 256 + threadIdx.x) * 4; e < n; e += gridDim.x * 1024) {
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    const uint32_t m = min(4u, n - e);
    if (a.vec_in && m == 4) {
      const float4 v = *reinterpret_cast<const float4 *>(a.pic + e);
      o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
    } else {
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q)
        if (q < m) o[q] = a.pic[e + q];
    }
    if (KIND == kPostEq)
      tone4(reinterpret_cast<const float *>(s_tab), a.expfac, a.taylorlimit, o);
    if (a.out) {
      if (a.vec_in && m == 4) {
        *reinterpret_cast<float4 *>(a.out + e) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
          if (q < m) a.out[e + q] = o[q];
      }
    }
    if (a.rgb8) {
      if (a.vec_out == 4 && m == 4) {
        uint32_t w = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) w |= static_cast<uint32_t>(colour8(o[q])) << (8 * q);
        *reinterpret_cast<uint32_t *>(a.rgb8 + e) = w;
      } else {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
          if (q < m) a.rgb8[e + q] = colour8(o[q]);
      }
    }
  }
}

// TGA body through LDS: block (bx, by) owns the pixels [kTX bx, kTX bx + kTX) x
// [kTY by, kTY by + kTY); the bytes are put into LDS in the file's order, so
// that a row leaves in 16-byte words.  HBM-bound at large images (4096^2: 96 us
// with every lookup behind a branch, 49 with four values side by side and the
// table in LDS; 2048^2: 30 -> 17 us, of which about 5 are the launch; 128 x 32
// and 64 x 32 tiles, whose columns are whole 128-byte lines, measured 52 / 48
// and 18 / 18 us, and leave small images too few blocks).
constexpr int kTX = 64, kTY = 16;

template <PostKind KIND>
__global__ __launch_bounds__(256) void k_post_tga(PostArgs a) {
  constexpr int kRow = 3 * kTX + 16;      // LDS bytes per pixel row (padded, 16-byte words)
  constexpr int kCol = 3 * kTY / 4;       // groups of four values per pixel column
  constexpr int kPer = kTX * kCol / 256;  // groups per thread
  static_assert(kTX * kCol % 256 == 0, "whole groups per thread");
  __shared__ __align__(16) uint8_t tile[kTY * kRow];
  __shared__ float4 s_tab[KIND == kPostEq ? 512 : 1];
  const int ix0 = blockIdx.x * kTX, iy0 = blockIdx.y * kTY;
  const int nx = min(kTX, a.xres - ix0), ny = min(kTY, a.yres - iy0);
  // read: per pixel column ix, the 3 ny floats of iy0.. are contiguous; full
  // columns of a 4-aligned image go as float4, all of a thread's loads issued
  // before its stores (out may be pic)
  const bool vec = ny == kTY && a.vec_in;
  float v[kPer][4] = {};
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int f = threadIdx.x + 256 * k, r = f / kCol, w0 = 4 * (f - r * kCol);
    const float *src = a.pic + (static_cast<int64_t>(ix0 + r) * a.yres + iy0) * 3 + w0;
    if (r < nx && vec) {
      const float4 t = *reinterpret_cast<const float4 *>(src);
      v[k][0] = t.x, v[k][1] = t.y, v[k][2] = t.z, v[k][3] = t.w;
    } else if (r < nx) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (w0 + q < 3 * ny) v[k][q] = src[q];
    }
  }
  if (KIND == kPostEq) stage_table(s_tab, a.exptab);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int f = threadIdx.x + 256 * k, r = f / kCol, w0 = 4 * (f - r * kCol);
    if (r >= nx) continue;
    const int ix = ix0 + r;
    float(&o)[4] = v[k];
    if (KIND == kPostEq)
      tone4(reinterpret_cast<const float *>(s_tab), a.expfac, a.taylorlimit, o);
    int il = w0 / 3, c = w0 - 3 * il;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (vec || il < ny) {
        if (KIND == kPostGeneral) o[q] = post_value(a, o[q], ix, iy0 + il, c);
        tile[il * kRow + 3 * r + 2 - c] = colour8(o[q]);
      }
      if (++c == 3) {
        c = 0;
        ++il;
      }
    }
    if (a.out) {
      float *dst = a.out + (static_cast<int64_t>(ix) * a.yres + iy0) * 3 + w0;
      if (vec) {
        *reinterpret_cast<float4 *>(dst) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (w0 + q < 3 * ny) dst[q] = o[q];
      }
    }
  }
  __syncthreads();
  // write: per row iy, the 3 nx bytes of ix0.. are contiguous (B, G, R); full
  // rows of a 16- or 4-aligned output go as 16-byte or 32-bit words
  auto rows = [&](auto word, int per_row) {
    typedef decltype(word) W;
    for (int f = threadIdx.x; f < ny * per_row; f += 256) {
      const int il = f / per_row, w = f - il * per_row;
      reinterpret_cast<W *>(a.rgb8 + (static_cast<int64_t>(iy0 + il) * a.xres + ix0) * 3)[w] =
          reinterpret_cast<const W *>(&tile[il * kRow])[w];
    }
  };
  if (nx == kTX && a.vec_out == 16) rows(uint4{}, 3 * kTX / 16);
  else if (nx == kTX && a.vec_out == 4) rows(uint32_t{}, 3 * kTX / 4);
  else rows(uint8_t{}, 3 * nx);
}

}  // namespace

void launch_post(const PostArgs &a, int layout, hipStream_t s) {
  const bool plain = !a.adjust && a.nbars == 0;
  auto at = [](const void *p, uintptr_t m) { return reinterpret_cast<uintptr_t>(p) % m == 0; };
  PostArgs b = a;
  if (layout == 1 && a.rgb8) {
    const dim3 grid((a.xres + kTX - 1) / kTX, (a.yres + kTY - 1) / kTY);
    // float4 columns need every column start (ix yres + iy0) 3 on a 16-byte
    // boundary; word rows need (iy xres + ix0) 3 on a word boundary
    b.vec_in = a.yres % 4 == 0 && at(a.pic, 16) && at(a.out, 16);
    b.vec_out = a.xres % 16 == 0 && at(a.rgb8, 16) ? 16 : a.xres % 4 == 0 && at(a.rgb8, 4) ? 4 : 1;
    if (!plain) k_post_tga<kPostGeneral><<<grid, 256, 0, s>>>(b);
    else if (a.a_eq_e) k_post_tga<kPostEq><<<grid, 256, 0, s>>>(b);
    else k_post_tga<kPostPlain><<<grid, 256, 0, s>>>(b);
    hip_check(hipGetLastError(), "k_post_tga launch");
    return;
  }
  const int64_t n = static_cast<int64_t>(a.xres) * a.yres * 3;
  if (plain) {
    b.vec_in = at(a.pic, 16) && at(a.out, 16);
    b.vec_out = at(a.rgb8, 4) ? 4 : 1;
    const unsigned g = static_cast<unsigned>(std::min<int64_t>((n + 1023) / 1024, 2048));
    if (a.a_eq_e) k_post_stream<kPostEq><<<g, 256, 0, s>>>(b);
    else k_post_stream<kPostPlain><<<g, 256, 0, s>>>(b);
    hip_check(hipGetLastError(), "k_post_stream launch");
    return;
  }
  const int64_t g = std::min<int64_t>((n + 255) / 256, 1 << 16);
  k_post_xmajor<<<static_cast<unsigned>(std::max<int64_t>(g, 1)), 256, 0, s>>>(a);
  hip_check(hipGetLastError(), "k_post_xmajor launch");
}

}  // namespace splhip
