// Memory microbenchmarks for gfx950 (measurement only; not part of the render
// library): the chip's practical peaks that the bench sets kernels against,
// and known-size kernels for scaling profiler counters.
//
// LDS reads: every workgroup fills 33 KiB of LDS (4 workgroups, 16 waves per
// CU), then each wave reads 4-, 8- or 16-byte words (ds_read_b32 / b64 / b128)
// from 16 places 1 KiB apart, by immediate offsets from one address per lane:
// linear (64 lanes, consecutive words: no bank conflict), or 4 distinct words
// (lane l that of l % 4, as a splat reads the constants of 4 particles).  Every
// word that is read goes into a checksum (one VALU operation, below the issue
// limit) that is written at the end: a part of a vector that nothing uses would
// be left out of the read.  Reads per launch and wave = iters * 16.
//
// HBM copy: dst[i] = src[i] over n 16-byte vectors, grid-stride, each lane
// moving four vectors per step with all four loads issued before the stores.
// Bytes per launch = 2 * 16 * n (read + write).
#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

constexpr int kLdsBytes = 33 * 1024;
constexpr int kReads = 16;  // per iteration, 1 KiB apart

template <typename T, bool FOUR>
__global__ __launch_bounds__(256, 4) void k_lds_read(uint32_t *out, int iters) {
  __shared__ uint4 buf[kLdsBytes / 16];
  const int t = threadIdx.x, lane = t & 63;
  for (int i = t; i < kLdsBytes / 16; i += 256)
    buf[i] = make_uint4(i, i * 3u + 1u, i * 5u + 2u, i * 7u + 3u);
  __syncthreads();
  uint32_t acc = 0;
  uint32_t x = FOUR ? lane & 3 : lane;  // the lane's word: at most 1 KiB, then 2 KiB on and back
  for (int k = 0; k < iters; ++k) {
#pragma unroll
    for (int j = 0; j < kReads; ++j) {
      const T v = reinterpret_cast<const T *>(buf)[x + j * (1024 / sizeof(T))];
      if constexpr (sizeof(T) == 16) acc ^= v.x ^ v.y ^ v.z ^ v.w;
      else if constexpr (sizeof(T) == 8) acc ^= v.x ^ v.y;
      else acc ^= v.x;
      asm volatile("" ::: "memory");  // one read each: not joined, not kept
    }
    x ^= 2048 / sizeof(T);
    asm volatile("" : "+v"(x));
  }
  out[static_cast<int64_t>(blockIdx.x) * 256 + t] = acc;
}

__global__ __launch_bounds__(256) void k_copy(const uint4 *__restrict__ src,
                                              uint4 *__restrict__ dst, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256 * 4;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 * 4 + threadIdx.x; i < n; i += stride) {
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t j = i + k * 256;
      v[k] = j < n ? src[j] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t j = i + k * 256;
      if (j < n) dst[j] = v[k];
    }
  }
}

}  // namespace

extern "C" {

// Times one launch of `grid` workgroups x `iters` iterations of reads of
// `words` 32-bit words per lane (1, 2 or 4; four != 0: 4 distinct ones per wave),
// after one warm-up launch, with HIP events on a stream of its own.  Returns 0
// and writes the milliseconds and the read instructions (of a wave each); a
// HIP error code otherwise.
int lds_peak_run(int device, int grid, int iters, int words, int four, float *ms,
                 double *instructions) {
  if (grid < 1 || iters < 1 || !ms || !instructions || (words != 1 && words != 2 && words != 4))
    return -1;
  if (hipSetDevice(device) != hipSuccess) return -2;
  uint32_t *out = nullptr;
  hipStream_t s = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = 0;
  if (hipMalloc(&out, static_cast<size_t>(grid) * 256 * 4) != hipSuccess) return -2;
  if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    rc = -2;
  } else {
    auto launch = [&]() {
      void (*kernel)(uint32_t *, int) =
          words == 4   ? (four ? k_lds_read<uint4, true> : k_lds_read<uint4, false>)
          : words == 2 ? (four ? k_lds_read<uint2, true> : k_lds_read<uint2, false>)
                       : (four ? k_lds_read<uint1, true> : k_lds_read<uint1, false>);
      kernel<<<grid, 256, 0, s>>>(out, iters);
    };
    launch();
    (void)hipEventRecord(e0, s);
    launch();
    (void)hipEventRecord(e1, s);
    if (hipEventSynchronize(e1) != hipSuccess || hipGetLastError() != hipSuccess) {
      rc = -2;
    } else {
      (void)hipEventElapsedTime(ms, e0, e1);
      *instructions = static_cast<double>(grid) * 4.0 * iters * kReads;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (s) (void)hipStreamDestroy(s);
  (void)hipFree(out);
  return rc;
}

// Copies `bytes` (a multiple of 16) between two device buffers it allocates:
// one warm-up launch, then `reps` launches timed with HIP events; writes the
// average milliseconds per launch.  grid = 0: 8 workgroups per CU.
int hbm_copy_run(int device, int64_t bytes, int reps, int grid, float *ms) {
  if (bytes <= 0 || (bytes & 15) || reps < 1 || !ms) return -1;
  if (hipSetDevice(device) != hipSuccess) return -2;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return -2;
  if (grid <= 0) grid = 8 * prop.multiProcessorCount;
  uint4 *a = nullptr, *b = nullptr;
  hipStream_t s = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = 0;
  const int64_t n = bytes / 16;
  if (hipMalloc(&a, bytes) != hipSuccess || hipMalloc(&b, bytes) != hipSuccess ||
      hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    rc = -2;
  } else {
    k_copy<<<grid, 256, 0, s>>>(a, b, n);
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < reps; ++r) k_copy<<<grid, 256, 0, s>>>(a, b, n);
    (void)hipEventRecord(e1, s);
    if (hipEventSynchronize(e1) != hipSuccess || hipGetLastError() != hipSuccess) {
      rc = -2;
    } else {
      (void)hipEventElapsedTime(ms, e0, e1);
      *ms /= reps;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (s) (void)hipStreamDestroy(s);
  if (a) (void)hipFree(a);
  if (b) (void)hipFree(b);
  return rc;
}

}  // extern "C"
