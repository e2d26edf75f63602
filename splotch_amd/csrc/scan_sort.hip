// Device-wide exclusive scan and stable LSD radix sort for wave64 (gfx950).
//
// Frames of up to a few million particles are bound by the number of launches
// (about 5 us each, most of them scans and sort passes), so both take as few
// as the size allows.
//
// Scan: up to 16384 elements in one workgroup; else reduce-then-scan over
// 4096-element tiles (256 threads x 16 items), two launches: a tile sums the
// tile sums before it itself (at most 8192 of them; beyond, they are scanned
// recursively first).  Each thread scans its 16 items serially, the 64 lanes
// of a wave combine their sums with a log-step shuffle scan, and the wave
// totals are combined through LDS.
//
// Radix sort: up to 4096 pairs in one workgroup and one launch, digit after
// digit in LDS.  Else per digit of up to 9 bits, (1) a per-tile digit
// histogram, (2) for more than 128 tiles an exclusive scan of the histograms
// in digit-major order (which makes the result stable); up to 128 tiles, the
// scatter's workgroups sum the histograms themselves, (3) a scatter: each wave
// ranks its keys in input order with a 64-lane "match any" on the digit (one
// ballot per bit), the rank among equal digits from a popcount under the lane
// mask, and a wave-private running count per digit; the tile is then staged in
// LDS in digit order and written out as contiguous per-digit runs.
#include "scan_sort.hpp"

#include <algorithm>
#include <type_traits>

namespace splhip {
namespace {

constexpr int kTile = 4096;
constexpr int kItems = 16;
constexpr int kMaxBits = 9;

struct LoadU32 {
  const uint32_t *p;
  __device__ __forceinline__ uint32_t operator()(int64_t i) const { return p[i]; }
};

struct LoadLow32 {  // of tile sums
  const uint64_t *p;
  __device__ __forceinline__ uint32_t operator()(int64_t i) const {
    return static_cast<uint32_t>(p[i]);
  }
};

struct LoadU8Bit {
  const uint8_t *p;
  uint8_t v;
  __device__ __forceinline__ uint32_t operator()(int64_t i) const { return (p[i] & v) ? 1u : 0u; }
};

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  return v;
}

__device__ __forceinline__ uint64_t wave_reduce(uint64_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Exclusive scan of one value per thread over a block of W waves.
template <int W = 4>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *s_w) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan(v, lane);
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  uint32_t woff = 0;
#pragma unroll
  for (int w = 0; w < W; ++w)
    if (w < wave) woff += s_w[w];
  __syncthreads();
  return woff + inc - v;
}

// The element count of a launch sized for `cap` elements: cap, or the device
// count *dn when it is given (at most cap).
__device__ __forceinline__ int64_t count_of(int64_t cap, const uint32_t *dn) {
  return dn ? min(cap, static_cast<int64_t>(*dn)) : cap;
}

// One or two scans of a launch (blockIdx.y), of the same element count.
template <class In>
struct Job {
  In in;
  uint32_t *out;
  uint32_t *total;    // optional: the sum of all elements ...
  uint64_t *total64;  // ... and in 64 bits
  uint64_t *partial;  // tile sums
  uint32_t *psum;     // their exclusive scan (null: the tiles add them up themselves)
};
template <class In>
struct Jobs {
  Job<In> j[2];
};

// A thread's kItems elements from base (a multiple of kItems) on, 0 past n, and
// their exclusive prefixes from `prefix` on: 16 bytes at a time where the array
// is aligned (element by element a wave's access is 64 lines long, 16 times).
template <class In>
__device__ __forceinline__ void load_items(const In &in, int64_t base, int64_t n,
                                           uint32_t (&v)[kItems]) {
  if constexpr (std::is_same<In, LoadU32>::value) {
    if ((reinterpret_cast<uintptr_t>(in.p) & 15u) == 0 && base + kItems <= n) {
      const uint4 *q = reinterpret_cast<const uint4 *>(in.p + base);
#pragma unroll
      for (int i = 0; i < kItems / 4; ++i) {
        const uint4 x = q[i];
        v[4 * i] = x.x;
        v[4 * i + 1] = x.y;
        v[4 * i + 2] = x.z;
        v[4 * i + 3] = x.w;
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) v[i] = (base + i < n) ? in(base + i) : 0u;
}
__device__ __forceinline__ uint32_t store_prefixes(uint32_t *out, int64_t base, int64_t n,
                                                   uint32_t prefix,
                                                   const uint32_t (&v)[kItems]) {
  if ((reinterpret_cast<uintptr_t>(out) & 15u) == 0 && base + kItems <= n) {
    uint4 *q = reinterpret_cast<uint4 *>(out + base);
#pragma unroll
    for (int i = 0; i < kItems / 4; ++i) {
      uint4 x;
      x.x = prefix;
      x.y = x.x + v[4 * i];
      x.z = x.y + v[4 * i + 1];
      x.w = x.z + v[4 * i + 2];
      prefix = x.w + v[4 * i + 3];
      q[i] = x;
    }
    return prefix;
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    if (base + i < n) out[base + i] = prefix;
    prefix += v[i];
  }
  return prefix;
}

// Sum of each tile, in 64 bits.
template <class In>
__global__ __launch_bounds__(256) void k_scan_reduce(Jobs<In> jobs, int64_t cap,
                                                     const uint32_t *dn) {
  __shared__ uint64_t s_w[4];
  const Job<In> &J = jobs.j[blockIdx.y];
  const int64_t n = count_of(cap, dn);
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
  uint64_t s = 0;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t idx = base + i * 256 + threadIdx.x;
    if (idx < n) s += J.in(idx);
  }
  s = wave_reduce(s);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) J.partial[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

template <class In>
__global__ __launch_bounds__(256) void k_scan_apply(Jobs<In> jobs, int64_t cap,
                                                    const uint32_t *dn) {
  __shared__ uint32_t s_w[4];
  __shared__ uint64_t s_p[4];
  const Job<In> &J = jobs.j[blockIdx.y];
  const int64_t n = count_of(cap, dn);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile + threadIdx.x * kItems;
  const bool last = blockIdx.x == gridDim.x - 1;
  // the elements of the tiles before this one
  const bool add_up = !J.psum || (last && J.total64);
  uint64_t before = 0;
  if (add_up) {
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += 256) before += J.partial[i];
    before = wave_reduce(before);
    if (lane == 0) s_p[wave] = before;
  }
  uint32_t v[kItems];
  uint32_t sum = 0;
  load_items(J.in, base, n, v);
#pragma unroll
  for (int i = 0; i < kItems; ++i) sum += v[i];
  const uint32_t excl = block_excl_scan(sum, s_w);
  before = add_up ? s_p[0] + s_p[1] + s_p[2] + s_p[3] : J.psum[blockIdx.x];
  uint32_t prefix = static_cast<uint32_t>(before) + excl;
  prefix = store_prefixes(J.out, base, n, prefix, v);
  if (last && threadIdx.x == 255) {
    if (J.total) *J.total = prefix;
    if (J.total64) *J.total64 = before + J.partial[blockIdx.x];
  }
}

// The whole scan in one workgroup, for at most kOneScan elements.
constexpr int kOneThreads = 1024;
constexpr int64_t kOneScan = kOneThreads * kItems;
template <class In>
__global__ __launch_bounds__(kOneThreads) void k_scan_one(Jobs<In> jobs, int64_t cap,
                                                          const uint32_t *dn) {
  __shared__ uint32_t s_w[kOneThreads / 64];
  __shared__ uint64_t s_p[kOneThreads / 64];
  const Job<In> &J = jobs.j[blockIdx.y];
  const int64_t n = count_of(cap, dn);
  const int64_t base = static_cast<int64_t>(threadIdx.x) * kItems;
  uint32_t v[kItems];
  uint32_t sum = 0;
  uint64_t wide = 0;
  load_items(J.in, base, n, v);
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    sum += v[i];
    wide += v[i];
  }
  if (J.total64) {
    wide = wave_reduce(wide);
    if ((threadIdx.x & 63) == 0) s_p[threadIdx.x >> 6] = wide;
  }
  const uint32_t prefix =
      store_prefixes(J.out, base, n, block_excl_scan<kOneThreads / 64>(sum, s_w), v);
  if (threadIdx.x == kOneThreads - 1) {
    if (J.total) *J.total = prefix;
    if (J.total64) {
      wide = 0;
      for (int w = 0; w < kOneThreads / 64; ++w) wide += s_p[w];
      *J.total64 = wide;
    }
  }
}

__global__ void k_set_totals(uint32_t *total, uint64_t *total64) {
  if (total) *total = 0;
  if (total64) *total64 = 0;
}

constexpr int64_t kDirectTiles = 8192;  // tile sums that a tile adds up itself

// n: the element count, or with dn the capacity the launches are sized for
// (the count itself then read from *dn on the device).
template <class In>
void scan_impl(Jobs<In> jobs, unsigned nj, int64_t n, Workspace &ws, hipStream_t s, int level,
               const uint32_t *dn) {
  if (n <= 0) {
    for (unsigned y = 0; y < nj; ++y)
      if (jobs.j[y].total || jobs.j[y].total64)
        k_set_totals<<<1, 1, 0, s>>>(jobs.j[y].total, jobs.j[y].total64);
    return;
  }
  if (n <= kOneScan) {
    k_scan_one<In><<<dim3(1, nj), kOneThreads, 0, s>>>(jobs, n, dn);
    return;
  }
  const int64_t nb = (n + kTile - 1) / kTile;
  if (level >= 4) throw HipError{hipErrorInvalidValue, "scan too deep"};
  uint64_t *partial = ws.get_as<uint64_t>(S_SCAN0 + level, 4 * static_cast<size_t>(nb));
  for (unsigned y = 0; y < nj; ++y) {
    jobs.j[y].partial = partial + 2 * y * nb;
    jobs.j[y].psum = nullptr;
  }
  const dim3 grid(static_cast<unsigned>(nb), nj);
  k_scan_reduce<In><<<grid, 256, 0, s>>>(jobs, n, dn);
  if (nb > kDirectTiles) {
    Jobs<LoadLow32> up{};
    for (unsigned y = 0; y < nj; ++y) {
      jobs.j[y].psum = reinterpret_cast<uint32_t *>(partial + (2 * y + 1) * nb);
      up.j[y].in.p = jobs.j[y].partial;
      up.j[y].out = jobs.j[y].psum;
    }
    scan_impl(up, nj, nb, ws, s, level + 1, nullptr);
  }
  k_scan_apply<In><<<grid, 256, 0, s>>>(jobs, n, dn);
}

// ITEMS: keys per thread; a tile is 256 ITEMS keys.
template <int BITS, int ITEMS>
__global__ __launch_bounds__(256) void k_rs_hist(const uint32_t *keys, int64_t cap,
                                                 const uint32_t *dn, int shift, uint32_t *hist,
                                                 int64_t nblocks, bool tile_major) {
  const int64_t n = count_of(cap, dn);
  constexpr int R = 1 << BITS;
  constexpr uint32_t M = R - 1;
  __shared__ uint32_t h[4][R];
  for (int i = threadIdx.x; i < 4 * R; i += 256) (&h[0][0])[i] = 0;
  __syncthreads();
  const int wave = threadIdx.x >> 6;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (256 * ITEMS);
#pragma unroll 4
  for (int i = 0; i < ITEMS; ++i) {
    const int64_t idx = base + i * 256 + threadIdx.x;
    if (idx < n) atomicAdd(&h[wave][(keys[idx] >> shift) & M], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += 256)
    hist[tile_major ? static_cast<int64_t>(blockIdx.x) * R + d
                    : static_cast<int64_t>(d) * nblocks + blockIdx.x] =
        h[0][d] + h[1][d] + h[2][d] + h[3][d];
}

// Ranks a wave's ITEMS keys (striped: item it of lane l is input it * 64 + l)
// by digit, in input order: rk[it] = rank among the wave's equal digits, counts
// per digit in wh (zeroed by the caller).
template <int BITS, int ITEMS>
__device__ __forceinline__ void wave_rank(const uint32_t (&kk)[ITEMS], const bool (&ok)[ITEMS],
                                          int shift, int lane, uint32_t *wh,
                                          uint32_t (&rk)[ITEMS]) {
  constexpr uint32_t M = (1u << BITS) - 1;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const uint32_t d = (kk[it] >> shift) & M;
    uint64_t m = __ballot(ok[it]);
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t rank_in = __popcll(m & lt);
    const uint32_t cnt = __popcll(m);
    // the lowest lane of each peer group reserves cnt slots; peers read its base
    const int leader = __ffsll(static_cast<long long>(m)) - 1;
    uint32_t old = 0;
    if (ok[it] && rank_in == 0) old = atomicAdd(&wh[d], cnt);
    old = __shfl(old, leader & 63, 64);
    rk[it] = old + rank_in;
  }
}

// Digit totals of the block's W waves (wh[w][d] counts) to the wave offsets
// within each digit (wh) and the start of each digit's run (dstart).
template <int R, int W = 4>
__device__ __forceinline__ void digit_starts(uint32_t (*wh)[R], uint32_t *dstart, uint32_t *s_w) {
  constexpr int DPT = (R + 64 * W - 1) / (64 * W);  // digits per thread in the block scan
  uint32_t tot[DPT];
  uint32_t tsum = 0;
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int d = threadIdx.x * DPT + j;
    uint32_t acc = 0;
    if (d < R) {
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const uint32_t t = wh[w][d];
        wh[w][d] = acc;
        acc += t;
      }
    }
    tot[j] = acc;
    tsum += acc;
  }
  uint32_t start = block_excl_scan<W>(tsum, s_w);
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int d = threadIdx.x * DPT + j;
    if (d < R) dstart[d] = start;
    start += tot[j];
  }
}

// DIRECT: hist holds the tiles' own histograms, tile-major, and the workgroup
// sums them to its digits' global starts; else their digit-major scan.
template <int BITS, bool DIRECT, int ITEMS>
__global__ __launch_bounds__(256) void k_rs_scatter(const uint32_t *kin, const uint32_t *vin,
                                                    uint32_t *kout, uint32_t *vout, int64_t cap,
                                                    const uint32_t *dn, int shift,
                                                    const uint32_t *hist, int64_t nblocks) {
  const int64_t n = count_of(cap, dn);
  constexpr int R = 1 << BITS, TILE = 256 * ITEMS;
  constexpr uint32_t M = R - 1;
  constexpr int DPT = (R + 255) / 256;
  __shared__ uint32_t wh[4][R];   // per-wave digit counts -> offsets
  __shared__ uint32_t dstart[R];  // block-local start of each digit run
  __shared__ uint32_t gbase[R];   // global start of (digit, this tile)
  __shared__ uint32_t sk[TILE], sv[TILE];
  __shared__ uint32_t s_w[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t tbase = static_cast<int64_t>(blockIdx.x) * TILE;
  if (tbase >= n) return;  // a tile past the device count (uniform)
  for (int i = threadIdx.x; i < 4 * R; i += 256) (&wh[0][0])[i] = 0;
  if (DIRECT) {
    // thread t: digits [t DPT, t DPT + DPT), counts below this tile and in all
    uint32_t below[DPT], all[DPT], sum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = threadIdx.x * DPT + j;
      below[j] = all[j] = 0;
      if (d < R) {
#pragma unroll 8
        for (int b = 0; b < static_cast<int>(nblocks); ++b) {
          const uint32_t h = hist[static_cast<int64_t>(b) * R + d];
          all[j] += h;
          below[j] += b < static_cast<int>(blockIdx.x) ? h : 0u;
        }
      }
      sum += all[j];
    }
    uint32_t start = block_excl_scan(sum, s_w);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const int d = threadIdx.x * DPT + j;
      if (d < R) gbase[d] = start + below[j];
      start += all[j];
    }
  } else {
    for (int d = threadIdx.x; d < R; d += 256)
      gbase[d] = hist[static_cast<int64_t>(d) * nblocks + blockIdx.x];
  }
  __syncthreads();
  const int64_t base = tbase + wave * (TILE / 4);
  uint32_t kk[ITEMS], vv[ITEMS], rk[ITEMS];
  bool ok[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int64_t idx = base + it * 64 + lane;
    ok[it] = idx < n;
    kk[it] = ok[it] ? kin[idx] : 0u;
    vv[it] = ok[it] ? vin[idx] : 0u;
  }
  wave_rank<BITS, ITEMS>(kk, ok, shift, lane, wh[wave], rk);
  __syncthreads();
  digit_starts<R>(wh, dstart, s_w);
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    if (ok[it]) {
      const uint32_t d = (kk[it] >> shift) & M;
      const uint32_t lp = dstart[d] + wh[wave][d] + rk[it];
      sk[lp] = kk[it];
      sv[lp] = vv[it];
    }
  }
  __syncthreads();
  const int cnt = static_cast<int>(min<int64_t>(TILE, n - tbase));
  for (int i = threadIdx.x; i < cnt; i += 256) {
    const uint32_t key = sk[i];
    const uint32_t d = (key >> shift) & M;
    const uint32_t pos = gbase[d] + (static_cast<uint32_t>(i) - dstart[d]);
    kout[pos] = key;
    vout[pos] = sv[i];
  }
}

// The whole sort in one workgroup, for at most kTile pairs: digits of 8 bits
// (the last pass's digit is cut at end_bit).  1024 threads with 4 pairs each: a
// wave ranks its keys 64 at a time (256 threads with 16 pairs: 8.4 us for one
// digit of 1000 keys, 5 with 1024).
constexpr int kOneItems = kTile / kOneThreads;
__global__ __launch_bounds__(kOneThreads) void k_rs_one(const uint32_t *kin, const uint32_t *vin,
                                                uint32_t *kout, uint32_t *vout, int64_t cap,
                                                const uint32_t *dn, int begin_bit, int end_bit) {
  const int n = static_cast<int>(count_of(cap, dn));
  constexpr int R = 256, W = kOneThreads / 64;
  __shared__ uint32_t wh[W][R], dstart[R], sk[kTile], sv[kTile], s_w[W];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = wave * (kTile / W);
  uint32_t kk[kOneItems], vv[kOneItems], rk[kOneItems];
  bool ok[kOneItems];
#pragma unroll
  for (int it = 0; it < kOneItems; ++it) {
    const int idx = base + it * 64 + lane;
    ok[it] = idx < n;
    kk[it] = ok[it] ? kin[idx] : 0u;
    vv[it] = ok[it] ? vin[idx] : 0u;
  }
  const uint32_t keep = end_bit < 32 ? (1u << end_bit) - 1u : ~0u;
  for (int shift = begin_bit; shift < end_bit; shift += 8) {
    for (int i = threadIdx.x; i < W * R; i += kOneThreads) (&wh[0][0])[i] = 0;
    __syncthreads();
    uint32_t dk[kOneItems];
#pragma unroll
    for (int it = 0; it < kOneItems; ++it) dk[it] = kk[it] & keep;
    wave_rank<8, kOneItems>(dk, ok, shift, lane, wh[wave], rk);
    __syncthreads();
    digit_starts<R, W>(wh, dstart, s_w);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kOneItems; ++it) {
      if (ok[it]) {
        const uint32_t d = (dk[it] >> shift) & (R - 1);
        const uint32_t lp = dstart[d] + wh[wave][d] + rk[it];
        sk[lp] = kk[it];
        sv[lp] = vv[it];
      }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kOneItems; ++it) {
      const int idx = base + it * 64 + lane;
      if (ok[it]) {
        kk[it] = sk[idx];
        vv[it] = sv[idx];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int it = 0; it < kOneItems; ++it) {
    const int idx = base + it * 64 + lane;
    if (ok[it]) {
      kout[idx] = kk[it];
      vout[idx] = vv[it];
    }
  }
}

constexpr int64_t kDirectSort = 128;  // tiles whose histograms a scatter workgroup sums itself

template <int BITS, int ITEMS>
void rs_pass(const uint32_t *sk, const uint32_t *sv, uint32_t *dk, uint32_t *dv, int64_t n,
             const uint32_t *dn, int shift, int64_t nb, uint32_t *hist, Workspace &ws,
             hipStream_t s) {
  const bool direct = nb <= kDirectSort;
  const unsigned g = static_cast<unsigned>(nb);
  k_rs_hist<BITS, ITEMS><<<g, 256, 0, s>>>(sk, n, dn, shift, hist, nb, direct);
  if (direct) {
    k_rs_scatter<BITS, true, ITEMS><<<g, 256, 0, s>>>(sk, sv, dk, dv, n, dn, shift, hist, nb);
  } else {
    scan_u32(hist, hist, (int64_t(1) << BITS) * nb, nullptr, ws, s);
    k_rs_scatter<BITS, false, ITEMS><<<g, 256, 0, s>>>(sk, sv, dk, dv, n, dn, shift, hist, nb);
  }
  hip_check(hipGetLastError(), "radix sort launch");
}

// Sorts of up to kSmallSort pairs take tiles of 1024 (128 of them, as many as a
// scatter sums the histograms of): a wave ranks its keys 64 at a time, one LDS
// update after another, which is a pass's time where the tiles do not fill the
// GPU (20k ordered at 257 x 193: 325 -> 295 us; 16 captured thumbnails 861 -> 842
// us, 851 up to 65536 pairs only).
constexpr int64_t kSmallSort = 131072;
constexpr int kSmallItems = 4;

template <int ITEMS>
int radix_sort_tiled(uint32_t *k0, uint32_t *v0, uint32_t *k1, uint32_t *v1, int64_t n,
                     int begin_bit, int end_bit, Workspace &ws, hipStream_t s,
                     const uint32_t *dn) {
  const int64_t nb = (n + 256 * ITEMS - 1) / (256 * ITEMS);
  const int bits = end_bit - begin_bit;
  const int passes = (bits + kMaxBits - 1) / kMaxBits;
  const int width = (bits + passes - 1) / passes;  // <= 9
  uint32_t *hist = ws.get_as<uint32_t>(S_HIST, (size_t(1) << width) * static_cast<size_t>(nb));
  int cur = 0;
  for (int shift = begin_bit; shift < end_bit; shift += width) {
    const int w = std::min(width, end_bit - shift);
    const uint32_t *sk = cur ? k1 : k0;
    const uint32_t *sv = cur ? v1 : v0;
    uint32_t *dk = cur ? k0 : k1;
    uint32_t *dv = cur ? v0 : v1;
    switch (w) {
#define SPLHIP_PASS(B) rs_pass<B, ITEMS>(sk, sv, dk, dv, n, dn, shift, nb, hist, ws, s)
      case 1: SPLHIP_PASS(1); break;
      case 2: SPLHIP_PASS(2); break;
      case 3: SPLHIP_PASS(3); break;
      case 4: SPLHIP_PASS(4); break;
      case 5: SPLHIP_PASS(5); break;
      case 6: SPLHIP_PASS(6); break;
      case 7: SPLHIP_PASS(7); break;
      case 8: SPLHIP_PASS(8); break;
      default: SPLHIP_PASS(9); break;
#undef SPLHIP_PASS
    }
    cur ^= 1;
  }
  return cur;
}

}  // namespace

void scan_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *total, Workspace &ws,
              hipStream_t s, const uint32_t *dn, uint64_t *total64) {
  scan_impl(Jobs<LoadU32>{{{{in}, out, total, total64, nullptr, nullptr}, {}}}, 1, n, ws, s, 0, dn);
  hip_check(hipGetLastError(), "scan_u32 launch");
}

void scan_u32_pair(const uint32_t *in0, uint32_t *out0, uint32_t *total0, uint64_t *total64,
                   const uint32_t *in1, uint32_t *out1, uint32_t *total1, int64_t n, Workspace &ws,
                   hipStream_t s, const uint32_t *dn) {
  scan_impl(Jobs<LoadU32>{{{{in0}, out0, total0, total64, nullptr, nullptr},
                           {{in1}, out1, total1, nullptr, nullptr, nullptr}}},
            2, n, ws, s, 0, dn);
  hip_check(hipGetLastError(), "scan_u32_pair launch");
}

void scan_u8bit(const uint8_t *flags, uint8_t bits, uint32_t *out, int64_t n, uint32_t *total,
                Workspace &ws, hipStream_t s) {
  scan_impl(Jobs<LoadU8Bit>{{{{flags, bits}, out, total, nullptr, nullptr, nullptr}, {}}}, 1, n, ws,
            s, 0, nullptr);
  hip_check(hipGetLastError(), "scan_u8bit launch");
}

int radix_sort_pairs(uint32_t *k0, uint32_t *v0, uint32_t *k1, uint32_t *v1, int64_t n,
                     int begin_bit, int end_bit, Workspace &ws, hipStream_t s,
                     const uint32_t *dn) {
  if (n <= 1 || end_bit <= begin_bit) return 0;
  if (n <= kTile) {
    k_rs_one<<<1, kOneThreads, 0, s>>>(k0, v0, k1, v1, n, dn, begin_bit, end_bit);
    hip_check(hipGetLastError(), "k_rs_one launch");
    return 1;
  }
  return n <= kSmallSort
             ? radix_sort_tiled<kSmallItems>(k0, v0, k1, v1, n, begin_bit, end_bit, ws, s, dn)
             : radix_sort_tiled<kItems>(k0, v0, k1, v1, n, begin_bit, end_bit, ws, s, dn);
}

}  // namespace splhip
