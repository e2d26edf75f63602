// Device-wide exclusive scan and stable LSD radix sort (key/value u32 pairs),
// written for wave64: wave-level scans over 64 lanes, wave-local digit
// ranking with ballots; tiles of 1024 elements (small inputs) or 4096 per 256-thread
// workgroup, and inputs of one tile in one workgroup.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "workspace.hpp"

namespace splhip {

// out[i] = sum_{j<i} in[j] over n elements (in == out allowed).  total /
// total64 (device, optional): the grand total in 32 and 64 bits.  Scratch:
// S_SCAN0+level.  dn (device, optional): the element count is min(n, *dn),
// read on the device (launches sized for n elements; no host wait).
void scan_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *total, Workspace &ws,
              hipStream_t s, const uint32_t *dn = nullptr, uint64_t *total64 = nullptr);

// Two scans of n elements each in the launches of one (total64: of the first).
void scan_u32_pair(const uint32_t *in0, uint32_t *out0, uint32_t *total0, uint64_t *total64,
                   const uint32_t *in1, uint32_t *out1, uint32_t *total1, int64_t n, Workspace &ws,
                   hipStream_t s, const uint32_t *dn = nullptr);

// Same with in[i] = ((flags[i] & bits) != 0).
void scan_u8bit(const uint8_t *flags, uint8_t bits, uint32_t *out, int64_t n, uint32_t *total,
                Workspace &ws, hipStream_t s);

// Stable sort of (keys, vals) by key bits [begin_bit, end_bit).  Ping-pongs
// between (k0,v0) and (k1,v1); returns 0 if the result is in (k0,v0), 1 if in
// (k1,v1).  Scratch: S_HIST and the scan slots.  dn (device, optional): the
// pair count is min(n, *dn), read on the device.
int radix_sort_pairs(uint32_t *k0, uint32_t *v0, uint32_t *k1, uint32_t *v1, int64_t n,
                     int begin_bit, int end_bit, Workspace &ws, hipStream_t s,
                     const uint32_t *dn = nullptr);

}  // namespace splhip
