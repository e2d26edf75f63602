// Launch wrappers of the render kernels (kernels.hip, splat8.hip).
//
// Every stage works on a batch of jobs (views); a plain render is a batch of
// one.  Particles of all jobs are concatenated (job j owns global indices
// [pbase[j], pbase[j+1])), a pass's particles stay job-major through
// compaction and the depth sort (job j owns pass positions [mo[j], mo[j+1])),
// and the units (tiles or 8x8 blocks) of job j are numbered from ubase[j].
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "common.hpp"

namespace splhip {

// Per-job projection inputs (device table, one entry per job).
struct ProjectArgs {
  const float *x, *y, *z, *hsml, *inten, *col, *c1, *c2;
  const uint8_t *type;
  int64_t n;
  int64_t poff;  // first global particle index of the job
  splhip_camera cam;
  float smooth_fac[kMaxTypes];
  float brightness[kMaxTypes];
  int32_t col_vector[kMaxTypes];
  int32_t pass_code[kMaxTypes];  // 1: ordered pass, 2: additive pass, 0: not rendered
  int32_t pal_n[kMaxTypes];
  int32_t pal_stride;
  int32_t ntypes;
  int32_t sort_type;
  const double *pal_x;
  const float *pal_rgb;
  float bfak, rfac;
};

// Particle-parallel launches over jobs: jobs get whole blocks of kPerBlock
// particles; blk[j] is the first block of job j (blk[nj] = grid size).
// (256: a particle per thread; with 1024, four one after another, 20k particles at
// 257 x 193 take 302 us, 288 here, and larger frames 1 % more)
constexpr int kPerBlock = 256;

struct SplatArgs {
  const uint32_t *bin_off;  // [nunits+1]
  const uint32_t *ent;      // entries: slot in recs
  const Rec *recs;
  const float *exptab;      // 2048 floats
  const JobSplat *jobs;     // per-job geometry, image and flags
  const uint32_t *ubase;    // [nj+1] first unit of each job
  int nj;
  int pass;                 // 0 ordered, 1 additive
  float rfac, h2sigma, expfac, taylorlimit;
  uint32_t prio_len;  // splat8: lists at least this long run at raised wave priority
  uint64_t *trace;    // splat8: optional per-item {start, end, len | chan << 32, hw id}
  uint32_t heavy_len; // splat8: lists at least this long go to the producer/consumer kernel
  uint32_t stage_len; // lists at least this long are staged (0xffffffff: none)
  // (device, optional) nonzero: the pass has a particle with a non-finite q_c,
  // so no list goes to the producer/consumer kernel (it applies every particle
  // to the whole block with zero operands, and (l - q) * 0 is NaN there)
  const uint32_t *qbad;
  const uint32_t *seg;  // (optional) per unit: nonzero = walked in segments, no items
};

// tot: ntot words set to 0 beside.
void launch_project(const ProjectArgs *jobs, const uint32_t *blk, int nj, uint32_t nblocks,
                    Rec *rec, uint8_t *act, uint32_t *tot, uint32_t ntot, hipStream_t s);
// Compaction of one pass (act & code) into pass order; keys (optional): the
// depth-sort key of each job's sort_type.
void launch_compact(const ProjectArgs *jobs, const uint32_t *blk, int nj, uint32_t nblocks,
                    const uint8_t *act, uint8_t code, const uint32_t *pos, const Rec *rec,
                    uint32_t *keys, uint32_t *vals, hipStream_t s);
// Device counts: a launcher given an optional `const uint32_t *d*` pointer
// sizes its grid for the host count (then a capacity) and reads the actual
// count from that device word (at most the capacity), so that no host wait
// is needed between the stage that counts and the stage that consumes.
//
// Per pass mo[j] = pos[pbase[j]] (pass particles before job j), mo[nj] = *total;
// with js also the jobs' pass flags from them.
struct PassOffsets {
  const uint32_t *pos[2], *total[2];
  uint32_t *mo[2];  // null: pass absent
};
void launch_pass_offsets(const PassOffsets &a, const uint32_t *pbase, int nj, int64_t n,
                         JobSplat *js, hipStream_t s);
// keys[i] = job of global particle index vals[i].
void launch_job_of_index(const uint32_t *vals, uint32_t m, const uint32_t *pbase, int nj,
                         uint32_t *keys, hipStream_t s, const uint32_t *dm = nullptr);
// cnt: entries per particle (units of the binned tiles); cnt16 (optional):
// the regions of 2^rsh x 2^rsh of those 8x8 blocks they cover.  qbad
// (optional, ordered pass): set to 1 when a particle's q_c = e_c / (e_c +
// gray_absorption) is not finite.
void launch_gather_count(const uint32_t *order, uint32_t m, const Rec *rec, Rec *recs,
                         uint32_t *cnt, uint32_t *cnt16, int rsh, const BinGeom *geoms,
                         const uint32_t *mo, int nj, uint32_t *qbad, hipStream_t s,
                         const uint32_t *dm = nullptr);
// rsh == 0: (unit, particle) entries; rsh > 0: (region | unit mask << rbits,
// particle) entries for regions of 2^rsh x 2^rsh blocks, regions of job j
// numbered from ubase[j] (then ubase holds the region bases).
void launch_emit(int rsh, int rbits, const Rec *recs, uint32_t m, const uint32_t *off,
                 uint32_t e, const BinGeom *geoms, const uint32_t *ubase, const uint32_t *mo,
                 int nj, uint32_t *keys, uint32_t *vals, hipStream_t s,
                 const uint32_t *dm = nullptr, const uint32_t *de = nullptr);
// Block lists from the sorted region lists (keys: region | mask << rbits,
// vals: particles; S x S blocks per region, S = 2 or 4; roff: region CSR;
// rbase / ubase: first region / unit of each job):
//   launch_split_chunks   per-chunk mask-bit counts ccnt[S^2 * split_chunks(e16)]
//   scan_u32(ccnt -> cpre, S^2 * nchunks, total at cpre[S^2 * nchunks])
//   launch_split_bounds   sx[S^2 * nregions] and the block list lengths ucnt
//   scan_u32(ucnt -> boff, nunits, total at boff[nunits])
//   launch_split_base     base[S^2 * nregions] from boff and sx (may be sx)
//   launch_split_scatter  the block lists ent, in list order
uint32_t split_chunks(uint32_t e16);
void launch_split_chunks(int S, const uint32_t *keys, uint32_t e16, int rbits, uint32_t *ccnt,
                         hipStream_t s, const uint32_t *de16 = nullptr);
void launch_split_bounds(int S, const uint32_t *roff, const uint32_t *keys, uint32_t nregions,
                         const uint32_t *cpre, uint32_t e16, int rbits, const uint32_t *rbase,
                         const uint32_t *ubase, const BinGeom *geoms, int nj, uint32_t *sx,
                         uint32_t *ucnt, hipStream_t s);
void launch_split_base(int S, uint32_t nregions, const uint32_t *rbase, const uint32_t *ubase,
                       const BinGeom *geoms, int nj, const uint32_t *sx, const uint32_t *boff,
                       uint32_t *base, hipStream_t s);
void launch_split_scatter(int S, const uint32_t *keys, const uint32_t *vals, uint32_t e16,
                          int rbits, const uint32_t *cpre, const uint32_t *base, uint32_t *ent,
                          hipStream_t s, const uint32_t *de16 = nullptr);
// kmask: the bits of a key that hold the bin (the rest ride along unsorted).
void launch_bin_offsets(const uint32_t *sorted_keys, uint32_t e, uint32_t nbins,
                        uint32_t *bin_off, hipStream_t s, uint32_t kmask = ~0u,
                        const uint32_t *de = nullptr);
void launch_map(const uint32_t *idx, const uint32_t *table, uint32_t *out, int64_t n,
                hipStream_t s);
void launch_fill(float *p, float v, int64_t n, hipStream_t s);
void launch_fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t s);
// Device-count pipeline helpers: zeros into the images of jobs with no particle
// in either pass (mo null: pass absent), and the capacity check of a pass (counts
// zeroed, bit set in *ovf when e64 > ecap or *e16 > e16cap).
void launch_fill_empty_jobs(const uint32_t *mo0, const uint32_t *mo1, int nj, const JobSplat *js,
                            hipStream_t s);
void launch_cap_check(uint32_t *m, uint32_t *e, const uint64_t *e64, uint32_t *e16,
                      uint64_t ecap, uint32_t e16cap, uint32_t bit, uint32_t *ovf,
                      hipStream_t s);
// pic[i] += add[i]
void launch_add_images(float *pic, const float *add, int64_t n, hipStream_t s);
// n <= 256 words from src to dst in host memory, then *flag = seq there.
void launch_publish(const uint32_t *src, uint32_t n, uint32_t *dst, uint32_t *flag, uint32_t seq,
                    hipStream_t s);
// A one-wave kernel that returns after `us` microseconds (bounded wait); at once
// where a device count n is given and is 0.
void launch_delay(uint32_t us, hipStream_t s, const uint32_t *n = nullptr);
// Host records staged chunk-major (chunk k: records [k C, k C + cnt_k), its
// ncol float columns of cnt_k values back to back, then cnt_k type bytes)
// into the SoA columns soa[q nn + i] and type[i].
void launch_unpack_records(const char *stage, int64_t n, int64_t C, int ncol, float *soa,
                           int64_t nn, uint8_t *type, hipStream_t s);

// Staging thresholds: level j = 0..kStageLevels-1 of a base length sl is
// sl * 2^(j/2) (odd levels times 181/128, about sqrt 2, rounded down).
constexpr int kStageLevels = 26;
__host__ __device__ inline uint64_t stage_level(uint32_t sl, int j) {
  const uint64_t b = static_cast<uint64_t>(sl) << (j >> 1);
  return (j & 1) ? (b * 181u) >> 7 : b;
}

// Wave-per-8x8-block splat (splat8.hip): work items (unit << 2 | channel,
// channel 3 = all), heaviest first.  heavy_cnt (device, optional): incremented
// once per unit whose list reaches a.heavy_len (one item); stage_cnt /
// stage_grp (optional, [kStageLevels] each): [j] once per unit whose list
// reaches stage_level(a.stage_len, j), and by its groups of 4 entries (at most); lmax
// (optional): the longest list of a unit with items.
void launch_items_count(const uint32_t *bin_off, uint32_t nunits, const SplatArgs &a,
                        int ordered, uint32_t split, uint32_t *cnt, uint32_t *heavy_cnt,
                        hipStream_t s, uint32_t *stage_cnt = nullptr,
                        uint32_t *stage_grp = nullptr, uint32_t *lmax = nullptr);
// keys: 8 bits, the longer lists first, by quarter octaves of the length (lists
// from the long-list length on before the others).
void launch_items_emit(const uint32_t *bin_off, uint32_t nunits, const SplatArgs &a, int ordered,
                       uint32_t split, const uint32_t *off, uint32_t *keys, uint32_t *vals,
                       hipStream_t s);
// Device item counts of a pass (all null: the host counts are exact).
struct ItemCounts {
  const uint32_t *items = nullptr;  // work items of the pass
  const uint32_t *heavy = nullptr;  // of which the long lists (sorted first)
  uint32_t heavy_cap = 0;           // the 8x8 splat skips min(*heavy, heavy_cap) items
  const uint32_t *first = nullptr;  // producer/consumer items: from *first on,
  const uint32_t *npc = nullptr;    // *npc of them (a grid sized for a capacity)
  const uint32_t *nsplit = nullptr; // long lists the 8x8 splat serves by channel
};
// With dc set, launch_splat8 is given the pass's whole item array and a grid
// for nitems (a capacity) and skips the first min(*dc.heavy, heavy_cap) items;
// launch_splat_pc is given the whole item array and npc = its capacity.  ppw
// (variant 4): particles per chunk of the walk, 1, 2, 4 or 8 (0: 8 for one
// channel, 8 additive / 4 ordered for all three).  nsplit (with dc:
// *dc.nsplit): the first nsplit of the 8x8 splat's items are long lists (one
// all-channel item each) left over by the staged and producer/consumer
// kernels; the 8x8 splat serves each as three one-channel items, so that
// three waves share its chain (a grid for nitems + 2 nsplit items).  beside: producer/
// consumer workgroups run at the same time.
void launch_splat8(bool additive, int variant, const uint32_t *items, uint32_t nitems,
                   const SplatArgs &a, hipStream_t s, const ItemCounts &dc = ItemCounts{},
                   int ppw = 0, uint32_t nsplit = 0, bool beside = false);
// Ordered lists walked in segments (splat8.hip): lists of at least 2 * seglen
// entries, cut where the sampled entries before the cut make every pixel's chain
// forget its start.  flag[u] says per unit whether its list is (the item kernels
// skip those: SplatArgs::seg).
struct SegCand {
  uint32_t unit, samples;  // first sample (192 floats each)
  uint32_t on;             // bit c: the list absorbs in channel c
};
struct SegList {
  uint32_t unit, first, n;  // first segment, segments
};
struct Seg {
  uint32_t list, e0, e1, warm, slot;  // entries, warm-up entries before e0, first kept state
  uint32_t chan;                      // 3: all
};
constexpr uint32_t kSegCheck = 1024;    // entries between a segment's kept states (192 floats)
constexpr uint32_t kSegSample = 2048;   // one batch of 64 is sampled in this many entries
constexpr uint32_t kSegWarm = 32;       // samples of the longest warm-up
// Device counts (zeroed before launch_seg_pick).
enum { SC_CAND, SC_CHUNK, SC_SAMPLE, SC_LIST, SC_SEG, SC_SLOT, SC_N };
struct SegArgs {
  uint32_t seglen, candcap, chunkcap, samplecap, segcap;
  uint32_t split, longest;  // samples from which a walk goes by channel / is not made
  uint32_t *flag, *cnt;
  SegCand *cand;      // [candcap]
  uint32_t *chunk;    // [chunkcap * 2]
  float *sample;      // [samplecap * 192]
  uint32_t *win;      // [samplecap]
  SegList *lists;     // [candcap]
  Seg *segs;          // [segcap]
};
// The capacities that a pass of etot entries cannot exceed.
void seg_caps(uint64_t etot, uint32_t seglen, SegArgs &g);
void launch_seg_pick(uint32_t nunits, const SegArgs &g, const SplatArgs &a, hipStream_t s);
// The segments (states: the slots counted, 192 floats each), then the lists' blocks.
void launch_seg_walk(const SegArgs &g, uint32_t nseg, float *states, const SplatArgs &a,
                     hipStream_t s);
void launch_seg_join(const SegArgs &g, uint32_t nlists, const float *states, const SplatArgs &a,
                     hipStream_t s);
// Staged lists (splat8.hip), the first n items of a pass (groups: an upper
// bound of their groups of 4 entries): list offsets into cbase / cbat ([n + 1]
// each); then, for lists [i0, i1) (called in two phases, [0, n1) and [n1, n)),
// each pixel's coverage per batch of 64 entries (masks) and the row counts of
// each batch and pixel column (rows), their scan (gofs; nrows[0] / nrows[1]
// counts on the device), the operands of the covering entries (ops:
// stage_floats floats in planes of stage_stride groups of 8 pixels), and the
// chains, one wave per list, channel and pixel column, which write the lists'
// blocks.  batches: stage_batches(groups, n), the room of masks (64 each) and
// of each phase's rows and gofs (8 each).  dn (device, optional): the staged
// lists are min(n, *dn) (n, i1 are capacities).
// Groups behind a plane's last stream that the chains' loads may run into
// (read ahead, never applied).
constexpr uint32_t kStagePad = 512;
uint64_t stage_floats(bool additive, uint64_t groups);
uint64_t stage_groups_in(bool additive, uint64_t bytes);  // the most with operands of `bytes`
uint64_t stage_stride(uint64_t groups);
uint64_t stage_batches(uint64_t groups, uint32_t n);
void launch_stage_base(const uint32_t *items, uint32_t n, uint32_t n1, uint32_t *cbase,
                       uint32_t *cbat, uint32_t *nrows, const SplatArgs &a, hipStream_t s,
                       const uint32_t *dn = nullptr);
void launch_stage_rows(const uint32_t *items, uint32_t i0, uint32_t i1, uint64_t batches,
                       const uint32_t *cbat, uint64_t *masks, uint32_t *rows, const SplatArgs &a,
                       hipStream_t s, const uint32_t *dn = nullptr);
void launch_stage_ops(bool additive, const uint32_t *items, uint32_t i0, uint32_t i1,
                      uint64_t batches, const uint32_t *cbase, const uint32_t *cbat,
                      const uint64_t *masks, const uint32_t *rows, const uint32_t *gofs,
                      float4 *ops, uint64_t stride, const SplatArgs &a, hipStream_t s,
                      const uint32_t *dn = nullptr);
void launch_stage_chain(bool additive, const uint32_t *items, uint32_t i0, uint32_t i1,
                        const uint32_t *cbase, const uint32_t *cbat, const uint32_t *rows,
                        const uint32_t *gofs, const float4 *ops, uint64_t stride,
                        const SplatArgs &a, hipStream_t s, const uint32_t *dn = nullptr);
// How a pass's staging length is chosen (stage_rule).
enum StageMode { kStageGiven, kStageAutoAdditive, kStageAutoOrdered };
// Device-count partition of a pass's long lists (one thread), as the host
// does it with exact counts (stage_rule): the staged lists stage_cnt[j] at
// the rule's level j (raised until they fit ns_cap and groups_cap), then at most heavy_max
// of the other lists from heavy_len on (the count heavy_cnt).  out[0] staged,
// out[1] producer/consumer, out[2] both, out[3] the first of the other long
// lists (one item each: from min(len0, heavy_len) entries on), which the 8x8
// splat serves by channel (split_lists).
struct PartitionArgs {
  const uint32_t *stage_cnt, *stage_grp, *heavy_cnt, *lmax;
  const uint64_t *etot;
  uint32_t len0;  // 0xffffffff: no staging
  StageMode mode;
  uint32_t ns_cap;
  uint64_t groups_cap;
  uint32_t heavy_max;  // 0: no producer/consumer workgroups
  uint32_t heavy_len;  // lists from this length on go to producer/consumer workgroups
  bool additive;
  uint32_t split;  // hip_split
};
// What an entry of a list costs, in ns (MI355X; a lone wave's walk 140 to 230 ordered,
// by absorption, 62 additive; by channel 100 to 118 and 54; in a producer/consumer
// workgroup 44 to 54 and 30).
struct ListRates {
  float walk, heavy;    // its walk by one wave, and in a producer/consumer workgroup
  float channels;       // the GPU's time for one walked by channel
  float staged, full;   // and for a staged one: typically covered, and in full
};
__host__ __device__ inline ListRates list_rates(bool additive) {
  return additive ? ListRates{62.f, 30.f, 0.15f, 0.165f, 0.28f}
                  : ListRates{190.f, 50.f, 0.16f, 0.2f, 0.65f};
}
// A pass's lists: count[j] and groups[j] (of 4 entries) of those from level j of
// len0 on, nheavy of those from heavy_len on.
struct ListCounts {
  const uint32_t *count, *groups;
  uint32_t len0, nheavy, heavy_max, heavy_len;
  uint64_t lmax, etot;
  __host__ __device__ float entries(int j) const { return 4.f * static_cast<float>(groups[j]); }
  __host__ __device__ bool enough_heavy() const { return heavy_max != 0u && nheavy <= heavy_max; }
  // Time of a list of `len` entries on its own, and of the longest shorter ones.
  __host__ __device__ float walk(float len, const ListRates &r) const {
    const float h = static_cast<float>(heavy_len);
    if (!enough_heavy() || len <= h) return len * r.walk;
    return len * r.heavy > h * r.walk ? len * r.heavy : h * r.walk;
  }
};
// The long lists after the first nheavy items (the staged ones, of `staged` groups,
// first) that the 8x8 splat serves by channel, of the nlong long lists: with
// hip_split given below its default (twice it in an additive pass), those from it on
// rounded down to a level of len0; else those from entries / kSplitRatio on.  Left to
// one wave, such a list (190 ns per entry ordered, by channel 105; additive 62 and 54)
// would outlast the pass (about 0.1 ns per entry over all CUs).  But walking a list by
// channel takes the GPU about twice the work: so not where that takes longer than the
// longest of these lists (16M particles at 2048^2, every leftover list by channel:
// 41.2 -> 48.2 ms; 1296 lists of 8000 ordered entries 1.6 and 2.5 ms, by absorption,
// 2.2 by channel, of 30k 5.0 and 8.3, and 7.1; 5184 of up to 30k additive ones 2.6, and
// 3.3), unless ordered lists that producer/consumer workgroups have no room for wait
// beside them (1104 of 100k: 28 ms by channel, 43 not; additive ones 14.6 and 14.0,
// 762 of 66k to 95k beside 4200 shorter 12.5 and 11.7).
constexpr uint32_t kSplitRatio = 2048;
constexpr uint32_t kSplitAuto = 32768;  // hip_split by default: the rule
__host__ __device__ inline uint32_t split_lists(const ListCounts &c, uint32_t nlong,
                                                uint32_t nheavy, uint32_t staged, float longest,
                                                bool additive, uint32_t split) {
  if (c.len0 == 0xffffffffu) return 0u;
  const bool given = split < kSplitAuto;
  const uint64_t from = given ? static_cast<uint64_t>(split) * (additive ? 2u : 1u)
                              : c.etot / kSplitRatio;
  int j = 0;
  while (j < kStageLevels - 1 && stage_level(c.len0, j + 1) <= from) ++j;
  const ListRates r = list_rates(additive);
  if (!given && (additive || c.nheavy <= c.heavy_max) &&
      (c.entries(j) - 4.f * static_cast<float>(staged)) * r.channels >= longest * r.walk)
    return 0u;
  const uint32_t n = c.count[j] < nlong ? c.count[j] : nlong;
  return n > nheavy ? n - nheavy : 0u;
}
// The staging level of a pass (-1: none): level 0 with a given length, else by
// the pass's entries and its longest list.  Lists are staged from the length on whose
// walk would outlast the pass, and not below a share of the longest list, whose chain
// bounds the pass anyway:
//   additive  from entries / 1300 (rounded down to a level) or the longest
//             list / 64 on (1M at 800^2, 5.2M entries, longest 165k: 1.23 ms
//             from 4096, 1.32 from 8192, 1.36 from 1024; 2M at 512^2: 2.35 ms
//             from 4096, 2.41 from 512)
//   ordered   from entries / 700 (rounded down) or the longest list / 16 on,
//             where the longest list bounds the pass: longest x 216 >= entries
//             (1.33M at 1279 x 719, 6.1M entries, longest 41k: 2.20 ms from
//             4096, 2.03 from 8192, 2.26 from 11585; 500k at 512^2, 1.5M
//             entries, longest 80k: 3.12 ms from 5793, 4.22 from 8192); else,
//             where it would still end after the rest in a producer/consumer
//             workgroup (108 clocks per entry against 0.25 per entry of the
//             pass: longest x 432 >= entries), the lists from entries / 432 on
//             (rounded down; 16M at 2048^2, 331M entries, longest 813k: 41.8
//             ms against 42.8 unstaged), whose operands compete least with
//             the rest; else none
// and none where the longest list is short: its walk costs less than the
// staged kernels' launches (20k ordered at 257 x 193, longest 1345 entries:
// 0.54 ms staged, 0.67 not).  From there the level rises while staging takes the GPU
// longer than the lists just below the next level take to walk, and past the longest
// list (none) where staging its like takes longer than its walk: a view in which every
// particle covers every block has hundreds of lists as long as the longest (1296 of
// 8000 additive entries: 3.5 ms staged, 0.97 not; 324 of 30k 3.2 and 2.1, ordered 7.1
// and 4.4).
__host__ __device__ inline int stage_rule(const ListCounts &c, StageMode mode) {
  if (mode == kStageGiven) return 0;
  const bool add = mode == kStageAutoAdditive;
  const uint64_t lmax = c.lmax, etot = c.etot;
  const uint32_t len0 = c.len0;
  if (lmax < (add ? 1536u : 512u)) return -1;
  int j = 0;
  if (add || lmax * 216u >= etot) {
    while (j < kStageLevels - 1 && stage_level(len0, j) * (add ? 64u : 16u) < lmax) ++j;
    while (j < kStageLevels - 1 && stage_level(len0, j + 1) * (add ? 1300u : 700u) <= etot) ++j;
  } else {
    if (lmax * 432u < etot || stage_level(len0, kStageLevels - 1) * 432u < etot) return -1;
    while (j < kStageLevels - 1 && stage_level(len0, j + 1) * 432u <= etot) ++j;
  }
  const ListRates r = list_rates(add);
  for (; j < kStageLevels && c.count[j] != 0u; ++j) {
    while (j < kStageLevels - 1 && c.count[j + 1] == c.count[j]) ++j;  // the same lists
    const uint64_t next = j < kStageLevels - 1 ? stage_level(len0, j + 1) : lmax;
    const bool last = next >= lmax;
    const float cost = c.entries(j) * (last ? r.full : r.staged);
    if (cost <= c.walk(static_cast<float>(last ? lmax : next), r)) return j;
  }
  return -1;
}
void launch_partition(const PartitionArgs &pa, uint32_t *out, hipStream_t s);
// Producer/consumer workgroups (splat8.hip), one per item: the first npc
// items, the units whose lists reach a.heavy_len.
void launch_splat_pc(bool additive, const uint32_t *items, uint32_t npc, const SplatArgs &a,
                     hipStream_t s, const ItemCounts &dc = ItemCounts{});
// Differentiable form (adjoint.hip): screen-space gradient accumulation over
// the forward's work items (gscr: n x 6 doubles, zeroed by the caller), the
// chain to the particle fields of job 0, and an FP64 fill.
// Backward work items: list segments of at most seglen entries per unit
// (cnt[u] segments; soff = exclusive scan of cnt).  A segment is one wave's
// serial walk, so short segments shorten the backward's critical path and its
// last, partly filled round of waves; an ordered one has 4.6 KB of FP64 state
// (500k ordered particles at 512^2, forward + backward: 2.97 ms with 512 entries,
// 2.41 with 256, 2.29 with 128, 2.39 with 64; 2M additive ones 2.15 ms with 256,
// 2.20 with 128).  Ordered passes past kAdjShort entries, which fill the GPU many
// times over, keep 256 and half the state.
constexpr uint32_t kAdjSeg = 256, kAdjSegOrdered = 128;
constexpr uint64_t kAdjShort = uint64_t(1) << 26;
inline uint32_t adjoint_seglen(bool additive, uint64_t entries) {
  return additive || entries > kAdjShort ? kAdjSeg : kAdjSegOrdered;
}
void launch_seg_count(const uint32_t *bin_off, uint32_t nunits, uint32_t seglen, uint32_t *cnt,
                      hipStream_t s);
void launch_seg_emit(const uint32_t *bin_off, uint32_t nunits, uint32_t nseg,
                     uint32_t seglen, const uint32_t *soff, uint32_t *seg_unit,
                     uint32_t *seg_first, hipStream_t s);
// part: 6 floats per list entry (the particle's screen-space partials over
// the entry's block); segstate: ordered mode only, nseg * 3 * 64 * 3 doubles.
void launch_adjoint(bool additive, const uint32_t *seg_unit, const uint32_t *seg_first,
                    uint32_t nseg, uint32_t seglen, const uint32_t *soff, uint32_t nunits,
                    const SplatArgs &a, const float *grad, float *part, double *segstate,
                    hipStream_t s);
// v[i] = i
void launch_iota(uint32_t *v, uint32_t n, hipStream_t s);
// gscr[order[s]] += sum over t in [poff[s], poff[s+1]) of part[jv[t]] (FP64,
// in that order), for the m particles of a pass.
void launch_reduce_parts(const uint32_t *poff, const uint32_t *jv, const float *part,
                         const uint32_t *order, uint32_t m, double *gscr, hipStream_t s);
void launch_chain(const ProjectArgs *jobs, int64_t n, const uint8_t *act, const double *gscr,
                  const splhip_grads &out, hipStream_t s);
void launch_zero_f64(double *p, int64_t n, hipStream_t s);
// G: region size (16, 32 or 64 px); additive: a_eq_e mode.  Single job.
void launch_splat(int G, bool additive, uint32_t nbins, const SplatArgs &a, hipStream_t s);

// Post-processing of a frame (post.hip): -expm1 when a_eq_e, colour_adjust
// when adjust, nbars colorbars of types bar_type[], then Colour8 bytes.
struct PostArgs {
  const float *pic;  // x-major RGB image
  float *out;        // post-processed float image (may be pic, or null)
  uint8_t *rgb8;     // bytes (null: none)
  int32_t xres, yres;
  int32_t a_eq_e, adjust, nbars;
  int32_t vec_in, vec_out;  // float4 image columns / bytes per word of a row (set by launch_post)
  int32_t bar_type[kMaxTypes];
  int32_t pal_n[kMaxTypes];
  int32_t pal_stride;
  double gamma, brightness, contrast;
  const double *pal_x;
  const float *pal_rgb;
  const float *exptab;
  float expfac, taylorlimit;
};
// layout 0: bytes in the image's x-major RGB order; 1: the TGA file body
// (rows iy ascending, B G R).
void launch_post(const PostArgs &a, int layout, hipStream_t s);

// particle_normalize over SoA fields (normalize.hip): flags[t] = intensity_log,
// color_log, color_asinh, color_is_vector; ovr_set / ovr[t] = intensity_min,
// intensity_max, color_min, color_max given as parameters.
struct NormArgs {
  int64_t n;
  float *I, *er, *eg, *eb;
  const float *r;
  const uint8_t *type;
  int32_t ntypes, norm_int;
  int32_t vector;  // some type has a vector colour (set by launch_normalize)
  int32_t flags[kMaxTypes][4];
  int32_t ovr_set[kMaxTypes][4];
  float ovr[kMaxTypes][4];
};
// Block-file ingest (ingest.hip): in place, byte swap when swap, then
// scale * v when scaled (else a multiply by one: only NaNs are quieted).
void launch_ingest_fix(float *d, int64_t n, int swap, int scaled, float scale, hipStream_t s);
void launch_fill_u8(uint8_t *p, uint8_t v, int64_t n, hipStream_t s);

// keys: 6 ntypes u32 of scratch; after the call they hold the per-type
// extremes as order-preserving keys (colour, intensity, size; min then max).
void launch_normalize(const NormArgs &a, uint32_t *keys, hipStream_t s);

}  // namespace splhip
