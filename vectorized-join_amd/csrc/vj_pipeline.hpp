// Descriptors of one join pipeline (a batch of one or more joins), shared by
// the host planner (vj_context.cpp) and the kernels (vj_join_kernels.hip).
//
// A join has two jobs: its build side (R) and its probe side (S). Each job is
// hashed and radix-partitioned on the same digits; the build+probe stage then
// draws (join, partition, R-chunk, S-chunk) tasks from a device work queue.
//
// Partitioning is count-then-scatter with exact destinations, so scatter
// blocks never wait on each other:
//  * A job's rows are cut into pass-1 tiles (T rows) grouped into segments,
//    and each segment into hsplit histogram rows of consecutive tiles (more
//    histogram blocks than segments when the segments alone would leave CUs
//    idle). The histogram kernel walks each row's tiles in order and records,
//    per tile, the exclusive prefix of its pass-1 digit counts inside the row
//    (tilepre), and per row the pass-1 digit counts (m1 row) and the
//    (pass-1, pass-2) digit counts (m2 row).
//  * Column scans over the rows turn m1 / m2 into per-row offsets, and a scan
//    over the column totals gives the partition bases.
//  * Pass 1 writes tile t's rows of digit d1 at
//      base[d1 << b2] + m1[row(t)][d1] + tilepre[t][d1] + rank.
//  * Pass 2 reads chunk (d1, g) = segment g's rows of pass-1 partition d1 (a
//    contiguous range of the pass-1 output, from row g * hsplit to the next
//    segment's) and writes its rows of digit d2 at
//      base[(d1 << b2) | d2] + m2[g * hsplit][(d1 << b2) | d2] + rank.
//
// HBM layout per partitioned job: SoA copies of the key columns plus a uint32
// row-id column, once after pass 1 ("mid", only for 2-pass jobs) and once
// after the last pass ("fin"). Partition q of a job occupies rows
// [base[q], base[q+1]) of "fin"; q = d1 * 2^b2 + d2 (pass-1 digit major).
//
// One-pass form (the exact layout's default up to kFanBits radix bits in all,
// whether the plan calls them one pass or two): no mid copy, no tile prefixes.
// Tile t of the pipeline belongs to group t % kXcds (the XCD its block runs
// on); k_fan_hist counts every job's rows by (group, partition), k_fan_plan
// turns the counts into partition bases and, inside each partition, one write
// cursor per group, and k_fan takes its rows' runs from its group's cursors
// with one device atomic per (tile, partition). The runs of one group's tiles
// follow each other in memory, so the lines they share fill up in one XCD's
// L2; partitions come out back to back, as after two passes.
//
// Region layout (2-pass pipelines that ask for it): no histogram and no scans.
// Every destination is a region of fixed capacity, and blocks reserve their
// runs in it with one device atomic per digit:
//  * pass 1 writes tile t's rows of digit d1 into region (d1, g) of "mid",
//    g = t / seg_tiles (the segment: segments spread the atomics over
//    2^b1 * nseg counters), rows [(d1 * nseg + g) * region1, + region1);
//  * pass 2 reads that region in tiles (chunk = (d1, g, tile k)) and writes
//    its rows of digit d2 into region q = (d1 << b2) | d2 of "fin", rows
//    [q * region2, + region2), counter m2[q].
// A run that does not fit its region goes to a one-tile trash area after the
// regions, and the counter keeps the full count, so an overflow is visible
// after the passes (k_tasks then schedules no task for the join and sets
// Ctl::overflow; the host runs the join again with the exact layout).
#pragma once
#include <stdint.h>

#include "vj_device.hpp"

namespace vj {

constexpr int kPassThreads = 512;   // radix pass kernels
constexpr int kPassWaves = kPassThreads / 64;
constexpr int kHistThreads = 1024;  // histogram kernel
constexpr int kMaxProbeThreads = 1024;  // build+probe kernel (512 or 1024 threads, see probe_threads)
constexpr int kMaxProbeWaves = kMaxProbeThreads / 64;
constexpr int kMaxSegments = 512;  // segments (histogram blocks) per job
constexpr int kMaxPassBits = 8;     // digits per pass <= 256
constexpr int kMaxHistBits = 14;    // 2D histogram in LDS: 2^14 x 4 B = 64 KiB
constexpr uint32_t kXcds = 8;       // accelerator dies (XCDs) of an MI355X
constexpr uint32_t kXcdGroup = 32;  // consecutive pass-2 chunks kept on one XCD
constexpr int kFanBits = 11;        // radix bits one pass can take (k_fan): 2^11 counters in LDS
constexpr int kFanThreads = 1024;   // one-pass kernels (k_fan_hist, k_fan_plan, k_fan)
constexpr uint32_t kFanPlanParts = 1u << kFanBits;  // partitions k_fan_plan handles: two per thread
static_assert(kFanPlanParts == 2 * kFanThreads, "k_fan_plan: two partitions per thread");

// Kernel shapes, chosen per pipeline by the planner or the autotuner.
//  tile  0: standard pass tile, 512 threads x pass_items rows (6 / 4 / 2 rows by
//           key bytes); 1: small tile, 512 threads x 2 rows (more blocks for
//           small tables); 2: large tile, 512 threads x 8 / 6 / 4 rows (longer
//           runs per digit; the region layout's tile).
//  table 0: standard build+probe block, 512 threads (up to four blocks per
//           CU) around an LDS table of build_cap rows; 1: wide block, 1024
//           threads (one block per CU) around a table of wide_cap rows, so a
//           partition four to eight times larger fits one build chunk.
__host__ __device__ constexpr int pass_items(int key_bytes, int tile = 0) {
    return tile == 1 ? 2
                     : (tile == 2 ? (key_bytes <= 8 ? 8 : (key_bytes <= 16 ? 6 : 4))
                                  : (key_bytes <= 8 ? 6 : (key_bytes <= 16 ? 4 : 2)));
}
// Rows per thread of the one-pass kernel k_fan. Large tiles (2^11 partitions)
// keep a run at a few rows: 12 of 8-byte keys is the largest tile whose keys
// fit the LDS (one block per CU); below that, 4096-row tiles leave room for
// two blocks per CU, whose phases overlap.
__host__ __device__ constexpr int fan_items(int key_bytes, int big) {
    return !big ? 4 : (key_bytes <= 8 ? 12 : (key_bytes <= 16 ? 8 : 6));
}
__host__ __device__ constexpr int fan_tile(int key_bytes, int big) { return kFanThreads * fan_items(key_bytes, big); }
constexpr int kTileShapes = 3;
__host__ __device__ constexpr int pass_tile(int key_bytes, int tile = 0) { return kPassThreads * pass_items(key_bytes, tile); }
__host__ __device__ constexpr int build_cap(int key_bytes) { return key_bytes <= 8 ? 2048 : 1024; }
// The build+probe block's LDS table: per build row its key, its 4-byte row id
// and a 2-byte link, and a power of two of 2-byte chain heads. Row entries are
// counted from 1 (entry 0 stands for the end of a chain), hence the + 1.
__host__ __device__ constexpr int table_bytes(int key_bytes, int cap, int heads) {
    return ((cap + 1) * (key_bytes + 6) + 15) / 16 * 16 + heads * 2;
}
constexpr int kTableBytes = 162 * 1000;  // of the 160 KiB of LDS per CU; the rest holds the task record
// Largest power of two <= 8192 whose table, with two heads per row, fits.
__host__ __device__ constexpr int wide_cap(int key_bytes) {
    int c = 8192;
    while (c > 1024 && table_bytes(key_bytes, c, 2 * c) > kTableBytes) c >>= 1;
    return c;
}
// table 2: the wide block around 8960 rows (keys of up to 8 bytes): what the
// LDS holds beside 2^14 heads. 2^11 partitions of a 2^24-row build average 8192
// rows; 8960 leave 8 standard deviations of their spread.
constexpr int kFullCap = 8960;
__host__ __device__ constexpr int probe_cap(int key_bytes, int table) {
    return table == 0 ? build_cap(key_bytes) : (table == 2 ? kFullCap : wide_cap(key_bytes));
}
// Chain heads: as many as keep the block's share of the LDS (a quarter of it
// for standard tables of up to 8-byte keys), two to four per row.
__host__ __device__ constexpr int probe_heads(int key_bytes, int table) {
    return table ? 16384 / (key_bytes > 24 ? 2 : (key_bytes > 16 ? 2 : 1)) : (key_bytes <= 4 ? 8192 : 4096);
}
__host__ __device__ constexpr int probe_table_bytes(int key_bytes, int table) {
    return table_bytes(key_bytes, probe_cap(key_bytes, table), probe_heads(key_bytes, table));
}
__host__ __device__ constexpr int probe_threads(int table) { return table ? 1024 : 512; }
constexpr int kProbeChunk = 16384;  // probe rows one walk of the build+probe kernel covers
static_assert(wide_cap(4) == 8192 && wide_cap(8) == 8192 && wide_cap(16) == 4096 && wide_cap(24) == 4096 && wide_cap(32) == 2048,
              "wide tables");
static_assert(probe_table_bytes(8, 1) <= kTableBytes && probe_table_bytes(8, 2) <= kTableBytes &&
                  probe_table_bytes(16, 1) <= kTableBytes && probe_table_bytes(24, 1) <= kTableBytes &&
                  probe_table_bytes(32, 1) <= kTableBytes,
              "tables fit the LDS");

struct JobDesc {
    TView in;                 // the caller's table
    // pass-1 output (2-pass jobs); one-pass form: [0] is null, or row-major 64-bit
    // keys that k_fan_hist reads in place of in's columns, which it fills
    void *mid_cols[4];
    uint32_t *mid_ids;
    void *fin_cols[4];        // last-pass output (partitioned jobs)
    uint32_t *fin_ids;
    uint32_t n;
    uint32_t b1, b2;          // radix bits of pass 1 / pass 2 (b1 == 0: not partitioned)
    uint32_t shift0;          // digit of pass 1 = (h >> shift0) & (2^b1 - 1)
    uint32_t base_off;        // u32 offset of the 2^(b1+b2)+1 partition bases in the base arena
    uint32_t p1_tiles;        // pass-1 tiles
    uint32_t seg_tiles;       // pass-1 tiles per segment
    uint32_t nseg;            // segments (pass-2 chunks of one pass-1 digit)
    uint32_t hsplit;          // histogram rows (blocks) per segment
    uint32_t hrow_tiles;      // pass-1 tiles per histogram row (ceil(seg_tiles / hsplit))
    uint32_t nrow;            // histogram rows = nseg * hsplit (= histogram blocks)
    // Region layout (0: exact layout): rows per pass-1 region (d1, segment),
    // rows per final region (partition), pass-2 chunks (tiles) per pass-1 region
    uint32_t region1, region2, region_tiles;
    // u32 offset of the partition ends in the base arena: partition q is rows
    // [base[base_off + q], base[end_off + q]) of fin (exact layout: end_off =
    // base_off + 1; region layout: a second array, both written by k_tasks)
    uint32_t end_off;
    uint32_t groups;          // one-pass form: write-cursor groups (kXcds, or 1 for few tiles)
    uint32_t pad_;
    uint64_t tilepre_off;     // u32 offset of tilepre [p1_tiles][2^b1] in the count arena
    uint64_t m1_off;          // u32 offset of m1 [nrow + 1][2^b1] (region layout: counters [2^b1][nseg];
                              // one-pass form: counts, then cursors [groups][2^(b1+b2)])
    uint64_t m2_off;          // u32 offset of m2 [nrow + 1][2^(b1+b2)] (2-pass jobs; region layout: counters [2^(b1+b2)])
    // Resident build sides. res_base != null: the job is already partitioned
    // (fin_* point at a resident table, res_base at its 2^(b1+b2)+1 bases) and
    // no hist / pass work is scheduled for it. keep_base != null: the bases
    // are also written there (the job's fin_* point at a table being kept).
    const uint32_t *res_base;
    uint32_t *keep_base;
};

struct JoinDesc {
    uint32_t job_r, job_s;
    uint32_t *out_r, *out_s;
    uint64_t cap;             // output capacity (pairs)
    uint32_t cap_r, cap_s;    // tuples per build chunk / probe chunk 
    uint32_t ptask_off;       // u64 offset of the per-partition task prefix (nparts + 1)
    uint32_t nparts;          // 2^(b1+b2)
    uint32_t slot_shift;      // hash bits consumed by partitioning (slot uses h >> slot_shift)
    uint32_t one_based;
    uint32_t part_off;        // u64 offset of the task-prefix blocks' partials [ceil(nparts / kTaskBlock)][4]
    uint32_t pad_;
};

constexpr uint32_t kTaskBlock = 1024;  // partitions per block of the task-prefix kernels

constexpr int kColScanCols = 64;     // columns per block of the column-scan kernel

// One block of the column-scan kernel: kColScanCols columns of one job's m1 or m2.
struct ColScanDesc {
    uint32_t job;
    uint32_t which;  // 1: m1, 2: m2
    uint32_t col0;
    uint32_t pad;
};

// Control words: the ticket is reset by k_bases (k_region_reset in the region
// layout), the total written by k_tasks (one join) or k_scan2, before the
// build+probe kernel reads them. overflow: a region of the region layout
// received more rows than it holds (set by k_tasks).
// done: build+probe blocks that have ended; the last one sets it back to 0.
// t0, t1: the device clock at the start of the first kernel (one-pass form) and
// at the end of the last block (written to the host's copy only).
struct Ctl {
    unsigned long long task_ticket;
    unsigned long long task_total;
    unsigned long long overflow;
    unsigned long long done;
    unsigned long long t0, t1;
};


struct PipeArgs {
    const JobDesc *jobs;
    const JoinDesc *joins;
    const ColScanDesc *colscan;     // [n_colscan]
    const uint32_t *hist_block0;    // [n_jobs + 1] prefix of nrow (host)
    const uint32_t *p1_tile0;       // [n_jobs + 1] prefix of p1_tiles (host)
    const uint32_t *p2_chunk0;      // [n_jobs + 1] prefix of pass-2 chunks (host)
    unsigned long long *join_tasks;   // [n_joins] (device)
    unsigned long long *task0;        // [n_joins + 1] (device)
    unsigned long long *out_count;    // [n_joins] (device)
    Ctl *ctl;
    uint32_t *counts;               // count arena: tilepre / m1 / m2 of every job
    uint32_t *base;
    unsigned long long *ptask;
    unsigned long long *taskmap;    // [taskmap_cap] task -> join << 32 | partition (tasks past it are searched)
    unsigned long long taskmap_cap;
    uint32_t max_nparts;            // partitions of the largest join
    uint32_t n_jobs, n_joins, n_colscan;
    uint32_t total_hist_blocks, total_p1_tiles, total_p2_chunks;
    uint32_t max_hist_bins;         // LDS bins of the histogram kernel
    uint32_t pass_tile;             // tuples per radix-pass tile (pass_tile(key bytes, tile shape))
    uint32_t regions;               // region layout (every job: two passes, 2^b1 a multiple of kXcds)
    uint32_t fan_bins;              // one-pass form: partitions of the largest job (0: another form)
    uint64_t count_words;           // one-pass form: words of the count arena (zeroed before k_fan_hist)
    // one-pass form: the descriptors' way from the host's staging buffer, in words of 8 bytes
    unsigned long long *up_dst;
    const unsigned long long *up_src;
    uint32_t up_words;
    // out_count and what follows it (to ctl's t0; t1 is taken then) goes to the host's buffer when build+probe ends
    uint32_t down_words;
    unsigned long long *down;
    HashCfg hash;
};

// One join without partitions (k_direct). count and done are zero before the
// launch and after it; the match count and the device clock at the start
// (count[1]) and the end are written to `down` (host memory).
struct DirectArgs {
    TView r, s;
    uint32_t *out_r, *out_s;
    uint64_t cap;
    uint32_t cap_s;  // probe rows per block
    uint32_t one_based;
    unsigned long long *count, *done, *down;
    HashCfg hash;
};

// The flat form (k_flat_build, k_flat_probe): slots of the table in 16-byte
// groups, zero before the build; links of equal keys, one per build row.
constexpr int kFlatThreads = 512;
// Probe blocks of a single join are large, since every block takes a turn at the
// one counter (join_into, us: 2^16 x 2^20 4-byte keys 51 with two atomics per
// block of 512 x 2 rows, 47 with one, 40 with one per 1024 x 4; 2^18 x 2^24,
// 512 x 8: 167, 1024 x 4: 161; 2^16 x 2^22 8-byte keys 94 / 90; 2^18 probe rows
// 4 x u32, 512 x 2: 81, 1024 x 2: 84). A batch's are of kFlatThreads and these rows
// per thread: its counters are as many as its joins (64 joins of up to 2048 int64
// rows, 512 x 8: 90, 1024 x 4: 103).
__host__ __device__ constexpr int flat_batch_rows(int key_bytes) { return key_bytes <= 8 ? 8 : 4; }
constexpr uint32_t kFlatChain = 64;                     // rows of one key followed link by link
constexpr unsigned long long kFlatGiveUp = 1ull << 63;  // in the count: a chain was longer
// The counter of a join: matches (below 2^32 rows x 65) and, above them, the
// blocks that have reserved their output (at most 2^22 of 1024 rows or more).
constexpr unsigned long long kFlatBlock = 1ull << 40;
constexpr uint64_t kFlatTableBytes = 4ull << 20;  // an XCD's L2
// All tables of a batch, beyond which the pipeline is the faster one (us a call,
// flat and pipeline, build sides log-uniform from 2^10, probe sides 4-16 times
// as large): 4-byte keys, 64 joins of up to 2^14 rows (8 MB) 105 / 150, of 2^16
// (21 MB) 186 / 219, of 2^18 (63 MB) 434 / 361, 16 of 2^18 (14 MB) 131 / 141;
// 8-byte keys, 20 joins of up to 2^15 rows (13 MB) 72 / 101, 16 of 2^16 (23 MB)
// 122 / 113, 64 of 2^16 (85 MB) 304 / 227; 4 x u32, 40 of 2^14 (18 MB)
// 118 / 158, of 2^16 (57 MB) 206 / 198; 2 x u64, 30 of 2^15 (24 MB) 124 / 159;
// two joins of 2048 rows 34 / 69.
__host__ __device__ constexpr uint64_t flat_batch_bytes(int key_bytes) { return (key_bytes > 4 && key_bytes <= 8 ? 16ull : 32ull) << 20; }
__host__ __device__ constexpr int flat_slot_bytes(int key_bytes) { return key_bytes <= 4 ? 8 : 16; }
// Build rows of the largest table: half full in pairs of 8-byte slots, a
// quarter in single 16-byte ones, whose chains grow sooner (join_into, us, flat and
// pipeline: 4-byte keys 2^18 x 2^24 162 / 180, 2^19 x 2^22 108 / 92; 8-byte keys
// 2^16 x 2^20 52 / 76, 2^16 x 2^22 85 / 100; 4 x u32 2^16 x 2^20 65 / 114). Twice
// as many rows of over 4 bytes, a table past an L2, where the probe side is of the
// build side's size or more and not past kFlatMaxProbe rows: 8-byte keys 2^17 x 2^20
// 65 / 74, 2^17 x 2^22 110 / 98, 2^18 x 2^20 84 / 75; 4 x u32 2^17 x 2^20 74 / 89,
// 2^17 x 2^22 162 / 136; 4 x u64 2^17 x 2^21 132 / 141.
__host__ __device__ constexpr uint64_t flat_max_rows(int key_bytes) {
    return kFlatTableBytes / flat_slot_bytes(key_bytes) / (key_bytes <= 4 ? 2 : 4);
}
constexpr uint64_t kFlatMaxProbe = 1ull << 21;
struct FlatArgs {
    TView r, s;
    uint32_t *slots;
    uint32_t *nxt;
    uint32_t *dup;      // set when two build rows have equal keys
    uint32_t mask;      // slots - 1
    uint32_t hshift;    // 32 - log2 of the slots (of the pairs for 4-byte keys)
    uint32_t *out_r, *out_s;
    uint64_t cap;
    uint32_t one_based;
    uint32_t zero_words;  // 16-byte words from `slots` on to clear before the build (the table, then dup)
    // the counter, zero before the launch (and after it where clock is set); host memory for the match count
    // (then the device clock at the start and the end); a single join's start on that clock
    unsigned long long *count, *down, *clock;
    HashCfg hash;
};

// A batch in the flat form: its joins' arguments in memory, a grid over all of
// their build blocks and one over their probe blocks.
struct FlatBatch {
    const FlatArgs *joins;
    const uint32_t *build0, *probe0;  // [n_joins + 1] prefixes of the joins' blocks
    uint32_t n_joins, build_blocks, probe_blocks;
    uint32_t up_words;                // the arguments' and prefixes' way from the host's buffer, in 8-byte words
    unsigned long long *up_dst;
    const unsigned long long *up_src;
    uint32_t *zero;                   // the tables and their dup words
    uint64_t zero_words;              // in 16-byte words
    unsigned long long *counts;
};

// Kernel launchers (vj_join_kernels.hip); all asynchronous on `s`.
struct LaunchShape {
    int hp, kw, nc;  // hash path, key width, key columns
    int cus;         // compute units of the device
    int tile, table; // kernel shapes (see pass_items / probe_cap)
    int fan_big;     // one-pass form: large tiles (see fan_items)
};

// The hashing stages (histogram, radix pass, build+probe), compiled once per
// hash path in its own translation unit (vj_join_fnv.hip, vj_join_xorhw.hip,
// vj_join_generic.hip) from vj_join_stages.hpp.
template <int HP> struct StageLaunch {
    static hipError_t hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
    static hipError_t pass(const PipeArgs &a, const LaunchShape &sh, int pass, hipStream_t s);
    static hipError_t fan_hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
    static hipError_t fan(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
    static hipError_t probe(const PipeArgs &a, const LaunchShape &sh, int blocks, hipStream_t s);
    static hipError_t direct(const DirectArgs &d, const LaunchShape &sh, int blocks, hipStream_t s);
    static hipError_t flat(const FlatArgs &a, const LaunchShape &sh, hipStream_t s);
    static hipError_t flat_batch(const FlatBatch &b, const LaunchShape &sh, hipStream_t s);
    static int probe_blocks_per_cu(const LaunchShape &sh);
};
extern template struct StageLaunch<HP_FNV>;
extern template struct StageLaunch<HP_XOR_HW>;
extern template struct StageLaunch<HP_GENERIC>;
hipError_t launch_hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
hipError_t launch_scan(const PipeArgs &a, hipStream_t s);
hipError_t launch_flat(const FlatArgs &a, const LaunchShape &sh, hipStream_t s);
hipError_t launch_flat_batch(const FlatBatch &b, const LaunchShape &sh, hipStream_t s);
hipError_t launch_direct(const DirectArgs &d, const LaunchShape &sh, int blocks, hipStream_t s);
hipError_t launch_fan_begin(const PipeArgs &a, hipStream_t s);
hipError_t launch_fan_hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
hipError_t launch_fan_plan(const PipeArgs &a, hipStream_t s);
hipError_t launch_fan(const PipeArgs &a, const LaunchShape &sh, hipStream_t s);
hipError_t launch_region_reset(const PipeArgs &a, hipStream_t s);
hipError_t launch_tasks(const PipeArgs &a, hipStream_t s);
hipError_t launch_reset_probe(const PipeArgs &a, hipStream_t s);
hipError_t launch_stage_copy(void *dst, const void *src, size_t bytes, hipStream_t s);
hipError_t launch_pass(const PipeArgs &a, const LaunchShape &sh, int pass, hipStream_t s);
hipError_t launch_probe(const PipeArgs &a, const LaunchShape &sh, int blocks, hipStream_t s);
int probe_blocks_per_cu(const LaunchShape &sh);
hipError_t launch_emit_hist(const uint32_t *base, uint32_t nb, uint32_t *hist, uint32_t *offsets, hipStream_t s);

}  // namespace vj
