// The join pipeline's hashing stages, templated on the hash path, the key
// shape and the kernel shapes:
//
//   k_hist   per segment of a job: per-tile pass-1 digit prefixes, the
//            segment's pass-1 and (pass-1, pass-2) digit counts (LDS)
//   k_pass   one radix pass over a tile (pass 1) or a (digit, segment) chunk
//            (pass 2)
//   k_fan_hist, k_fan  the one-pass form: counts per (group, partition), then
//            one pass of up to 2^11 partitions with atomically reserved runs
//   k_probe  persistent build + probe over (join, partition, R-chunk,
//            S-chunk) tasks from a device queue
//
// Included once per hash path (vj_join_fnv.hip, vj_join_xorhw.hip,
// vj_join_generic.hip), each of which instantiates StageLaunch<HP>, so the
// three paths compile in parallel. The reference's counterparts are
// histogram_kernel / prefix_sum_kernel / element_swap_kernel
// (src/join/join_provider.cu:315-380) and the build / probe / extract
// kernels (:382-608).
#pragma once
#include "vj_kernel_common.hpp"

namespace vj {

namespace {

// ---------------------------------------------------------------------------

// One block per segment. The block sweeps the segment one pass-1 tile at a
// time (all 1024 threads on one tile, coalesced), with one LDS atomic per row
// into the tile's pass-1 digit counters and, for 2-pass jobs, one into the
// segment's (pass-1, pass-2) histogram. Tile counters live in a ring of
// kHistRing tiles; every kHistRing tiles the ring is folded into the running
// in-segment prefix, which is stored per tile (tilepre).
constexpr int kHistRing = kHistThreads / 64;

template <int HP, int KW, int NC, int TV>
__global__ __launch_bounds__(kHistThreads) void k_hist(PipeArgs a) {
    constexpr int KB = KW * NC;
    constexpr int T = pass_tile(KB, TV);
    constexpr int U = T / kHistThreads;
    static_assert(U * kHistThreads == T, "a tile is a whole number of block sweeps");
    extern __shared__ uint32_t lds[];
    const uint32_t b = blockIdx.x, tid = threadIdx.x;
    const uint32_t j = upper_index(a.hist_block0, a.n_jobs, b);
    const JobDesc &job = a.jobs[j];
    const uint32_t g = b - a.hist_block0[j];
    const uint32_t n1 = 1u << job.b1, nb = 1u << (job.b1 + job.b2);
    const bool two = job.b2 > 0;
    uint32_t *h2 = lds;                    // [nb] (2-pass jobs)
    uint32_t *run = lds + (two ? nb : 0);  // [n1] running in-segment prefix
    uint32_t *th = run + n1;               // [kHistRing][n1] tile counts
    for (uint32_t i = tid; i < (two ? nb : 0) + n1 * (1 + kHistRing); i += kHistThreads) lds[i] = 0;
    __syncthreads();
    const uint32_t m1 = n1 - 1, m2 = (1u << job.b2) - 1, b2 = job.b2;
    const uint32_t s1 = job.shift0, s2 = job.shift0 + job.b1;
    const bool lo32 = s2 + b2 <= 32;  // every digit below bit 32 (joins): the low half of the hash suffices
    const HashCfg hc = a.hash;
    // histogram row g: the hrow_tiles tiles of segment g / hsplit starting at
    // its (g % hsplit)-th row (the last rows of a segment may be short or empty)
    const uint32_t sg = g / job.hsplit;
    const uint32_t s_end0 = (sg + 1) * job.seg_tiles;
    const uint32_t s_end = s_end0 < job.p1_tiles ? s_end0 : job.p1_tiles;
    const uint32_t r0 = sg * job.seg_tiles + (g - sg * job.hsplit) * job.hrow_tiles;
    const uint32_t t_begin = r0 < s_end ? r0 : s_end;
    const uint32_t t_end = t_begin + job.hrow_tiles < s_end ? t_begin + job.hrow_tiles : s_end;
    const gptr<uint32_t> tilepre = to_global(a.counts + job.tilepre_off);
    const GKeys<KW, NC> in = uniform_keys<KW, NC>(job.in);
    const uint32_t n = job.n;
    for (uint32_t t0 = t_begin; t0 < t_end; t0 += kHistRing) {
        const uint32_t kt = t_end - t0 < (uint32_t)kHistRing ? t_end - t0 : (uint32_t)kHistRing;
        for (uint32_t k = 0; k < kt; k++) {
            uint32_t *thk = th + k * n1;
            const uint32_t row_lo = (t0 + k) * T + tid;
            Key<KW, NC> key[U];
#pragma unroll
            for (int u = 0; u < U; u++) {  // all loads in flight at once (past the end: row 0 again)
                const uint32_t i = row_lo + u * kHistThreads;
                key[u] = load_key<KW, NC>(in, i < n ? i : 0u);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t i = row_lo + u * kHistThreads;
                if (i < n) {
                    const uint64_t h = lo32 ? (uint64_t)hash_key_lo<HP, KW, NC>(key[u], hc) : hash_key<HP, KW, NC>(key[u], hc);
                    const uint32_t d1 = (uint32_t)(h >> s1) & m1;
                    atomicAdd(&thk[d1], 1u);
                    if (two) atomicAdd(&h2[(d1 << b2) | ((uint32_t)(h >> s2) & m2)], 1u);
                }
            }
        }
        __syncthreads();
        if (tid < n1) {
            uint32_t acc = run[tid];
            for (uint32_t k = 0; k < kt; k++) {
                tilepre[(uint64_t)(t0 + k) * n1 + tid] = acc;
                acc += th[k * n1 + tid];
                th[k * n1 + tid] = 0;
            }
            run[tid] = acc;
        }
        __syncthreads();
    }
    const gptr<uint32_t> m1row = to_global(a.counts + job.m1_off + (uint64_t)g * n1);
    for (uint32_t d = tid; d < n1; d += kHistThreads) m1row[d] = run[d];
    if (two) {
        const gptr<uint32_t> m2row = to_global(a.counts + job.m2_off + (uint64_t)g * nb);
        for (uint32_t q = tid; q < nb; q += kHistThreads) m2row[q] = h2[q];
    }
}

// ---------------------------------------------------------------------------
// Radix pass
// ---------------------------------------------------------------------------

struct PassTile {
    TView src;
    void *dst_cols[4];
    uint32_t *dst_ids;
    uint32_t lo, hi;        // rows of src (pass 2: the whole chunk)
    uint32_t bins, shift;
    uint32_t job, local;    // job and tile (pass 1) / chunk (pass 2) index inside it
    uint32_t valid;
    // region layout (region == 0: exact layout): digit d's counter is
    // counts[rc0 + d * rstride], its region starts at row rrow0 + d * rdstride
    uint32_t region, rstride, rrow0, rdstride, trash;
    uint64_t rc0;
};

// Waves per SIMD the pass kernel is compiled for: 8 (64 VGPRs, four blocks per
// CU) for single 8-byte keys with FNV / XOR hashing; wider keys and the
// generic hash path get 6 (80 VGPRs, three blocks) to limit spills; the large
// tile (more rows per lane) 6, or 5 beyond 8-byte keys.
template <int HP, int KB, int TV> constexpr int pass_waves_per_simd() {
    return TV == 2 ? (KB <= 8 ? 6 : 5) : (KB <= 8 && HP != HP_GENERIC ? 8 : 6);
}

// Pass 1: one tile of a job. Pass 2: one (pass-1 digit, segment) chunk, in
// tile-sized steps; a running count per digit carries the destination.
// TV: tile shape (pass_items).
template <int HP, int KW, int NC, int TV>
__global__ __launch_bounds__(kPassThreads, (pass_waves_per_simd<HP, KW * NC, TV>())) void k_pass(PipeArgs a, int pass) {
    using KT = typename KeyT<KW>::T;
    constexpr int KB = KW * NC;
    constexpr int ITEMS = pass_items(KB, TV);
    constexpr int T = kPassThreads * ITEMS;
    constexpr int STAGE = (KB > 4 ? KB : 4) * T;  // key columns, then row ids, staged in turn
    extern __shared__ __align__(16) unsigned char smem[];
    KT *skeys = reinterpret_cast<KT *>(smem);                             // [NC][T]
    uint32_t *sids = reinterpret_cast<uint32_t *>(smem);                   // [T] (after the keys are out)
    uint32_t *wcnt = reinterpret_cast<uint32_t *>(smem + STAGE);           // [kPassWaves][256]
    uint32_t *loc = wcnt + kPassWaves * 256;                               // [256]
    uint32_t *gdst = loc + 256;                                            // [256] next destination row
    uint32_t *gdo = gdst + 256;                                            // [256] gdst - loc of the current tile
    uint8_t *sdig = reinterpret_cast<uint8_t *>(gdo + 256);                // [T]
    __shared__ PassTile ti;
    __shared__ uint32_t sh_scan[kPassWaves + 1];

    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (w == 0) {
        // Workgroups are dispatched round-robin over the XCDs. Consecutive
        // tiles go to one XCD, so that the runs adjacent tiles write to one
        // partition (which share cache lines) meet in the same L2: pass 1
        // gives each XCD one contiguous range of tiles; pass 2 deals out
        // groups of kXcdGroup consecutive chunks round-robin, so that a run of
        // heavy chunks (a skewed partition) is spread over all XCDs (block k
        // of XCD x takes chunk (k / G * 8 + x) * G + k % G).
        // In the region layout the runs into one final region arrive in
        // atomic order, so pass 2 keeps every chunk of a pass-1 digit d1 on
        // XCD d1 % kXcds instead: a region's partial lines then merge in one
        // L2. Each job's chunk count (2^b1 digits x c chunks) is a multiple of
        // kXcds; XCD x takes job j's digits x, x + kXcds, ... in turn.
        const uint32_t *pfx = pass == 1 ? a.p1_tile0 : a.p2_chunk0;
        const uint32_t total = pass == 1 ? a.total_p1_tiles : a.total_p2_chunks;
        const uint32_t x = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
        uint32_t b, valid, j;
        if (pass == 2 && a.regions) {
            valid = k * kXcds < total;
            j = valid ? wave_upper_index(pfx, a.n_jobs, k * kXcds) : 0;
            const JobDesc &jb = a.jobs[j];
            const uint32_t c = jb.nseg * jb.region_tiles, kk = k - pfx[j] / kXcds;
            b = valid ? pfx[j] + (x + kXcds * (kk / c)) * c + kk % c : total;
        } else {
            b = pass == 1 ? x * ((total + kXcds - 1) / kXcds) + k
                          : ((k / kXcdGroup) * kXcds + x) * kXcdGroup + k % kXcdGroup;
            valid = b < total;
            j = valid ? wave_upper_index(pfx, a.n_jobs, b) : 0;
        }
        if (lane == 0) {
            ti.valid = valid;
            ti.region = 0;
            if (valid) {
                const JobDesc &job = a.jobs[j];
                const uint32_t local = b - pfx[j];
                ti.job = j;
                ti.local = local;
                if (pass == 1) {
                    ti.src = job.in;
                    for (int c = 0; c < 4; c++) ti.dst_cols[c] = job.b2 ? job.mid_cols[c] : job.fin_cols[c];
                    ti.dst_ids = job.b2 ? job.mid_ids : job.fin_ids;
                    ti.lo = local * T;
                    ti.hi = ti.lo + T < job.n ? ti.lo + T : job.n;
                    ti.bins = 1u << job.b1;
                    ti.shift = job.shift0;
                    if (job.region1) {  // region (d1, g) of mid, g = this tile's segment
                        const uint32_t g = local / job.seg_tiles;
                        ti.region = job.region1;
                        ti.rc0 = job.m1_off + g;
                        ti.rstride = job.nseg;
                        ti.rrow0 = g * job.region1;
                        ti.rdstride = job.nseg * job.region1;
                        ti.trash = (job.nseg << job.b1) * job.region1;
                    }
                } else if (job.region1) {
                    // chunk = tile kt of pass-1 region (d1, g); digit d2's region is (d1 << b2) | d2 of fin
                    const uint32_t per = job.nseg * job.region_tiles;
                    const uint32_t d1 = local / per, r = local - d1 * per;
                    const uint32_t g = r / job.region_tiles, kt = r - g * job.region_tiles;
                    const uint32_t c1 = a.counts[job.m1_off + d1 * job.nseg + g];
                    const uint32_t filled = c1 < job.region1 ? c1 : job.region1;
                    const uint32_t start = (d1 * job.nseg + g) * job.region1;
                    for (int c = 0; c < 4; c++) ti.src.cols[c] = job.mid_cols[c];
                    ti.src.rowids = job.mid_ids;
                    ti.src.n = job.n;
                    for (int c = 0; c < 4; c++) ti.dst_cols[c] = job.fin_cols[c];
                    ti.dst_ids = job.fin_ids;
                    ti.lo = start + kt * T;
                    ti.hi = start + ((kt + 1) * T < filled ? (kt + 1) * T : filled);
                    ti.valid = kt * T < filled;
                    ti.bins = 1u << job.b2;
                    ti.shift = job.shift0 + job.b1;
                    ti.region = job.region2;
                    ti.rc0 = job.m2_off + (d1 << job.b2);
                    ti.rstride = 1;
                    ti.rrow0 = (d1 << job.b2) * job.region2;
                    ti.rdstride = job.region2;
                    ti.trash = (1u << (job.b1 + job.b2)) * job.region2;
                } else {
                    const uint32_t n1 = 1u << job.b1;
                    const uint32_t d1 = local / job.nseg, g = local - d1 * job.nseg;
                    const uint32_t p = a.base[job.base_off + (d1 << job.b2)];
                    const uint32_t *m1 = a.counts + job.m1_off;
                    for (int c = 0; c < 4; c++) ti.src.cols[c] = job.mid_cols[c];
                    ti.src.rowids = job.mid_ids;
                    ti.src.n = job.n;
                    for (int c = 0; c < 4; c++) ti.dst_cols[c] = job.fin_cols[c];
                    ti.dst_ids = job.fin_ids;
                    ti.lo = p + m1[(uint64_t)g * job.hsplit * n1 + d1];
                    ti.hi = p + m1[(uint64_t)(g + 1) * job.hsplit * n1 + d1];
                    ti.bins = 1u << job.b2;
                    ti.shift = job.shift0 + job.b1;
                }
            }
        }
    }
    __syncthreads();
    if (!ti.valid) return;
    if (tid < ti.bins && !ti.region) {  // first destination row of every digit (exact layout)
        const JobDesc &job = a.jobs[ti.job];
        const uint32_t *base = a.base + job.base_off;
        if (pass == 1) {
            const uint32_t n1 = 1u << job.b1, t = ti.local, sg = t / job.seg_tiles;
            const uint32_t g = sg * job.hsplit + (t - sg * job.seg_tiles) / job.hrow_tiles;  // histogram row
            gdst[tid] = base[tid << job.b2] + a.counts[job.m1_off + (uint64_t)g * n1 + tid] +
                        a.counts[job.tilepre_off + (uint64_t)t * n1 + tid];
        } else {
            const uint32_t nb = 1u << (job.b1 + job.b2);
            const uint32_t d1 = ti.local / job.nseg, g = ti.local - d1 * job.nseg;
            const uint32_t q = (d1 << job.b2) | tid;
            gdst[tid] = base[q] + a.counts[job.m2_off + (uint64_t)g * job.hsplit * nb + q];
        }
    }

    const uint32_t bins = ti.bins, shift = ti.shift, mask = bins - 1;
    const bool lo32 = shift + (uint32_t)__builtin_ctz(bins) <= 32;  // the digit lies in the hash's low half
    const GKeys<KW, NC> skeys_g = uniform_keys<KW, NC>(ti.src);  // source columns, in scalar registers
    const gptr<const uint32_t> sids_g = uniform_global(ti.src.rowids);
    gptr<KT> dcols[NC];  // destination columns
#pragma unroll
    for (int c = 0; c < NC; c++) dcols[c] = uniform_global(static_cast<KT *>(ti.dst_cols[c]));
    const gptr<uint32_t> dids = uniform_global(ti.dst_ids);
    const HashCfg hc = a.hash;
    for (uint32_t lo = ti.lo; lo < ti.hi; lo += T) {
        const uint32_t hi = lo + T < ti.hi ? lo + T : ti.hi;
        for (uint32_t i = tid; i < kPassWaves * 256; i += kPassThreads) wcnt[i] = 0;
        __syncthreads();

        // 1. load ITEMS rows per lane (wave w owns a contiguous 64*ITEMS segment), rank by digit
        Key<KW, NC> keys[ITEMS];
        uint32_t ids[ITEMS];
        uint32_t pk[ITEMS];  // digit | rank << 8, or ~0 for no row
        const uint32_t wbase = lo + w * 64 * ITEMS + lane;
        // every load issued before the first use (past the end: row lo again)
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t i = wbase + it * 64;
            keys[it] = load_key<KW, NC>(skeys_g, i < hi ? i : lo);
        }
        if (sids_g) {  // wave-uniform
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const uint32_t i = wbase + it * 64;
                ids[it] = sids_g[i < hi ? i : lo];
            }
        } else {
#pragma unroll
            for (int it = 0; it < ITEMS; it++) ids[it] = wbase + it * 64;
        }
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t i = wbase + it * 64;
            const bool valid = i < hi;
            uint32_t d = 0;
            if (valid) {
                const uint64_t h = lo32 ? (uint64_t)hash_key_lo<HP, KW, NC>(keys[it], hc) : hash_key<HP, KW, NC>(keys[it], hc);
                d = (uint32_t)(h >> shift) & mask;
            }
            const uint32_t r = valid ? atomicAdd(&wcnt[w * 256 + d], 1u) : 0u;
            pk[it] = valid ? (d | (r << 8)) : ~0u;
        }
        __syncthreads();

        // 2. per digit: wave prefixes, tile count, local offsets
        uint32_t cnt = 0;
        if (tid < bins) {
#pragma unroll
            for (int ww = 0; ww < kPassWaves; ww++) {
                uint32_t c = wcnt[ww * 256 + tid];
                wcnt[ww * 256 + tid] = cnt;
                cnt += c;
            }
        }
        uint32_t total;
        const uint32_t my_loc = block_excl_scan<uint32_t, kPassWaves>(cnt, sh_scan, &total);
        if (tid < bins) {
            loc[tid] = my_loc;
            uint32_t dst;
            if (ti.region) {  // reserve the run in the digit's region (a run that does not fit goes to the trash tile)
                const uint32_t got = cnt ? atomicAdd(a.counts + ti.rc0 + (uint64_t)tid * ti.rstride, cnt) : 0u;
                dst = (uint64_t)got + cnt <= ti.region ? ti.rrow0 + tid * ti.rdstride + got : ti.trash;
            } else {
                dst = gdst[tid];
            }
            gdo[tid] = dst - my_loc;  // output row of staged slot k = gdo[digit] + k
        }
        __syncthreads();

        // 3. stage the key columns in LDS ordered by digit; consecutive slots of
        //    one digit go to consecutive output rows
        uint32_t slot[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            slot[it] = ~0u;
            if (pk[it] != ~0u) {
                const uint32_t d = pk[it] & 255u;
                slot[it] = loc[d] + wcnt[w * 256 + d] + (pk[it] >> 8);
#pragma unroll
                for (int c = 0; c < NC; c++) skeys[c * T + slot[it]] = keys[it].c[c];
                sdig[slot[it]] = (uint8_t)d;
            }
        }
        __syncthreads();
        // 4. write the keys in slot order
        const uint32_t n = hi - lo;
        for (uint32_t k = tid; k < n; k += kPassThreads) {
            const uint32_t dst = gdo[sdig[k]] + k;
#pragma unroll
            for (int c = 0; c < NC; c++) dcols[c][dst] = skeys[c * T + k];
        }
        __syncthreads();
        // 5. the row ids, through the same staging buffer
#pragma unroll
        for (int it = 0; it < ITEMS; it++)
            if (slot[it] != ~0u) sids[slot[it]] = ids[it];
        __syncthreads();
        for (uint32_t k = tid; k < n; k += kPassThreads) dids[gdo[sdig[k]] + k] = sids[k];
        __syncthreads();
        if (tid < bins) gdst[tid] += cnt;  // next step of a pass-2 chunk
    }
}

// ---------------------------------------------------------------------------
// One-pass form
// ---------------------------------------------------------------------------

// Partition of a row: the pass-1 digit's bits above the pass-2 digit's, the
// numbering two passes would give (b2 == 0: the one digit).
__device__ __forceinline__ uint32_t fan_part(uint32_t h, uint32_t b1, uint32_t b2) {
    return ((h & ((1u << b1) - 1)) << b2) | ((h >> b1) & ((1u << b2) - 1));
}

// Rows per (group, partition). Each block sweeps every nper-th tile of one
// group with one LDS atomic per row, then adds its counters to the job's.
// HBM-bound: the keys once. Row-major keys (vj_join_rows) become columns on the
// way: as a kernel of its own in front this read them once more and took two
// launches (us a call with its consumer, before and now: 2^20 x 2^22 rows of 2 columns
// 343 / 325, of 3 390 / 362, 70000 x 300000 of 2 155 / 133).
template <int HP, int KW, int NC>
__global__ __launch_bounds__(kFanThreads, 8) void k_fan_hist(PipeArgs a) {
    using KT = typename KeyT<KW>::T;
    constexpr int KB = KW * NC;
    constexpr int U = KB <= 16 ? 4 : 2;  // rows per thread in flight
    extern __shared__ uint32_t lds[];    // [2^(b1+b2)]
    const uint32_t tid = threadIdx.x, b = blockIdx.x;
    const uint32_t j = upper_index(a.hist_block0, a.n_jobs, b);
    const JobDesc &job = a.jobs[j];
    const uint32_t b1 = job.b1, b2 = job.b2, nb = 1u << (b1 + b2), G = job.groups, n = job.n;
    const uint32_t local = b - a.hist_block0[j], g = local & (G - 1), nper = job.nrow / G;
    for (uint32_t q = tid; q < nb; q += kFanThreads) lds[q] = 0;
    __syncthreads();
    const GKeys<KW, NC> in = uniform_keys<KW, NC>(job.in);
    const HashCfg hc = a.hash;
    [[maybe_unused]] const gptr<const uint64_t> rows = uniform_global(static_cast<const uint64_t *>(job.mid_cols[0]));
    const uint32_t T = a.pass_tile, tiles = job.p1_tiles;
    // the group's tiles: those whose index over the whole pipeline is g modulo the group count
    for (uint32_t t = ((g - a.p1_tile0[j]) & (G - 1)) + G * (local / G); t < tiles; t += G * nper) {
        const uint32_t lo = t * T, hi = lo + T < n ? lo + T : n;
        for (uint32_t i0 = lo + tid; i0 < hi; i0 += kFanThreads * U) {
            Key<KW, NC> key[U];
#pragma unroll
            for (int u = 0; u < U; u++) {  // all loads in flight at once (past the end: the first row again)
                const uint32_t i = i0 + u * kFanThreads;
                const uint64_t r = i < hi ? i : i0;
                if constexpr (KW == 8 && NC > 1) {
                    if (rows) {  // block-uniform
#pragma unroll
                        for (int c = 0; c < NC; c++) key[u].c[c] = rows[r * NC + c];
                        continue;
                    }
                }
                key[u] = load_key<KW, NC>(in, r);
            }
            if constexpr (KW == 8 && NC > 1) {
                if (rows) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const uint32_t i = i0 + u * kFanThreads;
#pragma unroll
                        for (int c = 0; c < NC; c++)
                            if (i < hi) ((gptr<KT>)in.c[c])[i] = key[u].c[c];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u * kFanThreads < hi) atomicAdd(&lds[fan_part(hash_key_lo<HP, KW, NC>(key[u], hc), b1, b2)], 1u);
        }
    }
    __syncthreads();
    uint32_t *cnt = a.counts + job.m1_off + (uint64_t)g * nb;
    for (uint32_t q = tid; q < nb; q += kFanThreads) {
        const uint32_t c = lds[q];
        if (c) atomicAdd(cnt + q, c);
    }
}

// Per tile: rank the rows by partition (one LDS counter per partition), reserve
// each partition's run from the group's cursor, stage one column at a time in
// LDS in partition order and write it out in runs. Persistent: as soon as a
// column is staged its registers load the next tile's, so that the loads
// cross the write-out (with one large block per CU nothing else would).
// BIG: tile shape (fan_items).
template <int HP, int KW, int NC, int BIG>
__global__ __launch_bounds__(kFanThreads, (BIG || KW * NC > 16 ? 4 : 8)) void k_fan(PipeArgs a) {
    using KT = typename KeyT<KW>::T;
    constexpr int ITEMS = fan_items(KW * NC, BIG);
    constexpr int T = kFanThreads * ITEMS, WAVES = kFanThreads / 64;
    extern __shared__ __align__(16) unsigned char smem[];
    KT *skeys = reinterpret_cast<KT *>(smem);            // [T] one column (then the row ids) at a time
    uint32_t *sids = reinterpret_cast<uint32_t *>(smem);  // [T]
    uint16_t *spart = reinterpret_cast<uint16_t *>(smem + (size_t)T * KW);        // [T]
    uint32_t *cnt = reinterpret_cast<uint32_t *>(smem + (size_t)T * (KW + 2));    // [fan_bins] counts, then offsets
    uint32_t *gdo = cnt + a.fan_bins;                                             // [fan_bins]
    __shared__ uint32_t sh_scan[WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, total = a.total_p1_tiles;
    const HashCfg hc = a.hash;
    uint32_t b = blockIdx.x;  // tile over the whole pipeline; the grid is a multiple of kXcds: b stays on its XCD
    if (b >= total) return;
    uint32_t j = upper_index(a.p1_tile0, a.n_jobs, b);
    uint32_t lo = (b - a.p1_tile0[j]) * T, n = a.jobs[j].n;
    uint32_t rows = n - lo < (uint32_t)T ? n - lo : (uint32_t)T;
    Key<KW, NC> key[ITEMS];
    {
        const GKeys<KW, NC> in = uniform_keys<KW, NC>(a.jobs[j].in);
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {  // every load in flight at once (past the end: row lo again)
            const uint32_t i = it * kFanThreads + tid;
            key[it] = load_key<KW, NC>(in, lo + (i < rows ? i : 0u));
        }
    }
    for (uint32_t q = tid; q < a.fan_bins; q += kFanThreads) cnt[q] = 0;
    __syncthreads();
    while (true) {
        const JobDesc &job = a.jobs[j];
        const uint32_t b1 = job.b1, b2 = job.b2, nb = 1u << (b1 + b2);
        // the next tile, whose columns are loaded on the way
        const uint32_t b_next = b + gridDim.x;
        const bool more = b_next < total;
        uint32_t j_next = j;
        if (more && b_next >= a.p1_tile0[j + 1]) j_next = upper_index(a.p1_tile0, a.n_jobs, b_next);
        const uint32_t lo_next = more ? (b_next - a.p1_tile0[j_next]) * T : 0u, n_next = a.jobs[j_next].n;
        const uint32_t rows_next = !more ? 0u : (n_next - lo_next < (uint32_t)T ? n_next - lo_next : (uint32_t)T);
        const GKeys<KW, NC> in_next = uniform_keys<KW, NC>(a.jobs[j_next].in);
        // 1. partition and rank of every row
        uint32_t slot[ITEMS];  // partition | rank << kFanBits, then the row's slot in partition order
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t q = fan_part(hash_key_lo<HP, KW, NC>(key[it], hc), b1, b2);
            slot[it] = q;
            if (it * kFanThreads + tid < rows) slot[it] |= atomicAdd(&cnt[q], 1u) << kFanBits;
        }
        __syncthreads();
        // 2. each thread: its (two) partitions' runs reserved, their offsets in the tile
        const uint32_t per = nb > (uint32_t)kFanThreads ? 2u : 1u, q0 = tid * per;
        uint32_t c[2], got[2];
        uint32_t *cur = a.counts + job.m1_off + (uint64_t)(b & (job.groups - 1)) * nb;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            c[k] = (uint32_t)k < per && q0 + k < nb ? cnt[q0 + k] : 0u;
            got[k] = c[k] ? atomicAdd(cur + q0 + k, c[k]) : 0u;
        }
        uint32_t pre = wave_incl_scan(c[0] + c[1]);
        if (lane == 63) sh_scan[w] = pre;
        __syncthreads();
        pre -= c[0] + c[1];
#pragma unroll
        for (int k = 0; k < WAVES; k++) pre += (uint32_t)k < w ? sh_scan[k] : 0u;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            if ((uint32_t)k < per && q0 + k < nb) {
                cnt[q0 + k] = pre;
                gdo[q0 + k] = got[k] - pre;  // output row of slot s = gdo[partition] + s
                pre += c[k];
            }
        }
        __syncthreads();
        // 3. slots; the first key column staged with its rows' partitions
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            if (it * kFanThreads + tid < rows) {
                const uint32_t q = slot[it] & ((1u << kFanBits) - 1);
                slot[it] = cnt[q] + (slot[it] >> kFanBits);
                skeys[slot[it]] = key[it].c[0];
                spart[slot[it]] = (uint16_t)q;
            }
        }
        if (more) {  // block-uniform
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const uint32_t i = it * kFanThreads + tid;
                key[it].c[0] = in_next.c[0][lo_next + (i < rows_next ? i : 0u)];
            }
        }
        __syncthreads();
        // 4. columns out in slot order; each thread keeps its slots' output rows
        for (uint32_t q = tid; q < a.fan_bins; q += kFanThreads) cnt[q] = 0;
        uint32_t dst[ITEMS];
        {
            const gptr<KT> out = uniform_global(static_cast<KT *>(job.fin_cols[0]));
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const uint32_t s = it * kFanThreads + tid;
                if (s < rows) {
                    dst[it] = gdo[spart[s]] + s;
                    out[dst[it]] = skeys[s];
                }
            }
        }
#pragma unroll
        for (int col = 1; col < NC; col++) {
            __syncthreads();
#pragma unroll
            for (int it = 0; it < ITEMS; it++)
                if (it * kFanThreads + tid < rows) skeys[slot[it]] = key[it].c[col];
            if (more) {
#pragma unroll
                for (int it = 0; it < ITEMS; it++) {
                    const uint32_t i = it * kFanThreads + tid;
                    key[it].c[col] = in_next.c[col][lo_next + (i < rows_next ? i : 0u)];
                }
            }
            __syncthreads();
            const gptr<KT> out = uniform_global(static_cast<KT *>(job.fin_cols[col]));
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const uint32_t s = it * kFanThreads + tid;
                if (s < rows) out[dst[it]] = skeys[s];
            }
        }
        // 5. the row ids
        const gptr<const uint32_t> ids = uniform_global(job.in.rowids);
        __syncthreads();
        if (ids) {  // block-uniform
            uint32_t id[ITEMS];
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const uint32_t i = it * kFanThreads + tid;
                id[it] = ids[lo + (i < rows ? i : 0u)];
            }
#pragma unroll
            for (int it = 0; it < ITEMS; it++)
                if (it * kFanThreads + tid < rows) sids[slot[it]] = id[it];
        } else {
#pragma unroll
            for (int it = 0; it < ITEMS; it++)
                if (it * kFanThreads + tid < rows) sids[slot[it]] = lo + it * kFanThreads + tid;
        }
        __syncthreads();
        const gptr<uint32_t> out = uniform_global(job.fin_ids);
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t s = it * kFanThreads + tid;
            if (s < rows) out[dst[it]] = sids[s];
        }
        if (!more) return;
        b = b_next;
        j = j_next;
        lo = lo_next;
        rows = rows_next;
        // the staging buffer is written again after three barriers of the next
        // tile; its counters were cleared before the last two of this one
    }
}

// ---------------------------------------------------------------------------
// Build + probe
// ---------------------------------------------------------------------------

struct ProbeTask {
    TView r, s;
    uint32_t *out_r, *out_s;
    unsigned long long *count;
    uint64_t cap;
    unsigned long long out_base[4];  // first output row of walk k's matches (k & 3)
    uint32_t r_lo, r_n, s_lo, s_n;
    uint32_t nheads, hshift, shift, one_based;  // heads; 32 - their log2
    uint32_t dup;
    uint32_t done;
    uint32_t wave_count[4][kMaxProbeWaves];  // matches per wave of walk k (k & 3)
    // the join whose fixed fields the record holds (~0: none yet), its
    // sides' partition start / end offsets in base, chunk sizes, first task
    // and per-partition task prefix
    uint32_t jn, rb, re, sb, se, cap_r, cap_s;
    unsigned long long task0;
    const unsigned long long *pt;
};


// One task's parameters for the walks (all wave-uniform).
struct WalkArgs {
    GView s;
    gptr<uint32_t> out_r, out_s;
    uint64_t cap;
    uint32_t s_lo, s_end, hshift, shift, ob1;
    bool dup;
};

__device__ __forceinline__ WalkArgs walk_args(const ProbeTask &t) {
    WalkArgs w;
    w.s = uniform_view(t.s);
    w.out_r = uniform_global(t.out_r);
    w.out_s = uniform_global(t.out_s);
    w.cap = uniform((uint64_t)t.cap);
    w.s_lo = uniform(t.s_lo);
    w.s_end = w.s_lo + uniform(t.s_n < (uint32_t)kProbeChunk ? t.s_n : (uint32_t)kProbeChunk);
    w.hshift = uniform(t.hshift);
    w.shift = uniform(t.shift);
    w.ob1 = uniform(t.one_based);
    w.dup = false;  // known once the table is built
    return w;
}

// Writes a wave's matches straight to the join output: the matching lanes of
// one ballot take consecutive rows from `pos`, so every store instruction
// covers one contiguous run of each output column.
struct Emitter {
    unsigned long long pos;
    __device__ __forceinline__ void put(bool m, uint32_t r, uint32_t s, const WalkArgs &wa) {
        const uint64_t mb = __ballot(m);
        if (m) {
            const unsigned long long o = pos + lanes_below(mb);
            if (o < wa.cap) {
                wa.out_r[o] = r;
                wa.out_s[o] = s;
            }
        }
        pos += __builtin_popcountll(mb);
    }
};

// The block's LDS table of one build chunk: chained hashing. heads[h] is the
// first entry of chain h (0: none), key / id / nxt are indexed by entry
// (entry = chunk row + 1). Entries 1.. only: entry 0 reads as an end.
template <typename KT, int NC, int CAP> struct LdsTable {
    KT *key;         // [NC][CAP + 1]
    uint32_t *id;    // [CAP + 1]
    uint16_t *nxt;   // [CAP + 1]
    uint16_t *head;  // [heads]
    __device__ __forceinline__ bool eq(uint32_t e, const KT (&k)[NC]) const {
        bool r = true;
#pragma unroll
        for (int c = 0; c < NC; c++) r &= key[c * (CAP + 1) + e] == k[c];
        return r;
    }
    __device__ __forceinline__ bool eq(uint32_t e, uint32_t f) const {
        bool r = true;
#pragma unroll
        for (int c = 0; c < NC; c++) r &= key[c * (CAP + 1) + e] == key[c * (CAP + 1) + f];
        return r;
    }
};

// Walks over this wave's rows of the S chunk. The chunk holds up to
// kProbeChunk = ITERS x TH x U rows (TH threads per block, see ProbeShape); in
// iteration `it` lane `l` of wave `w` owns rows it*TH*U + w*64*U + u*64 + l.
// probe_walk finds each row's first matching entry, keeps it in registers and
// counts the row's matches (equal keys further down the chain); replay_walk
// then writes them. All U rows of a lane step down their chains together: one
// key and one link per row and step, with selects instead of branches, until
// the wave's longest chain ends (about three steps at four heads per row). A
// step is some 8 VALU instructions per row; buckets of tags read whole took
// about 35 per round and could not afford fewer than two slots per row.
// The S keys of the next iteration are loaded before the current one is
// probed, so one HBM round trip overlaps each iteration's probing (where
// registers allow, see PF); nk holds the first iteration's, loaded by the caller.

// A key's chain, from the low 32 hash bits above the partition digits (the
// digits are the same for every row of a partition): the top bits of their
// product with the golden ratio, which depend on all of them (FNV's low bits
// depend only on the keys' low bits, and custom_xor_hw mixes less).
__device__ __forceinline__ uint32_t chain_of(uint32_t lo, uint32_t shift, uint32_t hshift) {
    return ((lo >> shift) * 0x9E3779B1u) >> hshift;
}

template <int N> __device__ __forceinline__ uint32_t res_get(const uint32_t (&r)[N], int k) {
    return (r[k >> 1] >> ((k & 1) * 16)) & 0xFFFFu;
}
template <int N> __device__ __forceinline__ void res_set(uint32_t (&r)[N], int k, uint32_t v) {
    const int sh = (k & 1) * 16;
    r[k >> 1] = (r[k >> 1] & ~(0xFFFFu << sh)) | (v << sh);
}
// Block shape of the build+probe kernel for table shape PV (probe_threads).
template <int PV> struct ProbeShape {
    static constexpr int TH = probe_threads(PV);
    static constexpr int WAVES = TH / 64;
    static constexpr int U = PV ? 4 : 2;  // rows per lane and iteration (the wide block has half the waves, twice the registers)
    static constexpr int ITERS = kProbeChunk / (TH * U);
    static constexpr int RES = ITERS * U / 2;  // words of packed 16-bit results per lane
    static_assert(U % 2 == 0, "an iteration's results fill whole words");
    static_assert(ITERS * TH * U == kProbeChunk && WAVES <= kMaxProbeWaves, "probe chunk shape");
};

// First S row of this lane in iteration `it` of a walk with U rows per lane.
template <int U, int TH> __device__ __forceinline__ uint32_t walk_row(const WalkArgs &wa, int it) {
    return wa.s_lo + it * TH * U + (threadIdx.x >> 6) * 64 * U + lane_id();
}
// First S row of the wave in iteration `it` (wave-uniform).
template <int U, int TH> __device__ __forceinline__ uint32_t walk_wave_row(const WalkArgs &wa, int it) {
    return wa.s_lo + it * TH * U + uniform((uint32_t)(threadIdx.x >> 6)) * 64 * U;
}

// Loads this lane's S keys of iteration `it` (rows past the chunk are left alone).
template <int U, int TH, int KW, int NC>
__device__ __forceinline__ void walk_load(const WalkArgs &wa, int it, Key<KW, NC> (&k)[U]) {
    const uint32_t row = walk_row<U, TH>(wa, it);
#pragma unroll
    for (int u = 0; u < U; u++)
        if (row + u * 64 < wa.s_end) k[u] = load_key<KW, NC>(wa.s, row + u * 64);
}

template <int N> __device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

template <int HP, int KW, int NC, int PV, typename Tab>
__device__ __forceinline__ uint32_t probe_walk(const WalkArgs &wa, const HashCfg &hc, const Tab &tab,
                                               Key<KW, NC> (&nk)[ProbeShape<PV>::U],
                                               uint32_t (&res)[ProbeShape<PV>::RES]) {
    constexpr int TH = ProbeShape<PV>::TH, ITERS = ProbeShape<PV>::ITERS;
    constexpr int U = ProbeShape<PV>::U;
    // Next-iteration loads double the key registers; they are used where the
    // kernel stays within its register budget (single 8-byte key, or the wide
    // block's 128 VGPRs; FNV / XOR).
    constexpr bool PF = (KW * NC <= 8 || PV != 0) && HP != HP_GENERIC;
    const uint32_t hshift = wa.hshift, shift = wa.shift, s_end = wa.s_end;
    uint32_t total = 0;  // this lane's matches
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
        if (walk_wave_row<U, TH>(wa, it) >= s_end) break;  // wave-uniform
        const uint32_t row = walk_row<U, TH>(wa, it);
        Key<KW, NC> sk[U];
        if (!PF && it > 0) walk_load<U, TH, KW, NC>(wa, it, nk);
#pragma unroll
        for (int u = 0; u < U; u++) sk[u] = nk[u];
        if (PF && it + 1 < ITERS) walk_load<U, TH, KW, NC>(wa, it + 1, nk);
        uint32_t e[U], f[U];  // the row's next chain entry (0: done, or past the chunk); its match (0: none)
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t h = tab.head[chain_of(hash_key_lo<HP, KW, NC>(sk[u], hc), shift, hshift)];
            e[u] = row + u * 64 < s_end ? h : 0u;
            f[u] = 0;
        }
        while (true) {
            uint32_t any = 0;
#pragma unroll
            for (int u = 0; u < U; u++) any |= e[u];
            if (!__ballot(any != 0)) break;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t nx = tab.nxt[e[u]];
                const bool hit = tab.eq(e[u], sk[u].c) && e[u] != 0;
                f[u] = hit && f[u] == 0 ? e[u] : f[u];
                total += hit;
                e[u] = hit && !wa.dup ? 0u : nx;  // equal keys in the chunk: to the chain's end
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) res[(it * U + u) >> 1] |= f[u] << (((it * U + u) & 1) * 16);
    }
    return wave_sum<64>(total);
}

// Row ids of this lane's rows of iterations g .. g + G, matched or not, with
// clamped indexes: no per-row branches, and the loads are issued together (rows
// past the chunk, and all rows of iterations the walk skipped, hold no match:
// they read row s_lo).
template <int G, int PV>
__device__ __forceinline__ void load_ids(const WalkArgs &wa, int g, uint32_t (&sid)[G * ProbeShape<PV>::U]) {
    constexpr int U = ProbeShape<PV>::U, TH = ProbeShape<PV>::TH;
#pragma unroll
    for (int it = 0; it < G; it++) {
        const uint32_t row = walk_row<U, TH>(wa, g + it);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t i = row + u * 64;
            sid[it * U + u] = wa.s.rowids ? wa.s.rowids[i < wa.s_end ? i : wa.s_lo] : i;  // wave-uniform test
        }
    }
}

// Writes the matches probe_walk kept in iterations g .. g + G: each matched
// row's entry, then (when the build chunk has equal keys) the equal ones
// further down its chain. The build-side row ids come from LDS.
template <int G, int PV, typename Tab>
__device__ __forceinline__ void replay_group(const WalkArgs &wa, const Tab &tab, int g,
                                             const uint32_t (&res)[ProbeShape<PV>::RES],
                                             const uint32_t (&sid)[G * ProbeShape<PV>::U], Emitter &em) {
    constexpr int U = ProbeShape<PV>::U, TH = ProbeShape<PV>::TH;
    const uint32_t ob1 = wa.ob1;
#pragma unroll
    for (int it = 0; it < G; it++) {
        if (walk_wave_row<U, TH>(wa, g + it) >= wa.s_end) break;  // wave-uniform
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t f = res_get(res, (g + it) * U + u);
            em.put(f != 0, tab.id[f] + ob1, sid[it * U + u] + ob1, wa);
            if (wa.dup) {  // wave-uniform
                uint32_t x = tab.nxt[f];
                while (__ballot(x != 0)) {
                    em.put(x != 0 && tab.eq(x, f), tab.id[x] + ob1, sid[it * U + u] + ob1, wa);
                    x = tab.nxt[x];
                }
            }
        }
    }
}

// Waves per SIMD the probe kernel is compiled for. Standard table: 8 (64
// VGPRs, four blocks per CU) for single 8-byte keys with FNV / XOR hashing;
// wider keys and the generic hash path get 4 (128 VGPRs, two blocks per CU) so
// they do not spill. Wide table: one 16-wave block per CU, 4 waves per SIMD
// (128 VGPRs).
template <int HP, int KB, int PV> constexpr int probe_waves_per_simd() {
    return PV ? 4 : (KB <= 8 && HP != HP_GENERIC ? 8 : 4);
}

// The block's table in its dynamic LDS.
template <int KW, int NC, int PV>
__device__ __forceinline__ LdsTable<typename KeyT<KW>::T, NC, probe_cap(KW * NC, PV)> lds_table(unsigned char *smem) {
    using KT = typename KeyT<KW>::T;
    constexpr int CAP = probe_cap(KW * NC, PV);
    LdsTable<KT, NC, CAP> tab;
    tab.key = reinterpret_cast<KT *>(smem);
    tab.id = reinterpret_cast<uint32_t *>(tab.key + NC * (CAP + 1));
    tab.nxt = reinterpret_cast<uint16_t *>(tab.id + CAP + 1);
    tab.head = reinterpret_cast<uint16_t *>(smem + probe_table_bytes(KW * NC, PV) - 2 * probe_heads(KW * NC, PV));
    return tab;
}

// Chain heads of a task's table: four per row where the table has them, else at least 1.8.
__device__ __forceinline__ void set_heads(ProbeTask &t, uint32_t most) {
    uint32_t nh = 64;
    while (nh < 4 * t.r_n && nh < most) nh <<= 1;
    t.nheads = nh;
    t.hshift = (uint32_t)__builtin_clz(nh) + 1;
}

// Builds the table of task t's build chunk and joins its probe rows with it
// (block-wide; the record is complete). The caller's hooks run between the
// phases: after_build before the first walk, after_walk after it (wide block).
template <int HP, int KW, int NC, int PV, typename Build, typename Walk>
__device__ __forceinline__ void run_task(ProbeTask &t, const HashCfg &hc, unsigned char *smem, Build after_build, Walk after_walk) {
    constexpr int KB = KW * NC, CAP = probe_cap(KB, PV);
    constexpr int TH = ProbeShape<PV>::TH, WAVES = ProbeShape<PV>::WAVES;
    const auto tab = lds_table<KW, NC, PV>(smem);
    uint32_t *head2 = reinterpret_cast<uint32_t *>(tab.head);  // two heads per word
    uint32_t res[ProbeShape<PV>::RES];  // per probe row its first matching entry (0: none), two per word
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    Emitter em;
    em.pos = 0;
            constexpr int U = ProbeShape<PV>::U, ITERS = ProbeShape<PV>::ITERS;
            WalkArgs wa;
            Key<KW, NC> nk[U];
            if constexpr (PV != 0) {
                wa = walk_args(t);
                walk_load<U, TH, KW, NC>(wa, 0, nk);  // crosses the build
            }

            // build: load the R chunk, push every row on its chain, look for equal keys
            const uint32_t r_lo = t.r_lo, r_n = t.r_n, nheads = t.nheads, hshift = t.hshift, shift = t.shift;
            for (uint32_t i = tid; i < nheads / 2; i += TH) head2[i] = 0;
            if (tid == 0) {  // entry 0: the end of a chain
                tab.nxt[0] = 0;
                tab.id[0] = 0;
#pragma unroll
                for (int c = 0; c < NC; c++) tab.key[c * (CAP + 1)] = 0;
            }
            {
                // R rows in flight per lane (a task has r_n >= 1)
                constexpr int RB = PV && KB <= 16 ? 4 : 2;
                const GView rv = uniform_view(t.r);
                for (uint32_t i0 = 0; i0 < r_n; i0 += RB * TH) {
                    Key<KW, NC> rkey[RB];
                    uint32_t rrow[RB];
#pragma unroll
                    for (int r = 0; r < RB; r++) {
                        const uint32_t i = i0 + tid + r * TH;
                        const uint32_t row = r_lo + (i < r_n ? i : 0u);
                        rkey[r] = load_key<KW, NC>(rv, row);
                        rrow[r] = rv.rowids ? rv.rowids[row] : row;  // wave-uniform test
                    }
#pragma unroll
                    for (int r = 0; r < RB; r++) {
                        const uint32_t i = i0 + tid + r * TH;
                        if (i < r_n) {
#pragma unroll
                            for (int c = 0; c < NC; c++) tab.key[c * (CAP + 1) + i + 1] = rkey[r].c[c];
                            tab.id[i + 1] = rrow[r];
                        }
                    }
                }
            }
            __syncthreads();
            // push: the link is written before the compare-and-swap that publishes
            // the row (a half word swapped through its whole word)
            for (uint32_t i = tid + 1; i <= r_n; i += TH) {
                Key<KW, NC> k;
#pragma unroll
                for (int c = 0; c < NC; c++) k.c[c] = tab.key[c * (CAP + 1) + i];
                const uint32_t h = chain_of(hash_key_lo<HP, KW, NC>(k, hc), shift, hshift), sh = (h & 1) * 16;
                uint32_t old = head2[h >> 1];
                while (true) {
                    tab.nxt[i] = (uint16_t)(old >> sh);
                    const uint32_t got = atomicCAS(&head2[h >> 1], old, (old & ~(0xFFFFu << sh)) | (i << sh));
                    if (got == old) break;
                    old = got;
                }
            }
            __syncthreads();
            // equal keys in the chunk: whether a row's key comes again further down its chain
            for (uint32_t i = tid + 1; i <= r_n; i += TH) {
                uint32_t x = tab.nxt[i];
                while (x != 0 && !tab.eq(x, i)) x = tab.nxt[x];
                if (x != 0) t.dup = 1;
            }
            __syncthreads();

            // find and count every row's matches (kept in registers), reserve the
            // walk's output rows with one atomic, then write them
            if constexpr (PV == 0) {
                wa = walk_args(t);
                walk_load<U, TH, KW, NC>(wa, 0, nk);
            }
            wa.dup = uniform(t.dup) != 0;
            after_build();
#pragma unroll
            for (int k = 0; k < ProbeShape<PV>::RES; k++) res[k] = 0;  // results of skipped iterations read as no match
            uint32_t wc = probe_walk<HP, KW, NC, PV>(wa, hc, tab, nk, res);
            if (lane == 0) t.wave_count[0][w] = wc;
            if constexpr (PV == 0) {  // a task is one walk
                __syncthreads();
                if (tid == 0) {
                    uint32_t sum = 0;
                    for (int k = 0; k < WAVES; k++) sum += t.wave_count[0][k];
                    t.out_base[0] = sum ? atomicAdd(t.count, (unsigned long long)sum) : 0;
                }
                __syncthreads();
                if (wc) {
                    em.pos = t.out_base[0];
                    for (uint32_t k = 0; k < w; k++) em.pos += t.wave_count[0][k];
                    constexpr int G = 4;  // ids loaded four iterations at a time
                    static_assert(ITERS % G == 0, "replay groups");
#pragma unroll
                    for (int g = 0; g < ITERS; g += G) {
                        if (walk_wave_row<U, TH>(wa, g) >= wa.s_end) break;  // wave-uniform
                        uint32_t sid[G * U];
                        load_ids<G, PV>(wa, g, sid);
                        replay_group<G, PV>(wa, tab, g, res, sid, em);
                    }
                }
            } else {
                // A task may be several walks (one block per CU: nothing else hides
                // a walk's reservation or its first loads). While walk k + 1 runs,
                // the atomic that reserves walk k's rows and the loads of its row
                // ids are in flight; the first keys of walk k + 2 cross the writing
                // of walk k. One barrier per walk orders all of it. Four buffers:
                // a wave may still read walk k's counts while another posts walk
                // k + 2's.
                after_walk();
                const uint32_t task_end = uniform(t.s_lo + t.s_n), walks = (uniform(t.s_n) + kProbeChunk - 1) / kProbeChunk;
                auto advance = [&](WalkArgs &x) {
                    x.s_lo = x.s_end;
                    x.s_end = task_end - x.s_lo < (uint32_t)kProbeChunk ? task_end : x.s_lo + kProbeChunk;
                };
                WalkArgs wn = wa;  // the next walk, its first keys in nk
                if (walks > 1) {
                    advance(wn);
                    walk_load<U, TH, KW, NC>(wn, 0, nk);
                }
                __syncthreads();
                for (uint32_t k = 0; k < walks; k++) {
                    unsigned long long base = 0;
                    if (tid == 0) {
                        uint32_t sum = 0;
                        for (int x = 0; x < WAVES; x++) sum += t.wave_count[k & 3][x];
                        if (sum) base = atomicAdd(t.count, (unsigned long long)sum);
                    }
                    uint32_t done[ProbeShape<PV>::RES], sid[ITERS * U];
#pragma unroll
                    for (int x = 0; x < ProbeShape<PV>::RES; x++) done[x] = res[x];
                    load_ids<ITERS, PV>(wa, 0, sid);
                    const WalkArgs wd = wa;
                    const uint32_t wcd = wc;
                    if (k + 1 < walks) {
                        wa = wn;
#pragma unroll
                        for (int x = 0; x < ProbeShape<PV>::RES; x++) res[x] = 0;
                        wc = probe_walk<HP, KW, NC, PV>(wa, hc, tab, nk, res);
                        if (lane == 0) t.wave_count[(k + 1) & 3][w] = wc;
                        if (k + 2 < walks) {
                            advance(wn);
                            walk_load<U, TH, KW, NC>(wn, 0, nk);
                        }
                    }
                    if (tid == 0) t.out_base[k & 3] = base;
                    __syncthreads();
                    if (wcd) {
                        em.pos = t.out_base[k & 3];
                        for (uint32_t x = 0; x < w; x++) em.pos += t.wave_count[k & 3][x];
                        replay_group<ITERS, PV>(wd, tab, 0, done, sid, em);
                    }
                }
            }
    __syncthreads();
}

// Ends a block: the last one of the grid copies the counters (and what stands
// behind them, `words` in all) to the host's buffer, so that no copy has to
// follow the kernel, then the device clock, and clears the block count for the
// next launch. (The times of a join come from that clock: two event records around it
// cost 2 us of a call and up to 12 us of what its program launches next; join_into of
// 2^16 x 2^20 rows with a scatter of its result 80 us, without the events 68.) Only
// atomics touch the counters while blocks run, and this thread has the results
// of its own before it counts the block: no fence is needed (one writes the
// L2 back, in every block: 8-12 us of a 60 us launch).
__device__ __forceinline__ bool finish_block(uint32_t &flag, unsigned long long *done, unsigned long long *src,
                                             unsigned long long *dst, uint32_t words) {
    __syncthreads();
    if (threadIdx.x == 0) {
        flag = atomicAdd(done, 1ull) + 1 == gridDim.x;
    }
    __syncthreads();
    if (!flag) return false;
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x)
        dst[i] = __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x == 0) {
        dst[words] = wall_clock64();
        *done = 0;
    }
    return true;
}

// One join without partitions whose build side fits a table: one launch, the
// tables by value, no descriptors in memory, a block per probe chunk. Each
// block builds the whole table; up to some thousand rows that is cheaper than
// any partitioning (2^10 x 2^13 rows: 33 us of device work in five launches
// before, one launch now).
template <int HP, int KW, int NC, int PV>
__global__ __launch_bounds__(probe_threads(PV), (probe_waves_per_simd<HP, KW * NC, PV>())) void k_direct(DirectArgs d) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ ProbeTask t;
    if (threadIdx.x == 0) {
        t.r = d.r;
        t.s = d.s;
        t.out_r = d.out_r;
        t.out_s = d.out_s;
        t.count = d.count;
        t.cap = d.cap;
        t.r_lo = 0;
        t.r_n = (uint32_t)d.r.n;
        t.s_lo = blockIdx.x * d.cap_s;
        t.s_n = (uint32_t)d.s.n - t.s_lo < d.cap_s ? (uint32_t)d.s.n - t.s_lo : d.cap_s;
        t.shift = 0;
        t.one_based = d.one_based;
        t.dup = 0;
        set_heads(t, (uint32_t)probe_heads(KW * NC, PV));
        // (the result is waited for: the block is counted as ended after the clock has arrived)
        if (blockIdx.x == 0) t.done = (uint32_t)atomicExch(d.count + 1, (unsigned long long)wall_clock64());
    }
    __syncthreads();
    run_task<HP, KW, NC, PV>(t, d.hash, smem, [] {}, [] {});
    if (finish_block(t.done, d.done, d.count, d.down, 2)) {
        __syncthreads();
        if (threadIdx.x == 0) *d.count = 0;  // for the next join
    }
}

// PV: table shape (probe_cap, probe_threads).
template <int HP, int KW, int NC, int PV>
__global__ __launch_bounds__(probe_threads(PV), (probe_waves_per_simd<HP, KW * NC, PV>())) void k_probe(PipeArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ ProbeTask t;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const HashCfg hc = a.hash;
    const unsigned long long total = a.ctl->task_total;

    // Lane 0 of wave 0 holds the block's next task: block b's first is task b,
    // the following ones come from the queue (tickets count from the grid
    // size), fetched while the current one runs; no ticket is drawn when every
    // task is some block's first. In the wide block, with nothing else on the
    // CU to cover the set-up, the next task's map entry and partition bounds
    // are loaded along the way too (`ahead`: they are there).
    unsigned long long next_task = blockIdx.x, next_pt = 0;
    uint32_t next_q = 0, next_r0 = 0, next_r1 = 0, next_s0 = 0, next_s1 = 0, ahead = 0;
    if (tid == 0) t.jn = ~0u;  // read and written by this thread only (lane 0 of wave 0)
    while (true) {
        if (w == 0) {
            const unsigned long long task = __shfl(next_task, 0, 64);
            if (task >= total) {
                if (lane == 0) t.done = 1;
            } else {
                uint32_t jn = 0, q = 0;
                const bool ready = PV != 0 && uniform(ahead) != 0;
                if (ready) {
                    q = next_q;
                } else if (task < a.taskmap_cap) {  // wave-uniform
                    const unsigned long long e = a.taskmap[task];
                    jn = (uint32_t)(e >> 32);
                    q = (uint32_t)e;
                } else {
                    jn = wave_upper_index(a.task0, a.n_joins, task);
                    const JoinDesc &jd0 = a.joins[jn];
                    q = wave_upper_index(a.ptask + jd0.ptask_off, jd0.nparts, task - a.task0[jn]);
                }
                if (lane == 0) {
                    if (!ready && jn != t.jn) {  // a join's fixed fields, kept while its tasks follow each other
                        const JoinDesc &jd = a.joins[jn];
                        const JobDesc &jr = a.jobs[jd.job_r];
                        const JobDesc &js = a.jobs[jd.job_s];
                        if (jr.b1) {
                            for (int c = 0; c < 4; c++) t.r.cols[c] = jr.fin_cols[c];
                            t.r.rowids = jr.fin_ids;
                        } else {
                            t.r = jr.in;
                        }
                        if (js.b1) {
                            for (int c = 0; c < 4; c++) t.s.cols[c] = js.fin_cols[c];
                            t.s.rowids = js.fin_ids;
                        } else {
                            t.s = js.in;
                        }
                        t.rb = jr.base_off;
                        t.re = jr.end_off;
                        t.sb = js.base_off;
                        t.se = js.end_off;
                        t.cap_r = jd.cap_r;
                        t.cap_s = jd.cap_s;
                        t.task0 = a.task0[jn];
                        t.pt = a.ptask + jd.ptask_off;
                        t.shift = jd.slot_shift;
                        t.one_based = jd.one_based;
                        t.out_r = jd.out_r;
                        t.out_s = jd.out_s;
                        t.cap = jd.cap;
                        t.count = &a.out_count[jn];
                        t.jn = jn;
                    }
                    // the partition's sides and the task's chunks: one round of loads
                    const uint32_t cap_r = t.cap_r, cap_s = t.cap_s;
                    if (!ready) {
                        next_r0 = a.base[t.rb + q], next_s0 = a.base[t.sb + q];
                        next_r1 = a.base[t.re + q], next_s1 = a.base[t.se + q];
                        next_pt = t.pt[q];
                    }
                    const uint32_t r0 = next_r0, s0 = next_s0, nr = next_r1 - r0, ns = next_s1 - s0;
                    const uint32_t s_chunks = (ns + cap_s - 1) / cap_s;
                    const uint32_t k = (uint32_t)(task - t.task0 - next_pt);
                    const uint32_t rc = k / s_chunks, sc = k - rc * s_chunks;
                    t.r_lo = r0 + rc * cap_r;
                    t.r_n = nr - rc * cap_r < cap_r ? nr - rc * cap_r : cap_r;
                    t.s_lo = s0 + sc * cap_s;
                    t.s_n = ns - sc * cap_s < cap_s ? ns - sc * cap_s : cap_s;
                    set_heads(t, (uint32_t)probe_heads(KW * NC, PV));
                    t.dup = 0;
                    t.done = 0;
                }
            }
        }
        __syncthreads();
        if (t.done) break;
        if (tid == 0) next_task = total > gridDim.x ? gridDim.x + atomicAdd(&a.ctl->task_ticket, 1ull) : total;
        unsigned long long entry = ~0ull;  // the next task's map entry
        run_task<HP, KW, NC, PV>(
            t, hc, smem,
            [&] {
                if (PV != 0 && tid == 0 && next_task < total && next_task < a.taskmap_cap) entry = a.taskmap[next_task];
            },
            [&] {
                ahead = 0;
                if (tid == 0 && (uint32_t)(entry >> 32) == t.jn) {
                    next_q = (uint32_t)entry;
                    next_r0 = a.base[t.rb + next_q], next_s0 = a.base[t.sb + next_q];
                    next_r1 = a.base[t.re + next_q], next_s1 = a.base[t.se + next_q];
                    next_pt = t.pt[next_q];
                    ahead = 1;
                }
            });
    }
    (void)finish_block(t.done, &a.ctl->done, a.out_count, a.down, a.down_words);
}

// ---------------------------------------------------------------------------
// Flat form: one hash table in memory that an XCD's L2 holds
// ---------------------------------------------------------------------------

// Build sides of some thousand rows up to flat_max_rows: too many for an LDS
// table, so few that partitioning costs more in launches and passes than it
// saves. The table is open-addressed, at most half full: 8-byte slots {row + 1,
// key} for 4-byte keys, in pairs read with one 16-byte load, 16-byte slots
// {key, row + 1} for 8-byte keys, and {tag, row + 1} for wider ones, whose
// matches are verified against the build columns. Equal keys are chained behind
// the slot's row (nxt). Every probe row costs one random 16-byte read of the L2
// (measured 150 G rows/s over a table of up to 2 MiB, 131 at 4 MiB, 92 at 8
// MiB, 50 beyond), the probe side is read once and in order, and so are its
// matches written.

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// What a slot holds of a key: the key itself up to 8 bytes, else a 64-bit mix of it.
template <int KW, int NC> __device__ __forceinline__ uint64_t flat_word(const Key<KW, NC> &k) {
    if constexpr (KW * NC == 4) return k.c[0];
    else if constexpr (KW == 8 && NC == 1) return k.c[0];
    else if constexpr (KW == 4 && NC == 2) return (uint64_t)k.c[0] | (uint64_t)k.c[1] << 32;
    else {
        uint64_t m = 0;
#pragma unroll
        for (int c = 0; c < NC; c++) m = (m ^ (uint64_t)k.c[c]) * 0x9E3779B97F4A7C15ull + (m >> 29);
        return m;
    }
}

template <int HP, int KW, int NC> __device__ __forceinline__ void flat_build_block(const FlatArgs &a, uint32_t block) {
    const uint32_t i = block * kFlatThreads + threadIdx.x;
    if (i >= (uint32_t)a.r.n) return;
    const Key<KW, NC> k = load_key<KW, NC>(a.r, i);
    const uint32_t row = i + 1, lo = hash_key_lo<HP, KW, NC>(k, a.hash);
    // An empty slot takes the row; the slot of an equal key takes it by an
    // exchange (one atomic, however many rows of that key arrive) and the row
    // links to the one it replaced. Only the probe kernel follows links.
    uint32_t behind = 0;
    if constexpr (KW * NC == 4) {
        unsigned long long *slots = reinterpret_cast<unsigned long long *>(a.slots);
        const unsigned long long mine = (unsigned long long)flat_word(k) << 32 | row;
        uint32_t p = chain_of(lo, 0, a.hshift) * 2;  // slots of a pair fill in order
        while (true) {
            const unsigned long long got = atomicCAS(&slots[p], 0ull, mine);
            if (got == 0) break;
            if ((uint32_t)(got >> 32) == (uint32_t)(mine >> 32)) {
                behind = (uint32_t)atomicExch(&slots[p], mine);
                break;
            }
            p = (p + 1) & a.mask;
        }
    } else {
        uint32_t p = chain_of(lo, 0, a.hshift);
        while (true) {
            uint32_t *slot = a.slots + (uint64_t)p * 4;  // {word lo, word hi, row, -}
            const uint32_t got = atomicCAS(&slot[2], 0u, row);
            if (got == 0) {
                *reinterpret_cast<uint64_t *>(slot) = flat_word(k);  // the slot's key never changes again
                break;
            }
            // the occupant's key, from the build side itself (the slot may not hold it yet)
            if (key_eq<KW, NC>(k, load_key<KW, NC>(a.r, got - 1))) {
                behind = atomicExch(&slot[2], row);
                break;
            }
            p = (p + 1) & a.mask;
        }
    }
    a.nxt[i] = behind;
    if (behind) *a.dup = 1;
}

template <int HP, int KW, int NC> __global__ __launch_bounds__(kFlatThreads) void k_flat_build(FlatArgs a) {
    flat_build_block<HP, KW, NC>(a, blockIdx.x);
}

// `blocks`: of the join. One atomic per block reserves its output rows and
// counts it (kFlatBlock): the last block to reserve knows the join's count and
// hands it to the host, with the device clock.
template <int HP, int KW, int NC, int TH, int U>
__device__ __forceinline__ void flat_probe_block(const FlatArgs &a, uint32_t block, uint32_t blocks) {
    constexpr int WAVES = TH / 64;
    constexpr bool K4 = KW * NC == 4, WIDE = KW * NC > 8;
    __shared__ uint32_t wave_count[WAVES];
    __shared__ unsigned long long out_base;
    __shared__ uint32_t long_chain;
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    if (tid == 0) long_chain = 0;
    __syncthreads();
    const GKeys<KW, NC> sk = uniform_keys<KW, NC>(a.s), rk = uniform_keys<KW, NC>(a.r);
    const gptr<const u32x4> slots = (gptr<const u32x4>)a.slots;
    const gptr<const uint32_t> nxt = to_global(a.nxt);
    const uint32_t n = (uint32_t)a.s.n, mask = a.mask, hshift = a.hshift;
    const bool dup = *a.dup != 0;
    // a wave's rows are consecutive, and so are its matches
    const uint32_t row0 = block * (TH * U) + w * 64 * U + lane;
    Key<KW, NC> k[U];
#pragma unroll
    for (int u = 0; u < U; u++) k[u] = load_key<KW, NC>(sk, row0 + u * 64 < n ? row0 + u * 64 : 0u);
    uint32_t p[U], f[U];  // next slot (pair) to read, ~0: done; matched build row + 1
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t h = chain_of(hash_key_lo<HP, KW, NC>(k[u], a.hash), 0, hshift);
        p[u] = row0 + u * 64 < n ? h : ~0u;
        f[u] = 0;
    }
    while (true) {
        bool any = false;
#pragma unroll
        for (int u = 0; u < U; u++) any |= p[u] != ~0u;
        if (!__ballot(any)) break;
        u32x4 e[U];
#pragma unroll
        for (int u = 0; u < U; u++) e[u] = slots[p[u] != ~0u ? p[u] : 0u];  // rows that are done: one shared line
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool live = p[u] != ~0u;
            bool end;
            uint32_t hit;
            if constexpr (K4) {
                const uint32_t key = (uint32_t)k[u].c[0];
                hit = e[u].x && e[u].y == key ? e[u].x : (e[u].z && e[u].w == key ? e[u].z : 0u);
                end = e[u].x == 0 || e[u].z == 0;
            } else {
                const uint64_t word = flat_word(k[u]);
                hit = e[u].z && e[u].x == (uint32_t)word && e[u].y == (uint32_t)(word >> 32) ? e[u].z : 0u;
                end = e[u].z == 0;
                if constexpr (WIDE)
                    if (live && hit && !key_eq<KW, NC>(k[u], load_key<KW, NC>(rk, hit - 1))) hit = 0;  // another key of the same mix
            }
            f[u] = live ? hit : f[u];
            p[u] = !live || hit || end ? ~0u : (p[u] + 1) & (K4 ? mask >> 1 : mask);
        }
    }
    uint32_t c = 0, cu[U];  // matches of the lane, of each of its rows
#pragma unroll
    for (int u = 0; u < U; u++) {
        cu[u] = f[u] != 0;
        if (dup) {  // uniform: rows of an equal key behind the match
            uint32_t x = f[u];
            while (x && cu[u] <= kFlatChain) {
                x = nxt[x - 1];
                cu[u] += x != 0;
            }
            if (x) long_chain = 1;
        }
        c += cu[u];
    }
    c = wave_sum<64>(c);
    if (lane == 0) wave_count[w] = c;
    __syncthreads();
    if (tid == 0) {
        uint32_t sum = 0;
        for (int x = 0; x < WAVES; x++) sum += wave_count[x];
        // A key with too many rows to follow one by one: the host runs the join in the pipeline (with the top
        // bit of the count set nothing more is written).
        const unsigned long long gave_up = long_chain ? atomicOr(a.count, kFlatGiveUp) | kFlatGiveUp : 0;
        const unsigned long long got = atomicAdd(a.count, kFlatBlock | sum) | (gave_up & kFlatGiveUp);
        out_base = got & kFlatGiveUp ? kFlatGiveUp : got & (kFlatBlock - 1);
        if ((uint32_t)((got & ~kFlatGiveUp) / kFlatBlock) + 1 == blocks) {
            a.down[0] = (got & kFlatGiveUp) | ((got & (kFlatBlock - 1)) + sum);
            if (a.clock) {  // a single join; its counter is zero again for the next one
                a.down[1] = *a.clock;
                a.down[2] = wall_clock64();
                *a.count = 0;
            }
        }
    }
    const gptr<const uint32_t> rid = uniform_global(a.r.rowids), sid = uniform_global(a.s.rowids);
    uint32_t r[U], s[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t i = row0 + u * 64;
        s[u] = sid ? sid[i < n ? i : 0u] : i;
        r[u] = rid ? rid[f[u] ? f[u] - 1 : 0u] : f[u] - 1;
    }
    __syncthreads();
    if (c) {
        WalkArgs wa;
        wa.out_r = uniform_global(a.out_r);
        wa.out_s = uniform_global(a.out_s);
        wa.cap = uniform(a.cap);
        const uint32_t ob1 = a.one_based;
        Emitter em;
        em.pos = out_base;
        for (uint32_t x = 0; x < w; x++) em.pos += wave_count[x];
        if (!dup) {  // uniform
#pragma unroll
            for (int u = 0; u < U; u++) em.put(f[u] != 0, r[u] + ob1, s[u] + ob1, wa);
        } else {
            // each lane writes its rows' matches by itself, behind those of the lanes below: no state
            // of the wave is carried through a loop that lanes leave at different times
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t inc = wave_incl_scan(cu[u]);
                unsigned long long o = em.pos + inc - cu[u];
                uint32_t x = f[u], id = r[u];
                for (uint32_t m = 0; m < cu[u]; m++) {
                    if (o < wa.cap) {
                        wa.out_r[o] = id + ob1;
                        wa.out_s[o] = s[u] + ob1;
                    }
                    o++;
                    x = nxt[x - 1];
                    if (x) id = rid ? rid[x - 1] : x - 1;
                }
                em.pos += __shfl(inc, 63, 64);
            }
        }
    }
}

template <int HP, int KW, int NC, int TH, int U> __global__ __launch_bounds__(TH) void k_flat_probe(FlatArgs a) {
    flat_probe_block<HP, KW, NC, TH, U>(a, blockIdx.x, gridDim.x);
}

// A batch's blocks stand join after join in one line, of which each XCD takes
// one eighth from its start on: the few joins an XCD works on at a time have
// their tables in its L2 and in no other (a grid is a multiple of kXcds).
// The join and the block in it; false: past the line's end.
__device__ __forceinline__ bool flat_batch_at(const uint32_t *first, uint32_t n_joins, uint32_t total, uint32_t &j, uint32_t &block) {
    const uint32_t at = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
    if (at >= total) return false;
    j = uniform(wave_upper_index(first, n_joins, at));
    block = at - first[j];
    return true;
}

template <int HP, int KW, int NC> __global__ __launch_bounds__(kFlatThreads) void k_flat_build_batch(FlatBatch b) {
    uint32_t j, block;
    if (flat_batch_at(b.build0, b.n_joins, b.build_blocks, j, block)) flat_build_block<HP, KW, NC>(b.joins[j], block);
}

template <int HP, int KW, int NC> __global__ __launch_bounds__(kFlatThreads) void k_flat_probe_batch(FlatBatch b) {
    uint32_t j, block;
    if (flat_batch_at(b.probe0, b.n_joins, b.probe_blocks, j, block))
        flat_probe_block<HP, KW, NC, kFlatThreads, flat_batch_rows(KW * NC)>(b.joins[j], block, b.probe0[j + 1] - b.probe0[j]);
}

// Dispatch over the key shape (key width, key columns).
template <typename F> hipError_t dispatch_keys(const LaunchShape &sh, F &&f) {
#define VJ_CASE(KW, NC) \
    if (sh.kw == KW && sh.nc == NC) return f.template operator()<KW, NC>();
    VJ_CASE(4, 1) VJ_CASE(4, 2) VJ_CASE(4, 3) VJ_CASE(4, 4)
    VJ_CASE(8, 1) VJ_CASE(8, 2) VJ_CASE(8, 3) VJ_CASE(8, 4)
#undef VJ_CASE
    return hipErrorInvalidValue;
}

size_t pass_lds_bytes(int kw, int nc, int tile) {
    const int kb = kw * nc, T = pass_tile(kb, tile);
    return (size_t)T * (kb > 4 ? kb : 4) + (size_t)(kPassWaves * 256 + 768) * 4 + (size_t)T;
}

size_t probe_lds_bytes(int kw, int nc, int table) {
    return (size_t)probe_table_bytes(kw * nc, table);
}

size_t fan_lds_bytes(int kw, int nc, int big, uint32_t bins) {
    return (size_t)fan_tile(kw * nc, big) * (kw + 2) + (size_t)bins * 8;
}

}  // namespace

template <int HP> hipError_t StageLaunch<HP>::hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s) {
    const size_t lds = (size_t)a.max_hist_bins * 4;
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        if (sh.tile == 1)
            hipLaunchKernelGGL((k_hist<HP, KW, NC, 1>), dim3(a.total_hist_blocks), dim3(kHistThreads), lds, s, a);
        else if (sh.tile == 2)
            hipLaunchKernelGGL((k_hist<HP, KW, NC, 2>), dim3(a.total_hist_blocks), dim3(kHistThreads), lds, s, a);
        else
            hipLaunchKernelGGL((k_hist<HP, KW, NC, 0>), dim3(a.total_hist_blocks), dim3(kHistThreads), lds, s, a);
        return hipGetLastError();
    });
}

template <int HP> hipError_t StageLaunch<HP>::pass(const PipeArgs &a, const LaunchShape &sh, int pass, hipStream_t s) {
    const uint32_t total = pass == 1 ? a.total_p1_tiles : a.total_p2_chunks;
    const uint32_t groups = (total + kXcdGroup - 1) / kXcdGroup;  // pass 2: every XCD gets the same number of groups
    const uint32_t grid = pass == 1 ? (total + kXcds - 1) / kXcds * kXcds : (groups + kXcds - 1) / kXcds * kXcds * kXcdGroup;
    const size_t lds = pass_lds_bytes(sh.kw, sh.nc, sh.tile);
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        if (sh.tile == 1)
            hipLaunchKernelGGL((k_pass<HP, KW, NC, 1>), dim3(grid), dim3(kPassThreads), lds, s, a, pass);
        else if (sh.tile == 2)
            hipLaunchKernelGGL((k_pass<HP, KW, NC, 2>), dim3(grid), dim3(kPassThreads), lds, s, a, pass);
        else
            hipLaunchKernelGGL((k_pass<HP, KW, NC, 0>), dim3(grid), dim3(kPassThreads), lds, s, a, pass);
        return hipGetLastError();
    });
}

template <int HP> hipError_t StageLaunch<HP>::fan_hist(const PipeArgs &a, const LaunchShape &sh, hipStream_t s) {
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        hipLaunchKernelGGL((k_fan_hist<HP, KW, NC>), dim3(a.total_hist_blocks), dim3(kFanThreads), (size_t)a.fan_bins * 4, s, a);
        return hipGetLastError();
    });
}

template <int HP> hipError_t StageLaunch<HP>::fan(const PipeArgs &a, const LaunchShape &sh, hipStream_t s) {
    const size_t lds = fan_lds_bytes(sh.kw, sh.nc, sh.fan_big, a.fan_bins);
    // large tiles: one persistent block per CU; small ones: a block per tile, two at a time per CU
    const uint32_t cus = sh.cus >= (int)kXcds ? (uint32_t)sh.cus / kXcds * kXcds : kXcds;
    const dim3 g(sh.fan_big && a.total_p1_tiles > cus ? cus : a.total_p1_tiles);
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        if (sh.fan_big)
            hipLaunchKernelGGL((k_fan<HP, KW, NC, 1>), g, dim3(kFanThreads), lds, s, a);
        else
            hipLaunchKernelGGL((k_fan<HP, KW, NC, 0>), g, dim3(kFanThreads), lds, s, a);
        return hipGetLastError();
    });
}

template <int HP> int StageLaunch<HP>::probe_blocks_per_cu(const LaunchShape &sh) {
    const size_t lds = probe_lds_bytes(sh.kw, sh.nc, sh.table);
    int blocks = 1;
    (void)dispatch_keys(sh, [&]<int KW, int NC>() {
        int n = 0;
        hipError_t e;
        if (sh.table == 2) {
            if constexpr (KW * NC <= 8)
                e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_probe<HP, KW, NC, 2>, probe_threads(2), lds);
            else
                e = hipErrorInvalidValue;
        } else {
            e = sh.table ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_probe<HP, KW, NC, 1>, probe_threads(1), lds)
                         : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_probe<HP, KW, NC, 0>, probe_threads(0), lds);
        }
        if (e == hipSuccess && n > 0) blocks = n;
        return e;
    });
    return blocks > 8 ? 8 : blocks;
}

template <int HP> hipError_t StageLaunch<HP>::direct(const DirectArgs &d, const LaunchShape &sh, int blocks, hipStream_t s) {
    const size_t lds = probe_lds_bytes(sh.kw, sh.nc, sh.table);
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        if (sh.table)
            hipLaunchKernelGGL((k_direct<HP, KW, NC, 1>), dim3(blocks), dim3(probe_threads(1)), lds, s, d);
        else
            hipLaunchKernelGGL((k_direct<HP, KW, NC, 0>), dim3(blocks), dim3(probe_threads(0)), lds, s, d);
        return hipGetLastError();
    });
}

template <int HP> hipError_t StageLaunch<HP>::flat(const FlatArgs &a, const LaunchShape &sh, hipStream_t s) {
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        const uint32_t n = (uint32_t)a.s.n;
        hipLaunchKernelGGL((k_flat_build<HP, KW, NC>), dim3(((uint32_t)a.r.n + kFlatThreads - 1) / kFlatThreads), dim3(kFlatThreads), 0, s, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        auto probe = [&]<int TH, int U>() {
            hipLaunchKernelGGL((k_flat_probe<HP, KW, NC, TH, U>), dim3((n - 1) / (TH * U) + 1), dim3(TH), 0, s, a);
            return hipGetLastError();
        };
        // the largest blocks that leave no CU without one
        if (n <= 1u << 18) return probe.template operator()<512, 2>();
        if (n <= 1u << 19) return probe.template operator()<1024, 2>();
        return probe.template operator()<1024, 4>();
    });
}

template <int HP> hipError_t StageLaunch<HP>::flat_batch(const FlatBatch &b, const LaunchShape &sh, hipStream_t s) {
    auto grid = [](uint32_t blocks) { return dim3((blocks + kXcds - 1) / kXcds * kXcds); };
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        hipLaunchKernelGGL((k_flat_build_batch<HP, KW, NC>), grid(b.build_blocks), dim3(kFlatThreads), 0, s, b);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_flat_probe_batch<HP, KW, NC>), grid(b.probe_blocks), dim3(kFlatThreads), 0, s, b);
        return hipGetLastError();
    });
}

template <int HP> hipError_t StageLaunch<HP>::probe(const PipeArgs &a, const LaunchShape &sh, int blocks, hipStream_t s) {
    const size_t lds = probe_lds_bytes(sh.kw, sh.nc, sh.table);
    return dispatch_keys(sh, [&]<int KW, int NC>() {
        if (sh.table == 2) {
            if constexpr (KW * NC <= 8)
                hipLaunchKernelGGL((k_probe<HP, KW, NC, 2>), dim3(blocks), dim3(probe_threads(2)), lds, s, a);
            else
                return hipErrorInvalidValue;
        } else if (sh.table)
            hipLaunchKernelGGL((k_probe<HP, KW, NC, 1>), dim3(blocks), dim3(probe_threads(1)), lds, s, a);
        else
            hipLaunchKernelGGL((k_probe<HP, KW, NC, 0>), dim3(blocks), dim3(probe_threads(0)), lds, s, a);
        return hipGetLastError();
    });
}

}  // namespace vj
