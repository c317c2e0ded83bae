// Standalone hash kernel: vj_hash (replaces hash_func, src/hash/hash.cu:507-557).
//
// The reference walks a row-major buffer with one thread per row, so a wave
// reads 64 rows x row-width bytes with a stride; here key columns are SoA and
// each of the NC column loads of a wave is one contiguous 64 x KW-byte read.
// Every thread takes 16 bytes of each column at a time (two 8-byte or four
// 4-byte rows, vectors of element alignment) in two places per grid-stride
// step, so several wide loads are in flight. FNV and custom_xor_hw have kernels
// of their own; the other eleven kinds share one kernel per key shape, which
// branches on the kind once and then runs straight-line code for it. (A walk
// that looks the kind up at every word, through memory, took 217 us for 2e7 rows of
// 3 x u32 with custom_mult_xor_hw.) HBM-bound: bytes = n * (NC * KW +
// hash_bits / 8).
#include "vj_internal.hpp"

namespace vj {

namespace {

constexpr int kHashThreads = 256;
constexpr int kHashUnroll = 2;  // places per thread and step

// Reads and writes rows 16 bytes of a key column at a time; Row maps a key to its hash.
template <int KW, int NC, typename OutT, typename Row>
__device__ __forceinline__ void hash_rows(const TView &t, OutT *out_, Row row) {
    using KT = typename KeyT<KW>::T;
    constexpr int R = 16 / KW;                                        // rows per vector
    constexpr int OR = 16 / (int)sizeof(OutT) < R ? 16 / (int)sizeof(OutT) : R;  // rows per store
    typedef KT KV __attribute__((ext_vector_type(R), aligned(sizeof(KT))));
    typedef OutT OV __attribute__((ext_vector_type(OR), aligned(sizeof(OutT))));
    // key columns and output as global-address-space pointers (global_load /
    // global_store, counted on vmcnt only), copied out of the view once
    GKeys<KW, NC> in;
#pragma unroll
    for (int c = 0; c < NC; c++) in.c[c] = to_global(static_cast<const KT *>(t.cols[c]));
    const gptr<OutT> out = to_global(out_);
    const uint64_t n = t.n, whole = n / R;  // whole vectors
    const uint64_t stride = (uint64_t)gridDim.x * kHashThreads * kHashUnroll;
    for (uint64_t base = (uint64_t)blockIdx.x * kHashThreads * kHashUnroll + threadIdx.x; base < whole; base += stride) {
        KV k[kHashUnroll][NC];
#pragma unroll
        for (int u = 0; u < kHashUnroll; u++) {  // all loads in flight at once (past the end: the first again)
            const uint64_t v = base + (uint64_t)u * kHashThreads;
#pragma unroll
            for (int c = 0; c < NC; c++) k[u][c] = *(gptr<const KV>)(in.c[c] + (v < whole ? v : base) * R);
        }
#pragma unroll
        for (int u = 0; u < kHashUnroll; u++) {
            const uint64_t v = base + (uint64_t)u * kHashThreads;
            if (v < whole) {
#pragma unroll
                for (int r0 = 0; r0 < R; r0 += OR) {
                    OV o;
#pragma unroll
                    for (int r = 0; r < OR; r++) {
                        Key<KW, NC> key;
#pragma unroll
                        for (int c = 0; c < NC; c++) key.c[c] = k[u][c][r0 + r];
                        o[r] = row(key);
                    }
                    *(gptr<OV>)(out + v * R + r0) = o;
                }
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < n - whole * R) {  // the rows after the last whole vector
        const uint64_t i = whole * R + threadIdx.x;
        out[i] = row(load_key<KW, NC>(in, i));
    }
}

template <int HP, int KW, int NC, typename OutT>
__global__ __launch_bounds__(kHashThreads) void k_hash(TView t, HashCfg h, OutT *out) {
    hash_rows<KW, NC>(t, out, [&](const Key<KW, NC> &k) { return (OutT)hash_key<HP, KW, NC>(k, h); });
}

// One kind over 32-bit words (chunks of CB bits). WORDS: how a 4-byte column
// is widened (0: zero, 1: sign extension, 2: not at all); zero words fold.
template <int KIND, int CB, int KW, int NC, int WORDS, typename HT>
__device__ __forceinline__ void hash_kind_rows(const TView &t, HT *out) {
    hash_rows<KW, NC>(t, out, [&](const Key<KW, NC> &k) {
        Walker<HT> s;
        s.init(KIND, CB);
        constexpr int PER = KW == 4 && WORDS == 2 ? 1 : 2;  // words per column
#pragma unroll
        for (int round = 0; round < (KIND == HK_N_MULT_XOR_SHIFT ? 2 : 1); round++) {  // hash_func passes rounds = 2, hash.cu:526
#pragma unroll
            for (int i = 0; i < PER * NC; i++) {
                const uint64_t v = k.c[i / PER];
                uint32_t w = (uint32_t)v;
                if (PER == 2 && i % 2) w = KW == 8 ? (uint32_t)(v >> 32) : (WORDS == 1 ? (uint32_t)((int32_t)(uint32_t)v >> 31) : 0u);
                s.template step_as<KIND>(w);
                if ((i + 1) % (CB / 32) == 0) s.template chunk_end_as<KIND>();
            }
        }
        return s.hash;
    });
}

// Kinds whose steps depend on the chunk width get it at compile time.
template <int KIND, int KW, int NC, int WORDS, typename HT>
__device__ __forceinline__ void hash_kind_chunk(const TView &t, const HashCfg &h, HT *out) {
    constexpr bool by_chunk = KIND == HK_ADD_HW || KIND == HK_ADD_SHIFT || KIND == HK_XOR_SHIFT || KIND == HK_MULT_SHIFT ||
                              KIND == HK_MULT_XOR_SHIFT || KIND == HK_N_MULT_XOR_SHIFT;
    if (by_chunk && h.chunk_bits == 64) hash_kind_rows<KIND, by_chunk ? 64 : 32, KW, NC, WORDS>(t, out);
    else if (by_chunk && h.chunk_bits == 128) hash_kind_rows<KIND, by_chunk ? 128 : 32, KW, NC, WORDS>(t, out);
    else hash_kind_rows<KIND, 32, KW, NC, WORDS>(t, out);
}

template <int KW, int NC, int WORDS, typename HT>
__global__ __launch_bounds__(kHashThreads) void k_hash_kinds(TView t, HashCfg h, HT *out) {
    switch (h.kind) {  // uniform
#define VJ_KIND(K) \
    case K: hash_kind_chunk<K, KW, NC, WORDS>(t, h, out); break;
        VJ_KIND(HK_ADD) VJ_KIND(HK_ADD_SHIFT) VJ_KIND(HK_ADD_HW) VJ_KIND(HK_XOR) VJ_KIND(HK_XOR_SHIFT) VJ_KIND(HK_MULT)
        VJ_KIND(HK_MULT_SHIFT) VJ_KIND(HK_MULT_HW) VJ_KIND(HK_MULT_XOR_SHIFT) VJ_KIND(HK_N_MULT_XOR_SHIFT)
        VJ_KIND(HK_MULT_XOR_HW)
#undef VJ_KIND
    default: break;
    }
}

template <int HP, int KW, int NC, typename HT>
Err launch_typed(const TView &v, const HashCfg &h, HT *out, hipStream_t s, int cus) {
    const uint64_t per_block = (uint64_t)kHashThreads * kHashUnroll * (16 / KW);
    const uint64_t want = (v.n + per_block - 1) / per_block, cap = (uint64_t)cus * 16;
    const dim3 blocks((unsigned)(want < cap ? want : cap)), threads(kHashThreads);
    if (blocks.x == 0) return Err::ok();
    if constexpr (HP == HP_GENERIC) {
        if (h.chunk_bits != 8) {
            if (KW == 8 || (!h.native && !h.key_signed)) hipLaunchKernelGGL((k_hash_kinds<KW, NC, 0, HT>), blocks, threads, 0, s, v, h, out);
            else if (!h.native) hipLaunchKernelGGL((k_hash_kinds<KW, NC, KW == 4 ? 1 : 0, HT>), blocks, threads, 0, s, v, h, out);
            else hipLaunchKernelGGL((k_hash_kinds<KW, NC, KW == 4 ? 2 : 0, HT>), blocks, threads, 0, s, v, h, out);
            VJ_HIP_TRY(hipGetLastError());
            return Err::ok();
        }
    }
    hipLaunchKernelGGL((k_hash<HP, KW, NC, HT>), blocks, threads, 0, s, v, h, out);
    VJ_HIP_TRY(hipGetLastError());
    return Err::ok();
}

template <int HP, int KW, int NC>
Err launch_bits(const TView &v, const HashCfg &h, void *out, hipStream_t s, int cus) {
    return h.bits == 32 ? launch_typed<HP, KW, NC>(v, h, static_cast<uint32_t *>(out), s, cus)
                        : launch_typed<HP, KW, NC>(v, h, static_cast<uint64_t *>(out), s, cus);
}

template <int HP, int KW>
Err launch_nc(int nc, const TView &v, const HashCfg &h, void *out, hipStream_t s, int cus) {
    switch (nc) {
    case 1: return launch_bits<HP, KW, 1>(v, h, out, s, cus);
    case 2: return launch_bits<HP, KW, 2>(v, h, out, s, cus);
    case 3: return launch_bits<HP, KW, 3>(v, h, out, s, cus);
    case 4: return launch_bits<HP, KW, 4>(v, h, out, s, cus);
    }
    return Err::make(VJ_ERR_INVALID_ARGUMENT, "n_cols must be 1..4");
}

template <int HP>
Err launch_kw(const vj_table *t, const TView &v, const HashCfg &h, void *out, hipStream_t s, int cus) {
    if (t->key_width == 8) return launch_nc<HP, 8>(t->n_cols, v, h, out, s, cus);
    return launch_nc<HP, 4>(t->n_cols, v, h, out, s, cus);
}

}  // namespace

Err launch_hash(const vj_table *t, const HashCfg &h, void *out, hipStream_t s, int cus) {
    TView v = to_view(t);
    switch (hash_path(h)) {
    case HP_FNV: return launch_kw<HP_FNV>(t, v, h, out, s, cus);
    case HP_XOR_HW: return launch_kw<HP_XOR_HW>(t, v, h, out, s, cus);
    default: return launch_kw<HP_GENERIC>(t, v, h, out, s, cus);
    }
}

}  // namespace vj
