// rowstream.hpp - the rows of a block as the fused kernels read them: the WHERE on one row, and the
// streaming reader that the streaming phase 1 (twophase.hip) and the small-table kernel
// (smalltable.hip) share.
#pragma once

#include "groupby.hpp"

namespace qk {

// VV is VT, or a placeholder type when the table reads no value column.  MODE: 0 no WHERE,
// 1 row mask, 2 predicate list, 3 folded interval on the value column, 4 folded interval on
// another integer column, whose value (cv) and NULL bit (cn) the caller loaded.
template <typename VT, int MODE, typename VV>
__device__ __forceinline__ bool row_passes(const PredSet& preds, uint32_t vpred, const int8_t* mask,
                                           int64_t r, const VV& v, bool vn, int64_t cv = 0, bool cn = false) {
    if (MODE == 1) return mask[r] != 0;
    // & rather than &&: both sides are cheap and side-effect free, and a short circuit would
    // become a divergent branch per row
    if constexpr (MODE == 3 && VTraits<VT>::has) return !vn & in_range<VT>(preds.vr, v);
    if (MODE == 4) return !cn & col_in_range(preds, cv);
    if (MODE == 2) {
        for (int p = 0; p < preds.n; p++) {
            const qk_predicate& q = preds.p[p];
            bool pass;
            if constexpr (VTraits<VT>::has) {
                if ((vpred >> p) & 1u)
                    pass = !vn && pred_on_value(q, v, r);
                else
                    pass = eval_pred(q, r);
            } else {
                pass = eval_pred(q, r);
            }
            if (!pass) return false;
        }
    }
    return true;
}

// KT is the element type of a single integer key column, KeyPairI32 for two non-NULL int32
// key columns packed into one word (the first in the low half), or void for any key layout
// (read through the key spec's runtime switch).  With a typed key, the loads of a whole tile
// are issued before any of them is used.
struct KeyPairI32 {};
template <typename KT>
constexpr bool kPairKey = std::is_same<KT, KeyPairI32>::value;
template <typename KT>
constexpr bool kTypedKey = !std::is_same<KT, void>::value && !kPairKey<KT>;

// FP selects the aggregate states the LDS table keeps: kFieldsSum fixes them at sum + count
// (SUM, AVG, COUNT; no MIN/MAX) so that the loop carries no per-field tests; kFieldsAny reads
// them from `fields`.
constexpr int kFieldsAny = 0, kFieldsSum = 1;

// Whether the streaming reader reads these key columns: one int32 or int64 column, or two non-NULL
// int32 columns packed into one word.
inline bool stream_keys(const KeySpec& ks, const KeyCols& kc) {
    if (ks.single) return ks.nkeys == 1 && (ks.type[0] == QK_LONG || ks.type[0] == QK_INT);
    return ks.nkeys == 2 && ks.kw == 1 && ks.type[0] == QK_INT && ks.type[1] == QK_INT && ks.word[0] == 0 &&
           ks.shift[0] == 0 && ks.word[1] == 0 && ks.shift[1] == 32 && !kc.nm[0] && !kc.nm[1];
}

// ---- the streaming reader --------------------------------------------------------------------
//
// One typed key column (int32 or int64, nullable) or two non-NULL int32 key columns packed into one
// word, with no WHERE or a WHERE folded into an interval (on the value column or on one other integer
// column).  A wavefront takes chunks of kSChunk rows in parts of kSPart rows; lane l holds rows 2l and
// 2l+1 of every part, so every load instruction reads one contiguous 512 B (4-byte column) or 1 KB
// (8-byte column) range with 8- or 16-byte lanes, and a null bitmap costs one 32-bit load per part.
// The loads are buffer loads bounded by the resource's size: rows past the end read as zero and an
// absent bitmap is a resource of size zero, so no load needs a bounds test or a clamp, and the next
// chunk's loads are issued before the current chunk is aggregated.  Offsets are 32-bit bytes: every
// column of the block stays below 2^31 bytes.

// Blocks of at most this many rows can be streamed (8-byte columns and the prefetch past the end stay
// below 2^31 bytes).
constexpr int64_t kStreamMaxRows = (int64_t)1 << 27;

constexpr int kSRows = 4;                 // rows per lane per chunk
constexpr int kSParts = kSRows / 2;        // parts of a chunk: lane l holds rows 2l, 2l+1 of each
constexpr int kSChunk = 64 * kSRows;      // rows per wavefront per chunk
constexpr int kSPart = 128;               // rows per part

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int64_t bytes) {
    // word 3 = 0x00020000: the untyped 32-bit data format of raw buffer accesses on gfx9
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// The 32-bit words of one lane's kSRows rows of a column of E-byte elements: row j of the lane
// in w[j] (E = 4) or w[2j], w[2j+1] (E = 8).
template <int E>
struct LaneWords {
    uint32_t w[E * kSRows / 4];
};

// Every part of a lane's rows, the first at byte offset off, the next kSPart * E bytes further
// each (non-temporal: the columns are streamed once, and the lines of the cold regions being
// filled should stay in the L2).
__device__ __forceinline__ void ld_lane(__amdgpu_buffer_rsrc_t r, uint32_t off, LaneWords<4>& t) {
#pragma unroll
    for (int q = 0; q < kSParts; q++) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(off + q * kSPart * 4), 0, 2);
        t.w[2 * q] = v[0];
        t.w[2 * q + 1] = v[1];
    }
}
__device__ __forceinline__ void ld_lane(__amdgpu_buffer_rsrc_t r, uint32_t off, LaneWords<8>& t) {
#pragma unroll
    for (int q = 0; q < kSParts; q++) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off + q * kSPart * 8), 0, 2);
        t.w[4 * q] = v[0];
        t.w[4 * q + 1] = v[1];
        t.w[4 * q + 2] = v[2];
        t.w[4 * q + 3] = v[3];
    }
}

template <typename T>
__device__ __forceinline__ T word_elem(const uint32_t* w, int j) {
    if constexpr (sizeof(T) == 8) {
        const uint64_t u = (uint64_t)w[2 * j] | ((uint64_t)w[2 * j + 1] << 32);
        return __builtin_bit_cast(T, u);
    } else {
        return __builtin_bit_cast(T, w[j]);
    }
}

// A null bitmap's words for every part of a lane's rows: the lane's two rows of a part lie in
// one 32-bit word (2l is even), each part's word kSPart / 32 words after the previous one's.
struct LaneBits {
    uint32_t w[kSParts];
    __device__ __forceinline__ bool bit(int j, uint32_t sh) const {
        return (w[j >> 1] >> (sh + (uint32_t)(j & 1))) & 1u;
    }
};
__device__ __forceinline__ LaneBits no_bits() {
    LaneBits b;
#pragma unroll
    for (int q = 0; q < kSParts; q++) b.w[q] = 0u;
    return b;
}
__device__ __forceinline__ LaneBits ld_bits(__amdgpu_buffer_rsrc_t r, uint32_t boff) {
    LaneBits b;
#pragma unroll
    for (int q = 0; q < kSParts; q++)
        b.w[q] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(boff + q * (kSPart / 8)), 0, 0);
    return b;
}

// One lane's rows of a chunk: pass is false for rows past the end and rows the WHERE drops; a NULL
// key's key is 0.
template <typename VV>
struct StreamRows {
    uint64_t key[kSRows];
    VV val[kSRows];
    bool pass[kSRows], vnull[kSRows], knull[kSRows];
};

// Hands every row of the block to f, kSRows per lane at a time, on a grid of workgroups of BLOCK
// threads.  Control flow is uniform per wavefront: f is called with all 64 lanes.
template <typename VT, int MODE, typename KT, int BLOCK, typename F>
__device__ __forceinline__ void stream_rows(const KeyCols& kc, const VT* __restrict__ vals,
                                            const uint64_t* __restrict__ vnull, const PredSet& preds, int32_t n,
                                            F&& f) {
    constexpr bool HAS_V = VTraits<VT>::has;
    constexpr bool PAIR = kPairKey<KT>;
    using VV = typename std::conditional<HAS_V, VT, int>::type;
    constexpr int KE = PAIR ? 4 : (int)sizeof(KT);          // bytes per row of a key column
    constexpr int VE = HAS_V ? (int)sizeof(VV) : 4;         // bytes per row of the value column
    const int lane = threadIdx.x & 63;
    const int64_t bitmap_bytes = ((int64_t)n + 63) / 64 * 8;
    const __amdgpu_buffer_rsrc_t rk0 = make_rsrc(kc.col[0], (int64_t)n * KE);
    const __amdgpu_buffer_rsrc_t rk1 = make_rsrc(PAIR ? kc.col[1] : kc.col[0], PAIR ? (int64_t)n * KE : 0);
    const __amdgpu_buffer_rsrc_t rkn = make_rsrc(kc.nm[0], (!PAIR && kc.nm[0]) ? bitmap_bytes : 0);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vals, HAS_V ? (int64_t)n * VE : 0);
    const __amdgpu_buffer_rsrc_t rvn = make_rsrc(vnull, vnull ? bitmap_bytes : 0);
    const int CE = preds.rwide ? 8 : 4;
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(preds.rcol, MODE == 4 ? (int64_t)n * CE : 0);
    const __amdgpu_buffer_rsrc_t rcn = make_rsrc(preds.rnull, (MODE == 4 && preds.rnull) ? bitmap_bytes : 0);

    struct Chunk {
        LaneWords<KE> k0, k1;
        LaneWords<VE> v;
        LaneWords<8> c;
        LaneBits vb, kb, cb;
    };
    // the chunk's loads; a chunk past the end reads zeros
    auto load = [&](uint32_t chunk, Chunk& t) {
        const uint32_t row0 = chunk * (uint32_t)kSChunk + (uint32_t)lane * 2;
        ld_lane(rk0, row0 * KE, t.k0);
        if constexpr (PAIR) ld_lane(rk1, row0 * KE, t.k1);
        if constexpr (HAS_V) ld_lane(rv, row0 * VE, t.v);
        const uint32_t boff = (row0 >> 5) * 4;
        t.vb = ld_bits(rvn, boff);
        t.kb = PAIR ? no_bits() : ld_bits(rkn, boff);
        t.cb = no_bits();
        if constexpr (MODE == 4) {
            if (preds.rwide) {
                ld_lane(rc, row0 * 8, t.c);
            } else {
                LaneWords<4> c4;
                ld_lane(rc, row0 * 4, c4);
#pragma unroll
                for (int j = 0; j < kSRows; j++) t.c.w[j] = c4.w[j];
            }
            t.cb = ld_bits(rcn, boff);
        }
    };
    auto rows = [&](uint32_t chunk, const Chunk& t) {
        const uint32_t row0 = chunk * (uint32_t)kSChunk + (uint32_t)lane * 2;
        const uint32_t sh = row0 & 31;
        StreamRows<VV> o;
#pragma unroll
        for (int j = 0; j < kSRows; j++) {
            const bool vn = t.vb.bit(j, sh);
            const bool kn = t.kb.bit(j, sh);
            uint64_t kk;
            if constexpr (PAIR)
                kk = (uint64_t)t.k0.w[j] | ((uint64_t)t.k1.w[j] << 32);
            else
                kk = (uint64_t)(int64_t)word_elem<KT>(t.k0.w, j);
            VV v = 0;
            if constexpr (HAS_V) v = word_elem<VV>(t.v.w, j);
            int64_t cv = 0;
            if constexpr (MODE == 4)
                cv = preds.rwide ? word_elem<int64_t>(t.c.w, j) : (int64_t)word_elem<int32_t>(t.c.w, j);
            const bool cn = t.cb.bit(j, sh);
            const bool in_block = row0 + (uint32_t)((j >> 1) * kSPart + (j & 1)) < (uint32_t)n;
            o.key[j] = kn ? 0ull : kk;
            o.val[j] = v;
            o.pass[j] = in_block & row_passes<VT, MODE>(preds, 0u, nullptr, 0, v, vn, cv, cn);
            o.vnull[j] = vn;
            o.knull[j] = kn;
        }
        f(o);
    };
    // chunks are dealt to the wavefronts of the grid in turn; each wavefront loads its next
    // chunk before it aggregates the current one (two register sets, used alternately)
    const uint32_t nchunks = (uint32_t)(((int64_t)n + kSChunk - 1) / kSChunk);
    const uint32_t stride = gridDim.x * (uint32_t)(BLOCK / 64);
    uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6)));
    Chunk A, B;
    load(c, A);
    while (c < nchunks) {
        load(c + stride, B);
        rows(c, A);
        c += stride;
        if (c >= nchunks) break;
        load(c + stride, A);
        rows(c, B);
        c += stride;
    }
}

}  // namespace qk
