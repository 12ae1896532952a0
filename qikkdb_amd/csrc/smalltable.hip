// smalltable.hip - GROUP BY into a table whose every key fits a workgroup's LDS.
//
// The streaming reader's rows go straight into the workgroup's LDS table (no sample, no partitions, no
// second pass over rows); the workgroups' tables are then added up by k_gb_fold.
#include <algorithm>

#include "ldstable.hpp"
#include "rowstream.hpp"

namespace qk {

namespace {

constexpr int kSmallBlock = 512;

// Rows of one block into the LDS table (H a power of two, 32 - log2(H) = hshift).  A row costs one
// 64-bit LDS read and one 32-bit multiply to find its slot: the kernel is bound by the instructions it
// issues per row, once the lanes of a wave do not queue at the same words (lds_table copies).
template <typename VT, int MODE, typename KT, int FP>
__global__ void __launch_bounds__(kSmallBlock) k_gb_small(GView g, KeyCols kc, const VT* __restrict__ vals,
                                                          const uint64_t* __restrict__ vnull, PredSet preds,
                                                          int32_t n, uint32_t fields, int32_t H, int32_t hshift,
                                                          int32_t rbits, Partials out) {
    extern __shared__ __align__(16) uint64_t lds[];
    __shared__ unsigned int s_new;
    constexpr bool HAS_V = VTraits<VT>::has;
    constexpr bool REAL = VTraits<VT>::real;
    using VV = typename std::conditional<HAS_V, VT, int>::type;
    const uint32_t f = FP == kFieldsSum ? (fields & (F_CNT | F_CNTALL | F_SUM)) | F_SUM : fields;
    const Lds t = lds_carve(lds, H, rbits, f);
    if (threadIdx.x == 0) s_new = 0;
    lds_clear(t);
    __syncthreads();
    const int copy = threadIdx.x & ((1 << rbits) - 1);
    stream_rows<VT, MODE, KT, kSmallBlock>(kc, vals, vnull, preds, n, [&](const StreamRows<VV>& o) {
        uint32_t home[kSRows];
        uint64_t cur[kSRows];
#pragma unroll
        for (int j = 0; j < kSRows; j++) {
            home[j] = (((uint32_t)o.key[j] ^ (uint32_t)(o.key[j] >> 32)) * 0x9e3779b1u) >> hshift;
            cur[j] = __hip_atomic_load(&t.key[home[j]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
#pragma unroll
        for (int j = 0; j < kSRows; j++) {
            if (!o.pass[j]) continue;
            int s = (int)home[j];
            // an empty home matches the key equal to kEmpty, which lives in its side slot
            if ((cur[j] != o.key[j]) | o.knull[j] | (sizeof(KT) != 4 && o.key[j] == kEmpty))
                s = o.knull[j] ? lds_side(t, 0) : o.key[j] == kEmpty ? lds_side(t, 1) : lds_probe(t, o.key[j], home[j]);
            Part p;
            if constexpr (HAS_V) p = row_part<VT>(o.val[j], o.vnull[j]); else p = row_part<NoValue>(NoValue{}, o.vnull[j]);
            if (s >= 0) {
                lds_accum<REAL>(t, (s << rbits) | copy, p, f);
            } else {
                bool is_new = false;
                const int64_t gs = g_slot1(g, o.key[j], false, hash64(o.key[j]), &is_new);
                if (is_new) atomicAdd(&s_new, 1u);
                if (gs >= 0) g_accum_atomic(g, gs, p, f); else g_set_lost(g);
            }
        }
    });
    __syncthreads();
    lds_flush<1, REAL>(t, g, out, f, &s_new);
    __syncthreads();
    if (threadIdx.x == 0) g_count_new(g, s_new);
}

// Adds up the tables that a row kernel's workgroups left in `in` (`wgs` tables of T = H + 2 entries) and
// merges each group into the global table once, where every workgroup merging its own table would
// queue at the same few groups (1M rows, 1000 groups: 164 us, against 25 + 34 us).  An entry's
// place follows its key's hash up to a few probes, so a workgroup takes kFoldSlots neighbouring
// entries of every table; a key displaced over that border meets two workgroups, hence the atomics
// of add_entry.
constexpr int kFoldSlots = 16;
constexpr int kFoldBlock = 512;
constexpr int kFoldH = 128;
constexpr int kFoldBatch = 4;
template <int KW, bool REAL>
__global__ void __launch_bounds__(kFoldBlock) k_gb_fold(GView g, Partials in, int32_t T, int32_t wgs, uint32_t fields) {
    __shared__ uint64_t lds[(kFoldH + 2) * 5];
    __shared__ unsigned int s_new;
    Lds t = lds_carve(lds, kFoldH, 0, fields);
    for (int s = threadIdx.x; s < kFoldH + 2; s += blockDim.x) {
        t.key[s] = s < kFoldH ? kEmpty : 0ull;
        t.cnt[s] = 0;
        if (t.cntall) t.cntall[s] = 0;
        if (t.sum) t.sum[s] = 0;
        if (t.mn) t.mn[s] = ~0ull;
        if (t.mx) t.mx[s] = 0ull;
    }
    if (threadIdx.x == 0) s_new = 0;
    __syncthreads();
    const int s = blockIdx.x * kFoldSlots + threadIdx.x % kFoldSlots;
    const int side = s - (T - 2);  // 0 the NULL key's entry, 1 that of the key equal to kEmpty
    if (s < T) {
        // an entry mostly holds the same key in every table: it is added up in registers while it does
        uint64_t run = kEmpty;
        Part sum{};
        auto add = [&](uint64_t k, const Part& p) {
            if (k == kEmpty) return;
            const int ls = lds_find(t, side == 1 ? kEmpty : k, side == 0, hash64(k));
            if (ls >= 0) lds_accum<REAL>(t, ls, p, fields);
            else add_entry<KW, false>(g, k, side, p, fields, &s_new);
        };
        // kFoldBatch tables' entries at a time, key and states loaded together (an empty entry's states
        // are whatever memory holds, and are dropped)
        constexpr int kStep = kFoldBlock / kFoldSlots;
        for (int w0 = threadIdx.x / kFoldSlots; w0 < wgs; w0 += kFoldBatch * kStep) {
            uint64_t k[kFoldBatch];
            Part p[kFoldBatch];
#pragma unroll
            for (int i = 0; i < kFoldBatch; i++) {
                const int w = w0 + i * kStep;
                const int64_t at = (int64_t)min(w, wgs - 1) * T + s;
                k[i] = w < wgs ? to_g(in.key)[at] : kEmpty;
                p[i].cnt = to_g(in.cnt)[at];
                p[i].cntall = in.cntall ? to_g(in.cntall)[at] : 0ull;
                p[i].sum = in.sum ? to_g(in.sum)[at] : 0ull;
                p[i].mn = in.mn ? to_g(in.mn)[at] : ~0ull;
                p[i].mx = in.mx ? to_g(in.mx)[at] : 0ull;
            }
#pragma unroll
            for (int i = 0; i < kFoldBatch; i++) {
                if (k[i] == kEmpty) continue;
                if (k[i] != run) {
                    add(run, sum);
                    run = k[i];
                    sum = p[i];
                } else {
                    merge_part<REAL>(sum, p[i]);
                }
            }
        }
        add(run, sum);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kFoldH + 2; e += blockDim.x) {
        const uint64_t k = t.key[e];
        if (e < kFoldH ? k == kEmpty : k == 0ull) continue;
        add_entry<KW, false>(g, k, e - kFoldH, lds_fold<REAL>(t, e, 0), fields, &s_new);
    }
    __syncthreads();
    if (threadIdx.x == 0) g_count_new(g, s_new);
}

// ---- launch helpers -------------------------------------------------------------------------

template <typename VT, int MODE, typename KT, int FP>
int launch_small(const GView& g, const KeyCols& kc, const void* vals, const uint64_t* vnull, const PredSet& ps,
                 int64_t n, uint32_t fields, const LdsShape& L, hipStream_t s) {
    int hshift = 32;
    while ((1 << (32 - hshift)) < L.H) hshift--;
    auto kern = k_gb_small<VT, MODE, KT, FP>;
    const size_t lds = lds_table_bytes(L.H, L.rbits, fields);
    int occ = 0;
    QK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, kSmallBlock, lds));
    if (occ < 1) return fail(QK_ERROR, "group by: small-table launch (LDS %zu B) does not fit", lds);
    const int64_t grid = std::max<int64_t>(
        1, std::min<int64_t>({(int64_t)device_info().cus * occ, L.wgs_for(n),
                              (n + kSChunk * (kSmallBlock / 64) - 1) / (kSChunk * (kSmallBlock / 64))}));
    const Partials part = L.for_wgs(grid);
    kern<<<(unsigned)grid, kSmallBlock, lds, s>>>(g, kc, (const VT*)vals, vnull, ps, (int32_t)n, fields, L.H, hshift,
                                                  L.rbits, part);
    QK_HIP(hipGetLastError());
    return part.key ? fold_partials(g, L, (int32_t)grid, VTraits<VT>::real, fields, s) : QK_SUCCESS;
}

template <typename VT, typename KT, int FP>
int launch_small_m(int mode, const GView& g, const KeyCols& kc, const void* vals, const uint64_t* vnull,
                   const PredSet& ps, int64_t n, uint32_t fields, const LdsShape& L, hipStream_t s) {
    if (mode == 0) return launch_small<VT, 0, KT, FP>(g, kc, vals, vnull, ps, n, fields, L, s);
    if (mode == 4) return launch_small<VT, 4, KT, FP>(g, kc, vals, vnull, ps, n, fields, L, s);
    if constexpr (VTraits<VT>::has) return launch_small<VT, 3, KT, FP>(g, kc, vals, vnull, ps, n, fields, L, s);
    return fail(QK_ERROR, "value range filter without a value column");
}

template <typename VT>
int launch_small_k(int mode, const GView& g, const KeySpec& ks, const KeyCols& kc, const void* vals,
                   const uint64_t* vnull, const PredSet& ps, int64_t n, uint32_t fields, const LdsShape& L,
                   hipStream_t s) {
    const bool sum_only = (fields & F_SUM) && !(fields & (F_MIN | F_MAX));
#define QK_SMALL(KT)                                                                                        \
    (sum_only ? launch_small_m<VT, KT, kFieldsSum>(mode, g, kc, vals, vnull, ps, n, fields, L, s)           \
              : launch_small_m<VT, KT, kFieldsAny>(mode, g, kc, vals, vnull, ps, n, fields, L, s))
    if (!ks.single) return QK_SMALL(KeyPairI32);
    return ks.type[0] == QK_INT ? QK_SMALL(int32_t) : QK_SMALL(int64_t);
#undef QK_SMALL
}

}  // namespace

int fold_partials(const GView& g, const LdsShape& L, int32_t wgs, bool real, uint32_t fields, hipStream_t s) {
    const int T = L.H + 2;
    const unsigned grid = (unsigned)((T + kFoldSlots - 1) / kFoldSlots);
#define QK_FOLD(KW, REAL) k_gb_fold<KW, REAL><<<grid, kFoldBlock, 0, s>>>(g, L.part, T, wgs, fields)
    if (g.kw == 1) {
        if (real) QK_FOLD(1, true); else QK_FOLD(1, false);
    } else {
        if (real) QK_FOLD(2, true); else QK_FOLD(2, false);  // entries are slots, whatever the key's width
    }
#undef QK_FOLD
    QK_HIP(hipGetLastError());
    return QK_SUCCESS;
}

bool small_supported(const KeySpec& ks, const KeyCols& kc, int mode, int64_t n, const LdsShape& L) {
    return L.all && stream_keys(ks, kc) && (mode == 0 || mode == 3 || mode == 4) && n <= kStreamMaxRows;
}

int small_rows(const GView& g, const KeySpec& ks, const KeyCols& kc, int vtype, const void* vals,
               const uint64_t* vnull, const PredSet& ps, int mode, int64_t n, uint32_t fields, const LdsShape& L,
               hipStream_t s) {
    if (!vals) return launch_small_k<NoValue>(mode, g, ks, kc, vals, vnull, ps, n, fields, L, s);
    switch (vtype) {
    case QK_INT: return launch_small_k<int32_t>(mode, g, ks, kc, vals, vnull, ps, n, fields, L, s);
    case QK_LONG: return launch_small_k<int64_t>(mode, g, ks, kc, vals, vnull, ps, n, fields, L, s);
    case QK_FLOAT: return launch_small_k<float>(mode, g, ks, kc, vals, vnull, ps, n, fields, L, s);
    default: return launch_small_k<double>(mode, g, ks, kc, vals, vnull, ps, n, fields, L, s);
    }
}

}  // namespace qk
