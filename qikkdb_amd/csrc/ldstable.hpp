// ldstable.hpp - the hash table that a workgroup of the row kernels keeps in LDS, and the way from the
// workgroups' tables to the global one.
#pragma once

#include "groupby.hpp"

namespace qk {

constexpr int kLdsProbes = 8;    // LDS probe limit before a row goes to the global table

// ---- LDS table of the one-pass kernel ----------------------------------------------------
// Arrays of H hashed slots + 2 side slots (NULL key, key == kEmpty).  Every state is kept in
// 2^rbits copies, a lane adding to the copy of its number: with few groups the lanes of a wave
// would otherwise queue at the same LDS words (ten groups, 66.7M rows: 331 us with one copy).
// A multi-word key's entry holds its slot in the global table instead of the key.
struct Lds {
    uint64_t* key;
    uint64_t* sum;
    uint64_t* mn;
    uint64_t* mx;
    uint32_t* cnt;
    uint32_t* cntall;
    int32_t H, rbits;
};

constexpr int kMaxCopyBits = 5;

// Bytes of one copy of a slot's states; a slot takes 8 more for its key.
__host__ __device__ __forceinline__ int lds_state_bytes(uint32_t fields) {
    return 4 + ((fields & F_CNTALL) ? 4 : 0) + ((fields & F_SUM) ? 8 : 0) + ((fields & F_MIN) ? 8 : 0) +
           ((fields & F_MAX) ? 8 : 0);
}
__host__ __device__ __forceinline__ size_t lds_table_bytes(int32_t H, int32_t rbits, uint32_t fields) {
    return (size_t)(H + 2) * (8 + ((size_t)lds_state_bytes(fields) << rbits));
}

__device__ __forceinline__ Lds lds_carve(void* base, int32_t H, int32_t rbits, uint32_t fields) {
    Lds t;
    const size_t T = (size_t)(H + 2) << rbits;
    char* p = (char*)base;
    t.key = (uint64_t*)p; p += (size_t)(H + 2) * 8;
    t.sum = (fields & F_SUM) ? (uint64_t*)p : nullptr; p += (fields & F_SUM) ? T * 8 : 0;
    t.mn = (fields & F_MIN) ? (uint64_t*)p : nullptr; p += (fields & F_MIN) ? T * 8 : 0;
    t.mx = (fields & F_MAX) ? (uint64_t*)p : nullptr; p += (fields & F_MAX) ? T * 8 : 0;
    t.cnt = (uint32_t*)p; p += T * 4;
    t.cntall = (fields & F_CNTALL) ? (uint32_t*)p : nullptr;
    t.H = H;
    t.rbits = rbits;
    return t;
}

// Slot of a key from slot s on (inserting it when absent); -1 after kLdsProbes slots.
__device__ __forceinline__ int lds_probe(const Lds& t, uint64_t key, uint32_t s) {
#pragma unroll 1
    for (int p = 0; p < kLdsProbes; p++) {
        uint64_t cur = __hip_atomic_load(&t.key[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == key) return (int)s;
        if (cur == kEmpty) {
            unsigned long long old = atomicCAS((unsigned long long*)&t.key[s], (unsigned long long)kEmpty,
                                               (unsigned long long)key);
            if (old == kEmpty || old == key) return (int)s;
        }
        s = (s + 1 == (uint32_t)t.H) ? 0u : s + 1;
    }
    return -1;
}

// The side slot of the NULL key (side 0) or of the key equal to kEmpty (side 1), marked as used.
__device__ __forceinline__ int lds_side(const Lds& t, int side) {
    if (t.key[t.H + side] == 0ull) t.key[t.H + side] = 1ull;
    return t.H + side;
}

__device__ __forceinline__ int lds_find(const Lds& t, uint64_t key, bool knull, uint64_t h) {
    if (knull) return lds_side(t, 0);
    if (key == kEmpty) return lds_side(t, 1);
    return lds_probe(t, key, (uint32_t)(((h >> 32) * (uint64_t)(uint32_t)t.H) >> 32));
}

// Clears the table (every thread of the workgroup; the caller synchronises).
__device__ __forceinline__ void lds_clear(const Lds& t) {
    for (int s = threadIdx.x; s < t.H + 2; s += blockDim.x) t.key[s] = s < t.H ? kEmpty : 0ull;
    for (int e = threadIdx.x; e < (t.H + 2) << t.rbits; e += blockDim.x) {
        t.cnt[e] = 0;
        if (t.cntall) t.cntall[e] = 0;
        if (t.sum) t.sum[e] = 0;
        if (t.mn) t.mn[e] = ~0ull;
        if (t.mx) t.mx[e] = 0ull;
    }
}

// Adds one row to entry e = (slot << rbits) | copy.
template <bool REAL>
__device__ __forceinline__ void lds_accum(const Lds& t, int e, const Part& p, uint32_t fields) {
    if (p.cnt) atomicAdd(&t.cnt[e], (uint32_t)p.cnt);
    if (fields & F_CNTALL) atomicAdd(&t.cntall[e], (uint32_t)p.cntall);
    if (p.cnt) {
        if (fields & F_SUM) {
            if (REAL)
                atomicAdd((double*)&t.sum[e], __longlong_as_double((long long)p.sum));
            else
                atomicAdd((unsigned long long*)&t.sum[e], (unsigned long long)p.sum);
        }
        if (fields & F_MIN) atomicMin((unsigned long long*)&t.mn[e], (unsigned long long)p.mn);
        if (fields & F_MAX) atomicMax((unsigned long long*)&t.mx[e], (unsigned long long)p.mx);
    }
}

template <bool REAL>
__device__ __forceinline__ void merge_part(Part& a, const Part& b) {
    a.cnt += b.cnt;
    a.cntall += b.cntall;
    if (REAL)
        a.sum = (uint64_t)__double_as_longlong(__longlong_as_double((long long)a.sum) + __longlong_as_double((long long)b.sum));
    else
        a.sum += b.sum;
    a.mn = min(a.mn, b.mn);
    a.mx = max(a.mx, b.mx);
}

// The copies of slot s folded into one partial, from copy `first` on (the lanes of a wave start at
// different copies, so that their reads fall on different banks).
template <bool REAL>
__device__ __forceinline__ Part lds_fold(const Lds& t, int s, int first) {
    Part p;
    p.cnt = p.cntall = p.sum = p.mx = 0;
    p.mn = ~0ull;
    double d = 0.0;
    const int R = 1 << t.rbits;
    for (int i = 0; i < R; i++) {
        const int e = (s << t.rbits) | ((first + i) & (R - 1));
        p.cnt += t.cnt[e];
        if (t.cntall) p.cntall += t.cntall[e];
        if (t.sum) {
            if (REAL) d += __longlong_as_double((long long)t.sum[e]); else p.sum += t.sum[e];
        }
        if (t.mn) p.mn = min(p.mn, t.mn[e]);
        if (t.mx) p.mx = max(p.mx, t.mx[e]);
    }
    if (REAL) p.sum = (uint64_t)__double_as_longlong(d);
    return p;
}

// Merges one LDS entry (its key or, of a multi-word key, its global slot; side 0 and 1: the entries of
// the NULL key and of the key equal to kEmpty) into the global table.  READ as in g_accum_atomic.
template <int KW, bool READ>
__device__ __forceinline__ void add_entry(const GView& g, uint64_t k, int side, const Part& p, uint32_t fields,
                                          unsigned int* s_new) {
    bool is_new = false;
    int64_t gs;
    if (KW > 1) {
        gs = (int64_t)k;
    } else if (side == 0) {
        gs = g_slot1(g, 0ull, true, 0, &is_new);
    } else if (side == 1) {
        gs = g_slot1(g, kEmpty, false, 0, &is_new);
    } else {
        gs = g_slot1(g, k, false, hash64(k), &is_new);
    }
    if (is_new) atomicAdd(s_new, 1u);
    if (gs >= 0) g_accum_atomic<READ>(g, gs, p, fields); else g_set_lost(g);
}

// The workgroups' LDS tables in global memory: arrays [workgroup][H + 2] of keys (kEmpty: no entry)
// and of the states the table keeps.
struct Partials {
    uint64_t *key, *cnt, *cntall, *sum, *mn, *mx;
};

// The end of a row kernel's workgroup: its table to `out`, or, without one, into the global table.
template <int KW, bool REAL>
__device__ __forceinline__ void lds_flush(const Lds& t, const GView& g, const Partials& out, uint32_t fields,
                                          unsigned int* s_new) {
    for (int s = threadIdx.x; s < t.H + 2; s += blockDim.x) {
        const uint64_t k = t.key[s];
        const bool used = s < t.H ? k != kEmpty : k != 0ull;
        if (out.key) {
            const int64_t at = (int64_t)blockIdx.x * (t.H + 2) + s;
            out.key[at] = used ? k : kEmpty;
            if (used) {
                const Part p = lds_fold<REAL>(t, s, threadIdx.x);
                out.cnt[at] = p.cnt;
                if (t.cntall) out.cntall[at] = p.cntall;
                if (t.sum) out.sum[at] = p.sum;
                if (t.mn) out.mn[at] = p.mn;
                if (t.mx) out.mx[at] = p.mx;
            }
        } else if (used) {
            add_entry<KW, true>(g, k, s - t.H, lds_fold<REAL>(t, s, threadIdx.x), fields, s_new);
        }
    }
}

constexpr int64_t kMaxPartials = 512;  // workgroups whose tables k_gb_fold adds up
// Up to so many entries in all (workgroups x keys of the table) the workgroups merge their tables
// themselves: the atomics then take less than another launch does.
constexpr int64_t kDirectEntries = 32768;

// The one-pass kernel's LDS table: H slots (0: none) in 2^rbits copies.  all: it holds every key the
// table may; the workgroups' tables then go through `part` (null: straight to the global table), and
// a workgroup takes at least min_rows rows.  keys: those the table may hold.
struct LdsShape {
    int32_t H = 0, rbits = 0;
    bool all = false;
    int64_t min_rows = 0, keys = 0;
    Partials part{};

    // workgroups for n rows: min_rows each, but no fewer than 64 (82K rows, 651 groups of a wide key: 70 us
    // in 10 workgroups)
    int64_t wgs_for(int64_t n) const {
        const int64_t w = (n + min_rows - 1) / min_rows;
        return w < 64 ? 64 : (w > kMaxPartials ? kMaxPartials : w);
    }
    Partials for_wgs(int64_t wgs) const { return wgs * keys > kDirectEntries ? part : Partials{}; }
};

// Adds the tables that a row kernel's `wgs` workgroups left in L.part up into the global table.
int fold_partials(const GView& g, const LdsShape& L, int32_t wgs, bool real, uint32_t fields, hipStream_t s);

// The small-table kernel (smalltable.hip): whether it reads the block's columns, and its launch.
bool small_supported(const KeySpec& ks, const KeyCols& kc, int mode, int64_t n, const LdsShape& L);
int small_rows(const GView& g, const KeySpec& ks, const KeyCols& kc, int vtype, const void* vals,
               const uint64_t* vnull, const PredSet& ps, int mode, int64_t n, uint32_t fields, const LdsShape& L,
               hipStream_t s);

}  // namespace qk
