// reconstruct.hip - prefix sums and stream compaction.
//
// Counterparts of GPUReconstruct (QueryEngine/GPUCore/GPUReconstruct.cuh:29-71, :203-355,
// :486-624; GPUReconstruct.cu:8-43, :756-764).  The reference scans the mask with CUB and
// recomputes that scan for every compacted column; here the prefix sum is our own single-pass
// decoupled look-back (lookback.hpp), and compaction runs in two passes: the first turns the mask
// or the predicates into one bit per row and a count per tile, the second moves the kept rows of
// every column with offsets it takes from the bits and the counts.  The exact output size is
// needed between the two anyway, and no workgroup of the second waits for another.
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "lookback.hpp"
#include "pred.hpp"

namespace qk {

namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;                        // int8 items per thread
constexpr int kScanTile = kScanBlock * kScanItems;    // 4096 rows per tile

constexpr int kCBlock = 256;
constexpr int kMaxCols = 8;

// ---- inclusive / exclusive prefix sum of int8 values -> int32 ---------------------------
__global__ void __launch_bounds__(kScanBlock) k_scan_mask(const int8_t* __restrict__ mask,
                                                          int32_t* __restrict__ out, int64_t n,
                                                          int inclusive, uint64_t* status,
                                                          uint32_t* ticket, uint32_t epoch,
                                                          int64_t tiles) {
    __shared__ int64_t s_tile;
    __shared__ int32_t s_wave[kScanBlock / 64];
    __shared__ uint32_t s_excl;
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    if (t == 0) s_tile = lb_ticket(ticket, tiles);
    __syncthreads();
    const int64_t tile = s_tile;
    const int64_t r0 = tile * kScanTile + (int64_t)t * kScanItems;

    int32_t m[kScanItems];
    if (r0 + kScanItems <= n && (((uintptr_t)(mask + r0)) & 15u) == 0) {
        int4 v = *reinterpret_cast<const int4*>(mask + r0);
        const int8_t* b = reinterpret_cast<const int8_t*>(&v);
#pragma unroll
        for (int k = 0; k < kScanItems; k++) m[k] = b[k];
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++) m[k] = (r0 + k < n) ? mask[r0 + k] : 0;
    }
    int32_t tsum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) tsum += m[k];

    const int32_t incl = wave_incl_scan(tsum, lane);
    if (lane == 63) s_wave[wid] = incl;
    __syncthreads();
    int32_t woff = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / 64; w++) {
        if (w < wid) woff += s_wave[w];
        agg += s_wave[w];
    }
    if (wid == 0) {
        uint32_t e = lb_exclusive(status, epoch, tile, (uint32_t)agg);
        if (lane == 0) s_excl = e;
    }
    __syncthreads();
    int32_t run = (int32_t)s_excl + woff + (incl - tsum);
    int32_t o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        if (inclusive) {
            run += m[k];
            o[k] = run;
        } else {
            o[k] = run;
            run += m[k];
        }
    }
    if (r0 + kScanItems <= n && (((uintptr_t)(out + r0)) & 15u) == 0) {
#pragma unroll
        for (int q = 0; q < kScanItems / 4; q++)
            reinterpret_cast<int4*>(out + r0)[q] = make_int4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++)
            if (r0 + k < n) out[r0 + k] = o[k];
    }
}

// ---- reductions over a mask ------------------------------------------------------------
// Sum of the int8 values.
__global__ void __launch_bounds__(256) k_mask_reduce(const int8_t* __restrict__ mask, int64_t n,
                                                     unsigned long long* __restrict__ out) {
    __shared__ int64_t s_part[4];
    int64_t acc = 0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t vecs = n >> 4;
    const bool aligned = (((uintptr_t)mask) & 15u) == 0;
    if (aligned) {
        for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < vecs; v += stride) {
            int4 x = reinterpret_cast<const int4*>(mask)[v];
            const int8_t* b = reinterpret_cast<const int8_t*>(&x);
#pragma unroll
            for (int k = 0; k < 16; k++) acc += (int64_t)b[k];
        }
    }
    for (int64_t r = (aligned ? vecs * 16 : 0) + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
         r < n; r += stride)
        acc += (int64_t)mask[r];
    acc = wave_sum64(acc);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t s = s_part[0] + s_part[1] + s_part[2] + s_part[3];
        if (s) atomicAdd(out, (unsigned long long)s);
    }
}

// ---- stable compaction -------------------------------------------------------------------
//
// A wavefront holds 64 * STEPS consecutive rows, a tile is a workgroup's 256 * STEPS: STEPS is 16 for
// large inputs and 4 where those would leave most of the chip idle.

constexpr int kBigSteps = 16, kSmallSteps = 4;
constexpr int64_t kSmallRows = (int64_t)1 << 21;
// Up to so many tiles, every workgroup of the second pass adds the counts before its own tile up by
// itself, and the host their total; past that a kernel scans them.
constexpr int64_t kSelfScanTiles = 2048;

struct CompactCols {
    int32_t ncols;
    int32_t esize[kMaxCols];
    const void* in[kMaxCols];
    const uint64_t* in_null[kMaxCols];
    void* out[kMaxCols];
    uint64_t* out_null[kMaxCols];
};

// Null masks of n rows to be cleared.
struct NullMasks {
    int32_t n;
    uint64_t* m[kMaxCols];
};

// Bit per byte of 4 mask bytes: byte i non-zero -> bit i.
__device__ __forceinline__ uint32_t nonzero4(uint32_t x) {
    const uint32_t y = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u) >> 7;
    return (y | (y >> 7) | (y >> 14) | (y >> 21)) & 0xfu;
}

// Sum over the 4 wavefronts of a 256-thread workgroup of a value every lane of a wavefront holds.
__device__ __forceinline__ int32_t wg_sum4(int32_t v, int32_t* s_part) {
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    return s_part[0] + s_part[1] + s_part[2] + s_part[3];
}

// First pass over an int8 mask: each lane turns 16 mask bytes into 16 bits (a wavefront 1024 rows),
// so the pass reads 16 bytes per lane and load.  TILE 4096: one count per workgroup, TILE 1024: one
// per wavefront.
template <int TILE>
__global__ void __launch_bounds__(kCBlock) k_keep_mask(const int8_t* __restrict__ mask, int64_t n,
                                                       uint64_t* __restrict__ bits, int32_t* __restrict__ counts) {
    __shared__ int32_t s_part[kCBlock / 64];
    const int64_t lane16 = (int64_t)blockIdx.x * kCBlock + threadIdx.x;
    const int64_t r0 = lane16 * 16;
    uint32_t b = 0;
    if (r0 + 16 <= n && (((uintptr_t)mask) & 15u) == 0) {
        const int4 v = *reinterpret_cast<const int4*>(mask + r0);
        b = nonzero4((uint32_t)v.x) | nonzero4((uint32_t)v.y) << 4 | nonzero4((uint32_t)v.z) << 8 |
            nonzero4((uint32_t)v.w) << 12;
    } else {
        for (int k = 0; k < 16; k++)
            if (r0 + k < n && mask[r0 + k]) b |= 1u << k;
    }
    if (r0 < ((n + 63) & ~(int64_t)63)) reinterpret_cast<uint16_t*>(bits)[lane16] = (uint16_t)b;
    int32_t c = __popc(b);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
    if (TILE == 1024) {
        if ((threadIdx.x & 63) == 0 && r0 < n) counts[r0 / 1024] = c;
    } else {
        c = wg_sum4(c, s_part);
        if (threadIdx.x == 0) counts[blockIdx.x] = c;
    }
}

template <typename T, int STEPS>
__device__ __forceinline__ uint32_t rows_in_range(const RangeCol& c, int64_t r0, int64_t n) {
    T v[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; k++)
        v[k] = __builtin_nontemporal_load((const T*)c.col + min(r0 + k * 64, n - 1));
    uint32_t ok = 0;
#pragma unroll
    for (int k = 0; k < STEPS; k++) ok |= (in_range<T>(c.vr, v[k]) ? 1u : 0u) << k;
    return ok;
}

// First pass over predicates: row k * 64 + lane of the wavefront is bit k of `ok` while the columns are
// tested one after the other, a column's loads all in flight together; ballots then make the words.
// The outputs' null masks are cleared on the way (a fill of their own each took 4.7 us and its launch
// at 30M rows).
template <int STEPS>
__global__ void __launch_bounds__(kCBlock) k_keep_preds(RangeSet rs, PredSet preds, NullMasks clear, int64_t n,
                                                        uint64_t* __restrict__ bits, int32_t* __restrict__ counts) {
    __shared__ int32_t s_part[kCBlock / 64];
    const int lane = threadIdx.x & 63;
    const int64_t word0 = ((int64_t)blockIdx.x * (kCBlock / 64) + (threadIdx.x >> 6)) * STEPS;
    const int64_t nwords = (n + 63) >> 6;
    const int64_t r0 = word0 * 64 + lane;
    uint32_t ok = 0;
#pragma unroll
    for (int k = 0; k < STEPS; k++) ok |= (r0 + k * 64 < n ? 1u : 0u) << k;
    for (int i = 0; i < rs.n; i++) {
        const RangeCol& c = rs.c[i];
        if (c.nm) {
#pragma unroll
            for (int k = 0; k < STEPS; k++)
                ok &= ~((uint32_t)((c.nm[min(word0 + k, nwords - 1)] >> lane) & 1ull) << k);
        }
        switch (c.type) {
        case QK_INT8: ok &= rows_in_range<int8_t, STEPS>(c, r0, n); break;
        case QK_INT: ok &= rows_in_range<int32_t, STEPS>(c, r0, n); break;
        case QK_LONG: ok &= rows_in_range<int64_t, STEPS>(c, r0, n); break;
        case QK_FLOAT: ok &= rows_in_range<float, STEPS>(c, r0, n); break;
        default: ok &= rows_in_range<double, STEPS>(c, r0, n); break;
        }
    }
    for (int p = 0; p < preds.n; p++)
        for (int k = 0; k < STEPS; k++)
            if ((ok >> k) & 1u) ok &= ~((uint32_t)!eval_pred(preds.p[p], r0 + k * 64) << k);
    uint64_t word = 0;
    int32_t c = 0;
#pragma unroll
    for (int k = 0; k < STEPS; k++) {
        const uint64_t b = __ballot((ok >> k) & 1u);
        if (lane == k) word = b;
        c += __popcll(b);
    }
    if (lane < STEPS && word0 + lane < nwords) {
        bits[word0 + lane] = word;
        for (int i = 0; i < clear.n; i++) clear.m[i][word0 + lane] = 0;
    }
    c = wg_sum4(c, s_part);
    if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

// Exclusive prefix of the tiles' counts in place; *total gets their sum.  One workgroup.
__global__ void __launch_bounds__(1024) k_scan_counts(int32_t* counts, int64_t tiles, int32_t* total) {
    __shared__ int32_t s_wave[16];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    int32_t carry = 0;
    constexpr int kPer = 16;  // counts per thread and round, as four 16-byte accesses
    for (int64_t base = 0; base < tiles; base += 1024 * kPer) {
        const int64_t i0 = base + (int64_t)t * kPer;
        int32_t v[kPer], sum = 0;
        if (i0 + kPer <= tiles) {
#pragma unroll
            for (int q = 0; q < kPer / 4; q++) {
                const int4 x = reinterpret_cast<const int4*>(counts + i0)[q];
                v[4 * q] = x.x;
                v[4 * q + 1] = x.y;
                v[4 * q + 2] = x.z;
                v[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < kPer; k++) v[k] = i0 + k < tiles ? counts[i0 + k] : 0;
        }
#pragma unroll
        for (int k = 0; k < kPer; k++) sum += v[k];
        const int32_t incl = wave_incl_scan(sum, lane);
        if (lane == 63) s_wave[wid] = incl;
        __syncthreads();
        int32_t run = carry + incl - sum, all = 0;
#pragma unroll
        for (int w = 0; w < 16; w++) {
            if (w < wid) run += s_wave[w];
            all += s_wave[w];
        }
        carry += all;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int32_t x = v[k];
            v[k] = run;
            run += x;
        }
        if (i0 + kPer <= tiles) {
#pragma unroll
            for (int q = 0; q < kPer / 4; q++)
                reinterpret_cast<int4*>(counts + i0)[q] = make_int4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        } else {
#pragma unroll
            for (int k = 0; k < kPer; k++)
                if (i0 + k < tiles) counts[i0 + k] = v[k];
        }
        __syncthreads();
    }
    if (t == 0) *total = carry;
}

__device__ __forceinline__ uint64_t lane_word(uint64_t v, int lane) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

// The kept rows of one column of a wavefront: every kept row's element is loaded before any is stored.
template <typename T, int STEPS>
__device__ __forceinline__ void move_rows(T* __restrict__ out, const T* __restrict__ in, int64_t r0, uint32_t keep,
                                          const int64_t (&pos)[STEPS]) {
    T v[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; k++)
        if ((keep >> k) & 1u) v[k] = __builtin_nontemporal_load(in + r0 + k * 64);
#pragma unroll
    for (int k = 0; k < STEPS; k++)
        if ((keep >> k) & 1u) out[pos[k]] = v[k];
}

enum CompactOut { kColumns = 0, kIndex32 = 1, kIndex64 = 2 };

// Second pass: the kept rows of a tile go to [base, base + count) of every output.  SELF: `counts` are
// plain counts, and the tile adds the ones before it up; otherwise they are already offsets.
template <int OUT, int STEPS, bool SELF>
__global__ void __launch_bounds__(kCBlock) k_compact(const uint64_t* __restrict__ bits,
                                                     const int32_t* __restrict__ counts, CompactCols cols, int64_t n) {
    constexpr int W = kCBlock / 64;
    __shared__ int32_t s_part[W], s_cnt[W];
    __shared__ unsigned long long s_null[W * STEPS + 2];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    const int64_t tile = blockIdx.x;
    int32_t base = 0;
    if (SELF) {
        for (int64_t i = t; i < tile; i += kCBlock) base += counts[i];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) base += __shfl_xor(base, d, 64);
        base = wg_sum4(base, s_part);
    } else {
        base = counts[tile];
    }
    // lane k < STEPS holds word k of the wavefront and the kept rows before it
    const int64_t nwords = (n + 63) >> 6;
    const int64_t word0 = (tile * W + wid) * STEPS;
    const uint64_t word = (lane < STEPS && word0 + lane < nwords) ? bits[word0 + lane] : 0ull;
    const int32_t mine = __popcll(word);
    const int32_t incl = wave_incl_scan(mine, lane);
    if (lane == 63) s_cnt[wid] = incl;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
        if (w < wid) before += s_cnt[w];
        total += s_cnt[w];
    }
    const int32_t word_at = before + incl - mine;  // kept rows of the tile before word `lane`
    const uint64_t lt_mask = (1ull << lane) - 1;
    const int64_t r0 = word0 * 64 + lane;
    uint32_t keep = 0;
    int64_t pos[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; k++) {
        const uint64_t b = lane_word(word, k);
        keep |= (uint32_t)((b >> lane) & 1ull) << k;
        pos[k] = (int64_t)base + __builtin_amdgcn_readlane(word_at, k) + __popcll(b & lt_mask);
    }
    if (OUT != kColumns) {
#pragma unroll
        for (int k = 0; k < STEPS; k++) {
            if (!((keep >> k) & 1u)) continue;
            if (OUT == kIndex32) ((int32_t*)cols.out[0])[pos[k]] = (int32_t)(r0 + k * 64);
            else ((int64_t*)cols.out[0])[pos[k]] = r0 + k * 64;
        }
        return;
    }
    for (int c = 0; c < cols.ncols; c++) {
        switch (cols.esize[c]) {
        case 1: move_rows<int8_t, STEPS>((int8_t*)cols.out[c], (const int8_t*)cols.in[c], r0, keep, pos); break;
        case 2: move_rows<int16_t, STEPS>((int16_t*)cols.out[c], (const int16_t*)cols.in[c], r0, keep, pos); break;
        case 4: move_rows<int32_t, STEPS>((int32_t*)cols.out[c], (const int32_t*)cols.in[c], r0, keep, pos); break;
        default: move_rows<int64_t, STEPS>((int64_t*)cols.out[c], (const int64_t*)cols.in[c], r0, keep, pos); break;
        }
        if (!(cols.out_null[c] && cols.in_null[c])) continue;
        // null bits: lane k packs word k's kept bits together and ORs them into the tile's output
        // words in LDS; words inside the tile's range are then stored, the two at its ends (shared
        // with the neighbouring tiles, and cleared by the caller) added with atomics
        const int shift = base & 63;
        const int words = (shift + total + 63) >> 6;
        __syncthreads();
        for (int w = t; w < words; w += kCBlock) s_null[w] = 0;
        __syncthreads();
        uint64_t m = lane < STEPS && word ? cols.in_null[c][word0 + lane] & word : 0ull;
        uint64_t packed = 0;
        while (m) {
            const int b = __builtin_ctzll(m);
            packed |= 1ull << __popcll(word & ((1ull << b) - 1));
            m &= m - 1;
        }
        if (packed) {
            const int at = shift + word_at, off = at & 63;
            atomicOr(&s_null[at >> 6], (unsigned long long)(packed << off));
            if (off && (packed >> (64 - off))) atomicOr(&s_null[(at >> 6) + 1], (unsigned long long)(packed >> (64 - off)));
        }
        __syncthreads();
        unsigned long long* dst = (unsigned long long*)cols.out_null[c] + (base >> 6);
        for (int w = t; w < words; w += kCBlock) {
            if (w > 0 && w < words - 1) dst[w] = s_null[w];
            else if (s_null[w]) atomicOr(dst + w, s_null[w]);
        }
    }
}

// ---- one byte per row -> bit mask -------------------------------------------------------
__global__ void __launch_bounds__(256) k_compress_null_mask(const uint8_t* __restrict__ in,
                                                            uint64_t* __restrict__ out, int64_t n) {
    const int lane = threadIdx.x & 63;
    const int64_t words = (n + 63) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; w < words; w += nwaves) {
        const int64_t r = (w << 6) + lane;
        const uint64_t b = __ballot(r < n && (in[r] & 1u));
        if (lane == 0) out[w] = b;
    }
}

int grid_stride_blocks(int64_t items, int per_block) {
    const DeviceInfo& d = device_info();
    int64_t g = (items + per_block - 1) / per_block;
    int64_t cap = (int64_t)(d.cus > 0 ? d.cus : 64) * 8;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

// One compaction of n rows: bits and counts live in the stream's second scratch, which the call keeps
// to itself until its last kernel is queued.
struct Compaction {
    uint64_t* bits = nullptr;
    int32_t* counts = nullptr;
    int32_t* total = nullptr;
    int64_t n = 0, tiles = 0, kept = 0;
    bool small = false, self = false;
    std::unique_lock<std::mutex> hold;

    int begin(int64_t rows, hipStream_t s) {
        n = rows;
        small = n < kSmallRows;
        const int64_t tile = kCBlock * (small ? kSmallSteps : kBigSteps);
        tiles = (n + tile - 1) / tile;
        self = tiles <= kSelfScanTiles;
        const size_t word_bytes = (size_t)((n + 63) / 64) * 8;
        Scratch* sc = nullptr;
        QK_TRY(stream_scratch(s, 0, &sc, 1));
        hold = std::unique_lock<std::mutex>(sc->mu);
        QK_TRY(stream_scratch(s, word_bytes + (size_t)(tiles + 8) * 4 + 64, &sc, 1));
        bits = (uint64_t*)sc->ptr;
        counts = (int32_t*)((char*)sc->ptr + (word_bytes + 63) / 64 * 64);
        total = counts + (tiles + 3) / 4 * 4;
        return QK_SUCCESS;
    }

    // After the first pass: scans the counts and reads the number of kept rows back.
    int count(hipStream_t s) {
        if (self) return read_back_sum(s, counts, (int32_t)tiles, &kept);
        k_scan_counts<<<1, 1024, 0, s>>>(counts, tiles, total);
        QK_HIP(hipGetLastError());
        int32_t all = 0;
        QK_TRY(read_back_one(s, total, &all));
        kept = all;
        return QK_SUCCESS;
    }

    int by_mask(const int8_t* mask, int64_t rows, hipStream_t s) {
        QK_TRY(begin(rows, s));
        const unsigned grid = (unsigned)((n + 4095) / 4096);
        if (small) k_keep_mask<1024><<<grid, kCBlock, 0, s>>>(mask, n, bits, counts);
        else k_keep_mask<4096><<<grid, kCBlock, 0, s>>>(mask, n, bits, counts);
        QK_HIP(hipGetLastError());
        return count(s);
    }

    int by_preds(const RangeSet& rs, const PredSet& rest, const NullMasks& clear, int64_t rows, hipStream_t s) {
        QK_TRY(begin(rows, s));
        if (small) k_keep_preds<kSmallSteps><<<(unsigned)tiles, kCBlock, 0, s>>>(rs, rest, clear, n, bits, counts);
        else k_keep_preds<kBigSteps><<<(unsigned)tiles, kCBlock, 0, s>>>(rs, rest, clear, n, bits, counts);
        QK_HIP(hipGetLastError());
        return count(s);
    }

    template <int OUT>
    int move(const CompactCols& cols, hipStream_t s) {
        if (kept == 0) return QK_SUCCESS;
        const unsigned grid = (unsigned)tiles;
        if (small && self) k_compact<OUT, kSmallSteps, true><<<grid, kCBlock, 0, s>>>(bits, counts, cols, n);
        else if (small) k_compact<OUT, kSmallSteps, false><<<grid, kCBlock, 0, s>>>(bits, counts, cols, n);
        else if (self) k_compact<OUT, kBigSteps, true><<<grid, kCBlock, 0, s>>>(bits, counts, cols, n);
        else k_compact<OUT, kBigSteps, false><<<grid, kCBlock, 0, s>>>(bits, counts, cols, n);
        QK_HIP(hipGetLastError());
        return QK_SUCCESS;
    }
};

// ---- prefix sum without allocation ----------------------------------------------------------
// qk_prefix_sum_noalloc keeps its look-back state (ticket word + one status word per
// 4096-row tile) in this fixed array instead of the per-stream scratch, so the call never
// allocates.  Each device holds its own copy until the process ends; host code reaches it only
// through the address hipGetSymbolAddress returns for the current device.
constexpr int64_t kNoAllocMaxRows = (int64_t)1 << 30;
constexpr int64_t kNoAllocTiles = kNoAllocMaxRows / kScanTile;
constexpr size_t kNoAllocWords = kLbHeaderWords + kNoAllocTiles + 8;
static __device__ __align__(256) uint64_t scratch[kNoAllocWords];

struct NoAllocState {
    uint64_t* words = nullptr;  // device address of `scratch` on this device
    uint32_t epoch = 0;
};
std::mutex g_noalloc_mu;
std::map<int, NoAllocState> g_noalloc;

// Clears the ticket word before a launch (a kernel rather than a memset node, so the call can
// be captured into a graph).
__global__ void k_noalloc_arm(uint64_t* words) {
    if (threadIdx.x < kLbHeaderWords) words[threadIdx.x] = 0;
}

__global__ void k_noalloc_clear(uint64_t* words, size_t nwords) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += stride) words[i] = 0;
}

// Resolves this device's copy of `scratch` and clears it, once per device (the first call on
// the device; it synchronises the device, so that call should not be made under capture).
int noalloc_state(NoAllocState** out) {
    int dev = 0;
    QK_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    NoAllocState& st = g_noalloc[dev];
    if (!st.words) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(QK_RUNTIME_ERROR, "prefix_sum_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
        k_noalloc_clear<<<256, 256>>>((uint64_t*)p, kNoAllocWords);
        QK_HIP(hipGetLastError());
        QK_HIP(hipDeviceSynchronize());
        st.words = (uint64_t*)p;
    }
    *out = &st;
    return QK_SUCCESS;
}

}  // namespace

int prefix_noalloc_setup() {
    NoAllocState* st = nullptr;
    return noalloc_state(&st);
}

}  // namespace qk

using namespace qk;

extern "C" {

int qk_prefix_sum(const int8_t* mask, int32_t n, int32_t* out, int32_t inclusive, void* stream) {
    QK_TRY(ensure_init());
    if (n <= 0) return QK_SUCCESS;
    if (!mask || !out) return fail(QK_ERROR, "prefix_sum: null buffer");
    hipStream_t s = as_stream(stream);
    const int64_t tiles = ((int64_t)n + kScanTile - 1) / kScanTile;
    Scratch* sc = nullptr;
    QK_TRY(stream_scratch(s, lb_scratch_bytes(tiles), &sc));
    uint64_t* words = (uint64_t*)sc->ptr;
    const uint32_t epoch = ++sc->epoch;
    k_scan_mask<<<(unsigned)tiles, kScanBlock, 0, s>>>(mask, out, n, inclusive ? 1 : 0,
                                                       words + kLbHeaderWords, (uint32_t*)words,
                                                       epoch, tiles);
    QK_HIP(hipGetLastError());
    return QK_SUCCESS;
}

int qk_prefix_sum_noalloc(const int8_t* mask, int32_t n, int32_t* out, int32_t inclusive, void* stream) {
    QK_TRY(ensure_init());
    if (n <= 0) return QK_SUCCESS;
    if (!mask || !out) return fail(QK_ERROR, "prefix_sum_noalloc: null buffer");
    if ((int64_t)n > kNoAllocMaxRows)
        return fail(QK_ERROR, "prefix_sum_noalloc: %d rows exceed the fixed scratch's maximum of %lld rows",
                    n, (long long)kNoAllocMaxRows);
    NoAllocState* st = nullptr;
    QK_TRY(noalloc_state(&st));
    uint32_t epoch;
    {
        std::lock_guard<std::mutex> lk(g_noalloc_mu);
        epoch = ++st->epoch;
    }
    hipStream_t s = as_stream(stream);
    const int64_t tiles = ((int64_t)n + kScanTile - 1) / kScanTile;
    k_noalloc_arm<<<1, 64, 0, s>>>(st->words);
    QK_HIP(hipGetLastError());
    k_scan_mask<<<(unsigned)tiles, kScanBlock, 0, s>>>(mask, out, n, inclusive ? 1 : 0,
                                                       st->words + kLbHeaderWords, (uint32_t*)st->words,
                                                       epoch, tiles);
    QK_HIP(hipGetLastError());
    return QK_SUCCESS;
}

int qk_mask_sum(const int8_t* mask, int32_t n, int64_t* out_host, void* stream) {
    QK_TRY(ensure_init());
    if (!out_host) return fail(QK_ERROR, "mask_sum: null output");
    *out_host = 0;
    if (n <= 0) return QK_SUCCESS;
    if (!mask) return fail(QK_ERROR, "mask_sum: null mask");
    hipStream_t s = as_stream(stream);
    Scratch* sc = nullptr;
    QK_TRY(stream_scratch(s, 64, &sc));
    unsigned long long* ctr = (unsigned long long*)sc->ptr + 7;
    QK_HIP(hipMemsetAsync(ctr, 0, 8, s));
    k_mask_reduce<<<grid_stride_blocks(((int64_t)n + 15) / 16, 256), 256, 0, s>>>(mask, n, ctr);
    QK_HIP(hipGetLastError());
    return read_back_one(s, (const int64_t*)ctr, out_host);
}

int qk_reconstruct_col_keep(int32_t elem_size, const void* in, const int8_t* mask, int32_t n,
                            const uint64_t* in_null, void** out, int32_t* out_count,
                            uint64_t** out_null, void* stream) {
    QK_TRY(ensure_init());
    if (!out || !out_count) return fail(QK_ERROR, "reconstruct_col_keep: null output");
    if (elem_size != 1 && elem_size != 2 && elem_size != 4 && elem_size != 8)
        return fail(QK_ERROR, "reconstruct_col_keep: element size %d unsupported", elem_size);
    if (n <= 0) {  // GPUReconstruct.cuh:330-338
        *out = nullptr;
        *out_count = 0;
        if (out_null) *out_null = nullptr;
        return QK_SUCCESS;
    }
    if (!mask) {  // aliasing, no ownership transfer (GPUReconstruct.cuh:320-328)
        *out = const_cast<void*>(in);
        *out_count = n;
        if (out_null) *out_null = const_cast<uint64_t*>(in_null);
        return QK_SUCCESS;
    }
    if (!in) return fail(QK_ERROR, "reconstruct_col_keep: null input");
    hipStream_t s = as_stream(stream);
    Compaction cp;
    QK_TRY(cp.by_mask(mask, n, s));
    const int64_t kept = cp.kept;
    *out_count = (int32_t)kept;
    if (kept == 0) {  // GPUReconstruct.cuh:311-318
        *out = nullptr;
        if (out_null) *out_null = nullptr;
        return QK_SUCCESS;
    }
    void* o = nullptr;
    uint64_t* on = nullptr;
    QK_TRY(pool_alloc(&o, (size_t)kept * elem_size));
    const bool want_null = out_null && in_null;
    if (want_null) {
        int st = pool_alloc((void**)&on, (size_t)((kept + 63) / 64) * 8);
        if (st != QK_SUCCESS) {
            pool_free(o);
            return st;
        }
        QK_HIP(hipMemsetAsync(on, 0, (size_t)((kept + 63) / 64) * 8, s));
    }
    CompactCols cols{};
    cols.ncols = 1;
    cols.esize[0] = elem_size;
    cols.in[0] = in;
    cols.in_null[0] = want_null ? in_null : nullptr;
    cols.out[0] = o;
    cols.out_null[0] = on;
    int st = cp.move<kColumns>(cols, s);
    if (st != QK_SUCCESS) {
        pool_free(o);
        pool_free(on);
        return st;
    }
    *out = o;
    if (out_null) *out_null = on;
    return QK_SUCCESS;
}

int qk_generate_indexes_keep(const int8_t* mask, int32_t n, int32_t index_size, void** out,
                             int32_t* out_count, void* stream) {
    QK_TRY(ensure_init());
    if (!out || !out_count) return fail(QK_ERROR, "generate_indexes: null output");
    if (!mask) return fail(QK_ERROR, "inMask cannot be nullptr in GenerateIndexes");  // :558-562
    if (index_size != 4 && index_size != 8)
        return fail(QK_ERROR, "generate_indexes: index size must be 4 or 8");
    *out = nullptr;
    *out_count = 0;
    if (n <= 0) return QK_SUCCESS;
    hipStream_t s = as_stream(stream);
    Compaction cp;
    QK_TRY(cp.by_mask(mask, n, s));
    const int64_t kept = cp.kept;
    *out_count = (int32_t)kept;
    if (kept == 0) return QK_SUCCESS;
    void* o = nullptr;
    QK_TRY(pool_alloc(&o, (size_t)kept * index_size));
    CompactCols cols{};
    cols.ncols = 1;
    cols.out[0] = o;
    int st = index_size == 4 ? cp.move<kIndex32>(cols, s) : cp.move<kIndex64>(cols, s);
    if (st != QK_SUCCESS) {
        pool_free(o);
        return st;
    }
    *out = o;
    return QK_SUCCESS;
}

int qk_compress_null_mask(const uint8_t* in, int32_t n, uint64_t** out, void* stream) {
    QK_TRY(ensure_init());
    if (!out) return fail(QK_ERROR, "compress_null_mask: null output");
    *out = nullptr;
    if (n <= 0) return QK_SUCCESS;
    if (!in) return fail(QK_ERROR, "compress_null_mask: null input");
    const int64_t words = ((int64_t)n + 63) / 64;
    uint64_t* o = nullptr;
    QK_TRY(pool_alloc((void**)&o, (size_t)words * 8));
    hipStream_t s = as_stream(stream);
    k_compress_null_mask<<<grid_stride_blocks(words, 4), 256, 0, s>>>(in, o, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        pool_free(o);
        return fail(QK_RUNTIME_ERROR, "compress_null_mask launch: %s", hipGetErrorString(e));
    }
    *out = o;
    return QK_SUCCESS;
}

int qk_where_compact(int32_t npreds, const qk_predicate* preds, int32_t ncols,
                     const int32_t* elem_sizes, const void* const* cols, const uint64_t* const* col_nulls,
                     int32_t n, void* const* outs, uint64_t* const* out_nulls, int32_t* out_count,
                     void* stream) {
    QK_TRY(ensure_init());
    if (!out_count) return fail(QK_ERROR, "where_compact: null count output");
    *out_count = 0;
    if (ncols < 0 || ncols > kMaxCols) return fail(QK_ERROR, "where_compact: at most %d columns", kMaxCols);
    PredSet ps{};
    QK_TRY(check_preds(npreds, preds, &ps));
    if (n <= 0) return QK_SUCCESS;
    CompactCols cc{};
    cc.ncols = ncols;
    for (int c = 0; c < ncols; c++) {
        const int es = elem_sizes[c];
        if (es != 1 && es != 2 && es != 4 && es != 8)
            return fail(QK_ERROR, "where_compact: element size %d unsupported", es);
        if (!cols[c] || !outs[c]) return fail(QK_ERROR, "where_compact: null column %d", c);
        cc.esize[c] = es;
        cc.in[c] = cols[c];
        cc.in_null[c] = col_nulls ? col_nulls[c] : nullptr;
        cc.out[c] = outs[c];
        cc.out_null[c] = (out_nulls && cc.in_null[c]) ? out_nulls[c] : nullptr;
    }
    hipStream_t s = as_stream(stream);
    NullMasks clear{};
    for (int c = 0; c < ncols; c++)
        if (cc.out_null[c]) clear.m[clear.n++] = cc.out_null[c];
    RangeSet rs{};
    PredSet rest{};
    fold_columns(ps, &rs, &rest);
    Compaction cp;
    QK_TRY(cp.by_preds(rs, rest, clear, n, s));
    *out_count = (int32_t)cp.kept;
    return cp.move<kColumns>(cc, s);
}

}  // extern "C"
