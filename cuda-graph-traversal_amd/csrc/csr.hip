// CSR construction from the tuple list and the isolated-vertex query.
// Reference: src/traversal.cu:15-73 (degree / rowstart / fill kernels),
// :342-410 (oned_graph_from_tuple_graph, oned_graph_is_vertex_isolated).
//
// Steps: (1) both directions of every non-loop tuple edge are put in row order,
// small lists through a degree histogram and per-row cursors, large ones by a
// partition in passes; (2) a three-phase exclusive scan of the row lengths
// gives u64 row offsets; (3) each row is sorted ascending by the key
// (f32 weight bits << 32 | column), which makes the CSR deterministic and puts
// light edges first in every row. Rows are sorted by a thread (<= 16 entries) or a wave (<= 512); longer ones are
// split by weight into bins that a wave sorts.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "common.hpp"

namespace g500 {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ u64 make_key(u32 col, f32 w) { return ((u64)__float_as_uint(w) << 32) | col; }

// Tuples with an endpoint >= n are skipped and flagged (the entry point then
// fails) instead of indexing out of bounds.
__global__ __launch_bounds__(256) void degree_kernel(const Packed_Edge *__restrict__ edges, u64 ne, u64 n,
                                                     u32 *__restrict__ deg, u32 *__restrict__ bad) {
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < ne; i += (u64)gridDim.x * blockDim.x) {
        Packed_Edge e = edges[i];
        if (e.v0 >= n || e.v1 >= n) {
            atomicOr(bad, 1u);
            continue;
        }
        if (e.v0 == e.v1) continue;
        atomicAdd(&deg[e.v0], 1u);
        atomicAdd(&deg[e.v1], 1u);
    }
}

// Exclusive scan over the block; *total receives the block sum.
template <int BLOCK>
__device__ __forceinline__ u64 block_exclusive_scan(u64 v, u64 *total) {
    __shared__ u64 wtot[BLOCK / kWave];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const u64 x = wave_inclusive_scan(v);
    if (lane == kWave - 1) wtot[wave] = x;
    __syncthreads();
    if (wave == 0) {
        const u64 t = wave_inclusive_scan(lane < BLOCK / kWave ? wtot[lane] : (u64)0);
        if (lane < BLOCK / kWave) wtot[lane] = t;
    }
    __syncthreads();
    u64 before = wave ? wtot[wave - 1] : 0;
    *total = wtot[BLOCK / kWave - 1];
    __syncthreads();
    return before + x - v;
}

__global__ __launch_bounds__(kScanBlock) void scan_tile_sums(const u32 *__restrict__ deg, u64 n,
                                                             u64 *__restrict__ tile_sums) {
    const u64 base = (u64)blockIdx.x * kScanTile;
    u64 s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        u64 i = base + threadIdx.x + (u64)j * kScanBlock;
        if (i < n) s += deg[i];
    }
    u64 tot;
    block_exclusive_scan<kScanBlock>(s, &tot);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// Single block: exclusive scan of the tile sums in place; rowstarts[n] = total.
__global__ __launch_bounds__(1024) void scan_tile_offsets(u64 *__restrict__ tile_sums, u64 ntiles,
                                                          u64 *__restrict__ rowstarts, u64 n) {
    u64 carry = 0;
    for (u64 b = 0; b < ntiles; b += 1024) {
        u64 i = b + threadIdx.x;
        u64 v = i < ntiles ? tile_sums[i] : 0;
        u64 tot;
        u64 ex = block_exclusive_scan<1024>(v, &tot);
        if (i < ntiles) tile_sums[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) rowstarts[n] = carry;
}

__global__ __launch_bounds__(kScanBlock) void scan_write(const u32 *__restrict__ deg, u64 n,
                                                         const u64 *__restrict__ tile_off,
                                                         u64 *__restrict__ rowstarts) {
    const u64 base = (u64)blockIdx.x * kScanTile + (u64)threadIdx.x * kScanItems;
    u32 d[kScanItems];
    u64 s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        d[j] = base + j < n ? deg[base + j] : 0;
        s += d[j];
    }
    u64 tot;
    u64 run = tile_off[blockIdx.x] + block_exclusive_scan<kScanBlock>(s, &tot);
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        if (base + j < n) rowstarts[base + j] = run;
        run += d[j];
    }
}

__global__ __launch_bounds__(256) void fill_kernel(const Packed_Edge *__restrict__ edges,
                                                   const f32 *__restrict__ ew, u64 ne, u64 n,
                                                   const u64 *__restrict__ rowstarts,
                                                   u32 *__restrict__ cursor, u32 *__restrict__ col,
                                                   f32 *__restrict__ cw) {
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < ne; i += (u64)gridDim.x * blockDim.x) {
        Packed_Edge e = edges[i];
        if (e.v0 == e.v1 || e.v0 >= n || e.v1 >= n) continue;
        f32 w = ew[i];
        u64 p0 = rowstarts[e.v0] + atomicAdd(&cursor[e.v0], 1u);
        u64 p1 = rowstarts[e.v1] + atomicAdd(&cursor[e.v1], 1u);
        col[p0] = (u32)e.v1;
        cw[p0] = w;
        col[p1] = (u32)e.v0;
        cw[p1] = w;
    }
}

// ------------------------------------------------------- partition into rows
// Rows filled through cursors in tuple order (degree_kernel, fill_kernel) cost
// two random atomics and a random 8-byte write per entry: 34 ms of a 90 ms S23
// construction (7.9 ms now). Large tuple lists are instead split by row in two or three
// passes of at most kPartBins buckets per tile, high bits first: a block takes
// a tile of entries, ranks them per bucket in LDS, reserves one run per bucket
// with one atomic, and writes the runs from LDS in bucket order, so that
// neighbouring lanes write neighbouring entries. The last pass's buckets are
// the rows. Each pass is a histogram (4-8 bytes read per entry), a scan and a
// scatter (12 read, 12 or 8 written); order inside a bucket does not matter,
// the rows are sorted afterwards.
constexpr int kPartThreads = 1024, kPartItems = 8, kPartTile = kPartThreads * kPartItems;
constexpr u32 kPartBins = 2048;

struct PartArgs {
    const Packed_Edge *edges;  // pass 1: tuples (two entries each, loops dropped), else null
    const f32 *ew;
    const u32 *row_in, *col_in, *w_in;
    u64 count;                 // tuples or entries
    u64 n;
    u32 shift;                 // bucket = row >> shift
    u64 *next;                 // next free position per bucket (not the last pass)
    const u64 *rs;             // last pass: row offsets
    u32 *used;                 //   and entries placed per row
    u32 *row_out, *col_out, *w_out;  // row_out null in the last pass
};

__device__ __forceinline__ u64 part_reserve(const PartArgs &a, u32 bucket, u32 k) {
    return a.next ? atomicAdd((unsigned long long *)&a.next[bucket], (unsigned long long)k)
                  : a.rs[bucket] + atomicAdd(&a.used[bucket], k);
}

template <bool TUPLES>
__global__ __launch_bounds__(kPartThreads) void partition_kernel(PartArgs a) {
    __shared__ u32 s_row[kPartTile], s_col[kPartTile], s_w[kPartTile];
    __shared__ u32 bins[kPartBins];  // counts, then the bucket's first place in the tile
    __shared__ u64 dst[kPartBins];   // the bucket's reserved run
    __shared__ u32 wave_sum_[kPartThreads / kWave];
    __shared__ u32 s_lo, s_hi;
    const u32 tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    constexpr u64 kPer = TUPLES ? kPartTile / 2 : kPartTile;
    for (u64 t0 = (u64)blockIdx.x * kPer; t0 < a.count; t0 += (u64)gridDim.x * kPer) {
        u32 row[kPartItems], col[kPartItems], w[kPartItems];
        bool ok[kPartItems];
        if (tid == 0) {
            s_lo = ~0u;
            s_hi = 0;
        }
        if (TUPLES) {
#pragma unroll
            for (int k = 0; k < kPartItems; k += 2) {
                const u64 i = t0 + (u64)(k / 2) * kPartThreads + tid;
                Packed_Edge e = {0, 0};
                u32 wb = 0;
                if (i < a.count) {
                    e = a.edges[i];
                    wb = __float_as_uint(a.ew[i]);
                }
                ok[k] = ok[k + 1] = e.v0 != e.v1 && e.v0 < a.n && e.v1 < a.n;
                row[k] = col[k + 1] = (u32)e.v0;
                row[k + 1] = col[k] = (u32)e.v1;
                w[k] = w[k + 1] = wb;
            }
        } else {
#pragma unroll
            for (int k = 0; k < kPartItems; ++k) {
                const u64 i = t0 + (u64)k * kPartThreads + tid;
                ok[k] = i < a.count;
                row[k] = ok[k] ? a.row_in[i] : 0;
                col[k] = ok[k] ? a.col_in[i] : 0;
                w[k] = ok[k] ? a.w_in[i] : 0;
            }
        }
        u32 lo = ~0u, hi = 0;
#pragma unroll
        for (int k = 0; k < kPartItems; ++k)
            if (ok[k]) {
                lo = min(lo, row[k] >> a.shift);
                hi = max(hi, row[k] >> a.shift);
            }
        lo = wave_min(lo);
        hi = ~wave_min(~hi);
        __syncthreads();
        if (lane == 0) {
            atomicMin(&s_lo, lo);
            atomicMax(&s_hi, hi);
        }
        __syncthreads();
        lo = s_lo;
        hi = s_hi;
        if (lo > hi || hi - lo >= kPartBins) {
            // no entries, or a stretch of almost empty buckets: entry by entry
#pragma unroll
            for (int k = 0; k < kPartItems; ++k)
                if (ok[k]) {
                    const u64 g = part_reserve(a, row[k] >> a.shift, 1);
                    a.col_out[g] = col[k];
                    a.w_out[g] = w[k];
                    if (a.row_out) a.row_out[g] = row[k];
                }
            __syncthreads();  // s_lo and s_hi are set again by the next tile
            continue;
        }
        const u32 nb = hi - lo + 1;
        for (u32 b = tid; b < kPartBins; b += kPartThreads) bins[b] = 0;
        __syncthreads();
        u32 rank[kPartItems];
#pragma unroll
        for (int k = 0; k < kPartItems; ++k) rank[k] = ok[k] ? atomicAdd(&bins[(row[k] >> a.shift) - lo], 1u) : 0;
        __syncthreads();
        static_assert(kPartBins == 2 * kPartThreads, "two buckets per thread");
        const u32 c0 = bins[2 * tid], c1 = bins[2 * tid + 1];
        const u32 incl = wave_inclusive_scan(c0 + c1);
        if (lane == kWave - 1) wave_sum_[wave] = incl;
        __syncthreads();
        u32 before = incl - c0 - c1, total = 0;
        for (u32 i = 0; i < kPartThreads / kWave; ++i) {
            before += i < wave ? wave_sum_[i] : 0u;
            total += wave_sum_[i];
        }
        bins[2 * tid] = before;
        bins[2 * tid + 1] = before + c0;
        if (2 * tid < nb && c0) dst[2 * tid] = part_reserve(a, lo + 2 * tid, c0);
        if (2 * tid + 1 < nb && c1) dst[2 * tid + 1] = part_reserve(a, lo + 2 * tid + 1, c1);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPartItems; ++k)
            if (ok[k]) {
                const u32 p = bins[(row[k] >> a.shift) - lo] + rank[k];
                s_row[p] = row[k];
                s_col[p] = col[k];
                s_w[p] = w[k];
            }
        __syncthreads();
        for (u32 p = tid; p < total; p += kPartThreads) {
            const u32 r = s_row[p], b = (r >> a.shift) - lo;
            const u64 g = dst[b] + (p - bins[b]);
            a.col_out[g] = s_col[p];
            a.w_out[g] = s_w[p];
            if (a.row_out) a.row_out[g] = r;
        }
        __syncthreads();
    }
}

// Words after pass 1's bucket counts.
constexpr u32 kPartBad = kPartBins, kPartSeen = kPartBins + 1, kPartNear = kPartBins + 2, kPartWords = kPartBins + 3;

// Entries per bucket of pass 1, from the tuples; flags endpoints out of range.
// Every eighth block also counts its tuples with one before them in the wave,
// and those of them whose endpoints both lie next to, but not on, the endpoints
// of the one before (see tuples_are_near): a sample, since all waves' counts
// would queue at these two words for longer than the pass takes.
constexpr u64 kNearVertices = 16;  // a 64-byte line of the degrees
__device__ __forceinline__ bool near_but_not_on(u64 a, u64 b) { return a - b + kNearVertices <= 2 * kNearVertices && a != b; }
__global__ __launch_bounds__(1024) void partition_count_tuples(const Packed_Edge *__restrict__ edges, u64 ne, u64 n,
                                                               u32 shift, u32 *__restrict__ counts) {
    __shared__ u32 h[kPartBins], pairs[2];
    for (u32 b = threadIdx.x; b < kPartBins; b += blockDim.x) h[b] = 0;
    if (threadIdx.x < 2) pairs[threadIdx.x] = 0;
    __syncthreads();
    const u32 lane = lane_id();
    const u64 step = (u64)gridDim.x * blockDim.x;
    u32 seen = 0, near = 0;
    for (u64 i0 = (u64)blockIdx.x * blockDim.x + (threadIdx.x - lane); i0 < ne; i0 += step) {
        const u64 i = i0 + lane;
        const Packed_Edge e = edges[min(i, ne - 1)];
        if (blockIdx.x % 8 == 0) {
            const int before = lane ? (int)lane - 1 : 0;
            const u64 p0 = shfl64(e.v0, before), p1 = shfl64(e.v1, before);
            const bool pair = lane && i < ne;
            seen += pair;
            near += pair && near_but_not_on(e.v0, p0) && near_but_not_on(e.v1, p1);
        }
        if (i >= ne) continue;
        if (e.v0 >= n || e.v1 >= n) {
            atomicOr(&counts[kPartBad], 1u);
            continue;
        }
        if (e.v0 == e.v1) continue;
        atomicAdd(&h[(u32)(e.v0 >> shift)], 1u);
        atomicAdd(&h[(u32)(e.v1 >> shift)], 1u);
    }
    if (blockIdx.x % 8 == 0) {
        seen = wave_sum(seen);
        near = wave_sum(near);
        if (lane == 0) {
            atomicAdd(&pairs[0], seen);
            atomicAdd(&pairs[1], near);
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 && pairs[threadIdx.x]) atomicAdd(&counts[threadIdx.x ? kPartNear : kPartSeen], pairs[threadIdx.x]);
    for (u32 b = threadIdx.x; b < kPartBins; b += blockDim.x)
        if (h[b]) atomicAdd(&counts[b], h[b]);
}

// Entries per bucket of a later pass, from the rows of the pass before: a
// block's tile lies in few parents, so its buckets are counted in LDS.
constexpr u32 kCountBins = 4096;
constexpr int kCountItems = 16;
__global__ __launch_bounds__(1024) void partition_count_rows(const u32 *__restrict__ rows, u64 count, u32 shift,
                                                             u32 *__restrict__ counts) {
    __shared__ u32 h[kCountBins];
    __shared__ u32 s_lo, s_hi;
    constexpr u64 kPer = 1024 * kCountItems;
    for (u64 t0 = (u64)blockIdx.x * kPer; t0 < count; t0 += (u64)gridDim.x * kPer) {
        if (threadIdx.x == 0) {
            s_lo = ~0u;
            s_hi = 0;
        }
        for (u32 b = threadIdx.x; b < kCountBins; b += blockDim.x) h[b] = 0;
        u32 b[kCountItems], lo = ~0u, hi = 0;
#pragma unroll
        for (int k = 0; k < kCountItems; ++k) {
            const u64 i = t0 + (u64)k * 1024 + threadIdx.x;
            b[k] = i < count ? rows[i] >> shift : 0u;
        }
        auto valid = [&](int k) { return t0 + (u64)k * 1024 + threadIdx.x < count; };
#pragma unroll
        for (int k = 0; k < kCountItems; ++k)
            if (valid(k)) {
                lo = min(lo, b[k]);
                hi = max(hi, b[k]);
            }
        lo = wave_min(lo);
        hi = ~wave_min(~hi);
        __syncthreads();
        if (lane_id() == 0) {
            atomicMin(&s_lo, lo);
            atomicMax(&s_hi, hi);
        }
        __syncthreads();
        lo = s_lo;
        hi = s_hi;
        const bool narrow = hi - lo < kCountBins;
#pragma unroll
        for (int k = 0; k < kCountItems; ++k)
            if (valid(k)) atomicAdd(narrow ? &h[b[k] - lo] : &counts[b[k]], 1u);
        __syncthreads();
        if (narrow)
            for (u32 q = threadIdx.x; q <= hi - lo; q += blockDim.x)
                if (h[q]) atomicAdd(&counts[lo + q], h[q]);
        __syncthreads();
    }
}

// ------------------------------------------------------------------ row sort
// Tiers by row length: 2..16 a thread, 17..64 / 128 / 256 / 512 a wave with 1
// / 2 / 4 / 8 entries per lane; longer rows are split by weight into bins of
// about kBinEntries, which a wave sorts too (see the long rows below).
constexpr int kWaveTiers = 4;            // 64 << t entries
constexpr u32 kLongRow = 512;            // rows above it are long
constexpr u32 kSegBlock = 4096;          // longest segment that one block sorts in LDS
struct SortLists {
    CounterLine<u32> n[kWaveTiers];      // rows per wave tier
    CounterLine<u64> longs;              // packed hub counter of the long rows
    CounterLine<u64> long_entries;       // their entries
    CounterLine<u64> huge_entries;       //   of those above kSegBlock
    CounterLine<u32> nblock, nradix;     // segments for the block and radix sorts
    CounterLine<u64> notisolated;
};
// Rows of a tier's list are at least `least` entries long, so M entries have
// at most this many of them.
static u64 tier_cap(u64 n, u64 m, u64 least) { return MIN(n, m / least + 1); }

struct TierLists {
    u32 *rows[kWaveTiers];
    u32 *long_row, *long_len;
    u64 *long_off;
    u64 long_cap;
};

// The lists are staged in LDS per tile of rows, one atomic per list and tile
// (one per wave and list on neighbouring counters took 3.4 ms at S23, this 0.6).
constexpr int kClassifyTile = 1024;
__global__ __launch_bounds__(1024) void classify_rows(const u64 *__restrict__ rs, u64 n, SortLists *L, TierLists t,
                                                      u32 *__restrict__ error) {
    __shared__ u32 stage[kWaveTiers][kClassifyTile];
    __shared__ u32 cnt[kWaveTiers], base[kWaveTiers];
    u32 nonzero = 0;
    u64 longs = 0, huge = 0;
    for (u64 v0 = (u64)blockIdx.x * kClassifyTile; v0 < n; v0 += (u64)gridDim.x * kClassifyTile) {
        if (threadIdx.x < kWaveTiers) cnt[threadIdx.x] = 0;
        __syncthreads();
        for (int k = 0; k < kClassifyTile; k += 1024) {
            const u64 v = v0 + k + threadIdx.x;
            const u64 d = v < n ? rs[v + 1] - rs[v] : 0;
            nonzero += d > 0;
            const bool is_long = d > kLongRow;
            if (is_long) {
                longs += d;
                huge += d > kSegBlock ? d : 0;
            }
            hub_append(&L->longs.v, t.long_row, t.long_off, t.long_len, is_long, (u32)v, (u32)d, t.long_cap, error);
            if (d > 16 && !is_long) {
                const int tier = d <= 64 ? 0 : d <= 128 ? 1 : d <= 256 ? 2 : 3;
                stage[tier][atomicAdd(&cnt[tier], 1u)] = (u32)v;
            }
        }
        __syncthreads();
        if (threadIdx.x < kWaveTiers)
            base[threadIdx.x] = cnt[threadIdx.x] ? atomicAdd(&L->n[threadIdx.x].v, cnt[threadIdx.x]) : 0;
        __syncthreads();
        for (int q = 0; q < kWaveTiers; ++q)
            for (u32 i = threadIdx.x; i < cnt[q]; i += 1024) t.rows[q][base[q] + i] = stage[q][i];
        __syncthreads();
    }
    const u32 tot = wave_sum(nonzero);
    longs = wave_sum(longs);
    huge = wave_sum(huge);
    if (lane_id() == 0) {
        if (tot) atomicAdd((unsigned long long *)&L->notisolated.v, (unsigned long long)tot);
        if (longs) atomicAdd((unsigned long long *)&L->long_entries.v, (unsigned long long)longs);
        if (huge) atomicAdd((unsigned long long *)&L->huge_entries.v, (unsigned long long)huge);
    }
}

// Tier 0: rows of 2..16 entries, one thread each, bitonic network in registers.
__global__ __launch_bounds__(256) void sort_rows_thread(const u64 *__restrict__ rs, u64 n,
                                                        u32 *__restrict__ col, f32 *__restrict__ cw) {
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (u64)gridDim.x * blockDim.x) {
        const u64 b = rs[v];
        const u32 d = (u32)(rs[v + 1] - b);
        if (d < 2 || d > 16) continue;
        u64 k[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) k[i] = (u32)i < d ? make_key(col[b + i], cw[b + i]) : ~0ull;
#pragma unroll
        for (int size = 2; size <= 16; size <<= 1)
#pragma unroll
            for (int stride = size / 2; stride > 0; stride >>= 1)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int j = i ^ stride;
                    if (j > i) {
                        const bool up = (i & size) == 0;
                        if ((k[i] > k[j]) == up) {
                            u64 t = k[i];
                            k[i] = k[j];
                            k[j] = t;
                        }
                    }
                }
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if ((u32)i < d) {
                col[b + i] = (u32)k[i];
                cw[b + i] = __uint_as_float((u32)(k[i] >> 32));
            }
    }
}

// Ascending bitonic sort of a wave's 64 E keys, E per lane, key p in lane p / E:
// strides below E stay in a lane's registers, the others are 21 lane exchanges
// of each key for any E.
template <int E>
__device__ __forceinline__ void wave_sort(u64 (&x)[E]) {
    const u32 lane = lane_id();
#pragma unroll
    for (int size = 2; size <= kWave * E; size <<= 1)
#pragma unroll
        for (int stride = size / 2; stride > 0; stride >>= 1) {
            if (stride >= E) {
                const bool lower = (lane & (u32)(stride / E)) == 0;
                const bool up = (lane * E & (u32)size) == 0;  // size > stride >= E: the lane alone decides
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    const u64 y = shfl_xor64(x[i], stride / E);
                    x[i] = (lower == up) ? (x[i] < y ? x[i] : y) : (x[i] < y ? y : x[i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    const int j = i ^ stride;
                    if (j > i) {
                        const bool up = ((lane * E + (u32)i) & (u32)size) == 0;
                        if ((x[i] > x[j]) == up) {
                            const u64 t = x[i];
                            x[i] = x[j];
                            x[j] = t;
                        }
                    }
                }
            }
        }
}

// Sorts src[0, len) (len <= 64 E) into dst; they may be the same place.
template <int E>
__device__ __forceinline__ void wave_sort_segment(const u32 *src_col, const u32 *src_w, u32 *col, u32 *w, u32 len) {
    const u32 lane = lane_id();
    u64 x[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const u32 p = (u32)i * kWave + lane;
        x[i] = p < len ? ((u64)src_w[p] << 32) | src_col[p] : ~0ull;
    }
    wave_sort(x);
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const u32 p = lane * E + (u32)i;
        if (p < len) {
            col[p] = (u32)x[i];
            w[p] = (u32)(x[i] >> 32);
        }
    }
}

// Rows of the wave tiers, in place, the longest first.
struct TierCounts {
    u32 n[kWaveTiers];
};
__global__ __launch_bounds__(256) void sort_rows_wave(const u64 *__restrict__ rs, TierLists t, TierCounts k, u32 *col,
                                                      u32 *w) {
    const u32 waves = gridDim.x * (blockDim.x / kWave);
    u32 r = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    auto tier = [&](auto entries, int q) {
        for (; r < k.n[q]; r += waves) {
            const u32 v = t.rows[q][r];
            const u64 b = rs[v];
            wave_sort_segment<decltype(entries)::value>(col + b, w + b, col + b, w + b, (u32)(rs[v + 1] - b));
        }
        r -= k.n[q];
    };
    static_assert(kWaveTiers == 4, "one call per tier");
    tier(std::integral_constant<int, 8>(), 3);
    tier(std::integral_constant<int, 4>(), 2);
    tier(std::integral_constant<int, 2>(), 1);
    tier(std::integral_constant<int, 1>(), 0);
}

// Segments that a wave does not sort: a block's bitonic sort in LDS up to
// kSegBlock entries, a block's radix sort above. They are whole long rows, or
// bins of rows whose weights are far from evenly spread (many equal ones). A
// bin's entries are still in the scratch pair, and its sort reads them there:
// the wave that finds it too long would copy it alone (a row of 1e6 equal
// weights: 6.9 of 24.3 ms).
struct Segment {
    u64 at;       // in the columns and weights
    u64 scratch;  // in the scratch pair (whole rows: radix only)
    u32 len;
    u32 in_scratch;  // where the entries are: 0 at, 1 scratch
};
constexpr u32 kSegThreads = 1024;
__device__ __forceinline__ void block_sort(u64 *keys, const u32 *from_col, const u32 *from_w, u32 *col, u32 *w, u32 d) {
    u32 P = 128;
    while (P < d) P <<= 1;
    for (u32 i = threadIdx.x; i < P; i += kSegThreads) keys[i] = i < d ? ((u64)from_w[i] << 32) | from_col[i] : ~0ull;
    __syncthreads();
    for (u32 size = 2; size <= P; size <<= 1)
        for (u32 stride = size >> 1; stride > 0; stride >>= 1) {
            for (u32 t = threadIdx.x; t < P / 2; t += kSegThreads) {
                const u32 i = 2 * stride * (t / stride) + (t % stride), j = i + stride;
                const bool up = (i & size) == 0;
                const u64 a = keys[i], c = keys[j];
                if ((a > c) == up) {
                    keys[i] = c;
                    keys[j] = a;
                }
            }
            __syncthreads();
        }
    for (u32 i = threadIdx.x; i < d; i += kSegThreads) {
        col[i] = (u32)keys[i];
        w[i] = (u32)(keys[i] >> 32);
    }
    __syncthreads();
}
__global__ __launch_bounds__(kSegThreads) void sort_segments_block(const Segment *__restrict__ segs, const u32 *__restrict__ nsegs,
                                                           u32 *__restrict__ col, u32 *__restrict__ w,
                                                           const u32 *__restrict__ s_col,
                                                           const u32 *__restrict__ s_w) {
    __shared__ u64 keys[kSegBlock];
    const u32 count = *nsegs;
    for (u32 r = blockIdx.x; r < count; r += gridDim.x) {
        const u64 b = segs[r].at;
        const u32 *from_col = segs[r].in_scratch ? s_col + segs[r].scratch : col + b;
        const u32 *from_w = segs[r].in_scratch ? s_w + segs[r].scratch : w + b;
        block_sort(keys, from_col, from_w, col + b, w + b, segs[r].len);
    }
}

// Segments longer than kSegBlock entries, one 1024-thread block each, stable
// LSD radix sort on 8-bit digits ping-ponging between the segment (column /
// weight-bit arrays) and a scratch pair, from where the entries are. Digits
// cover the column bits, then the weight bits.
constexpr int kRadixBlock = 1024;
constexpr int kRadixWaves = kRadixBlock / kWave;

__device__ __forceinline__ u32 digit_of(u32 lo, u32 hi, int shift) {
    return shift < 32 ? (lo >> shift) & 0xFF : (hi >> (shift - 32)) & 0xFF;
}

struct RadixLds {
    u32 base[256];
    u32 wcnt[kRadixWaves][256];
};
// Sorts the d entries of pair a, or of pair b with in_b set, into a.
__device__ __forceinline__ void block_radix(RadixLds &lds, u32 *a_lo, u32 *a_hi, u32 *b_lo, u32 *b_hi, int in_b, u32 d,
                                            int col_passes) {
    const int wave = threadIdx.x / kWave;
    const int npass = col_passes + 4;
    for (int pass = 0; pass < npass; ++pass) {
        const bool from_b = (pass + in_b) & 1;
        const int shift = pass < col_passes ? 8 * pass : 32 + 8 * (pass - col_passes);
        const u32 *src_lo = from_b ? b_lo : a_lo, *src_hi = from_b ? b_hi : a_hi;
        u32 *dst_lo = from_b ? a_lo : b_lo, *dst_hi = from_b ? a_hi : b_hi;
        if (threadIdx.x < 256) lds.base[threadIdx.x] = 0;
        __syncthreads();
        for (u32 i = threadIdx.x; i < d; i += kRadixBlock)
            atomicAdd(&lds.base[digit_of(src_lo[i], src_hi[i], shift)], 1u);
        __syncthreads();
        if (threadIdx.x < 256) {  // exclusive scan of the 256 bins, 4 waves
            u32 x = lds.base[threadIdx.x];
            const u32 incl = wave_inclusive_scan(x);
            lds.wcnt[0][threadIdx.x] = incl;  // staging of wave-inclusive sums
        }
        __syncthreads();
        if (threadIdx.x < 256) {
            u32 add = 0;
            for (int w = 0; w < (int)(threadIdx.x / kWave); ++w) add += lds.wcnt[0][w * kWave + kWave - 1];
            lds.base[threadIdx.x] = add + lds.wcnt[0][threadIdx.x] - lds.base[threadIdx.x];
        }
        __syncthreads();
        for (u32 t0 = 0; t0 < d; t0 += kRadixBlock) {
            const u32 i = t0 + threadIdx.x;
            const bool valid = i < d;
            u32 lo = 0, hi = 0, dg = 0;
            if (valid) {
                lo = src_lo[i];
                hi = src_hi[i];
                dg = digit_of(lo, hi, shift);
            }
            for (int k = threadIdx.x; k < kRadixWaves * 256; k += kRadixBlock) (&lds.wcnt[0][0])[k] = 0;
            u64 peers = ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                const u64 m = ballot((dg >> bit) & 1);
                peers &= ((dg >> bit) & 1) ? m : ~m;
            }
            const u32 rank = mask_rank(peers);
            __syncthreads();
            if (valid && rank == 0) lds.wcnt[wave][dg] = (u32)__popcll(peers);
            __syncthreads();
            if (threadIdx.x < 256) {
                u32 run = lds.base[threadIdx.x];
                for (int w = 0; w < kRadixWaves; ++w) {
                    const u32 c = lds.wcnt[w][threadIdx.x];
                    lds.wcnt[w][threadIdx.x] = run;
                    run += c;
                }
                lds.base[threadIdx.x] = run;
            }
            __syncthreads();
            if (valid) {
                const u32 pos = lds.wcnt[wave][dg] + rank;
                dst_lo[pos] = lo;
                dst_hi[pos] = hi;
            }
            __syncthreads();
        }
    }
    if ((npass + in_b) & 1) {  // result sits in the scratch pair: copy back
        for (u32 i = threadIdx.x; i < d; i += kRadixBlock) {
            a_lo[i] = b_lo[i];
            a_hi[i] = b_hi[i];
        }
    }
    __syncthreads();
}
__global__ __launch_bounds__(kRadixBlock) void sort_segments_radix(
    const Segment *__restrict__ segs, const u32 *__restrict__ nsegs, u32 *__restrict__ col, u32 *__restrict__ wbits,
    u32 *__restrict__ s_lo, u32 *__restrict__ s_hi, int col_passes) {
    __shared__ RadixLds lds;
    const u32 count = *nsegs;
    for (u32 r = blockIdx.x; r < count; r += gridDim.x)
        block_radix(lds, col + segs[r].at, wbits + segs[r].at, s_lo + segs[r].scratch, s_hi + segs[r].scratch,
                    (int)segs[r].in_scratch, segs[r].len, col_passes);
}

// ------------------------------------------------------------- without lists
// For arenas that hold the rows but not the lists of them beside the sort's
// scratch (up to 32 bytes a vertex and 1 an entry in 20): a block walks `per`
// rows, its waves sort those of 17..512 entries and the block the longer ones.
struct UnlistedCounts {
    u64 notisolated, huge_entries, scratch_used;
};
__global__ __launch_bounds__(256) void count_rows(const u64 *__restrict__ rs, u64 n, UnlistedCounts *k) {
    u64 nonzero = 0, huge = 0;
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (u64)gridDim.x * blockDim.x) {
        const u64 d = rs[v + 1] - rs[v];
        nonzero += d > 0;
        huge += d > kSegBlock ? d : 0;
    }
    nonzero = wave_sum(nonzero);
    huge = wave_sum(huge);
    if (lane_id() == 0 && nonzero) atomicAdd((unsigned long long *)&k->notisolated, (unsigned long long)nonzero);
    if (lane_id() == 0 && huge) atomicAdd((unsigned long long *)&k->huge_entries, (unsigned long long)huge);
}

constexpr u32 kUnlistedRows = 1024;  // at most, per block at a time
__global__ __launch_bounds__(kSegThreads) void sort_rows_unlisted(const u64 *__restrict__ rs, u64 n, u32 per, u32 *col,
                                                                  u32 *w, u32 *s_col, u32 *s_w, UnlistedCounts *k,
                                                                  int col_passes) {
    static_assert(kSegThreads == (u32)kRadixBlock, "one block shape for both sorts");
    __shared__ u64 keys[kSegBlock];
    __shared__ RadixLds radix;
    __shared__ u32 longs[kUnlistedRows], nlongs;
    __shared__ u64 place;
    const u32 wave = threadIdx.x / kWave;
    for (u64 v0 = (u64)blockIdx.x * per; v0 < n; v0 += (u64)gridDim.x * per) {
        if (threadIdx.x == 0) nlongs = 0;
        __syncthreads();
        for (u32 r = wave; r < per && v0 + r < n; r += kSegThreads / kWave) {
            const u64 b = rs[v0 + r], d = rs[v0 + r + 1] - b;
            u32 *c = col + b, *x = w + b;
            if (d > kLongRow) {
                if (lane_id() == 0) longs[atomicAdd(&nlongs, 1u)] = r;
            } else if (d > 256) {
                wave_sort_segment<8>(c, x, c, x, (u32)d);
            } else if (d > 64) {
                wave_sort_segment<4>(c, x, c, x, (u32)d);
            } else if (d > 16) {
                wave_sort_segment<1>(c, x, c, x, (u32)d);
            }
        }
        __syncthreads();
        for (u32 i = 0; i < nlongs; ++i) {
            const u64 b = rs[v0 + longs[i]];
            const u32 d = (u32)(rs[v0 + longs[i] + 1] - b);
            if (d <= kSegBlock) {
                block_sort(keys, col + b, w + b, col + b, w + b, d);
            } else {
                if (threadIdx.x == 0)
                    place = atomicAdd((unsigned long long *)&k->scratch_used, (unsigned long long)d);
                __syncthreads();
                block_radix(radix, col + b, w + b, s_col + place, s_w + place, 0, d, col_passes);
            }
        }
        __syncthreads();  // nlongs is set again for the next rows
    }
}

// ----------------------------------------------------------------- long rows
// Rows above kLongRow entries (three quarters of the entries at S23) are split
// by weight: row r of d entries has K = ceil(d / kBinEntries) bins, linear in
// the weight between the row's smallest and largest (a monotone map, so the
// bins are in order), its entries are scattered by bin into scratch, and a
// wave sorts each bin into the row. Rows with negative or non-finite weights
// are one bin. Rows lie in a flattened space padded to kHubChunk entries
// (hub_append); chunk c of it stands for 256 entries of its row and, for the
// row's first K chunks, for a bin. Before, rows of 65..4096 entries were
// sorted by a block's bitonic sort in LDS and longer ones by one block's
// radix sort each: 20 ms at S23, now 5.3 with the wave tiers.
constexpr u32 kBinEntries = 384;  // on average; a wave sorts up to 512 (six deviations above it for uniform weights)
constexpr int kLongBlock = 512, kLongChunks = 4;  // a wave takes 4 chunks, a block a span of 32
constexpr u64 kLongSpan = (u64)kLongChunks * (kLongBlock / kWave);
constexpr u32 kLongBins = 8192;  // bins counted in LDS at a time

struct LongRows {
    const u64 *rs;
    const u32 *row, *len;
    const u64 *off;
    u64 nrows, nchunks;
    u32 *chunk_row;    // [nchunks] slot of the row
    u32 *wlo, *whi;    // [nrows] smallest and largest weight bits
    u32 *count;        // [nchunks] entries per bin
    u64 *bin_off;      // [nchunks + 1] the bin's place in the scratch
    u32 *used;         // [nchunks] entries placed
    u32 *col, *w;      // the CSR
    u32 *s_col, *s_w;  // scratch
};

__device__ __forceinline__ u32 long_bins(u32 len) { return (len + kBinEntries - 1) / kBinEntries; }

// The slot of every chunk's row; clears the row's weight range.
__global__ __launch_bounds__(256) void long_chunk_rows(LongRows a) {
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    for (u64 r = wave; r < a.nrows; r += nw) {
        const u64 c0 = a.off[r] / kHubChunk, k = (a.len[r] + kHubChunk - 1) / kHubChunk;
        for (u64 c = lane_id(); c < k; c += kWave) a.chunk_row[c0 + c] = (u32)r;
        if (lane_id() == 0) {
            a.wlo[r] = ~0u;
            a.whi[r] = 0;
        }
    }
}

// A lane's 4 entries of chunk c (false beyond the row's end).
struct LongChunk {
    u64 at[4];
    bool ok[4];
};
__device__ __forceinline__ u32 long_chunk(const LongRows &a, u64 c, LongChunk &k) {
    const u32 r = a.chunk_row[c];
    const u32 in_row = (u32)(c * kHubChunk - a.off[r]) + lane_id(), len = a.len[r];
    const u64 b = a.rs[a.row[r]];
#pragma unroll
    for (u32 q = 0; q < 4; ++q) {
        k.ok[q] = in_row + q * kWave < len;
        k.at[q] = b + in_row + q * kWave;
    }
    return r;
}

__global__ __launch_bounds__(256) void long_weight_range(LongRows a) {
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    for (u64 c = wave; c < a.nchunks; c += nw) {
        LongChunk k;
        const u32 r = long_chunk(a, c, k);
        u32 lo = ~0u, hi = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (k.ok[q]) {
                const u32 wb = a.w[k.at[q]];
                lo = min(lo, wb);
                hi = max(hi, wb);
            }
        lo = wave_min(lo);
        hi = ~wave_min(~hi);
        if (lane_id() == 0) {  // a plain read may be stale, the wrong way only for skipping nothing
            if (lo < ld_relaxed(&a.wlo[r])) atomicMin(&a.wlo[r], lo);
            if (hi > ld_relaxed(&a.whi[r])) atomicMax(&a.whi[r], hi);
        }
    }
}

// Bin of a weight in its row: first bin, bins, and the linear map.
struct LongMap {
    u32 first, bins;
    f32 lo, scale;
    __device__ __forceinline__ u32 bin(u32 wb) const {
        return first + min((u32)((__uint_as_float(wb) - lo) * scale), bins - 1);
    }
};
__device__ __forceinline__ LongMap long_map(const LongRows &a, u32 r) {
    LongMap m;
    m.first = (u32)(a.off[r] / kHubChunk);
    m.bins = long_bins(a.len[r]);
    const u32 lo = a.wlo[r], hi = a.whi[r];
    m.lo = __uint_as_float(lo);
    m.scale = (f32)m.bins / (__uint_as_float(hi) - m.lo);
    if (hi >= 0x7F800000u || !(m.scale < 1e30f)) {  // negative or not finite, or (almost) all equal: one bin
        m.lo = 0.0f;
        m.scale = 0.0f;
        m.bins = 1;
    }
    return m;
}

// Counts (SCATTER false) or places (true) the entries of a span of chunks by
// bin. The bins of the span's rows are ranked in LDS, kLongBins of them at a
// time (rows above 3.1e6 entries have more; their entries are read again for
// each), with one global atomic per bin and span: entries of one bin that each
// made their own would queue at its counter, 11 ns each (a row of 4e6 equal
// weights: 91 of 158 ms).
template <bool SCATTER>
__global__ __launch_bounds__(kLongBlock) void long_bin_kernel(LongRows a) {
    __shared__ u32 h[kLongBins];
    const u32 wave = threadIdx.x / kWave;
    auto count_span = [&](u64 c0, u64 c1, u32 lo, u32 nb) {  // bins [lo, lo + nb)
        for (u32 b = threadIdx.x; b < nb; b += kLongBlock) h[b] = 0;
        __syncthreads();
        u32 bin[kLongChunks][4], rank[kLongChunks][4], wb[kLongChunks][4], cv[kLongChunks][4];
        bool ok[kLongChunks][4];
#pragma unroll
        for (int g = 0; g < kLongChunks; ++g) {
            const u64 c = c0 + (u64)wave * kLongChunks + g;
            LongChunk k;
            u32 r = 0;
            if (c < c1) r = long_chunk(a, c, k);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                ok[g][q] = c < c1 && k.ok[q];
                wb[g][q] = ok[g][q] ? a.w[k.at[q]] : 0;
                if (SCATTER) cv[g][q] = ok[g][q] ? a.col[k.at[q]] : 0;
            }
            if (c < c1) {
                const LongMap m = long_map(a, r);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    bin[g][q] = ok[g][q] ? m.bin(wb[g][q]) - lo : 0;
                    ok[g][q] = ok[g][q] && bin[g][q] < nb;
                }
            }
        }
        u32 *cnt = (SCATTER ? a.used : a.count) + lo;
#pragma unroll
        for (int g = 0; g < kLongChunks; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) rank[g][q] = ok[g][q] ? atomicAdd(&h[bin[g][q]], 1u) : 0;
        __syncthreads();
        for (u32 b = threadIdx.x; b < nb; b += kLongBlock)
            if (h[b]) h[b] = atomicAdd(&cnt[b], h[b]);
        __syncthreads();
        if (SCATTER) {
#pragma unroll
            for (int g = 0; g < kLongChunks; ++g)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (ok[g][q]) {
                        const u64 p = a.bin_off[lo + bin[g][q]] + rank[g][q] + h[bin[g][q]];
                        a.s_col[p] = cv[g][q];
                        a.s_w[p] = wb[g][q];
                    }
            __syncthreads();
        }
    };
    for (u64 c0 = (u64)blockIdx.x * kLongSpan; c0 < a.nchunks; c0 += (u64)gridDim.x * kLongSpan) {
        const u64 c1 = min(c0 + kLongSpan, a.nchunks);
        const u32 r0 = a.chunk_row[c0], r1 = a.chunk_row[c1 - 1];
        const u32 lo = (u32)(a.off[r0] / kHubChunk), hi = (u32)(a.off[r1] / kHubChunk) + long_bins(a.len[r1]);
        for (u32 b = lo; b < hi; b += kLongBins) count_span(c0, c1, b, min(hi - b, kLongBins));
    }
}

// Sorts every bin into its row; a bin too long for a wave is listed for the
// block and radix sorts.
__global__ __launch_bounds__(256) void long_sort_bins(LongRows a, SortLists *L, Segment *__restrict__ block_segs,
                                                      Segment *__restrict__ radix_segs) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    for (u64 c = wave; c < a.nchunks; c += nw) {
        const u32 len = a.count[c];
        if (!len) continue;
        const u32 r = a.chunk_row[c];
        const u64 from = a.bin_off[c];
        const u64 to = a.rs[a.row[r]] + (from - a.bin_off[a.off[r] / kHubChunk]);
        if (len <= 4 * kWave) {
            wave_sort_segment<4>(a.s_col + from, a.s_w + from, a.col + to, a.w + to, len);
        } else if (len <= 8 * kWave) {
            wave_sort_segment<8>(a.s_col + from, a.s_w + from, a.col + to, a.w + to, len);
        } else if (lane == 0) {
            const Segment s = {to, from, len, 1};
            if (len <= kSegBlock) block_segs[atomicAdd(&L->nblock.v, 1u)] = s;
            else radix_segs[atomicAdd(&L->nradix.v, 1u)] = s;
        }
    }
}

// Few long rows, or no room for the scratch of them all: each is a segment of its own
// (scratch places in list order for those above kSegBlock entries).
__global__ __launch_bounds__(256) void long_rows_as_segments(LongRows a, SortLists *L, Segment *__restrict__ block_segs,
                                                             Segment *__restrict__ radix_segs, u64 *scratch_used) {
    for (u64 r = (u64)blockIdx.x * blockDim.x + threadIdx.x; r < a.nrows; r += (u64)gridDim.x * blockDim.x) {
        Segment s = {a.rs[a.row[r]], 0, a.len[r], 0};
        if (s.len <= kSegBlock) {
            block_segs[atomicAdd(&L->nblock.v, 1u)] = s;
        } else {
            s.scratch = atomicAdd((unsigned long long *)scratch_used, (unsigned long long)s.len);
            radix_segs[atomicAdd(&L->nradix.v, 1u)] = s;
        }
    }
}

// ---------------------------------------------------------------- relabeling
// Traversal copy of the CSR with vertices renumbered by decreasing degree
// (exact up to kDegKeys - 1, above that in one class). In Kronecker graphs a
// few percent of the vertices hold most edge endpoints; numbering them first
// packs the labels, bitmap words and masks that traversals probe most into a
// small, cache-resident range. Entry order inside each row is unchanged, so
// rows stay sorted by weight.
constexpr u32 kDegKeys = 4096;
constexpr int kRelabelBlock = 1024;
constexpr int kRelabelItems = 8;

__device__ __forceinline__ u32 degree_key(const u64 *rs, u64 v) {
    const u64 d = rs[v + 1] - rs[v];
    return kDegKeys - 1 - (u32)(d < kDegKeys - 1 ? d : kDegKeys - 1);
}

__global__ __launch_bounds__(kRelabelBlock) void relabel_count(const u64 *__restrict__ rs, u64 n,
                                                               u32 *__restrict__ counts) {
    __shared__ u32 h[kDegKeys];
    for (u32 k = threadIdx.x; k < kDegKeys; k += blockDim.x) h[k] = 0;
    __syncthreads();
    const u64 base = (u64)blockIdx.x * kRelabelBlock * kRelabelItems;
    for (int j = 0; j < kRelabelItems; ++j) {
        const u64 v = base + (u64)j * kRelabelBlock + threadIdx.x;
        if (v < n) atomicAdd(&h[degree_key(rs, v)], 1u);
    }
    __syncthreads();
    for (u32 k = threadIdx.x; k < kDegKeys; k += blockDim.x)
        if (h[k]) atomicAdd(&counts[k], h[k]);
}

// Single block: exclusive scan of the key counts into cursors.
__global__ __launch_bounds__(1024) void relabel_offsets(const u32 *__restrict__ counts, u32 *__restrict__ cursor) {
    u64 carry = 0;
    for (u32 b = 0; b < kDegKeys; b += 1024) {
        const u32 k = b + threadIdx.x;
        const u64 v = counts[k];
        u64 tot;
        const u64 ex = block_exclusive_scan<1024>(v, &tot);
        cursor[k] = (u32)(carry + ex);
        carry += tot;
    }
}

// Each block reserves one range per key for its tile, then ranks its
// vertices inside the ranges (order inside a key class is not specified).
__global__ __launch_bounds__(kRelabelBlock) void relabel_scatter(const u64 *__restrict__ rs, u64 n,
                                                                 u32 *__restrict__ cursor, u32 *__restrict__ perm,
                                                                 u32 *__restrict__ iperm, u32 *__restrict__ deg_t) {
    __shared__ u32 h[kDegKeys], base[kDegKeys];
    for (u32 k = threadIdx.x; k < kDegKeys; k += blockDim.x) h[k] = 0;
    __syncthreads();
    const u64 tile = (u64)blockIdx.x * kRelabelBlock * kRelabelItems;
    u32 key[kRelabelItems];
    for (int j = 0; j < kRelabelItems; ++j) {
        const u64 v = tile + (u64)j * kRelabelBlock + threadIdx.x;
        key[j] = v < n ? degree_key(rs, v) : 0;
        if (v < n) atomicAdd(&h[key[j]], 1u);
    }
    __syncthreads();
    for (u32 k = threadIdx.x; k < kDegKeys; k += blockDim.x) {
        base[k] = h[k] ? atomicAdd(&cursor[k], h[k]) : 0;
        h[k] = 0;
    }
    __syncthreads();
    for (int j = 0; j < kRelabelItems; ++j) {
        const u64 v = tile + (u64)j * kRelabelBlock + threadIdx.x;
        if (v >= n) continue;
        const u32 pos = base[key[j]] + atomicAdd(&h[key[j]], 1u);
        perm[v] = pos;
        iperm[pos] = (u32)v;
        deg_t[pos] = (u32)(rs[v + 1] - rs[v]);
    }
}

// Largest row p of [0, n) with rs[p] <= k (rows before it may be empty).
__device__ __forceinline__ u64 row_at(const u64 *rs, u64 n, u64 k) {
    u64 lo = 0, hi = n;
    while (hi - lo > 1) {
        const u64 mid = lo + (hi - lo) / 2;
        if (rs[mid] <= k) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Rows of the traversal copy. Bound by the gather of the columns' new ids
// (4 random bytes an entry); what remains is to keep many of them in flight:
// a lane per short row and a block per longer one took 7.5 ms at S23, this 4.2.
struct RelabelArgs {
    const u64 *rs;
    const u32 *col;
    const f32 *w;
    const u32 *perm, *iperm;
    const u64 *rs_t;
    u32 *col_t;
    f32 *w_t;
    u64 nlong, n;
    u64 span;  // entries of a wave's piece of the long rows
    u32 per;   // short rows per wave
};

// Rows longer than a wave, [0, nlong): spans of the copy's entries, a wave
// walks the row pieces of its span.
constexpr int kRelabelSteps = 8;
__global__ __launch_bounds__(256) void relabel_rows_long(RelabelArgs a) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    const u64 total = a.rs_t[a.nlong];
    for (u64 s0 = wave * a.span; s0 < total; s0 += nw * a.span) {
        const u64 s1 = min(s0 + a.span, total);
        u64 p = row_at(a.rs_t, a.nlong, s0);
        for (u64 k = s0; k < s1; ++p) {
            const u64 e = min(a.rs_t[p + 1], s1);
            const u64 from = a.rs[a.iperm[p]] - a.rs_t[p];  // source position - copy's position
            for (; k < e; k += kRelabelSteps * kWave) {
                u32 c[kRelabelSteps];
                f32 wk[kRelabelSteps];
#pragma unroll
                for (int q = 0; q < kRelabelSteps; ++q) {
                    const u64 i = k + (u64)q * kWave + lane;
                    c[q] = i < e ? a.col[from + i] : 0;
                    wk[q] = i < e ? a.w[from + i] : 0.0f;
                }
#pragma unroll
                for (int q = 0; q < kRelabelSteps; ++q) c[q] = a.perm[c[q]];
#pragma unroll
                for (int q = 0; q < kRelabelSteps; ++q) {
                    const u64 i = k + (u64)q * kWave + lane;
                    if (i < e) {
                        a.col_t[i] = c[q];
                        a.w_t[i] = wk[q];
                    }
                }
            }
            k = e;
        }
    }
}

// The other rows: a wave takes `per` of them and gives each G lanes, the power
// of two that holds the longest (neighbours have the same length in this order).
__global__ __launch_bounds__(256) void relabel_rows_short(RelabelArgs a) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    for (u64 p0 = a.nlong + wave * a.per; p0 < a.n; p0 += nw * a.per) {
        const bool mine = lane < a.per && p0 + lane < a.n;
        const u64 to = mine ? a.rs_t[p0 + lane] : 0;
        const u32 len = mine ? (u32)(a.rs_t[p0 + lane + 1] - to) : 0;
        const u64 from = len ? a.rs[a.iperm[p0 + lane]] : 0;
        const u32 longest = ~wave_min(~len);
        if (!longest) continue;
        u32 G = 1;
        while (G < longest) G <<= 1;
        const u32 step = kWave / G, k = lane & (G - 1);
        for (u32 r = 0; r < a.per; r += 4 * step) {  // four groups of rows in flight
            u32 c[4];
            f32 wk[4];
            u64 o[4];
            bool in[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u32 j = r + (u32)q * step + lane / G, js = j & (kWave - 1);
                const u32 lj = __shfl(len, (int)js);
                const u64 f = shfl64(from, (int)js);
                o[q] = shfl64(to, (int)js) + k;
                in[q] = j < (u32)kWave && k < lj;
                c[q] = in[q] ? a.col[f + k] : 0;
                wk[q] = in[q] ? a.w[f + k] : 0.0f;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) c[q] = a.perm[c[q]];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (in[q]) {
                    a.col_t[o[q]] = c[q];
                    a.w_t[o[q]] = wk[q];
                }
        }
    }
}

// Units of a kernel's work that one wave takes at a time: `most`, halved down
// to `least` while that leaves waves of the chip without any.
static u64 wave_share(u64 units, u64 least, u64 most) {
    u64 share = most;
    while (share > least && units / share < (u64)ctx().num_cus * 32) share /= 2;
    return share;
}

// ---------------------------------------------------------------- SSSP copy
// An entry (u, v, w) of the traversal copy is left out of the SSSP copy when
// a two-hop path u-x-v through one of the kPruneHubs highest-degree vertices
// (ties to the smaller traversal id) is lighter by more than kPruneMargin:
// hw[u][x] + hw[v][x] + kPruneMargin < w, with hw[y][x] the lightest weight of
// an entry (y, x) (+inf without one), summed in f64 (exact for f32 weights
// below kPruneMaxWeight that are multiples of 2^-31, as generated weights are;
// otherwise off by far less than the margin).
//
// Why distances do not change: both hops of a dropped entry are lighter than
// it, so by induction on weight every dropped entry is beaten by a path of
// kept entries that is lighter by more than (hops - 1) margins. Along that
// path f32 rounding costs at most half an ulp per addition, and comparing
// with fl(d + w) costs another half: with every value below 2048 + 2, an ulp
// is at most 2^-12, and (h - 1) * 2^-10 > (h + 1) * 2^-13 for every h >= 2.
// So fl(d(u) + w) is never below what the kept path gives v, the entry never
// decides a distance, and the f32 fixpoint (the distances) is the same with
// or without it. Parents stay valid for the full graph's certificate.
constexpr int kPruneHubs = 32;
constexpr double kPruneMargin = 1.0 / 1024.0;
constexpr f32 kPruneMaxWeight = 2.0f;

// The hubs' traversal ids, by slot.
struct HubIds {
    u32 id[kPruneHubs];
    u32 count;
};

// hw[y][slot of x] (f32 bits; non-negative floats order as their bits) from
// the hubs' own rows: the graph is symmetric, so entry (x, y, w) stands for
// (y, x, w). Reading every row for its entries to hubs took 2.8 ms at S23,
// this 0.2.
__global__ __launch_bounds__(256) void prune_hub_weights(const u64 *__restrict__ rs, const u32 *__restrict__ col,
                                                         const f32 *__restrict__ w, HubIds hubs,
                                                         u32 *__restrict__ hw) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    const u32 x = blockIdx.y;
    const u64 b = rs[hubs.id[x]], e = rs[hubs.id[x] + 1];
    for (u64 k = b + (u64)blockIdx.x * blockDim.x + threadIdx.x; k < e; k += stride)
        atomicMin(&hw[(u64)col[k] * kPruneHubs + x], __float_as_uint(w[k]));
}

// Row u's hub weights, and their minimum (an entry lighter than it plus the
// margin cannot be beaten).
struct HubRow {
    f32 h[kPruneHubs];
    f32 hmin;
};
__device__ __forceinline__ void load_hub_row(const u32 *hw, u64 u, HubRow &r) {
    const uint4 *p = reinterpret_cast<const uint4 *>(hw + u * kPruneHubs);
    r.hmin = __uint_as_float(0x7F800000u);
#pragma unroll
    for (int q = 0; q < kPruneHubs / 4; ++q) {
        const uint4 c = p[q];
        r.h[4 * q] = __uint_as_float(c.x);
        r.h[4 * q + 1] = __uint_as_float(c.y);
        r.h[4 * q + 2] = __uint_as_float(c.z);
        r.h[4 * q + 3] = __uint_as_float(c.w);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.hmin = fminf(r.hmin, r.h[4 * q + i]);
    }
}

// Whether entry (u, v, w) of row u is beaten by a two-hop path through a hub.
__device__ __forceinline__ bool prune_entry(const HubRow &r, const u32 *hw, u32 v, f32 w) {
    if (!(w < kPruneMaxWeight) || !((double)r.hmin + kPruneMargin < (double)w)) return false;
    const uint4 *p = reinterpret_cast<const uint4 *>(hw + (u64)v * kPruneHubs);
    double best = __builtin_inf();
#pragma unroll
    for (int q = 0; q < kPruneHubs / 4; ++q) {
        const uint4 c = p[q];
        best = fmin(best, (double)r.h[4 * q] + (double)__uint_as_float(c.x));
        best = fmin(best, (double)r.h[4 * q + 1] + (double)__uint_as_float(c.y));
        best = fmin(best, (double)r.h[4 * q + 2] + (double)__uint_as_float(c.z));
        best = fmin(best, (double)r.h[4 * q + 3] + (double)__uint_as_float(c.w));
    }
    return best + kPruneMargin < (double)w;
}

// The hub table in 8 bits: q = ceil(127 w) of a weight below kPruneMaxWeight,
// 255 without one (or a heavier one). The least sum S of two rows' q bounds the
// least sum of weights: it is at most S / 127 (S <= 253, both below 255), and
// at least (S - 2) / 127. Where that settles an entry, its 32-byte row
// replaces a 128-byte one, and the rows of the few thousand vertices that hold
// half of all endpoints stay in an L2; about 2 % of the entries are left to
// the exact rows. With `quant` null every entry takes the exact rows.
constexpr f32 kQuant = 127.0f;
__global__ __launch_bounds__(256) void prune_quantise(const u32 *__restrict__ hw, u64 n, u32 *__restrict__ quant) {
    // a lane per 4 hubs
    const u64 total = n * (kPruneHubs / 4);
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (u64)gridDim.x * blockDim.x) {
        const uint4 c = reinterpret_cast<const uint4 *>(hw)[i];
        const u32 b[4] = {c.x, c.y, c.z, c.w};
        u32 q = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const f32 w = __uint_as_float(b[k]);
            q |= (w < kPruneMaxWeight ? (u32)ceil((double)w * (double)kQuant) : 255u) << (8 * k);
        }
        quant[i] = q;
    }
}

// A vertex's 8-bit row as 16-bit pairs.
typedef unsigned short Pair16 __attribute__((ext_vector_type(2)));
struct QuantRow {
    Pair16 p[kPruneHubs / 2];
};
__device__ __forceinline__ void load_quant_row(const u32 *quant, u64 v, QuantRow &r) {
    const uint4 *q = reinterpret_cast<const uint4 *>(quant + v * (kPruneHubs / 4));
    const uint4 x = q[0], y = q[1];
    const u32 d[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        r.p[2 * i] = __builtin_bit_cast(Pair16, d[i] & 0x00FF00FFu);
        r.p[2 * i + 1] = __builtin_bit_cast(Pair16, (d[i] >> 8) & 0x00FF00FFu);
    }
}
__device__ __forceinline__ u32 quant_sum(const QuantRow &a, const QuantRow &b) {
    Pair16 m = a.p[0] + b.p[0];
#pragma unroll
    for (int i = 1; i < kPruneHubs / 2; ++i) m = __builtin_elementwise_min(m, a.p[i] + b.p[i]);
    return min((u32)m.x, (u32)m.y);
}

// Whether entry (u, v, w) is kept; ru: u's 8-bit row (when there is a table).
__device__ __forceinline__ bool keep_entry(const u32 *hw, const u32 *quant, const QuantRow &ru, u32 u, u32 v, f32 w) {
    if (!(w < kPruneMaxWeight)) return true;
    if (quant) {
        QuantRow rv;
        load_quant_row(quant, v, rv);
        const f32 s = (f32)quant_sum(ru, rv);
        constexpr f32 kSlack = 1e-5f;  // far above the rounding of these comparisons, all below 8
        if (s <= 253.0f && s / kQuant + (f32)kPruneMargin + kSlack < w) return false;
        if ((s - 2.0f) / kQuant + (f32)kPruneMargin - kSlack >= w) return true;
    }
    HubRow r;
    load_hub_row(hw, u, r);
    return !prune_entry(r, hw, v, w);
}

// The kept entries as bits over the traversal copy's entry positions.
struct PruneArgs {
    const u64 *rs;
    const u32 *col;
    const f32 *w;
    const u32 *hw, *quant;
    u64 *bits;  // zero at the start
    u64 nlong, n;
    u64 span;   // entries of a wave's piece of the long rows
    u32 per;    // short rows per wave
};

// `mask`: the kept ones of 64 consecutive entries from position k on.
__device__ __forceinline__ void put_bits(u64 *bits, u64 k, u64 mask) {
    const u32 s = (u32)(k & 63);
    atomicOr((unsigned long long *)&bits[k >> 6], (unsigned long long)(mask << s));
    if (s && mask >> (64 - s)) atomicOr((unsigned long long *)&bits[(k >> 6) + 1], (unsigned long long)(mask >> (64 - s)));
}

// Rows longer than a wave, [0, nlong): the entries in spans over the grid, a
// wave walks the row pieces of its span, so that a row's own table row is
// read once per piece and the longest rows spread over the chip.
constexpr int kPruneSteps = 4;
__global__ __launch_bounds__(256) void prune_keep_long(PruneArgs a) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    const u64 total = a.rs[a.nlong];
    for (u64 s0 = wave * a.span; s0 < total; s0 += nw * a.span) {
        const u64 s1 = min(s0 + a.span, total);
        u64 u = row_at(a.rs, a.nlong, s0);
        for (u64 k = s0; k < s1; ++u) {
            const u64 e = min(a.rs[u + 1], s1);
            QuantRow ru = {};
            if (a.quant) load_quant_row(a.quant, u, ru);
            for (; k < e; k += kPruneSteps * kWave) {
                u32 v[kPruneSteps];
                f32 wk[kPruneSteps];
                bool in[kPruneSteps];
#pragma unroll
                for (int q = 0; q < kPruneSteps; ++q) {
                    const u64 i = k + (u64)q * kWave + lane;
                    in[q] = i < e;
                    v[q] = in[q] ? a.col[i] : 0;
                    wk[q] = in[q] ? a.w[i] : 0.0f;
                }
#pragma unroll
                for (int q = 0; q < kPruneSteps; ++q) {
                    const u64 m = ballot(in[q] && keep_entry(a.hw, a.quant, ru, (u32)u, v[q], wk[q]));
                    if (lane == 0 && m) put_bits(a.bits, k + (u64)q * kWave, m);
                }
            }
            k = e;
        }
    }
}

// The other rows: a wave takes `per` of them and gives each G lanes, the power
// of two that holds the longest (neighbours have the same length in this order).
__global__ __launch_bounds__(256) void prune_keep_short(PruneArgs a) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    for (u64 u0 = a.nlong + wave * a.per; u0 < a.n; u0 += nw * a.per) {
        const u64 mine = min(u0 + lane, a.n - 1);
        const u64 b = a.rs[mine];
        const u32 len = lane < a.per && u0 + lane < a.n ? (u32)(a.rs[mine + 1] - b) : 0;
        const u32 longest = ~wave_min(~len);
        if (!longest) continue;
        u32 G = 1;
        while (G < longest) G <<= 1;
        for (u32 r = 0; r < a.per; r += kWave / G) {
            const u32 j = r + lane / G, k = lane & (G - 1);
            const u64 bj = shfl64(b, (int)j);
            const u32 lj = __shfl(len, (int)j);
            bool keep = false;
            if (k < lj) {
                const u64 u = u0 + j;
                QuantRow ru = {};
                if (a.quant) load_quant_row(a.quant, u, ru);
                keep = keep_entry(a.hw, a.quant, ru, (u32)u, a.col[bj + k], a.w[bj + k]);
            }
            const u64 m = ballot(keep) >> (lane & ~(G - 1));
            const u64 own = G == (u32)kWave ? m : m & ((1ull << G) - 1);
            if (k == 0 && own) put_bits(a.bits, bj, own);
        }
    }
}

// Compaction by the bits, in entry order, so without rows: kept entries per
// tile of 8 words, their scan, then rows offsets and entries from the tiles.
constexpr u64 kKeepTile = 512;
__device__ __forceinline__ u64 keep_word(const u64 *bits, u64 word, u64 m) {
    return word * 64 < m ? bits[word] : 0ull;
}
__global__ __launch_bounds__(256) void prune_count(const u64 *__restrict__ bits, u64 m, u64 ntiles,
                                                   u32 *__restrict__ counts) {
    for (u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x; t < ntiles; t += (u64)gridDim.x * blockDim.x) {
        u32 c = 0;
#pragma unroll
        for (u64 i = 0; i < kKeepTile / 64; ++i) c += (u32)__popcll(keep_word(bits, t * (kKeepTile / 64) + i, m));
        counts[t] = c;
    }
}
__global__ __launch_bounds__(256) void prune_rowstarts(const u64 *__restrict__ rs, u64 n, const u64 *__restrict__ bits,
                                                       const u64 *__restrict__ tile_off, u64 *__restrict__ rs_s) {
    for (u64 u = (u64)blockIdx.x * blockDim.x + threadIdx.x; u <= n; u += (u64)gridDim.x * blockDim.x) {
        const u64 k = rs[u], t = k / kKeepTile;
        u64 o = tile_off[t];
        for (u64 i = t * (kKeepTile / 64); i < k / 64; ++i) o += (u64)__popcll(bits[i]);
        if (k & 63) o += (u64)__popcll(bits[k / 64] & ((1ull << (k & 63)) - 1));
        rs_s[u] = o;
    }
}
__global__ __launch_bounds__(256) void prune_compact(const u32 *__restrict__ col, const f32 *__restrict__ w, u64 m,
                                                     const u64 *__restrict__ bits, const u64 *__restrict__ tile_off,
                                                     u64 ntiles, u32 *__restrict__ col_s, f32 *__restrict__ w_s) {
    const u32 lane = lane_id();
    const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / kWave, nw = (u64)gridDim.x * blockDim.x / kWave;
    constexpr int kWords = kKeepTile / 64;
    for (u64 t = wave; t < ntiles; t += nw) {
        u64 word[kWords], o[kWords + 1];
        o[0] = tile_off[t];
#pragma unroll
        for (int i = 0; i < kWords; ++i) {
            word[i] = keep_word(bits, t * kWords + i, m);
            o[i + 1] = o[i] + (u64)__popcll(word[i]);
        }
        u32 c[kWords];
        f32 wk[kWords];
#pragma unroll
        for (int i = 0; i < kWords; ++i) {
            const u64 k = t * kKeepTile + (u64)i * 64 + lane;
            const bool keep = (word[i] >> lane) & 1;
            c[i] = keep ? col[k] : 0;
            wk[i] = keep ? w[k] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kWords; ++i)
            if ((word[i] >> lane) & 1) {
                const u64 at = o[i] + mask_rank(word[i]);
                col_s[at] = c[i];
                w_s[at] = wk[i];
            }
    }
}

// Exclusive scan of counts[0, n) into offsets[0, n], the total last.
static void scan_counts(const u32 *counts, u64 n, u64 *tiles, u64 *offsets, hipStream_t s) {
    const u64 ntiles = (n + kScanTile - 1) / kScanTile;
    scan_tile_sums<<<(unsigned)ntiles, kScanBlock, 0, s>>>(counts, n, tiles);
    scan_tile_offsets<<<1, 1024, 0, s>>>(tiles, ntiles, offsets, n);
    scan_write<<<(unsigned)ntiles, kScanBlock, 0, s>>>(counts, n, tiles, offsets);
    G500_HIP(hipGetLastError());
}
static u64 scan_tile_bytes(u64 n) { return ((n + kScanTile - 1) / kScanTile + 1) * sizeof(u64); }

// Builds g's SSSP copy from its traversal copy (rows longer than kWave
// entries, the first nlong, are walked in pieces; the first ntop rows are the
// degree class above the exact range, in no particular order). Each entry is
// judged once, into a bit; the kept ones are then compacted in entry order
// (23.6 ms at S23 with two hub tables and two exact judgements, now 5.5).
// Scratch: the 8-bit hub table, the bits and their tile offsets lie where the
// copy's entries will (at most the traversal copy's size), followed by the
// hub table; before the entries are written, the bits move into the hub
// table's place.
void build_sssp_copy(Worker_State *ws, Oned_Graph *g, u64 nlong, u64 ntop) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, m = g->nlocaledges;
    const u64 ntiles = (m + kKeepTile - 1) / kKeepTile;
    auto align = [](u64 x) { return (x + 255) & ~255ull; };
    // bits (and a word beyond, for the last row's end), tile counts, scan tiles, tile offsets
    const u64 bits_bytes = align((m / 64 + 2) * sizeof(u64)), off_bytes = align((ntiles + 1) * sizeof(u64));
    const u64 kept_bytes = bits_bytes + off_bytes, count_bytes = align(ntiles * sizeof(u32)) + align(scan_tile_bytes(ntiles));
    const u64 table_bytes = align(n * kPruneHubs * sizeof(u32)), quant_bytes = align(n * kPruneHubs);
    const u64 entry_bytes = 2 * align(MAX(m, (u64)1) * sizeof(u32));
    // The copy is an optimization: without arena room for row offsets, entries
    // at full size and the hub table (and a reserve of 8 bytes a vertex and
    // 8 MiB) the graph keeps none, and SSSP relaxes the traversal copy. The bits
    // and their counts always fit in that room, the 8-bit table beside them
    // except on graphs of fewer than 5 entries a vertex. On graphs of hundreds of
    // entries a vertex, whose bits outgrow the hub table, the room left for the
    // entries may be less than full size: the kept ones are held against it.
    const u64 start = ws->gpu_arena.used, room = ws->gpu_arena.reserved - start;
    const u64 least = (n + 1) * 8 + m * 8 + n * kPruneHubs * 4 + n * 8 + (8u << 20);
    auto no_room = [&](u64 bytes) {
        fprintf(stderr, "libg500: no arena room for the SSSP copy (%llu bytes); SSSP relaxes the traversal copy\n",
                (unsigned long long)bytes);
        ws->gpu_arena.used = start;
    };
    if (least > room) return no_room(least);
    const u64 high_bytes = MAX(table_bytes, kept_bytes);
    const u64 low_room = room - (align((n + 1) * 8) + high_bytes + 1024);
    // the hubs: the kPruneHubs largest degrees among the first max(ntop, kPruneHubs)
    // rows (every later row is no longer), ties to the smaller id
    const u64 nhead = MIN(n, MAX(ntop, (u64)kPruneHubs));
    std::vector<u64> head(nhead + 1);
    G500_HIP(hipMemcpyAsync(head.data(), g->rowstarts_t, (nhead + 1) * sizeof(u64), hipMemcpyDeviceToHost, s));
    sync();
    if (failed()) return;
    std::vector<u32> ids(nhead);
    for (u64 i = 0; i < nhead; ++i) ids[i] = (u32)i;
    HubIds hubs = {};
    hubs.count = (u32)MIN(nhead, (u64)kPruneHubs);
    std::partial_sort(ids.begin(), ids.begin() + hubs.count, ids.end(), [&](u32 x, u32 y) {
        const u64 dx = head[x + 1] - head[x], dy = head[y + 1] - head[y];
        return dx != dy ? dx > dy : x < y;
    });
    u64 hub_longest = 1, hub_entries = 0;
    for (u32 i = 0; i < hubs.count; ++i) {
        hubs.id[i] = ids[i];
        hub_longest = MAX(hub_longest, head[ids[i] + 1] - head[ids[i]]);
        hub_entries += head[ids[i] + 1] - head[ids[i]];
    }
    // The 8-bit table costs 160 bytes a vertex and pays where many rows reach a
    // hub; a row that reaches none keeps its entries by its exact row alone.
    // Whole construction with / without it, us, by hub entries a vertex: S20 0.07
    // 1204 / 1197, 0.14 1375 / 1366, 0.21 1233 / 1254, 0.63 2250 / 2380, 1.1 3297 / 3516; 4e6
    // uniform vertices (none) with 12e6 edges 2663 / 2354, with 64e6 11509 / 10397; a
    // path of 1e7 2529 / 2170.
    const bool quantised = hub_entries >= n / 8 && kept_bytes + count_bytes + quant_bytes <= low_room;
    u64 *rs_s = (u64 *)arena_alloc(ws, (n + 1) * sizeof(u64), "SSSP row offsets");
    if (failed()) return;
    const u64 mark = ws->gpu_arena.used;
    const u64 quant_used = quantised ? quant_bytes : 0;
    const u64 low_bytes = MIN(low_room, MAX(entry_bytes, kept_bytes + count_bytes + quant_used));
    u8 *low = (u8 *)arena_alloc(ws, low_bytes, "SSSP prune scratch");
    u8 *high = (u8 *)arena_alloc(ws, high_bytes, "SSSP prune hub table");
    if (failed()) return;
    u64 *bits = (u64 *)low, *tile_off = (u64 *)(low + bits_bytes);
    u32 *counts = (u32 *)(low + kept_bytes);
    u64 *tiles = (u64 *)(low + kept_bytes + align(ntiles * sizeof(u32)));
    u32 *quant = quantised ? (u32 *)(low + kept_bytes + count_bytes) : nullptr;
    u32 *hw = (u32 *)high;
    G500_HIP(hipMemsetD32Async(hw, 0x7F800000u, n * kPruneHubs, s));
    G500_HIP(hipMemsetAsync(bits, 0, bits_bytes, s));
    prune_hub_weights<<<dim3(grid_for(hub_longest, 256, 256), hubs.count), 256, 0, s>>>(g->rowstarts_t, g->column_t,
                                                                                      g->weights_t, hubs, hw);
    if (quant)
        prune_quantise<<<grid_for(n * (kPruneHubs / 4), 256, (u64)c.num_cus * 32), 256, 0, s>>>(hw, n, quant);
    const PruneArgs a = {g->rowstarts_t, g->column_t, g->weights_t, hw, quant, bits, nlong, n, wave_share(m, 256, 4096),
                         (u32)wave_share(n - nlong, 1, kWave)};
    if (nlong) prune_keep_long<<<grid_for(m / a.span * kWave + kWave, 256, (u64)c.num_cus * 16), 256, 0, s>>>(a);
    if (nlong < n) prune_keep_short<<<grid_for((n - nlong) / a.per * kWave + kWave, 256, (u64)c.num_cus * 16), 256, 0, s>>>(a);
    prune_count<<<grid_for(ntiles, 256, (u64)c.num_cus * 16), 256, 0, s>>>(bits, m, ntiles, counts);
    G500_HIP(hipGetLastError());
    if (ntiles) scan_counts(counts, ntiles, tiles, tile_off, s);
    else G500_HIP(hipMemsetAsync(tile_off, 0, sizeof(u64), s));
    u64 m_s = 0;
    G500_HIP(hipMemcpyAsync(&m_s, tile_off + ntiles, sizeof(u64), hipMemcpyDeviceToHost, s));
    G500_HIP(hipMemcpyAsync(high, low, kept_bytes, hipMemcpyDeviceToDevice, s));
    sync();
    if (failed()) return;
    const u64 kept_entries = 2 * align(MAX(m_s, (u64)1) * sizeof(u32));
    if (kept_entries > low_bytes) return no_room(kept_entries - low_bytes + room);
    ws->gpu_arena.used = mark;
    u32 *col_s = (u32 *)arena_alloc(ws, MAX(m_s, (u64)1) * sizeof(u32), "SSSP columns");
    f32 *w_s = (f32 *)arena_alloc(ws, MAX(m_s, (u64)1) * sizeof(f32), "SSSP weights");
    if (failed()) return;
    bits = (u64 *)high;
    tile_off = (u64 *)(high + bits_bytes);
    prune_rowstarts<<<grid_for(n + 1, 256, (u64)c.num_cus * 32), 256, 0, s>>>(g->rowstarts_t, n, bits, tile_off, rs_s);
    if (ntiles)
        prune_compact<<<grid_for(ntiles * kWave, 256, (u64)c.num_cus * 32), 256, 0, s>>>(
            g->column_t, g->weights_t, m, bits, tile_off, ntiles, col_s, w_s);
    G500_HIP(hipGetLastError());
    sync();
    if (failed()) return;
    g->rowstarts_s = rs_s;
    g->column_s = col_s;
    g->weights_s = w_s;
}

// Builds g's traversal copy (perm, iperm, rowstarts_t, column_t, weights_t)
// on the library stream; scratch is taken above the arena mark and released.
void build_traversal_copy(Worker_State *ws, Oned_Graph *g) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, m = g->nlocaledges;
    g->perm = (u32 *)arena_alloc(ws, n * sizeof(u32), "traversal ids");
    g->iperm = (u32 *)arena_alloc(ws, n * sizeof(u32), "original ids");
    g->rowstarts_t = (u64 *)arena_alloc(ws, (n + 1) * sizeof(u64), "traversal row offsets");
    g->column_t = (u32 *)arena_alloc(ws, m * sizeof(u32), "traversal columns");
    g->weights_t = (f32 *)arena_alloc(ws, m * sizeof(f32), "traversal weights");
    const u64 mark = ws->gpu_arena.used;
    u32 *counts = (u32 *)arena_alloc(ws, 2 * kDegKeys * sizeof(u32), "relabel counts");
    u32 *deg_t = (u32 *)arena_alloc(ws, n * sizeof(u32), "relabel degrees");
    const u64 ntiles = (n + kScanTile - 1) / kScanTile;
    u64 *tiles = (u64 *)arena_alloc(ws, (ntiles + 1) * sizeof(u64), "relabel scan tiles");
    if (failed()) return;
    u32 *cursor = counts + kDegKeys;
    const unsigned nblk = (unsigned)((n + (u64)kRelabelBlock * kRelabelItems - 1) / ((u64)kRelabelBlock * kRelabelItems));
    G500_HIP(hipMemsetAsync(counts, 0, kDegKeys * sizeof(u32), s));
    relabel_count<<<nblk, kRelabelBlock, 0, s>>>(g->rowstarts, n, counts);
    relabel_offsets<<<1, 1024, 0, s>>>(counts, cursor);
    relabel_scatter<<<nblk, kRelabelBlock, 0, s>>>(g->rowstarts, n, cursor, g->perm, g->iperm, deg_t);
    scan_tile_sums<<<(unsigned)ntiles, kScanBlock, 0, s>>>(deg_t, n, tiles);
    scan_tile_offsets<<<1, 1024, 0, s>>>(tiles, ntiles, g->rowstarts_t, n);
    scan_write<<<(unsigned)ntiles, kScanBlock, 0, s>>>(deg_t, n, tiles, g->rowstarts_t);
    G500_HIP(hipGetLastError());
    // rows longer than kWave entries: keys below kDegKeys - 1 - kWave
    u32 hc[kDegKeys];
    G500_HIP(hipMemcpyAsync(hc, counts, sizeof(hc), hipMemcpyDeviceToHost, s));
    sync();
    u64 nlong = 0;
    for (u32 k = 0; k < kDegKeys - 1 - (u32)kWave; ++k) nlong += hc[k];
    const RelabelArgs a = {g->rowstarts, g->column, g->weights, g->perm, g->iperm, g->rowstarts_t, g->column_t,
                           g->weights_t, nlong, n, wave_share(m, 512, 4096), (u32)wave_share(n - nlong, 1, kWave)};
    if (nlong)
        relabel_rows_long<<<grid_for(m / a.span * kWave + kWave, 256, (u64)c.num_cus * 16), 256, 0, s>>>(a);
    if (nlong < n)
        relabel_rows_short<<<grid_for((n - nlong) / a.per * kWave + kWave, 256, (u64)c.num_cus * 16), 256, 0, s>>>(a);
    G500_HIP(hipGetLastError());
    sync();
    ws->gpu_arena.used = mark;
    if (c.sssp_prune && !failed()) build_sssp_copy(ws, g, nlong, hc[0]);
}

// Tuple lists below this take the direct path, where the partition's launches
// cost more than scattered accesses in cache. Whole construction, direct /
// partition, us: 48 Ki tuples (3000 uniform vertices) 490 / 520, S12 (64 Ki)
// 876 / 800, S14 1259 / 1045, S16 2346 / 1762, S18 5046 / 3673, S20 14348 / 11278,
// S22 47674 / 34400.
constexpr u64 kPartitionTuples = 1ull << 16;
// So do lists below this with at most two tuples a vertex, whose atomics seldom
// meet: 1e5 tuples over 1e5 vertices, a path 378 / 432, uniform 379 / 398; 3e5 over
// 1e5 uniform 417 / 406, 1e6 over 5e5 684 / 684, 2e6 over 2e6 1240 / 1078.
constexpr u64 kPartitionSparse = 1ull << 18;
// And lists of any length whose tuples lie near the ones before them (meshes,
// paths and bands numbered along themselves): a wave's atomics and writes then
// share lines, without meeting on a vertex, which the partition cannot better.
// A 1000 x 1000 grid 633 / 771, 4000 x 4000 4585 / 6016, a path of 1e7 2439 / 3038, a
// binary tree of 1e7 (half of the tuples near) 3100 / 3631; a band of five entries
// after another at each vertex (one in five near) 1363 / 1141. Half of that last
// but one case's share is the line.
static bool tuples_are_near(u32 seen, u32 near) { return (u64)near * 8 >= (u64)seen * 3; }

static bool bad_endpoints(u64 n) {
    fail("oned_graph_from_tuple_graph: tuple endpoint outside [0, %llu)", (unsigned long long)n);
    return false;
}

// Row offsets, columns and weights (rows unsorted) through per-row cursors.
static bool fill_direct(Worker_State *ws, const Tuple_Graph *tg, Oned_Graph *g) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, ne = tg->edges_size;
    const u64 mark = ws->gpu_arena.used;
    u32 *deg = (u32 *)arena_alloc(ws, n * sizeof(u32), "CSR degrees");
    u64 *tiles = (u64 *)arena_alloc(ws, scan_tile_bytes(n) + 16, "CSR scan tiles");
    if (failed()) return false;
    u32 *bad = (u32 *)((u8 *)tiles + scan_tile_bytes(n));
    G500_HIP(hipMemsetAsync(deg, 0, n * sizeof(u32), s));
    G500_HIP(hipMemsetAsync(bad, 0, sizeof(u32), s));
    if (ne) degree_kernel<<<grid_for(ne, 256, (u64)c.num_cus * 64), 256, 0, s>>>(tg->edges, ne, n, deg, bad);
    scan_counts(deg, n, tiles, g->rowstarts, s);
    u64 m = 0;
    u32 hbad = 0;
    G500_HIP(hipMemcpyAsync(&m, g->rowstarts + n, sizeof(u64), hipMemcpyDeviceToHost, s));
    G500_HIP(hipMemcpyAsync(&hbad, bad, sizeof(u32), hipMemcpyDeviceToHost, s));
    sync();
    if (hbad) return bad_endpoints(n);
    if (failed()) return false;
    // the scratch moves above the column and weight arrays, to be released afterwards
    ws->gpu_arena.used = mark;
    g->nlocaledges = m;
    g->column = (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR columns");
    g->weights = (f32 *)arena_alloc(ws, m * sizeof(f32), "CSR weights");
    const u64 mark_fill = ws->gpu_arena.used;
    u32 *cursor = (u32 *)arena_alloc(ws, n * sizeof(u32), "CSR cursors");
    if (failed()) return false;
    G500_HIP(hipMemsetAsync(cursor, 0, n * sizeof(u32), s));
    if (ne)
        fill_kernel<<<grid_for(ne, 256, (u64)c.num_cus * 64), 256, 0, s>>>(tg->edges, tg->weights, ne, n,
                                                                          g->rowstarts, cursor, g->column,
                                                                          g->weights);
    G500_HIP(hipGetLastError());
    ws->gpu_arena.used = mark_fill;
    return !failed();
}

// Whether the partition path is tried: lists above the limits whose entry counts
// fit 32 bits (below 2^31 tuples), when the arena has room for its scratch (16
// bytes an entry beside the columns and weights, 5 a vertex, and 64 MiB for
// offsets and rounding; the copies built later need as much).
static bool partition_pays(const Worker_State *ws, u64 n, u64 ne) {
    const u64 room = ws->gpu_arena.reserved - ws->gpu_arena.used;
    return ne >= kPartitionTuples && (ne >= kPartitionSparse || ne > 2 * n) && 2 * ne < (1ull << 32) &&
           2 * ne * 24 + n * 5 + (64ull << 20) <= room;
}

// The same arrays by partition (see partition_kernel), unless the tuples turn
// out to be near each other.
static bool fill_partitioned(Worker_State *ws, const Tuple_Graph *tg, Oned_Graph *g) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, ne = tg->edges_size;
    const u64 mark = ws->gpu_arena.used;
    u32 bits = 1;
    while (bits < 32 && (1ull << bits) < n) ++bits;
    // two passes up to 2^18 rows, else three; at most 11 bits each
    const u32 d1 = bits <= 18 ? (bits + 1) / 2 : (bits + 2) / 3;
    const u32 shift1 = bits - d1, shift2 = bits <= 18 ? 0 : shift1 / 2;
    const u64 nb1 = ((n - 1) >> shift1) + 1, nb2 = ((n - 1) >> shift2) + 1;
    // pass 1's counts, whose sum is the number of entries
    std::vector<u32> h(kPartWords);
    std::vector<u64> first(nb1 + 1);
    u32 *count1 = (u32 *)arena_alloc(ws, kPartWords * sizeof(u32), "CSR partition counts");
    if (failed()) return false;
    G500_HIP(hipMemsetAsync(count1, 0, kPartWords * sizeof(u32), s));
    partition_count_tuples<<<(unsigned)c.num_cus * 2, 1024, 0, s>>>(tg->edges, ne, n, shift1, count1);
    G500_HIP(hipGetLastError());
    G500_HIP(hipMemcpyAsync(h.data(), count1, kPartWords * sizeof(u32), hipMemcpyDeviceToHost, s));
    sync();
    if (failed()) return false;
    if (h[kPartBad]) return bad_endpoints(n);
    if (tuples_are_near(h[kPartSeen], h[kPartNear])) {
        ws->gpu_arena.used = mark;
        return fill_direct(ws, tg, g);
    }
    u64 m = 0;
    for (u64 b = 0; b < nb1; ++b) {
        first[b] = m;
        m += h[b];
    }
    ws->gpu_arena.used = mark;
    g->nlocaledges = m;
    g->column = (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR columns");
    g->weights = (f32 *)arena_alloc(ws, m * sizeof(f32), "CSR weights");
    const u64 mark_fill = ws->gpu_arena.used;
    u64 *next1 = (u64 *)arena_alloc(ws, nb1 * sizeof(u64), "CSR partition offsets");
    u32 *deg = (u32 *)arena_alloc(ws, n * sizeof(u32), "CSR degrees");
    u64 *tiles = (u64 *)arena_alloc(ws, scan_tile_bytes(n), "CSR scan tiles");
    // the last pass's input, and pass 1's rows when there are three
    u32 *row2 = (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR partition rows");
    u32 *col2 = (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR partition columns");
    u32 *w2 = (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR partition weights");
    u32 *row1 = shift2 ? (u32 *)arena_alloc(ws, m * sizeof(u32), "CSR partition rows") : nullptr;
    u64 *next2 = shift2 ? (u64 *)arena_alloc(ws, (nb2 + 1) * sizeof(u64), "CSR partition offsets") : nullptr;
    if (failed()) return false;
    const unsigned max_blocks = (unsigned)c.num_cus;  // a block's LDS fills a CU
    const unsigned count_blocks = grid_for(m, 1024 * kCountItems, (u64)c.num_cus * 4);
    auto pass = [&](auto tuples, PartArgs a) {
        constexpr bool kTuples = decltype(tuples)::value;
        partition_kernel<kTuples><<<grid_for(a.count, kTuples ? kPartTile / 2 : kPartTile, max_blocks), kPartThreads,
                                    0, s>>>(a);
    };
    PartArgs a = {};
    a.edges = tg->edges;
    a.ew = tg->weights;
    a.count = ne;
    a.n = n;
    a.shift = shift1;
    a.next = next1;
    G500_HIP(hipMemcpyAsync(next1, first.data(), nb1 * sizeof(u64), hipMemcpyHostToDevice, s));
    if (shift2) {
        a.row_out = row1;
        a.col_out = g->column;
        a.w_out = (u32 *)g->weights;
        pass(std::true_type(), a);
        G500_HIP(hipMemsetAsync(deg, 0, nb2 * sizeof(u32), s));
        partition_count_rows<<<count_blocks, 1024, 0, s>>>(row1, m, shift2, deg);
        scan_counts(deg, nb2, tiles, next2, s);
        a.edges = nullptr;
        a.row_in = row1;
        a.col_in = g->column;
        a.w_in = (const u32 *)g->weights;
        a.count = m;
        a.shift = shift2;
        a.next = next2;
    }
    a.row_out = row2;
    a.col_out = col2;
    a.w_out = w2;
    if (shift2) pass(std::false_type(), a);
    else pass(std::true_type(), a);
    G500_HIP(hipMemsetAsync(deg, 0, n * sizeof(u32), s));
    partition_count_rows<<<count_blocks, 1024, 0, s>>>(row2, m, 0, deg);
    scan_counts(deg, n, tiles, g->rowstarts, s);
    G500_HIP(hipMemsetAsync(deg, 0, n * sizeof(u32), s));
    a.edges = nullptr;
    a.row_in = row2;
    a.col_in = col2;
    a.w_in = w2;
    a.count = m;
    a.shift = 0;
    a.next = nullptr;
    a.rs = g->rowstarts;
    a.used = deg;
    a.row_out = nullptr;
    a.col_out = g->column;
    a.w_out = (u32 *)g->weights;
    pass(std::false_type(), a);
    G500_HIP(hipGetLastError());
    sync();  // `first` is read by the copy
    ws->gpu_arena.used = mark_fill;
    return !failed();
}

// Fewer entries in long rows than this are sorted as whole rows, in fewer
// launches. Whole construction, whole rows / bins, us: S10 646 / 690, S14 (2.5e5
// entries in long rows) 1088 / 928, S15 1359 / 1155, S16 1745 / 1393.
constexpr u64 kLongMin = 1 << 17;

// 8-bit digits of the columns.
static int column_passes(u64 n) {
    int bits = 1;
    while (bits < 32 && (1ull << bits) < n) ++bits;
    return (bits + 7) / 8;
}

// sort_rows in the least room: three counters, and a scratch for the rows above
// kSegBlock entries.
static bool sort_rows_without_lists(Worker_State *ws, Oned_Graph *g) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, mark = ws->gpu_arena.used;
    u32 *col = g->column, *w = (u32 *)g->weights;
    UnlistedCounts *k = (UnlistedCounts *)arena_alloc(ws, sizeof(UnlistedCounts), "sort counts");
    if (failed()) return false;
    G500_HIP(hipMemsetAsync(k, 0, sizeof(UnlistedCounts), s));
    count_rows<<<grid_for(n, 256, (u64)c.num_cus * 16), 256, 0, s>>>(g->rowstarts, n, k);
    G500_HIP(hipGetLastError());
    UnlistedCounts h = {};
    G500_HIP(hipMemcpyAsync(&h, k, sizeof(h), hipMemcpyDeviceToHost, s));
    sync();
    if (failed()) return false;
    g->notisolated = h.notisolated;
    u32 *s_col = nullptr, *s_w = nullptr;
    if (h.huge_entries) {
        s_col = (u32 *)arena_alloc(ws, h.huge_entries * sizeof(u32), "sort scratch");
        s_w = (u32 *)arena_alloc(ws, h.huge_entries * sizeof(u32), "sort scratch");
        if (failed()) return false;
    }
    const u64 blocks = (u64)c.num_cus * 2;
    const u32 per = (u32)MAX((u64)1, MIN((u64)kUnlistedRows, n / (4 * blocks)));
    sort_rows_thread<<<grid_for(n, 256, (u64)c.num_cus * 32), 256, 0, s>>>(g->rowstarts, n, col, g->weights);
    sort_rows_unlisted<<<grid_for(n, (int)per, blocks), kSegThreads, 0, s>>>(g->rowstarts, n, per, col, w, s_col, s_w, k,
                                                                            column_passes(n));
    G500_HIP(hipGetLastError());
    ws->gpu_arena.used = mark;
    return !failed();
}

// Sorts every row by (weight bits, column) and counts the rows with entries.
static bool sort_rows(Worker_State *ws, Oned_Graph *g) {
    Context &c = ctx();
    const hipStream_t s = c.stream;
    const u64 n = g->nlocalverts, m = g->nlocaledges;
    const u64 mark = ws->gpu_arena.used;
    u32 *col = g->column, *w = (u32 *)g->weights;
    auto room = [&]() { return ws->gpu_arena.reserved - MIN(ws->gpu_arena.used + 255, ws->gpu_arena.reserved); };
    u64 caps[kWaveTiers], lists = sizeof(SortLists) + (kWaveTiers + 6) * 256;
    for (int q = 0; q < kWaveTiers; ++q) lists += (caps[q] = tier_cap(n, m, q ? 32u << q : 17)) * sizeof(u32);
    TierLists t;
    t.long_cap = tier_cap(n, m, kLongRow + 1);
    const u64 block_cap = tier_cap(m, m, kLongRow + 1), radix_cap = tier_cap(m, m, kSegBlock + 1);
    lists += t.long_cap * (2 * sizeof(u32) + sizeof(u64)) + (block_cap + radix_cap) * sizeof(Segment);
    if (lists > room()) return sort_rows_without_lists(ws, g);
    SortLists *L = (SortLists *)arena_alloc(ws, sizeof(SortLists) + 256, "sort lists");
    for (int q = 0; q < kWaveTiers; ++q) t.rows[q] = (u32 *)arena_alloc(ws, caps[q] * sizeof(u32), "sort tier");
    t.long_row = (u32 *)arena_alloc(ws, t.long_cap * sizeof(u32), "long rows");
    t.long_len = (u32 *)arena_alloc(ws, t.long_cap * sizeof(u32), "long row lengths");
    t.long_off = (u64 *)arena_alloc(ws, t.long_cap * sizeof(u64), "long row offsets");
    Segment *block_segs = (Segment *)arena_alloc(ws, block_cap * sizeof(Segment), "block segments");
    Segment *radix_segs = (Segment *)arena_alloc(ws, radix_cap * sizeof(Segment), "radix segments");
    if (failed()) return false;
    u32 *error = (u32 *)(L + 1);
    G500_HIP(hipMemsetAsync(L, 0, sizeof(SortLists) + 256, s));
    classify_rows<<<grid_for(n, kClassifyTile, (u64)c.num_cus * 2), 1024, 0, s>>>(g->rowstarts, n, L, t, error);
    sort_rows_thread<<<grid_for(n, 256, (u64)c.num_cus * 32), 256, 0, s>>>(g->rowstarts, n, col, g->weights);
    G500_HIP(hipGetLastError());
    SortLists h;
    G500_HIP(hipMemcpyAsync(&h, L, sizeof(h), hipMemcpyDeviceToHost, s));
    sync();
    if (failed()) return false;
    if (2 * (MAX(h.huge_entries.v, (u64)1) * sizeof(u32) + 256) > room()) {
        ws->gpu_arena.used = mark;
        return sort_rows_without_lists(ws, g);
    }
    g->notisolated = h.notisolated.v;
    TierCounts k;
    u64 nwave = 0;
    for (int q = 0; q < kWaveTiers; ++q) nwave += k.n[q] = h.n[q].v;
    if (nwave)
        sort_rows_wave<<<grid_for(nwave * kWave, 256, (u64)c.num_cus * 32), 256, 0, s>>>(g->rowstarts, t, k, col, w);
    LongRows a = {};
    a.nrows = hub_count(h.longs.v);
    a.nchunks = hub_total(h.longs.v) / kHubChunk;
    if (a.nrows) {
        a.rs = g->rowstarts;
        a.row = t.long_row;
        a.len = t.long_len;
        a.off = t.long_off;
        a.col = col;
        a.w = w;
        const u64 per_chunk = 3 * sizeof(u32) + sizeof(u64), slack = 16 * 256 + scan_tile_bytes(a.nchunks);
        const bool bins = h.long_entries.v >= kLongMin && h.long_entries.v * 8 + a.nchunks * per_chunk + a.nrows * 8 + slack <= room();
        const u64 scratch = MAX(bins ? h.long_entries.v : h.huge_entries.v, (u64)1);
        a.s_col = (u32 *)arena_alloc(ws, scratch * sizeof(u32), "sort scratch");
        a.s_w = (u32 *)arena_alloc(ws, scratch * sizeof(u32), "sort scratch");
        if (failed()) return false;
        if (bins) {
            a.chunk_row = (u32 *)arena_alloc(ws, a.nchunks * sizeof(u32), "long row chunks");
            a.count = (u32 *)arena_alloc(ws, a.nchunks * sizeof(u32), "long row bin counts");
            a.used = (u32 *)arena_alloc(ws, a.nchunks * sizeof(u32), "long row bins filled");
            a.bin_off = (u64 *)arena_alloc(ws, (a.nchunks + 1) * sizeof(u64), "long row bin offsets");
            a.wlo = (u32 *)arena_alloc(ws, a.nrows * sizeof(u32), "long row weights");
            a.whi = (u32 *)arena_alloc(ws, a.nrows * sizeof(u32), "long row weights");
            u64 *tiles = (u64 *)arena_alloc(ws, scan_tile_bytes(a.nchunks), "long row scan tiles");
            if (failed()) return false;
            const unsigned waves = grid_for(a.nchunks * kWave, 256, (u64)c.num_cus * 32);
            const unsigned spans = grid_for(a.nchunks, (int)kLongSpan, (u64)c.num_cus * 8);
            long_chunk_rows<<<grid_for(a.nrows * kWave, 256, (u64)c.num_cus * 16), 256, 0, s>>>(a);
            G500_HIP(hipMemsetAsync(a.count, 0, a.nchunks * sizeof(u32), s));
            G500_HIP(hipMemsetAsync(a.used, 0, a.nchunks * sizeof(u32), s));
            long_weight_range<<<waves, 256, 0, s>>>(a);
            long_bin_kernel<false><<<spans, kLongBlock, 0, s>>>(a);
            scan_counts(a.count, a.nchunks, tiles, a.bin_off, s);
            long_bin_kernel<true><<<spans, kLongBlock, 0, s>>>(a);
            long_sort_bins<<<waves, 256, 0, s>>>(a, L, block_segs, radix_segs);
        } else {
            long_rows_as_segments<<<grid_for(a.nrows, 256, 1024), 256, 0, s>>>(a, L, block_segs, radix_segs,
                                                                              (u64 *)(error + 2));
        }
        G500_HIP(hipGetLastError());
        // The kernels read how many segments there are: waiting for the counts would cost more than an empty launch.
        // Grids for the most that there can be, a whole row each or, in bins, any number of a row's: by rows alone one
        // block would sort every over-full bin of a lone row (ms, a row of 4e6 entries: squared uniform weights 27.6, now
        // 3.9; 255 different ones 63, now 1.9).
        const u64 most_block = bins ? tier_cap(a.nchunks, h.long_entries.v, kLongRow + 1) : a.nrows;
        const u64 most_radix = bins ? tier_cap(a.nchunks, h.long_entries.v, kSegBlock + 1) : a.nrows;
        sort_segments_block<<<(unsigned)MIN(most_block, (u64)c.num_cus * 4), kSegThreads, 0, s>>>(
            block_segs, &L->nblock.v, col, w, a.s_col, a.s_w);
        if (bins || h.huge_entries.v)
            sort_segments_radix<<<(unsigned)MIN(most_radix, (u64)c.num_cus * 2), kRadixBlock, 0, s>>>(
                radix_segs, &L->nradix.v, col, w, a.s_col, a.s_w, column_passes(n));
    }
    G500_HIP(hipGetLastError());
    ws->gpu_arena.used = mark;  // release the scratch
    return !failed();
}

}  // namespace g500

using namespace g500;

extern "C" {

Oned_Graph oned_graph_from_tuple_graph(Worker_State *ws, Tuple_Graph *tg, u64 nglobalverts) {
    Context &c = ctx();
    Oned_Graph g;
    memset(&g, 0, sizeof(g));
    const u64 n = nglobalverts;
    g.nglobalverts = n;
    g.nlocalverts = n;
    if (n == 0 || n > (1ull << 32)) {
        fail("oned_graph_from_tuple_graph: %llu vertices outside [1, 2^32]", (unsigned long long)n);
        return g;
    }
    const u64 ne = tg->edges_size;
    g.rowstarts = (u64 *)arena_alloc(ws, (n + 1) * sizeof(u64), "CSR row offsets");
    if (failed()) return g;
    timer_start();
    if (!(partition_pays(ws, n, ne) ? fill_partitioned(ws, tg, &g) : fill_direct(ws, tg, &g))) return g;
    if (!sort_rows(ws, &g)) return g;
    if (c.relabel) build_traversal_copy(ws, &g);
    timer_stop();
    return g;
}

b32 oned_graph_is_vertex_isolated(Worker_State *ws, const Oned_Graph *g, u64 global_vertex) {
    (void)ws;
    if (global_vertex >= g->nglobalverts) {
        fail("Vertex %llu is outside graph vertex range [0, %llu)", (unsigned long long)global_vertex,
             (unsigned long long)g->nglobalverts);
        return 1;
    }
    u64 r[2];
    g500_copy_to_host(r, g->rowstarts + global_vertex, sizeof(r));
    return r[0] == r[1];
}

void oned_graph_free(Oned_Graph *g) {
    if (g) memset(g, 0, sizeof(*g));
}

}  // extern "C"
