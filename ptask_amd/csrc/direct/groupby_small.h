// groupby_small.h -- the groupby of a few thousand rows in one block (and, over many keys, a second
// launch for the offsets), for the direct calls of libptk_groupby.so.
//
// The seven passes of the graph's pipeline take 44 us or more however few the rows: seven dependent
// launches of 2.5 to 6 us, and 21 for the partition, one block that ranks four quarter chunks.  A block of
// 1024 threads orders up to GB_SMALL_ROWS rows in LDS instead: a stable radix sort
// of (key, value) by eight key bits a pass (wave ballots, as gb_partition_chunks), then the group records
// from the sorted rows.  Per call, us: 500 rows over 256 keys 9.6 (44.2 with the pipeline), 4000 over 1024
// 15.5 (47.0), 4000 over 262144 31 (99), 8000 over 1024 21 (50).  With sixteen rows a thread (128 KB of
// LDS, registers spilled) 16,000 rows took 48 to 61, no less than the pipeline's 56 to 60: eight it is.  Outputs are those of the pipeline, bit for bit (positions are ranks in row order
// at every pass; per-group sums are differences of wrapping int64 prefix sums).
#pragma once

#include "groupby_body.h"

namespace ptk_groupby {

#define GB_SMALL_THREADS 1024
#define GB_SMALL_WAVES (GB_SMALL_THREADS / 64)
#define GB_SMALL_RPT 8                                         // rows per thread; four when that is enough
#define GB_SMALL_ROWS (GB_SMALL_THREADS * GB_SMALL_RPT)        // most rows
#define GB_SMALL_KEYS 4096                                     // most keys whose offsets the block forms itself

template <int RPT>
struct GbSmallLds {
    int2 row[GB_SMALL_THREADS * (RPT + 1)];  // row p at p + p / RPT: a thread's RPT rows start on their own banks
    union {
        unsigned short wcnt[GB_SMALL_WAVES][256];  // per wave and digit: rows, then the wave's base
        unsigned off[GB_SMALL_KEYS];               // per key: rows, then the offset
    } u;
    unsigned base[256];
    unsigned red[GB_SMALL_WAVES];
    unsigned long long red64[GB_SMALL_WAVES];
};

// Exclusive prefixes over the block of a count and of a wrapping sum, and their totals.
__device__ __forceinline__ void gb_small_scan(unsigned c, unsigned long long s, unsigned *red, unsigned long long *red64,
                                              unsigned &cbefore, unsigned long long &sbefore, unsigned &ctotal,
                                              unsigned long long &stotal) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned ci = wave_incl32(c);
    const unsigned long long si = wave_incl(s);
    __syncthreads();
    if (lane == 63) {
        red[w] = ci;
        red64[w] = si;
    }
    __syncthreads();
    cbefore = ci - c, sbefore = si - s, ctotal = 0, stotal = 0;
    for (int q = 0; q < GB_SMALL_WAVES; ++q) {
        if (q < w) cbefore += red[q], sbefore += red64[q];
        ctotal += red[q], stotal += red64[q];
    }
}

// One block of GB_SMALL_THREADS; n <= GB_SMALL_THREADS * RPT.  Writes groups, outKeys, outVals and, for
// numKeys < GB_SMALL_KEYS, offsets.
template <int RPT>
__device__ __forceinline__ void gb_small(const int *keys, const int *vals, int n, int numKeys, long long *offsets,
                                         long long *groups, int *outKeys, int *outVals, GbSmallLds<RPT> &L) {
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned long long below = (1ull << lane) - 1ull;
    auto at = [](unsigned p) { return p + p / RPT; };
    // wave w, step s: the 64 rows from first + 64 s on, in row order
    const int first = w * 64 * RPT + lane;
    int2 x[RPT];
    unsigned use = 0;  // bit s: x[s] is a row
    unsigned bad = 0;
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const unsigned r = (unsigned)(first + 64 * s), c = r < (unsigned)n ? r : (unsigned)n - 1u;
        x[s] = make_int2(keys[c], vals[c]);
    }
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        if (first + 64 * s >= n) continue;
        if (x[s].x >= 0 && x[s].x <= numKeys) use |= 1u << s;
        else ++bad;
    }
    unsigned valid = 0;
    // the passes: the first also closes the gaps of the dropped rows, so there is at least one
    const int bits = numKeys > 0 ? 32 - __builtin_clz((unsigned)numKeys) : 1;
    for (int shift = 0; shift < bits; shift += 8) {
        for (int i = tid; i < GB_SMALL_WAVES * 256 / 2; i += GB_SMALL_THREADS) ((unsigned *)L.u.wcnt)[i] = 0;
        __syncthreads();
        unsigned rk[RPT];
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const bool on = (use >> s) & 1u;
            const unsigned d = ((unsigned)x[s].x >> shift) & 255u;
            const unsigned long long peers = gb_match<8>(d, on);
            unsigned old = 0;
            if (on) old = L.u.wcnt[w][d];
            if (on && (peers & below) == 0) L.u.wcnt[w][d] = (unsigned short)(old + __popcll(peers));
            rk[s] = old + (unsigned)__popcll(peers & below);
            __builtin_amdgcn_sched_barrier(0);  // one step at a time: keeps the ballots' masks few
        }
        __syncthreads();
        if (tid < 256) {  // wave bases and the digit's rows
            unsigned t = 0;
#pragma unroll
            for (int v = 0; v < GB_SMALL_WAVES; ++v) {
                const unsigned c = L.u.wcnt[v][tid];
                L.u.wcnt[v][tid] = (unsigned short)t;
                t += c;
            }
            L.base[tid] = t;
        }
        valid = gb_lds_exscan(L.base, 256, L.red);
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const unsigned d = ((unsigned)x[s].x >> shift) & 255u;
            if ((use >> s) & 1u) L.row[at(L.base[d] + L.u.wcnt[w][d] + rk[s])] = x[s];
        }
        __syncthreads();
        if (shift + 8 < bits) {
            use = 0;
#pragma unroll
            for (int s = 0; s < RPT; ++s) {
                if ((unsigned)(first + 64 * s) < valid) use |= 1u << s;
                x[s] = L.row[at((unsigned)first) + s * (64 + 64 / RPT)];  // at(first + 64 s)
            }
        }
    }
    // the grouped rows
    for (unsigned i = tid; i < valid; i += GB_SMALL_THREADS) {
        const int2 v = L.row[at(i)];
        outKeys[i] = v.x;
        outVals[i] = v.y;
    }
    // thread t owns rows t RPT .. : the first rows of groups among them, and the values' prefix sums
    const unsigned p0 = (unsigned)tid * RPT, p1 = p0 + RPT < valid ? p0 + RPT : valid;
    const int2 *mine = &L.row[at(p0)];
    const int prev0 = p0 > 0 && p0 < valid ? L.row[at(p0 - 1)].x : -1;
    unsigned heads = 0;
    unsigned long long sum = 0;
    int prev = prev0;
    for (unsigned p = p0; p < p1; ++p) {
        const int2 v = mine[p - p0];
        heads += v.x != prev;
        prev = v.x;
        sum += (unsigned long long)(long long)v.y;
    }
    unsigned g, G;
    unsigned long long before, total;
    gb_small_scan(heads, sum, L.red, L.red64, g, before, G, total);
    // records {key, first row, sum of the values before it}, turned into {key, count, sum} below
    prev = prev0;
    for (unsigned p = p0; p < p1; ++p) {
        const int2 v = mine[p - p0];
        if (v.x != prev) {
            long long *r = groups + 3 + 3 * (long long)g;
            r[0] = v.x;
            r[1] = p;
            r[2] = (long long)before;
            ++g;
        }
        prev = v.x;
        before += (unsigned long long)(long long)v.y;
    }
    const bool own = numKeys < GB_SMALL_KEYS;
    if (own)
        for (int k = tid; k <= numKeys; k += GB_SMALL_THREADS) L.u.off[k] = 0;
    const unsigned long long errors = block_sum(bad, L.red64);
    __syncthreads();
    for (unsigned g0 = 0; g0 < G; g0 += GB_SMALL_THREADS) {
        const unsigned q = g0 + tid;
        long long *r = groups + 3 + 3 * (long long)q;
        long long key = 0, a = 0, b = 0, sa = 0, sb = 0;
        if (q < G) {
            key = r[0], a = r[1], sa = r[2];
            b = q + 1 < G ? r[4] : (long long)valid;
            sb = q + 1 < G ? r[5] : (long long)total;
        }
        __syncthreads();  // every record of this round, and the next round's first, has been read
        if (q < G) {
            r[1] = b - a;
            r[2] = (long long)((unsigned long long)sb - (unsigned long long)sa);
            if (own) L.u.off[key] = (unsigned)(b - a);
        }
    }
    if (tid == 0) {
        groups[0] = G;
        groups[1] = valid;
        groups[2] = (long long)errors;
    }
    if (own) {
        gb_lds_exscan(L.u.off, numKeys + 1, L.red);
        for (int k = tid; k <= numKeys; k += GB_SMALL_THREADS) offsets[k] = L.u.off[k];
    }
}

// offsets[k] for every key from the sorted keys: the first of the groups[1] rows whose key is at least k.
// Four keys a thread, their searches interleaved (a search is a chain of dependent loads).
__device__ __forceinline__ void gb_small_offsets(const int *__restrict__ sorted, const long long *__restrict__ groups,
                                                 int numKeys, long long *__restrict__ offsets) {
    const int rows = (int)groups[1];
    const int k0 = (int)blockIdx.x * 4 * (int)blockDim.x + (int)threadIdx.x;
    int lo[4] = {0, 0, 0, 0};
    int step = 1;
    while (step < rows) step *= 2;
    for (; step > 0; step /= 2)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = lo[i] + step;  // rows [0, lo) are below the key
            if (m <= rows && sorted[m - 1] < k0 + i * (int)blockDim.x) lo[i] = m;
        }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (k0 + i * (int)blockDim.x <= numKeys) offsets[k0 + i * (int)blockDim.x] = lo[i];
}

}  // namespace ptk_groupby

template <int RPT>
__global__ void __launch_bounds__(GB_SMALL_THREADS)
GroupbySmall(const int *keys, const int *vals, int n, int numKeys, long long *offsets, long long *groups, int *outKeys,
             int *outVals) {
    __shared__ ptk_groupby::GbSmallLds<RPT> L;
    if (n < 1 || n > GB_SMALL_THREADS * RPT || blockDim.x != GB_SMALL_THREADS || blockIdx.x != 0) return;
    ptk_groupby::gb_small<RPT>(keys, vals, n, numKeys, offsets, groups, outKeys, outVals, L);
}

static __global__ void __launch_bounds__(256)
GroupbySmallOffsets(const int *sorted, const long long *groups, int numKeys, long long *offsets) {
    ptk_groupby::gb_small_offsets(sorted, groups, numKeys, offsets);
}
