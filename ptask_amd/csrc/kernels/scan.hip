// scan.hip -- exclusive prefix sums as PTask task kernels (code object scan.hsaco).
//
// Semantics (reference oracle host_pfxsum, ptaskUnitTest/pfxsum.cpp:56-69): out[0] = 0,
// out[i] = out[i-1] + in[i-1], in two's-complement int32 (wrapping) arithmetic.
//
//   pfxsum(int* pin, int* pout, int N)           -- the reference task ABI (pfxsum.cu:21-25,
//       formal indices pin 0, pout 1, N 2 as cpfxsum.cpp wires them).  Any N >= 0: one block
//       walks the array in chunks of 2*blockDim with a running carry; extra blocks exit.  The
//       reference kernel is limited to 256 elements (pfxsum.cu:6); this one is not.
//   PfxScanReduce(const int* pin, int N, int* tileSums)          -- large N, pass 1: one total
//       per tile of PFX_TILE elements.
//   PfxScanApply(const int* pin, int N, const int* tileSums, int* pout) -- pass 2: each block
//       sums the totals before its tile, then scans its tile.  12 B of HBM traffic per element.
//   *64 variants: int64 elements.
//
// Wave-level scans and sums run over DPP (row shifts and row broadcasts: no LDS), then one LDS
// exchange of the per-wave totals.  Integer addition is associative, so the result is exact
// regardless of the reduction order.
//
// Both passes of the large scan are a block's latency (load, reduce, store) times the rounds of
// blocks, so a block does as little in sequence as it can: 16-byte accesses, the tile's loads issued
// before the earlier tiles' totals are read, one barrier per tile.  8M int32: 8.9 and 13.2 us; 12.4 and
// 27.4 with 4-byte accesses, shuffles, and the totals and the tile one after the other (six barriers). 500,000:
// 2.6 and 3.2 us against 3.3 and 5.6, 40,000: 2.5 and 3.0 against 3.2 and 5.8; below a million elements the
// two launches are most of a scan.
#include <hip/hip_runtime.h>

#define PFX_TILE 4096  // elements per tile of the large scan (1024 threads x 4)

// v of the lane that the DPP control names, 0 where there is none or the row is masked out.
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T lane_dpp(T v) {
    if constexpr (sizeof(T) == 8) {
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROWS, 0xF, false);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, ROWS, 0xF, false);
        return ((T)hi << 32) | lo;
    } else {
        return (T)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
    }
}

template <typename T>
__device__ __forceinline__ T wave_inclusive(T v) {
    v += lane_dpp<0x111, 0xF>(v);  // row_shr:1, 2, 4, 8: within the rows of 16 lanes
    v += lane_dpp<0x112, 0xF>(v);
    v += lane_dpp<0x114, 0xF>(v);
    v += lane_dpp<0x118, 0xF>(v);
    v += lane_dpp<0x142, 0xA>(v);  // row_bcast:15: the last lane of rows 0 and 2 into rows 1 and 3
    v += lane_dpp<0x143, 0xC>(v);  // row_bcast:31: lane 31 into rows 2 and 3
    return v;
}

// The value of one lane, in every lane.
template <typename T>
__device__ __forceinline__ T lane_value(T v, int lane) {
    if constexpr (sizeof(T) == 8)
        return ((T)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), lane) << 32) |
               (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
    else
        return (T)__builtin_amdgcn_readlane((int)v, lane);
}

template <typename T>
__device__ __forceinline__ T wave_total(T v) {
    return lane_value(wave_inclusive(v), 63);
}

// Block-wide exclusive scan of one value per thread (blockDim.x a multiple of 64, <= 1024).
// Returns the exclusive prefix; *total receives the block total.
template <typename T>
__device__ inline T block_exclusive(T v, T *total) {
    __shared__ T waveSums[16];
    __shared__ T blockTotal;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    T inc = wave_inclusive(v);
    if (lane == 63 || (int)threadIdx.x == (int)blockDim.x - 1) waveSums[wave] = inc;
    __syncthreads();
    if (wave == 0) {
        T s = lane < nw ? waveSums[lane] : T(0);
        T si = wave_inclusive(s);
        if (lane < nw) waveSums[lane] = si - s;  // exclusive prefix of the wave totals
        if (lane == nw - 1) blockTotal = si;
    }
    __syncthreads();
    T res = waveSums[wave] + inc - v;
    *total = blockTotal;
    __syncthreads();  // the shared slots are reused by the next call
    return res;
}

// One block scans the whole array, two elements per thread per chunk, carrying the running sum.
// Launch contract of every kernel here: blockDim.x a multiple of 64 (whole wavefronts), at most
// 1024, blockDim.y == blockDim.z == 1.
__device__ inline bool block_ok() { return (blockDim.x & 63) == 0 && blockDim.y == 1 && blockDim.z == 1; }

template <typename T>
__device__ inline void single_block_scan(const T *__restrict__ in, T *__restrict__ out, long long n) {
    if (!block_ok() || blockIdx.x != 0 || blockIdx.y != 0 || blockIdx.z != 0) return;
    T carry = 0;
    const long long chunk = 2ll * blockDim.x;
    for (long long base = 0; base < n; base += chunk) {
        const long long i0 = base + 2ll * threadIdx.x, i1 = i0 + 1;
        const T a = i0 < n ? in[i0] : T(0), b = i1 < n ? in[i1] : T(0);
        T tot;
        T ex = block_exclusive<T>(a + b, &tot);
        if (i0 < n) out[i0] = carry + ex;
        if (i1 < n) out[i1] = carry + ex + a;
        carry += tot;
    }
}

// int32 with wrapping adds: compute in unsigned arithmetic (defined overflow), store the bits.
extern "C" __global__ void __launch_bounds__(1024) pfxsum(int *pin, int *pout, int N) {
    single_block_scan<unsigned>((const unsigned *)pin, (unsigned *)pout, N < 0 ? 0 : N);
}

extern "C" __global__ void __launch_bounds__(1024) pfxsum64(long long *pin, long long *pout, int N) {
    single_block_scan<unsigned long long>((const unsigned long long *)pin, (unsigned long long *)pout,
                                          N < 0 ? 0 : N);
}

// Elements [base, base + PER) of in, zeros from n on; 16-byte loads when `vec` (in is 16-byte aligned,
// and base is a multiple of 16 bytes by construction).
template <int PER, typename T>
__device__ __forceinline__ void load_run(const T *__restrict__ in, long long base, long long n, bool vec, T (&v)[PER]) {
    constexpr int V = 16 / (int)sizeof(T);
    if (vec && base + PER <= n) {
        typedef T Vec __attribute__((ext_vector_type(V)));
#pragma unroll
        for (int q = 0; q < PER; q += V) {
            const Vec x = *(const Vec *)(in + base + q);
#pragma unroll
            for (int e = 0; e < V; ++e) v[q + e] = x[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < PER; ++e) v[e] = base + e < n ? in[base + e] : T(0);
    }
}

// Tile sums; the two parities of `part` let a block's next tile begin without a second barrier.
template <typename T>
__device__ __forceinline__ void tile_reduce(const T *__restrict__ in, long long n, T *__restrict__ tileSums) {
    __shared__ T part[2][16];
    if (!block_ok()) return;
    const long long ntiles = (n + PFX_TILE - 1) / PFX_TILE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    const bool vec = ((unsigned long long)in & 15ull) == 0;
    int b = 0;
    for (long long t = blockIdx.x; t < ntiles; t += gridDim.x, b ^= 1) {
        const long long base = t * PFX_TILE;
        T s = 0;
        for (int e = 4 * (int)threadIdx.x; e < PFX_TILE; e += 4 * (int)blockDim.x) {
            T v[4];
            load_run<4>(in, base + e, n, vec, v);
            s += (v[0] + v[1]) + (v[2] + v[3]);
        }
        s = wave_total(s);
        if (lane == 0) part[b][wave] = s;
        __syncthreads();
        if (wave == 0) {
            const T tot = wave_total(lane < nw ? part[b][lane] : T(0));
            if (lane == 0) tileSums[t] = tot;
        }
    }
}

// One tile per block and round, PER consecutive elements a thread.  `pre` is this thread's part of the
// totals before the tile: it grows by the totals between the block's tiles, each read once.
template <int PER, typename T>
__device__ __forceinline__ void tile_apply_per(const T *__restrict__ in, long long n, const T *__restrict__ tileSums,
                                               T *__restrict__ out) {
    __shared__ T part[2][2][16];
    const long long ntiles = (n + PFX_TILE - 1) / PFX_TILE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    const bool vin = ((unsigned long long)in & 15ull) == 0, vout = ((unsigned long long)out & 15ull) == 0;
    T pre = 0;
    long long u0 = 0;
    int b = 0;
    for (long long t = blockIdx.x; t < ntiles; t += gridDim.x, b ^= 1) {
        const long long base = t * PFX_TILE + (long long)threadIdx.x * PER;
        T v[PER];
        load_run<PER>(in, base, n, vin, v);
        for (long long u = u0 + threadIdx.x; u < t; u += blockDim.x) pre += tileSums[u];
        u0 = t;
        T s = 0;
#pragma unroll
        for (int e = 0; e < PER; ++e) s += v[e];
        const T inc = wave_inclusive(s), wpre = wave_total(pre);
        if (lane == 63) {
            part[b][0][wave] = inc;
            part[b][1][wave] = wpre;
        }
        __syncthreads();
        // the totals before the tile and of the waves before this one
        const T before = lane < nw ? part[b][1][lane] + (lane < wave ? part[b][0][lane] : T(0)) : T(0);
        T run = wave_total(before) + inc - s;
        constexpr int V = 16 / (int)sizeof(T);
        if (vout && base + PER <= n) {
            typedef T Vec __attribute__((ext_vector_type(V)));
#pragma unroll
            for (int q = 0; q < PER; q += V) {
                Vec x;
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    x[e] = run;
                    run += v[q + e];
                }
                *(Vec *)(out + base + q) = x;
            }
        } else {
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                if (base + e < n) out[base + e] = run;
                run += v[e];
            }
        }
    }
}

template <typename T>
__device__ __forceinline__ void tile_apply(const T *__restrict__ in, long long n, const T *__restrict__ tileSums,
                                           T *__restrict__ out) {
    if (!block_ok()) return;
    switch (PFX_TILE / (int)blockDim.x) {  // a multiple of 64 that divides PFX_TILE: a power of two
        case 4: tile_apply_per<4>(in, n, tileSums, out); break;
        case 8: tile_apply_per<8>(in, n, tileSums, out); break;
        default: tile_apply_per<16>(in, n, tileSums, out); break;
    }
}

extern "C" __global__ void __launch_bounds__(1024) PfxScanReduce(int *pin, int N, int *tileSums) {
    tile_reduce<unsigned>((const unsigned *)pin, N < 0 ? 0 : N, (unsigned *)tileSums);
}

extern "C" __global__ void __launch_bounds__(1024) PfxScanApply(int *pin, int N, int *tileSums, int *pout) {
    if (PFX_TILE % blockDim.x != 0 || PFX_TILE / blockDim.x > 16) return;  // geometry contract
    tile_apply<unsigned>((const unsigned *)pin, N < 0 ? 0 : N, (const unsigned *)tileSums, (unsigned *)pout);
}

extern "C" __global__ void __launch_bounds__(1024) PfxScanReduce64(long long *pin, int N, long long *tileSums) {
    tile_reduce<unsigned long long>((const unsigned long long *)pin, N < 0 ? 0 : N,
                                    (unsigned long long *)tileSums);
}

extern "C" __global__ void __launch_bounds__(1024) PfxScanApply64(long long *pin, int N, long long *tileSums,
                                                                  long long *pout) {
    if (PFX_TILE % blockDim.x != 0 || PFX_TILE / blockDim.x > 16) return;
    tile_apply<unsigned long long>((const unsigned long long *)pin, N < 0 ? 0 : N,
                                   (const unsigned long long *)tileSums, (unsigned long long *)pout);
}
