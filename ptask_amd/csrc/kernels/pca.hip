// pca.hip -- Gram-Schmidt PCA (NIPALS with deflation) as PTask task kernels (pca.hsaco).
//
// Semantics follow ptaskUnitTest/pca_cpu.cpp:267-424 (the host reference the unrolled BLAS graph
// of ptaskUnitTest/graphcupca.cpp is checked against); the decomposition into kernels is the
// build's own.  The reference runs, per component k and inner iteration, separate BLAS-2 tasks
// (dgemv R^T t, dgemv for the Gram-Schmidt step, dnrm2, dscal, dgemv R p, dnrm2, dscal) and a
// rank-1 dger per component.  Here the matrix R lives row-major in HBM and every pass over it
// does as much as one read allows:
//   PcaStart    t_{k-1} = R p_{k-1} and deflation by component k-1 (R -= t p^T, written back),
//               fused with p = R^T R[:,k]: the last inner iteration's t = R p of component k-1
//               is formed in the same read of R that deflates it
//   PcaGram     p = R^T (R p) in one read of R: each 8-row slab's t = R_slab p is reduced inside
//               the block and immediately used for R_slab^T t (the reference's t = R p, |t|,
//               t /= |t|, p = R^T t -- the scaling by 1/|t| is undone by the next normalisation)
//   PcaDeflate  t_K-1 = R p and R -= t p^T by the last component (the residual the reference returns)
// T[:,k] holds t = R p_k, which is the reference's final L_k (t / L_k) (pca_cpu.cpp:385-386 and
// 404-408) without the two rounding steps.  The small steps are single kernels: PcaReduce +
// PcaOrthonormalize (sum the per-block p partials in a fixed order, p -= P_<k (P_<k^T p),
// p /= |p|) and PcaFinish (L_k = |t| from the per-block |t|^2 partials).  All reductions are
// fixed-order, so results are bitwise reproducible.  Dot products and norms of length-N and
// length-M vectors are binary64.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ptk_pca.h"

// Tolerance-checked binary32 work: let the compiler fuse multiply-adds (the build default is off).
#pragma clang fp contract(fast)

#define PCA_LOAD_COLS 128  // columns of a tile of PcaLoad

enum { PCA_START = 0, PCA_GRAM = 1, PCA_DEFLATE = 3 };

__device__ inline bool pca_ok(const PCA_DIMS &d) {
    return d.M >= 1 && d.N >= 1 && d.N <= PTK_PCA_MAX_N && d.K >= 1 && d.K <= PTK_PCA_MAX_K &&
           d.K <= d.N && d.J >= 1 && d.ld == ptk_pca_ld(d.N) && d.Mp == ptk_pca_mp(d.M) && d.G >= 1 &&
           d.GR >= 1 && d.GR <= d.G && d.k >= 0 && d.k < d.K;
}

__device__ inline double *pca_L(float *S, const PCA_DIMS &d) { return (double *)((char *)S + ptk_pca_off_L(&d)); }
__device__ inline double *pca_tn(float *S, const PCA_DIMS &d) { return (double *)((char *)S + ptk_pca_off_tn(&d)); }
__device__ inline double *pca_red(float *S, const PCA_DIMS &d) { return (double *)((char *)S + ptk_pca_off_red(&d)); }
__device__ inline float *pca_P(float *S, const PCA_DIMS &d) { return (float *)((char *)S + ptk_pca_off_P(&d)); }
__device__ inline float *pca_part(float *S, const PCA_DIMS &d) { return (float *)((char *)S + ptk_pca_off_part(&d)); }

__device__ inline float f4get(const float4 &v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }
__device__ inline float f4dot(const float4 &a, const float4 &b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

// ---- PcaLoad: X (column-major M x N) -> R (row-major Mp x ld), rows optionally centred; T and S
// cleared.  Grid Mp/64 blocks of 256; block b owns rows 64b .. 64b+63.  With few rows only some CUs
// have a block and the time is its chain of round trips and address arithmetic: 32 loads in flight
// per thread from scalar column addresses take 24.3 us at 3000 x 700 (8 and 16 from per-lane 64-bit
// products took 39.0, and 64 in flight give no more); at 65536 x 2048 it is two reads and a write of
// the matrix at 4.5 TB/s, 359 us, as before.
extern "C" __global__ void __launch_bounds__(256)
PcaLoad(const float *__restrict__ X, PCA_DIMS d, float *__restrict__ R, float *__restrict__ T,
        float *__restrict__ S) {
    __shared__ double sSum[4][64];
    __shared__ double sMean[64];
    __shared__ float tile[PCA_LOAD_COLS][65];
    if (!pca_ok(d) || blockDim.x != 256 || (int)gridDim.x != d.Mp / 64) return;
    const int tid = threadIdx.x, M = d.M, N = d.N, ld = d.ld;
    const long long r0 = (long long)blockIdx.x * 64;
    // Column c0 + 4 j is one wave's, row r one lane's: a column's address is a scalar, the lane's
    // offset from it the same 32 bits in every load (the rows past the last read the last).
    const int r = tid & 63, c0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned ro = (unsigned)(r0 + r < M ? r : M - 1 - r0);
    const bool mv = r0 + r < M;
    constexpr int kLoads = PCA_LOAD_COLS / 4;
    float v[kLoads];
    auto load = [&](int n0) {  // columns n0 + c0 + 4 j; past the last, the last
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int n = n0 + c0 + 4 * j;
            v[j] = (X + ((long long)(n < N ? n : N - 1) * M + r0))[ro];
        }
    };
    load(0);
    {
        // row sums, added in column order
        double s = 0;
        if (d.center)
            for (int n0 = 0; n0 < N; n0 += PCA_LOAD_COLS) {
                if (n0 > 0) load(n0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < kLoads; ++j)
                    if (n0 + c0 + 4 * j < N) s += (double)v[j];
            }
        sSum[c0][r] = s;
    }
    if (d.center && N > PCA_LOAD_COLS) load(0);
    __syncthreads();
    if (tid < 64) sMean[tid] = d.center ? (sSum[0][tid] + sSum[1][tid] + sSum[2][tid] + sSum[3][tid]) / N : 0.0;
    __syncthreads();
    // 64 x PCA_LOAD_COLS tiles through LDS; the next tile's loads are issued before the current tile
    // is stored
    const double mean = sMean[r];
    const int w0 = __builtin_amdgcn_readfirstlane(tid / PCA_LOAD_COLS), wc = tid % PCA_LOAD_COLS;
    for (int n0 = 0; n0 < ld; n0 += PCA_LOAD_COLS) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int c = c0 + 4 * j;
            tile[c][r] = (n0 + c < N && mv) ? (float)((double)v[j] - mean) : 0.f;
        }
        __syncthreads();
        if (n0 + PCA_LOAD_COLS < ld) load(n0 + PCA_LOAD_COLS);
        __builtin_amdgcn_sched_barrier(0);
        if (n0 + wc < ld)
#pragma unroll 8
            for (int rr = w0; rr < 64; rr += 256 / PCA_LOAD_COLS) (R + ((r0 + rr) * ld + n0))[(unsigned)wc] = tile[wc][rr];
        __syncthreads();
    }
    const long long nT = (long long)d.K * d.Mp, nS = ptk_pca_state_bytes(&d) / 4;
    const long long step = (long long)gridDim.x * 256;
    for (long long i = (long long)blockIdx.x * 256 + tid; i < nT; i += step) T[i] = 0.f;
    for (long long i = (long long)blockIdx.x * 256 + tid; i < nS; i += step) S[i] = 0.f;
}

// ---- the row passes.  Block of 256; thread t owns float4 column chunks t + 256 c (c < NCH); a
// slab of RB rows is held in registers, its RB row dot products are reduced across the block
// (wave shuffles, then a double-buffered LDS exchange, one barrier per slab).
//
// Deflation by component dk (PcaStart of component k deflates k - 1; PcaDeflate deflates the
// last): the rows' scores t = R p_dk are the block-reduced dot products of the rows about to be
// deflated (pca_cpu.cpp:380-401 computes t = R p, L = |t|, t /= L and R -= L t p^T; L t is t
// before the scaling, so no separate pass computes it); t goes to T[:, dk] and its squares to
// the block's tn partial (PcaFinish takes L_dk = |t| from them); then R -= t p_dk^T.
template <int NCH, int RB, int MODE>
__device__ __forceinline__ void pca_row_pass(float *__restrict__ R, float *__restrict__ T,
                                             float *__restrict__ S, const PCA_DIMS &d) {
    __shared__ float sRed[2][4][RB];
    __shared__ float sCol[2][RB];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ld = d.ld, ld4 = ld >> 2, k = d.k;
    const long long Mp = d.Mp;
    float *P = pca_P(S, d);
    int cix[NCH];
    bool cv[NCH];
    float4 wv4[NCH], acc[NCH];  // the vector the rows are dotted with: p_k (Gram) or p_dk (deflation)
    const bool deflate = (MODE == PCA_START && k > 0) || MODE == PCA_DEFLATE;
    const bool rowdot = MODE == PCA_GRAM || deflate;
    const int dk = MODE == PCA_START ? k - 1 : k;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        cix[c] = tid + 256 * c;
        cv[c] = cix[c] < ld4;
        const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        wv4[c] = (rowdot && cv[c]) ? ((const float4 *)(P + (long long)(MODE == PCA_GRAM ? k : dk) * ld))[cix[c]] : z;
        acc[c] = z;
    }
    // p_dk at column k: every thread forms column k of the deflated rows from the exchanged
    // pre-deflation values, as the column's owner deflates it (the same fused multiply-add)
    const float pk = (MODE == PCA_START && deflate) ? P[(long long)dk * ld + k] : 0.f;
    const int ck = k >> 2, ce = k & 3, cowner = ck & 255, creg = ck >> 8;
    const long long nslab = Mp / RB;
    int buf = 0;
    double tsq = 0;
    for (long long s = blockIdx.x; s < nslab; s += gridDim.x) {
        const long long r0 = s * RB;
        float4 x[RB][NCH];
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int c = 0; c < NCH; ++c)
                x[i][c] = cv[c] ? ((const float4 *)(R + (r0 + i) * ld))[cix[c]] : make_float4(0.f, 0.f, 0.f, 0.f);
        if (rowdot) {
            float v[RB];
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                v[i] = 0.f;
#pragma unroll
                for (int c = 0; c < NCH; ++c) v[i] += f4dot(x[i][c], wv4[c]);
#pragma unroll
                for (int off = 32; off >= 1; off >>= 1) v[i] += __shfl_xor(v[i], off, 64);
            }
            if (lane == 0) {
#pragma unroll
                for (int i = 0; i < RB; ++i) sRed[buf][wv][i] = v[i];
            }
        }
        if (MODE == PCA_START && tid == cowner) {
            // column k of the rows (before any deflation), from the thread that owns it
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                float xv = 0.f;
#pragma unroll
                for (int c = 0; c < NCH; ++c)
                    if (c == creg) xv = f4get(x[i][c], ce);
                sCol[buf][i] = xv;
            }
        }
        __syncthreads();
        float red[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i)
            red[i] = rowdot ? sRed[buf][0][i] + sRed[buf][1][i] + sRed[buf][2][i] + sRed[buf][3][i] : 0.f;
        if (deflate) {
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const float a = red[i];  // t of row r0 + i
#pragma unroll
                for (int c = 0; c < NCH; ++c) {
                    if (!cv[c]) continue;
                    x[i][c].x = fmaf(-a, wv4[c].x, x[i][c].x);
                    x[i][c].y = fmaf(-a, wv4[c].y, x[i][c].y);
                    x[i][c].z = fmaf(-a, wv4[c].z, x[i][c].z);
                    x[i][c].w = fmaf(-a, wv4[c].w, x[i][c].w);
                    ((float4 *)(R + (r0 + i) * ld))[cix[c]] = x[i][c];
                }
            }
            if (tid == 0) {
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    T[(long long)dk * Mp + r0 + i] = red[i];
                    tsq += (double)red[i] * (double)red[i];
                }
            }
        }
        if (MODE == PCA_DEFLATE) {
            buf ^= 1;
            continue;
        }
        float t[RB];  // Start: column k of the (deflated) residual; Gram: R_slab p_k
#pragma unroll
        for (int i = 0; i < RB; ++i)
            t[i] = MODE == PCA_GRAM ? red[i] : (deflate ? fmaf(-red[i], pk, sCol[buf][i]) : sCol[buf][i]);
        buf ^= 1;
#pragma unroll
        for (int c = 0; c < NCH; ++c)
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                acc[c].x = fmaf(x[i][c].x, t[i], acc[c].x);
                acc[c].y = fmaf(x[i][c].y, t[i], acc[c].y);
                acc[c].z = fmaf(x[i][c].z, t[i], acc[c].z);
                acc[c].w = fmaf(x[i][c].w, t[i], acc[c].w);
            }
    }
    if (deflate && tid == 0) pca_tn(S, d)[blockIdx.x] = tsq;
    if (MODE != PCA_DEFLATE) {
        float *part = pca_part(S, d) + (long long)blockIdx.x * ld;
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (cv[c]) ((float4 *)part)[cix[c]] = acc[c];
    }
}

template <int MODE>
__device__ __forceinline__ void pca_row_dispatch(float *R, float *T, float *S, const PCA_DIMS &d) {
    switch ((d.ld / 4 + 255) / 256) {
        case 1: pca_row_pass<1, 8, MODE>(R, T, S, d); break;
        case 2: pca_row_pass<2, 8, MODE>(R, T, S, d); break;
        case 3: pca_row_pass<3, 4, MODE>(R, T, S, d); break;
        default: pca_row_pass<4, 4, MODE>(R, T, S, d); break;
    }
}

extern "C" __global__ void __launch_bounds__(256)
PcaStart(float *__restrict__ R, float *__restrict__ T, float *__restrict__ S, PCA_DIMS d) {
    if (!pca_ok(d) || blockDim.x != 256 || (int)gridDim.x != d.G) return;
    pca_row_dispatch<PCA_START>(R, T, S, d);
}

extern "C" __global__ void __launch_bounds__(256)
PcaGram(float *__restrict__ R, float *__restrict__ S, PCA_DIMS d) {
    if (!pca_ok(d) || blockDim.x != 256 || (int)gridDim.x != d.G) return;
    pca_row_dispatch<PCA_GRAM>(R, nullptr, S, d);
}

// After the last component: t_k = R p_k into T[:, k] and the tn partials, R -= t_k p_k^T for
// k = d.k (pca_cpu.cpp:380-401 of the final k).
extern "C" __global__ void __launch_bounds__(256)
PcaDeflate(float *__restrict__ R, float *__restrict__ T, float *__restrict__ S, PCA_DIMS d) {
    if (!pca_ok(d) || blockDim.x != 256 || (int)gridDim.x != d.G) return;
    pca_row_dispatch<PCA_DEFLATE>(R, T, S, d);
}

// ---- PcaReduce: red[g][n] = sum of part[b][n] over the g-th of GR contiguous groups of the G
// rows.  Grid (ceil(ld/64), GR) blocks of 256 (64 columns x 4 interleaved row subsets).  The
// loads read clamped, always valid rows unconditionally, sixteen at a time, so they issue together
// (384 rows in 8 groups are 12 per thread: one round trip); the sums take the valid terms in row order.
extern "C" __global__ void __launch_bounds__(256)
PcaReduce(float *__restrict__ S, PCA_DIMS d) {
    __shared__ double sh[4][64];
    if (!pca_ok(d) || blockDim.x != 256 || (int)gridDim.x != (d.ld + 63) / 64 || (int)gridDim.y != d.GR) return;
    const int tid = threadIdx.x, c = tid & 63, sub = tid >> 6, g = blockIdx.y, ld = d.ld;
    const int col = blockIdx.x * 64 + c, cc = col < ld ? col : ld - 1;
    const int lo = (int)((long long)g * d.G / d.GR), hi = (int)((long long)(g + 1) * d.G / d.GR);
    const float *part = pca_part(S, d);
    double s = 0;
    for (int b0 = lo + sub; b0 < hi; b0 += 64) {
        float x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int b = b0 + 4 * u < hi ? b0 + 4 * u : hi - 1;
            x[u] = part[(long long)b * ld + cc];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (b0 + 4 * u < hi) s += (double)x[u];
    }
    sh[sub][c] = col < ld ? s : 0.0;
    __syncthreads();
    if (sub == 0 && col < ld) pca_red(S, d)[(long long)g * ld + col] = sh[0][c] + sh[1][c] + sh[2][c] + sh[3][c];
}

// ---- PcaOrthonormalize: one block of 1024.  p = sum of the GR rows of red; classical
// Gram-Schmidt against the components before k (U = P_<k^T p, then p -= P_<k U: pca_cpu.cpp:356-372);
// p *= 1/|p| (dnrm2 + dscal: pca_cpu.cpp:374-376); P[k] = p.
//
// One block, so its time is a chain of latencies and what one CU can load and exchange, and the
// kernel is built to keep that chain short: a thread owns EPT consecutive columns, the loads of the
// first CH rows of P are issued together with those of red and stay in registers for both uses, and
// the dot products are reduced by halving (below), not each on its own.  Average over k = 0 .. 15
// at 2048 columns: 7.2 us, and 5.3 us over k = 0 .. 3 at 700 columns; 12.0 and 8.4 us with a shuffle
// tree per dot product (2 x 6 x k LDS exchanges in each of the 16 waves) and the rows of P loaded
// again for the second use.

// 16 lanes of a DPP row: a value from the lane that mirrors this one in its row, its half row, its
// quad, and its pair.
template <int CTRL>
__device__ __forceinline__ double pca_dpp(double v) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
constexpr int kRowMirror = 0x140, kHalfMirror = 0x141, kQuadMirror = 0x1B, kPairSwap = 0xB1;

// Sum of v over the 16 lanes of the row, in every lane.
__device__ __forceinline__ double pca_row_sum(double v) {
    v += pca_dpp<kRowMirror>(v);
    v += pca_dpp<kHalfMirror>(v);
    v += pca_dpp<kQuadMirror>(v);
    return v + pca_dpp<kPairSwap>(v);
}

// Sixteen sums over the row's lanes at once: lane l of the row gets the sum of v[l & 15].  At each step
// a lane gives its partner the half of the sums that the partner keeps: 15 exchanges and additions
// for all sixteen instead of 64.
__device__ __forceinline__ double pca_row_sum16(double (&v)[16], int l16) {
    auto step = [&](auto ctrl, int n, bool up) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < n) {
                const double give = up ? v[i] : v[i + n], keep = up ? v[i + n] : v[i];
                v[i] = keep + pca_dpp<decltype(ctrl)::value>(give);
            }
    };
    step(std::integral_constant<int, kRowMirror>{}, 8, (l16 & 8) != 0);
    step(std::integral_constant<int, kHalfMirror>{}, 4, (l16 & 4) != 0);
    step(std::integral_constant<int, kQuadMirror>{}, 2, (l16 & 2) != 0);
    step(std::integral_constant<int, kPairSwap>{}, 1, (l16 & 1) != 0);
    return v[0];
}

struct PcaOrthoLds {
    double w[64][PTK_PCA_MAX_K + 1];  // per DPP row of the block: its part of the dot products (rows
                                      // of an odd number of doubles: a column's parts spread over the banks)
    double u[PTK_PCA_MAX_K];
    double n[64];
};

// A load of E consecutive elements (E = 1, 2 or 4; aligned to as many).
template <int E, class T>
__device__ __forceinline__ void pca_load(const T *__restrict__ p, T (&v)[E]) {
    typedef T V __attribute__((ext_vector_type(E)));
    const V x = *(const V *)p;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = x[e];
}
template <>
__device__ __forceinline__ void pca_load<1, float>(const float *__restrict__ p, float (&v)[1]) { v[0] = *p; }
template <>
__device__ __forceinline__ void pca_load<1, double>(const double *__restrict__ p, double (&v)[1]) { v[0] = *p; }

template <int EPT>
__device__ inline void pca_orthonormalize(float *__restrict__ S, const PCA_DIMS &d, PcaOrthoLds &L) {
    constexpr int CH = 16;               // rows of P reduced together
    constexpr int RG = EPT == 4 ? 4 : 8; // rows of red loaded together
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, row = tid >> 4, ld = d.ld, k = d.k, GR = d.GR;
    const double *__restrict__ red = pca_red(S, d);
    float *P = pca_P(S, d);
    // columns n0 .. n0 + EPT - 1: ld is a multiple of 4, so all of them or none are in range; a
    // thread past the end reads the last ones and adds nothing
    const bool on = tid * EPT < ld;
    const int n0 = on ? tid * EPT : ld - EPT;
    // rows [j0, j0 + CH) of P below k, four at a time as far as they reach; the others as zeros
    float pv[CH][EPT];
    auto loadP = [&](int j0) {
#pragma unroll
        for (int q = 0; q < CH; q += 4) {
            if (j0 + q < k) {
#pragma unroll
                for (int i = q; i < q + 4; ++i) pca_load<EPT>(P + (long long)(j0 + i < k ? j0 + i : k - 1) * ld + n0, pv[i]);
            } else {
#pragma unroll
                for (int i = q; i < q + 4; ++i)
#pragma unroll
                    for (int e = 0; e < EPT; ++e) pv[i][e] = 0.f;
            }
        }
    };
    loadP(0);
    double p[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) p[e] = 0;
    for (int g0 = 0; g0 < GR; g0 += RG) {
        double rv[RG][EPT];
#pragma unroll
        for (int g = 0; g < RG; ++g) pca_load<EPT>(red + (long long)(g0 + g < GR ? g0 + g : GR - 1) * ld + n0, rv[g]);
#pragma unroll
        for (int g = 0; g < RG; ++g)
            if (g0 + g < GR)
#pragma unroll
                for (int e = 0; e < EPT; ++e) p[e] += rv[g][e];
    }
    if (!on)
#pragma unroll
        for (int e = 0; e < EPT; ++e) p[e] = 0;
    if (k > 0) {
        for (int j0 = 0; j0 < k; j0 += CH) {
            if (j0 > 0) loadP(j0);
            double v[CH];
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                v[i] = (double)pv[i][0] * p[0];  // a row past k - 1 may repeat it; its sum is not used
#pragma unroll
                for (int e = 1; e < EPT; ++e) v[i] = fma((double)pv[i][e], p[e], v[i]);
            }
            const double t = pca_row_sum16(v, l16);
            L.w[row][j0 + l16] = t;
        }
        __syncthreads();
        {   // U_j: sixteen threads a component, each four of the 64 rows' parts in order, then the row sum
            const int j = tid >> 4;  // 64 components
            double u = 0;
            if (j < k)
#pragma unroll
                for (int i = 0; i < 4; ++i) u += L.w[4 * l16 + i][j];
            u = pca_row_sum(u);
            if (l16 == 0) L.u[j] = j < k ? u : 0.0;
        }
        __syncthreads();
        // p -= P_<k U: each element's sum over j in order.  Only more than CH rows are loaded again.
        double s[EPT];
#pragma unroll
        for (int e = 0; e < EPT; ++e) s[e] = 0;
        for (int j0 = 0; j0 < k; j0 += CH) {
            if (k > CH) loadP(j0);
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const double u = L.u[j0 + i];  // 0 from k on
#pragma unroll
                for (int e = 0; e < EPT; ++e) s[e] = fma((double)pv[i][e], u, s[e]);
            }
        }
        if (on)
#pragma unroll
            for (int e = 0; e < EPT; ++e) p[e] -= s[e];
    }
    double v = 0;
#pragma unroll
    for (int e = 0; e < EPT; ++e) v = fma(p[e], p[e], v);
    v = pca_row_sum(v);
    if (l16 == 0) L.n[row] = v;
    __syncthreads();
    // |p|^2 from the 64 rows' parts: each DPP row four apiece in order, then the row sum
    double n2 = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) n2 += L.n[4 * l16 + i];
    const double inv = 1.0 / sqrt(pca_row_sum(n2));
    if (on) {
        typedef float V __attribute__((ext_vector_type(EPT)));
        V o;
#pragma unroll
        for (int e = 0; e < EPT; ++e) o[e] = (float)(p[e] * inv);
        *(V *)(P + (long long)k * ld + n0) = o;
    }
}

extern "C" __global__ void __launch_bounds__(1024)
PcaOrthonormalize(float *__restrict__ S, PCA_DIMS d) {
    __shared__ PcaOrthoLds L;
    if (!pca_ok(d) || blockDim.x != 1024 || gridDim.x != 1) return;
    if (d.ld <= 2048) pca_orthonormalize<2>(S, d, L);
    else pca_orthonormalize<4>(S, d, L);
}

// ---- PcaFinish: L_k = sqrt(sum of the G tn partials) (pca_cpu.cpp:385), one block of 256
// summing in a fixed order.
extern "C" __global__ void __launch_bounds__(256)
PcaFinish(float *__restrict__ S, PCA_DIMS d) {
    __shared__ double sh[256];
    if (!pca_ok(d) || blockDim.x != 256 || gridDim.x != 1) return;
    const int tid = threadIdx.x;
    const double *tn = pca_tn(S, d);
    double s = 0;
    for (int b = tid; b < d.G; b += 256) s += tn[b];
    sh[tid] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) sh[tid] += sh[tid + w];
        __syncthreads();
    }
    if (tid == 0) pca_L(S, d)[d.k] = sqrt(sh[0]);
}
#include "pca_blas.h"
