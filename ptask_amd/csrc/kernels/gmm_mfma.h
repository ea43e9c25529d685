// gmm_mfma.h -- GmmAccumulate with its products on the matrix cores (v_mfma_f32_16x16x4f32), every
// operand in registers.
//
//   GmmAccumulateMfma(const float* X, GMM_DIMS d, const double* model, double* partials)
//     Same arguments and partial-row format as GmmAccumulate (gmm_body.h), so GmmFinalize and every
//     caller are unchanged; only the rounding differs, and the tiles go to the first
//     GMM_MFMA_ROWS rows.
//
// A wave works alone on groups of 16 points, with coordinates centred on g (the mean of the
// component means, one per-dimension vector per launch: x' = x - g, c'_k = mu_k - g):
//   E-step  the squared Mahalanobis distances of its 16 points to all components as one product
//           [x'^2 | x'] (16 x 2W) . [iv ; -2 iv c'] (2W x Kp)  + sum_m iv c'^2.  The right-hand
//           operand is the same for every point: it stays in registers for the whole launch.
//   log-sum-exp  of each point, in the product's own output layout: lane (l4, l16) holds points
//           4 l4 + r (r < 4) against components 16 kt + l16, so a point's components are a few
//           registers of the 16 lanes of one DPP row.  Base 2 throughout.
//   M-step  the moments about g as one product  R^T (Kp x 16) . [x' | x'^2] (16 x 2W).  The
//           responsibilities are its left operand exactly as the E-step leaves them: lane (l4,
//           l16) supplies A[component l16][point 4 l4 + r], one product per r (which four points
//           form a product's inner dimension is free, as long as both operands agree).
// So nothing passes through LDS between the products and no wave waits for another.
//
// The expansion in the E-step cancels (|x'|^2 iv against the distance); it runs only while every
// reciprocal variance is at most GMM_MFMA_IV_LIMIT.  Otherwise (the first EM step, var = 1e-10) the
// block runs GmmAccumulate's body, its M-phase on the matrix cores in binary64.
//
// Sums are binary32 over at most 128 points of one wave (in MFMA order), then binary64 (LDS for the
// block, or registers where the moments are few), converted once per block to moments about the
// table centres c = mu_k:  su = A1 - c' W,  suu = A2 - 2 c' A1 + c'^2 W.  The order of every sum is
// a fixed function of (N, blocks): bitwise reproducible run to run.
//
// Bound: the matrix cores (8 N D K flops per step; 32 cycles of a SIMD per product).  Two waves per
// SIMD (at most 256 registers) cover each other's log-sum-exp, about a quarter of the products'
// issue time at D = 32, K = 64.  Measured there with N = 2M, 768 blocks: 304 us per launch on average (328
// with the tiles on all 768 rows, 313 without the log-sum-exp's priority), 70% of the rate of a large
// matrix product; 612 us when tiles of coordinates and responsibilities passed through
// LDS between the products (four barriers a tile, an LDS read per operand).  N = 50,001, D = 16, K = 24
// (one tile per block): 13.1 us, 27.8 before, when every block first built the operand in LDS.
#pragma once

#include "gmm_body.h"

typedef float gmm_f4 __attribute__((ext_vector_type(4)));

#define GMM_MFMA_IV_LIMIT 1.0e3f
#define GMM_GROUP 16  // points per wave and product
// Partial rows that receive tiles; further ones are zero.  512 blocks are resident at once (two on each
// of 256 CUs): of 768 the last 256 would have a CU each to themselves, where one wave per SIMD does not
// cover its own log-sum-exp.
#define GMM_MFMA_ROWS 512
// doubles per component row of the block's moment sums (2 W moments): the four rows a wave's store
// touches then start 32 banks apart
#define GMM_ACC_STRIDE(W) (2 * (W) + 4)

struct GmmMfmaShared {
    union {
        GmmShared valu;                                // the steps before the E-step expansion is safe
        double acc[KMAX * GMM_ACC_STRIDE(DMAX)];       // the block's moment sums about g
    } u;
    float g[DMAX];
    double w[4][KMAX];
    double ll[4];
    unsigned turn;  // additions to acc made so far by the block's waves
};

// Max and sum of four values over the 16 lanes of a DPP row; every lane gets the results.  Rotating
// by 8, 4, 2 and 1 the four chains are interleaved, so an operand is always three instructions old
// (a DPP operand may be read two after it is written): written as instructions because the
// compiler takes the chains one after the other with a wait and a move per step.
#define GMM_DPP4(OP, N)                                              \
    OP " %0, %0, %0 row_ror:" N " row_mask:0xf bank_mask:0xf\n\t"    \
    OP " %1, %1, %1 row_ror:" N " row_mask:0xf bank_mask:0xf\n\t"    \
    OP " %2, %2, %2 row_ror:" N " row_mask:0xf bank_mask:0xf\n\t"    \
    OP " %3, %3, %3 row_ror:" N " row_mask:0xf bank_mask:0xf\n\t"
#define GMM_ROW4(OP) "s_nop 1\n\t" GMM_DPP4(OP, "8") GMM_DPP4(OP, "4") GMM_DPP4(OP, "2") GMM_DPP4(OP, "1")
__device__ __forceinline__ void gmm_row_max4(float (&v)[4]) {
    asm(GMM_ROW4("v_max_f32_dpp") : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}
__device__ __forceinline__ void gmm_row_sum4(float (&v)[4]) {
    asm(GMM_ROW4("v_add_f32_dpp") : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}

// One partial row.  W = 8 DC dimensions (D rounded up to 8), KT component tiles of 16.  Returns
// false, having written nothing, when the E-step expansion is not safe (uniform over the block).
template <int DC, int KT>
__device__ __forceinline__ bool gmm_mfma_tiles(const float *__restrict__ X, const GMM_DIMS &d,
                                               const double *__restrict__ model, double *__restrict__ row,
                                               long long t0, long long t1, long long tstep, GmmMfmaShared &sh) {
#pragma clang fp contract(fast)
    constexpr int W = 8 * DC, NF = 2 * DC;            // dimensions; dimensions per lane of the E-step
    constexpr int JT = DC;                            // 16-wide tiles of the 2 W moments
    constexpr int NS = W % 16 == 0 ? JT / 2 : JT;     // coordinate registers per point of the M-step
    constexpr bool kRegAcc = KT * JT <= 4;            // binary64 sums in registers
    constexpr int kStride = GMM_ACC_STRIDE(W);
    constexpr float kLog2e = 1.44269504088896340736f;
    const int D = d.D, K = d.K, Dp = ptk_gmm_dpad(&d);
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, l4 = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float *__restrict__ tab = (const float *)(model + ptk_gmm_table(&d));

    // ---- per launch: the centre and the E-step operand of this lane's dimensions f0 .. f0 + NF - 1, those
    // from l4 NF on.  Where these run past D the lane starts earlier, at dimensions of lanes before it, with
    // zeros in the operand there: it then loads coordinates of its point only.  (One dimension is fewer
    // than NF: the second of a lane's is none of the point's.)
    const int f0 = D < NF ? 0 : min(l4 * NF, D - NF);
    float g[NF], b1[KT][NF], b2[KT][NF], ek[KT];
    bool big = false;
    {
        double s[NF];
#pragma unroll
        for (int i = 0; i < NF; ++i) s[i] = 0;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            const int k = kt * 16 + l16;
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                const bool in = k < K && f0 + i < D, on = in && f0 + i >= l4 * NF;
                const float *e = tab + 2 * (k < K ? k : 0) * Dp + (f0 + i < D ? f0 + i : 0);
                const float mu = e[0], iv = e[Dp];
                b1[kt][i] = in ? mu : 0.f;
                b2[kt][i] = on ? iv : 0.f;
                if (on && !(iv <= GMM_MFMA_IV_LIMIT)) big = true;
                s[i] += (double)b1[kt][i];
            }
        }
        if (__builtin_expect(__any(big), 0)) return false;  // unlikely: the other body's code lies behind this one's
        if (t0 >= t1) {  // a row without a tile
            for (int i = tid; i < K + 2 * K * D + 1; i += 256) row[i] = 0;
            return true;
        }
#pragma unroll
        for (int i = 0; i < NF; ++i) {
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) s[i] += __shfl_xor(s[i], off, 64);
            g[i] = (float)(s[i] / K);
        }
        if (wv == 0 && l16 == 0)
#pragma unroll
            for (int i = 0; i < NF; ++i)
                if (f0 + i >= l4 * NF && f0 + i < D) sh.g[f0 + i] = g[i];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            const int k = kt * 16 + l16;
            double q = 0;
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                const float mu = b1[kt][i], iv = b2[kt][i];
                const double cp = (double)mu - (double)g[i];
                q += (double)iv * cp * cp;
                b1[kt][i] = -2.f * iv * (mu - g[i]);
            }
            q += __shfl_xor(q, 16, 64);
            q += __shfl_xor(q, 32, 64);
            // log2 of the responsibilities: a component past the last gets weight 0
            ek[kt] = k < K ? (float)(((double)tab[2 * K * Dp + k] - 0.5 * q) * 1.44269504088896340736) : -INFINITY;
        }
    }
    for (int i = tid; i < KT * 16 * kStride; i += 256) sh.u.acc[i] = 0;
    if (tid == 0) sh.turn = 0;
    __syncthreads();
    // ---- the M-step's coordinates of this lane: moment column 16 jt + l16 is dimension jd of point
    // 4 l4 + r, squared from column W on
    int jd[NS];
    float gm[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int c = 16 * j + l16, m = c < W ? c : c - W;
        jd[j] = m < D ? m : D - 1;  // a column past D is never read back
        gm[j] = sh.g[jd[j]];
    }

    gmm_f4 acc[KT][JT];
    double dacc[kRegAcc ? KT : 1][kRegAcc ? JT : 1][4];
    float w[KT];
    double dw[KT], ll = 0;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        w[kt] = 0.f;
        dw[kt] = 0;
#pragma unroll
        for (int jt = 0; jt < JT; ++jt) {
            acc[kt][jt] = gmm_f4{0.f, 0.f, 0.f, 0.f};
            if (kRegAcc)
#pragma unroll
                for (int r = 0; r < 4; ++r) dacc[kt][jt][r] = 0;
        }
    }
    // this wave's binary32 sums (at most 128 points) into the binary64 ones
    auto *lacc = (__attribute__((address_space(3))) double *)sh.u.acc;
    auto *lturn = (__attribute__((address_space(3))) unsigned *)&sh.turn;
    auto flush = [&]() {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            dw[kt] += (double)w[kt];
            w[kt] = 0.f;
#pragma unroll
            for (int jt = 0; jt < JT; ++jt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (kRegAcc) dacc[kt][jt][r] += (double)acc[kt][jt][r];
                    else __builtin_amdgcn_ds_atomic_fadd_f64(lacc + (16 * kt + 4 * l4 + r) * kStride + 16 * jt + l16,
                                                             (double)acc[kt][jt][r]);
                }
                acc[kt][jt] = gmm_f4{0.f, 0.f, 0.f, 0.f};
            }
        }
    };

    // Wave wv takes points [32 wv, 32 wv + 32) of each 128-point tile, as two groups: group n of the
    // wave is points 16 (n & 1) .. of tile t0 + (n >> 1) tstep.  A group's coordinates are loaded
    // while the group before it computes, through a buffer that ends with the last point (what lies past it
    // reads as 0), so a group is always the same loads, whatever D and its alignment.
    float xe[NF], xm[NS][4];
    auto base = [&](long long t, int q) { return t * TILE + 32 * wv + 16 * q; };
    auto group = [&](long long p0) {
        const long long left = ((long long)d.N - p0) * D * 4;
        const int bytes = left < 0 ? 0 : (int)min(left, (long long)GMM_GROUP * DMAX * 4);
        return __builtin_amdgcn_make_buffer_rsrc((void *)(X + (left > 0 ? p0 * D : 0)), (short)0, bytes, 0x00020000);
    };
    const int oe = (l16 * D + f0) * 4;
    int om[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) om[j] = (4 * l4 * D + jd[j]) * 4;
    auto loadE = [&](long long p0) {
        const auto rs = group(p0);
        constexpr int V = NF % 4 == 0 ? 4 : 2;
#pragma unroll
        for (int c = 0; c < NF; c += V) {
            if (V == 4) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, oe + 4 * c, 0, 0);
#pragma unroll
                for (int i = 0; i < V; ++i) xe[c + i] = __builtin_bit_cast(float, (unsigned)v[i]);
            } else {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, oe + 4 * c, 0, 0);
#pragma unroll
                for (int i = 0; i < V; ++i) xe[c + i] = __builtin_bit_cast(float, (unsigned)v[i]);
            }
        }
    };
    auto loadM = [&](long long p0) {
        const auto rs = group(p0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < NS; ++j)
                xm[j][r] = __builtin_bit_cast(float, (unsigned)__builtin_amdgcn_raw_buffer_load_b32(rs, om[j] + 4 * r * D, 0, 0));
    };
    int turn = 0;  // tiles of this wave so far
    if (t0 < t1) {
        loadE(base(t0, 0));
        loadM(base(t0, 0));
    }
    for (long long t = t0; t < t1; t += tstep) {
#pragma unroll 1
        for (int q = 0; q < 2; ++q) {
            const long long p0 = base(t, q);
            const long long pn = q == 0 ? base(t, 1) : t + tstep < t1 ? base(t + tstep, 0) : p0;
            const int np = (int)min((long long)GMM_GROUP, d.N - p0);  // valid points (<= 0: none)
            // ---- E-step
            float a1[NF], a2[NF];
            if (DC == 1 && D < NF) xe[NF - 1] = g[NF - 1];  // no dimension of the point's (see f0)
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                a1[i] = xe[i] - g[i];
                a2[i] = a1[i] * a1[i];
            }
            loadE(pn);
            gmm_f4 e[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) e[kt] = gmm_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NF; ++i)
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
                    e[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[i], b2[kt][i], e[kt], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NF; ++i)
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
                    e[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[i], b1[kt][i], e[kt], 0, 0, 0);
            // ---- log-sum-exp of point 4 l4 + r over the row's lanes; responsibilities into e
            // (ahead of the SIMD's other wave, whose products fill the matrix core meanwhile)
            __builtin_amdgcn_s_setprio(1);
            float mx[4], sum[4], lse[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                mx[r] = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    e[kt][r] = fmaf(-0.5f * kLog2e, e[kt][r], ek[kt]);
                    mx[r] = kt == 0 ? e[kt][r] : fmaxf(mx[r], e[kt][r]);
                }
            }
            gmm_row_max4(mx);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    e[kt][r] = __builtin_amdgcn_exp2f(e[kt][r] - mx[r]);
                    sum[r] = kt == 0 ? e[kt][r] : sum[r] + e[kt][r];
                }
            gmm_row_sum4(sum);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float inv = __builtin_amdgcn_rcpf(sum[r]);
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) e[kt][r] *= inv;
                lse[r] = mx[r] + __builtin_amdgcn_logf(sum[r]);
            }
            {   // the sixteen lanes of a row hold the same four values: lane l16 = r adds point r's
                const float v = l16 == 0 ? lse[0] : l16 == 1 ? lse[1] : l16 == 2 ? lse[2] : lse[3];
                if (l16 < 4 && 4 * l4 + l16 < np) ll += (double)v;
            }
            // ---- M-step
            // a point past the last, whose square may overflow, has responsibility 0 and lies at the centre
            if (__builtin_expect(np < GMM_GROUP, 0)) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (4 * l4 + r >= np) {
#pragma unroll
                        for (int kt = 0; kt < KT; ++kt) e[kt][r] = 0.f;
#pragma unroll
                        for (int j = 0; j < NS; ++j) xm[j][r] = gm[j];
                    }
            }
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) w[kt] += e[kt][r];
            float x1[NS][4], x2[NS][4];
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x1[j][r] = xm[j][r] - gm[j];
                    x2[j][r] = x1[j][r] * x1[j][r];
                }
            loadM(pn);
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int jt = 0; jt < JT; ++jt) {
                    const float b = NS == JT ? (16 * jt + l16 < W ? x1[jt % NS][r] : x2[jt % NS][r])
                                    : jt < NS ? x1[jt % NS][r] : x2[jt % NS][r];
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt)
                        acc[kt][jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(e[kt][r], b, acc[kt][jt], 0, 0, 0);
                }
        }
        // every fourth tile of the wave.  The waves take turns at the block's sums in tile order, so
        // that the order of the additions is fixed: turn n waits for turn n - 1, made by the wave
        // before at its previous tile (every wave of the block counts the same tiles, so each turn
        // comes).  A wave is held up only when another is behind by a tile; a barrier per tile would
        // have all four wait for the slowest each time.
        if (kRegAcc) {
            if ((turn & 3) == 3) flush();
        } else if ((turn & 3) == wv) {
            while (__hip_atomic_load(lturn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != (unsigned)turn)
                __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            flush();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            if (lane == 0) __hip_atomic_store(lturn, (unsigned)turn + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        ++turn;
    }
    if (kRegAcc) flush();
    __syncthreads();
#pragma unroll 1
    for (int v = 0; v < 4; ++v) {  // what is left, in wave order
        if (wv == v) {
            if (kRegAcc) {
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            sh.u.acc[(16 * kt + 4 * l4 + r) * kStride + 16 * jt + l16] += dacc[kt][jt][r];
            } else {
                flush();
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        double v = dw[kt];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (l4 == 0) sh.w[wv][16 * kt + l16] = v;
    }
    ll *= 0.69314718055994530942;  // base 2 to natural
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ll += __shfl_xor(ll, off, 64);
    if (lane == 0) sh.ll[wv] = ll;
    __syncthreads();

    // ---- the block's moments about the table centres, one partial row
    for (int i = tid; i < K * D; i += 256) {
        const int k = i / D, m = i - k * D;
        const double wk = sh.w[0][k] + sh.w[1][k] + sh.w[2][k] + sh.w[3][k];
        const double a1 = sh.u.acc[k * kStride + m], a2 = sh.u.acc[k * kStride + W + m];
        const double cp = (double)tab[2 * k * Dp + m] - (double)sh.g[m];
        row[K + i] = a1 - cp * wk;
        row[K + K * D + i] = a2 - 2.0 * cp * a1 + cp * cp * wk;
    }
    if (tid < K) row[tid] = sh.w[0][tid] + sh.w[1][tid] + sh.w[2][tid] + sh.w[3][tid];
    if (tid == 0) row[K + 2 * K * D] = sh.ll[0] + sh.ll[1] + sh.ll[2] + sh.ll[3];
    __syncthreads();  // a block may go on to another unit, which reuses sh
    return true;
}

template <int DC>
__device__ __forceinline__ bool gmm_mfma_comps(const float *__restrict__ X, const GMM_DIMS &d,
                                               const double *__restrict__ model, double *__restrict__ row,
                                               long long t0, long long t1, long long ts, GmmMfmaShared &sh) {
    switch ((d.K + 15) >> 4) {
        case 1: return gmm_mfma_tiles<DC, 1>(X, d, model, row, t0, t1, ts, sh);
        case 2: return gmm_mfma_tiles<DC, 2>(X, d, model, row, t0, t1, ts, sh);
        case 3: return gmm_mfma_tiles<DC, 3>(X, d, model, row, t0, t1, ts, sh);
        default: return gmm_mfma_tiles<DC, 4>(X, d, model, row, t0, t1, ts, sh);
    }
}

__device__ __forceinline__ void gmm_mfma_unit(const float *__restrict__ X, const GMM_DIMS &d,
                                              const double *__restrict__ model, double *__restrict__ partials,
                                              int b, GmmMfmaShared &sh) {
    const long long t1 = ((long long)d.N + TILE - 1) / TILE, ts = min(d.blocks, GMM_MFMA_ROWS), t0 = b < ts ? b : t1;
    double *row = partials + (long long)b * ptk_gmm_partial_stride(&d);
    bool done;
    switch ((d.D + 7) >> 3) {
        case 1: done = gmm_mfma_comps<1>(X, d, model, row, t0, t1, ts, sh); break;
        case 2: done = gmm_mfma_comps<2>(X, d, model, row, t0, t1, ts, sh); break;
        case 3: done = gmm_mfma_comps<3>(X, d, model, row, t0, t1, ts, sh); break;
        default: done = gmm_mfma_comps<4>(X, d, model, row, t0, t1, ts, sh); break;
    }
    if (!done) gmm_accumulate_unit<true>(X, d, model, partials, b, (int)ts, sh.u.valu);
}
