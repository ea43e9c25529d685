// fdtd_fused.h -- one full Yee step (H from old E, then E from new H) in a single pass.
//
// Traffic per cell-step: six fields read once, six written once (48 B), against 96 B for the
// six-task form.  Each cell's arithmetic is the expression of ptaskUnitTest/graphfdtd.cpp:185-312
// in the same order, so results are bit-identical to the six separate updates.
//
// Tiling.  A block owns a TI x TJ tile of (i,j) columns (thread (tx,ty) owns column
// (i0+tx, j0+ty)) and walks a slab of k planes upwards.  For every plane k it
//   1. computes new Hx,Hy,Hz of its own cells (old E at k and k+1; the plane k+1 values read
//      here are the plane k values of the next iteration and come back from cache) and writes
//      them out;
//   2. computes the one-cell halo on the low side that new E needs from other tiles: new Hx, Hz
//      on row j0-1 and new Hy, Hz on column i0-1 (bit-identical to what the owning tile writes);
//   3. after one barrier, computes new Ex,Ey,Ez from LDS (i-1 and j-1 neighbours) and from the
//      new Hx, Hy of plane k-1 that the thread carries.
// LDS is double-buffered by plane parity, so one barrier per plane suffices.
//
// The union domain is i in [0,Nx], j in [0,Ny], k in [0,Nz]; every load and store checks the
// extent of its own field (see include/ptk_fdtd.h).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "ptk_fdtd.h"

namespace ptk_fdtd {

struct Fields {
    const float *__restrict__ hx;
    const float *__restrict__ hy;
    const float *__restrict__ hz;
    const float *__restrict__ ex;
    const float *__restrict__ ey;
    const float *__restrict__ ez;
    float *__restrict__ ohx;
    float *__restrict__ ohy;
    float *__restrict__ ohz;
    float *__restrict__ oex;
    float *__restrict__ oey;
    float *__restrict__ oez;
};

// Flat offsets for each field's extents (i fastest), in 32-bit arithmetic: every field array
// must hold fewer than 2^31 elements (checked by the kernels before any access).
struct Ix {
    int Nx, Ny, Nz;
    __device__ int hx(int i, int j, int k) const { return i + (Nx + 1) * (j + Ny * k); }
    __device__ int hy(int i, int j, int k) const { return i + Nx * (j + (Ny + 1) * k); }
    __device__ int hz(int i, int j, int k) const { return i + Nx * (j + Ny * k); }
    __device__ int ex(int i, int j, int k) const { return i + Nx * (j + (Ny + 1) * k); }
    __device__ int ey(int i, int j, int k) const { return i + (Nx + 1) * (j + Ny * k); }
    __device__ int ez(int i, int j, int k) const { return i + (Nx + 1) * (j + (Ny + 1) * k); }
    // extents (graphfdtd.cpp:70-86)
    __device__ bool vhx(int i, int j, int k) const { return i <= Nx && j < Ny && k < Nz; }
    __device__ bool vhy(int i, int j, int k) const { return i < Nx && j <= Ny && k < Nz; }
    __device__ bool vhz(int i, int j, int k) const { return i < Nx && j < Ny && k <= Nz; }
    __device__ bool vex(int i, int j, int k) const { return i < Nx && j <= Ny && k <= Nz; }
    __device__ bool vey(int i, int j, int k) const { return i <= Nx && j < Ny && k <= Nz; }
    __device__ bool vez(int i, int j, int k) const { return i <= Nx && j <= Ny && k < Nz; }
};

struct Coef {
    float cH, cE, Cx, Cy, Cz;
};

__device__ inline Coef make_coef(const FDTD_PARAMS &p) {
    Coef c;
    c.cH = p.Dt / p.mu0;
    c.cE = p.Dt / p.eps0;
    c.Cx = p.Cx;
    c.Cy = p.Cy;
    c.Cz = p.Cz;
    return c;
}

// New Hx at (i,j,k) from old fields (graphfdtd.cpp:185-201).  Caller checks vhx.
__device__ inline float new_hx(const Fields &F, const Ix &X, const Coef &c, int i, int j, int k) {
    const float ey0 = F.ey[X.ey(i, j, k)], ey1 = F.ey[X.ey(i, j, k + 1)];
    const float ez0 = F.ez[X.ez(i, j, k)], ez1 = F.ez[X.ez(i, j + 1, k)];
    return F.hx[X.hx(i, j, k)] + c.cH * ((ey1 - ey0) * c.Cz - (ez1 - ez0) * c.Cy);
}
// New Hy (graphfdtd.cpp:204-221).  Caller checks vhy.
__device__ inline float new_hy(const Fields &F, const Ix &X, const Coef &c, int i, int j, int k) {
    const float ez0 = F.ez[X.ez(i, j, k)], ez1 = F.ez[X.ez(i + 1, j, k)];
    const float ex0 = F.ex[X.ex(i, j, k)], ex1 = F.ex[X.ex(i, j, k + 1)];
    return F.hy[X.hy(i, j, k)] + c.cH * ((ez1 - ez0) * c.Cx - (ex1 - ex0) * c.Cz);
}
// New Hz (graphfdtd.cpp:223-240).  Caller checks vhz.
__device__ inline float new_hz(const Fields &F, const Ix &X, const Coef &c, int i, int j, int k) {
    const float ex0 = F.ex[X.ex(i, j, k)], ex1 = F.ex[X.ex(i, j + 1, k)];
    const float ey0 = F.ey[X.ey(i, j, k)], ey1 = F.ey[X.ey(i + 1, j, k)];
    return F.hz[X.hz(i, j, k)] + c.cH * ((ex1 - ex0) * c.Cy - (ey1 - ey0) * c.Cx);
}

// TRUE when the largest field (the (Nx+1)(Ny+1)(Nz+1) union bounds them all) is addressable with
// 32-bit offsets.
__device__ inline bool fits_int32(const FDTD_PARAMS &p) {
    return (long long)(p.Nx + 1) * (p.Ny + 1) * (p.Nz + 1) < 2147483647ll;
}

// One tile of one time step over the k slab [k0, k1) of the union domain.
// LDS layout: [parity][field][TJ+1][TI+1], index [ty+1][tx+1] for own cells, row 0 and column 0
// for the low-side halo.
template <int TI, int TJ>
__device__ inline void fused_tile(const Fields &F, const FDTD_PARAMS &p, int i0, int j0, int k0, int k1,
                                  float (*lds)[3][TJ + 1][TI + 1]) {
    const Ix X{p.Nx, p.Ny, p.Nz};
    const Coef c = make_coef(p);
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = i0 + tx, j = j0 + ty;
    const bool own = i <= p.Nx && j <= p.Ny;  // inside the union domain
    const bool haloRow = ty == 0 && j0 >= 1 && i <= p.Nx;
    const bool haloCol = tx == 0 && i0 >= 1 && j <= p.Ny;

    // new Hx, Hy of this column on plane k0-1 (E at k0 needs them)
    float hxm = 0.f, hym = 0.f;
    if (own && k0 >= 1) {
        if (X.vhx(i, j, k0 - 1)) hxm = new_hx(F, X, c, i, j, k0 - 1);
        if (X.vhy(i, j, k0 - 1)) hym = new_hy(F, X, c, i, j, k0 - 1);
    }
    for (int k = k0; k < k1; ++k) {
        float (*s)[TJ + 1][TI + 1] = lds[k & 1];
        float hx = 0.f, hy = 0.f, hz = 0.f;
        if (own) {
            if (X.vhx(i, j, k)) {
                hx = new_hx(F, X, c, i, j, k);
                F.ohx[X.hx(i, j, k)] = hx;
            }
            if (X.vhy(i, j, k)) {
                hy = new_hy(F, X, c, i, j, k);
                F.ohy[X.hy(i, j, k)] = hy;
            }
            if (X.vhz(i, j, k)) {
                hz = new_hz(F, X, c, i, j, k);
                F.ohz[X.hz(i, j, k)] = hz;
            }
            s[0][ty + 1][tx + 1] = hx;
            s[1][ty + 1][tx + 1] = hy;
            s[2][ty + 1][tx + 1] = hz;
        }
        if (haloRow) {  // row j0-1: Hx and Hz
            const int jm = j0 - 1;
            s[0][0][tx + 1] = X.vhx(i, jm, k) ? new_hx(F, X, c, i, jm, k) : 0.f;
            s[2][0][tx + 1] = X.vhz(i, jm, k) ? new_hz(F, X, c, i, jm, k) : 0.f;
        }
        if (haloCol) {  // column i0-1: Hy and Hz
            const int im = i0 - 1;
            s[1][ty + 1][0] = X.vhy(im, j, k) ? new_hy(F, X, c, im, j, k) : 0.f;
            s[2][ty + 1][0] = X.vhz(im, j, k) ? new_hz(F, X, c, im, j, k) : 0.f;
        }
        __syncthreads();
        if (own) {
            // Ex (graphfdtd.cpp:243-264)
            if (X.vex(i, j, k)) {
                const float e = F.ex[X.ex(i, j, k)];
                float r = e;
                if (!(j < 1 || k < 1 || j > p.Ny - 1 || k > p.Nz - 1))
                    r = e + c.cE * ((hz - s[2][ty][tx + 1]) * c.Cy - (hy - hym) * c.Cz);
                F.oex[X.ex(i, j, k)] = r;
            }
            // Ey (graphfdtd.cpp:267-288)
            if (X.vey(i, j, k)) {
                const float e = F.ey[X.ey(i, j, k)];
                float r = e;
                if (!(i < 1 || k < 1 || i > p.Nx - 1 || k > p.Nz - 1))
                    r = e + c.cE * ((hx - hxm) * c.Cz - (hz - s[2][ty + 1][tx]) * c.Cx);
                F.oey[X.ey(i, j, k)] = r;
            }
            // Ez (graphfdtd.cpp:291-312)
            if (X.vez(i, j, k)) {
                const float e = F.ez[X.ez(i, j, k)];
                float r = e;
                if (!(i < 1 || j < 1 || i > p.Nx - 1 || j > p.Ny - 1))
                    r = e + c.cE * ((hy - s[1][ty + 1][tx]) * c.Cx - (hx - s[0][ty][tx + 1]) * c.Cy);
                F.oez[X.ez(i, j, k)] = r;
            }
        }
        hxm = hx;
        hym = hy;
    }
}

}  // namespace ptk_fdtd

namespace ptk_fdtd {

// ---- overlapped tiles: one whole step, one barrier per plane --------------------------------
//
// A block of 64 x R threads (R = blockDim.y, 3..MAXR) covers columns i0-1 .. i0+62 (lane l ->
// i = i0-1+l) and rows j0-1 .. j0+R-2 (wave r -> j = j0-1+r) and owns the inner 62 x (R-2)
// cells: it writes new H and E there only.  Every thread computes new H of its cell, so the
// i-1 / j-1 neighbours that an owned cell's new E needs are in the block; on the low edge these
// are cells of the neighbouring tile, recomputed bit for bit.  The old E that new H needs at
// i+1 / j+1 is likewise in the block.  New H of a cell outside a field's extent, or on the
// block's high edge, is formed from zeros or unrelated values and never reaches an output: an
// owned cell's new E reads new H only at in-extent cells of the block (graphfdtd.cpp:70-86).
//
// Per plane k a thread loads its own old H(k) and old E(k+1) once -- the plane k+1 values are
// carried to the next plane in registers, and both are prefetched two planes ahead -- so HBM
// sees each input once per tile (48 B per cell-step plus the overlap).  Neighbour values pass
// through LDS, double-buffered by plane parity:
//   H phase   new H(k) from registers and E(k) neighbours in e[k&1];
//             write new H(k) to h[k&1] and old E(k+1) to e[(k+1)&1];
//   barrier   (LDS only: loads in flight stay in flight);
//   E phase   new E(k) from registers (old E(k), new H(k), new H(k-1)) and h[k&1] neighbours.
// e[(k+1)&1] was last read in the H phase of plane k-1 and h[k&1] in the E phase of plane k-2,
// both before the barrier of plane k-1, so one barrier per plane orders every access.
// A slab [k0, k1) starts one plane early (k0-1) to form new H(k0-1) for E(k0).
#ifndef PTK_OVERLAP_AHEAD
#define PTK_OVERLAP_AHEAD 2  // planes of loads in flight ahead of the plane being computed (1 or 2)
#endif
#ifndef PTK_OVERLAP_STORE_POLICY
#define PTK_OVERLAP_STORE_POLICY 0  // cache-policy bits of the output stores
#endif

// LDS planes with one padding row and column on each side, so that the four neighbours of
// (r, l) are at fixed offsets from its slot: index [r + 1][l + 1].
template <int MAXR>
struct OverlapLds {
    float e[2][3][MAXR + 2][66];  // old Ex, Ey, Ez of a plane
    float h[2][3][MAXR + 2][66];  // new Hx, Hy, Hz of a plane
};

// Barrier that orders LDS accesses only; outstanding global loads are not waited for.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// x-neighbours across the lanes of one wave (a tile row): lane l reads lane l + 1 through the
// data-parallel-primitive mux (wave_shl:1), a VALU operand modifier instead of an LDS read.
// Lane 63 reads 0; it is a halo lane of every tile.
__device__ inline float lane_next(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xF, 0xF, false));
}

__device__ inline float lane_prev(float v) {  // lane l reads lane l - 1 (wave_shr:1), lane 0 reads 0
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xF, 0xF, false));
}

// Raw buffer access to one field array.  A byte offset at or beyond the array's size reads 0
// and drops a store (the buffer unit's range check), so a lane outside a field's extent issues
// the same instruction with bit 31 of its offset set instead of branching around it: every
// plane then issues a fixed sequence of memory instructions and the loads of later planes stay
// in flight across the barrier.  Arrays must hold fewer than 2^31 bytes.
constexpr unsigned kNoCell = 0x80000000u;

struct FieldBuf {
    __amdgpu_buffer_rsrc_t rs;
    __device__ float load(unsigned off) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
    }
    __device__ void store(unsigned off, float v) const {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, (int)off, 0,
                                              PTK_OVERLAP_STORE_POLICY);
    }
};

__device__ inline FieldBuf field_buf(const float *p, long long elems) {
    return FieldBuf{__builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)(elems * 4), 0x00020000)};
}

// TRUE when every field array is under 2^31 bytes (the buffer range check of overlap_tile).
__device__ inline bool fits_buffer(const FDTD_PARAMS &p) {
    return (long long)(p.Nx + 1) * (p.Ny + 1) * (p.Nz + 1) < (1ll << 29);
}

template <int MAXR>
__device__ inline void overlap_tile(const Fields &F, const FDTD_PARAMS &p, int i0, int j0, int k0, int k1,
                                    OverlapLds<MAXR> &L) {
    const Ix X{p.Nx, p.Ny, p.Nz};
    const Coef c = make_coef(p);
    const int R = (int)blockDim.y;
    const int l = (int)threadIdx.x, r = (int)threadIdx.y;
    const int i = i0 - 1 + l, j = j0 - 1 + r;
    const int Nx = p.Nx, Ny = p.Ny, Nz = p.Nz;
    const bool dom = i >= 0 && i <= Nx && j >= 0 && j <= Ny;
    const bool own = dom && l >= 1 && l <= 62 && r >= 1 && r <= R - 2;
    // byte offset of (i, j, 0) in each field, bit 31 set when the column is outside the field
    auto col = [](bool ok, int idx) { return ok ? 4u * (unsigned)idx : kNoCell; };
    const unsigned qHx = col(dom && j < Ny, X.hx(i, j, 0)), qHy = col(dom && i < Nx, X.hy(i, j, 0));
    const unsigned qHz = col(dom && i < Nx && j < Ny, X.hz(i, j, 0)), qEx = col(dom && i < Nx, X.ex(i, j, 0));
    const unsigned qEy = col(dom && j < Ny, X.ey(i, j, 0)), qEz = col(dom, X.ez(i, j, 0));
    const unsigned ownBit = own ? 0u : kNoCell;
    // byte plane strides
    const unsigned sHx = 4u * (Nx + 1) * Ny, sHy = 4u * Nx * (Ny + 1), sHz = 4u * Nx * Ny;
    const unsigned sEx = 4u * Nx * (Ny + 1), sEy = 4u * (Nx + 1) * Ny, sEz = 4u * (Nx + 1) * (Ny + 1);
    const FieldBuf bHx = field_buf(F.hx, (long long)(Nx + 1) * Ny * Nz), bHy = field_buf(F.hy, (long long)Nx * (Ny + 1) * Nz),
                   bHz = field_buf(F.hz, (long long)Nx * Ny * (Nz + 1)), bEx = field_buf(F.ex, (long long)Nx * (Ny + 1) * (Nz + 1)),
                   bEy = field_buf(F.ey, (long long)(Nx + 1) * Ny * (Nz + 1)), bEz = field_buf(F.ez, (long long)(Nx + 1) * (Ny + 1) * Nz);
    const FieldBuf wHx = field_buf(F.ohx, (long long)(Nx + 1) * Ny * Nz), wHy = field_buf(F.ohy, (long long)Nx * (Ny + 1) * Nz),
                   wHz = field_buf(F.ohz, (long long)Nx * Ny * (Nz + 1)), wEx = field_buf(F.oex, (long long)Nx * (Ny + 1) * (Nz + 1)),
                   wEy = field_buf(F.oey, (long long)(Nx + 1) * Ny * (Nz + 1)), wEz = field_buf(F.oez, (long long)(Nx + 1) * (Ny + 1) * Nz);
    // offset of plane k of a column: the plane test is uniform over the block (a scalar mask)
    auto at = [](unsigned q, unsigned s, int k, bool ok) { return (q + (unsigned)k * s) | (ok ? 0u : kNoCell); };
    // per-lane parts of the face tests of graphfdtd.cpp:243-312
    const bool jIn = j >= 1 && j <= Ny - 1, iIn = i >= 1 && i <= Nx - 1;

    // Register sets S_k = {old E(k+1), old H(k)}.  Plane k reads S_{k-1} (its E part is old
    // E(k)) and S_k, while the loads of the next PTK_OVERLAP_AHEAD sets are in flight: the sets
    // rotate through an unrolled loop body, so no set is ever copied.  A set S_k with k >= k1 is
    // never used and its loads are dropped.
    struct Set {
        float ex, ey, ez, hx, hy, hz;
    };
    auto load_set = [&](Set &S, int k) {
        const bool use = k < k1;
        S.ex = bEx.load(at(qEx, sEx, k + 1, use && k + 1 <= Nz));
        S.ey = bEy.load(at(qEy, sEy, k + 1, use && k + 1 <= Nz));
        S.ez = bEz.load(at(qEz, sEz, k + 1, use && k + 1 < Nz));
        S.hx = bHx.load(at(qHx, sHx, k, use && k < Nz));
        S.hy = bHy.load(at(qHy, sHy, k, use && k < Nz));
        S.hz = bHz.load(at(qHz, sHz, k, use && k <= Nz));
    };
    const int ks = k0 >= 1 ? k0 - 1 : 0;
    Set S0, S1, S2, S3;
    S0.ex = bEx.load(at(qEx, sEx, ks, ks <= Nz));  // old E(ks)
    S0.ey = bEy.load(at(qEy, sEy, ks, ks <= Nz));
    S0.ez = bEz.load(at(qEz, sEz, ks, ks < Nz));
    S0.hx = S0.hy = S0.hz = 0.f;
    load_set(S1, ks);
#if PTK_OVERLAP_AHEAD == 2
    load_set(S2, ks + 1);
#endif
    const int y = r + 1, x = l + 1;  // this thread's LDS slot
    L.e[ks & 1][0][y][x] = S0.ex;
    L.e[ks & 1][1][y][x] = S0.ey;
    L.e[ks & 1][2][y][x] = S0.ez;
    float hxm = 0.f, hym = 0.f;  // new Hx, Hy of plane k-1
    lds_barrier();
    // plane k: P = S_{k-1}, S = S_k; loads S_{k+PTK_OVERLAP_AHEAD} into N
    auto plane = [&](int k, const Set &P, const Set &S, Set &N) {
        const int b = k & 1;
        load_set(N, k + PTK_OVERLAP_AHEAD);
        const float ex = P.ex, ey = P.ey, ez = P.ez;  // old E(k)
        const float ezj = L.e[b][2][y + 1][x], ezi = L.e[b][2][y][x + 1];
        const float exj = L.e[b][0][y + 1][x], eyi = L.e[b][1][y][x + 1];
        // graphfdtd.cpp:185-240, in the reference's operation order
        const float hx = S.hx + c.cH * ((S.ey - ey) * c.Cz - (ezj - ez) * c.Cy);
        const float hy = S.hy + c.cH * ((ezi - ez) * c.Cx - (S.ex - ex) * c.Cz);
        const float hz = S.hz + c.cH * ((exj - ex) * c.Cy - (eyi - ey) * c.Cx);
        L.h[b][0][y][x] = hx;
        L.h[b][1][y][x] = hy;
        L.h[b][2][y][x] = hz;
        L.e[b ^ 1][0][y][x] = S.ex;
        L.e[b ^ 1][1][y][x] = S.ey;
        L.e[b ^ 1][2][y][x] = S.ez;
        lds_barrier();
        const float hzj = L.h[b][2][y - 1][x], hzi = L.h[b][2][y][x - 1];
        const float hyi = L.h[b][1][y][x - 1], hxj = L.h[b][0][y - 1][x];
        // graphfdtd.cpp:243-312: interior cells update, tangential faces copy through
        const bool kIn = k >= 1 && k <= Nz - 1;
        const float wx = ex + c.cE * ((hz - hzj) * c.Cy - (hy - hym) * c.Cz);
        const float wy = ey + c.cE * ((hx - hxm) * c.Cz - (hz - hzi) * c.Cx);
        const float wz = ez + c.cE * ((hy - hyi) * c.Cx - (hx - hxj) * c.Cy);
        const float vx = (jIn && kIn) ? wx : ex;
        const float vy = (iIn && kIn) ? wy : ey;
        const float vz = (iIn && jIn) ? wz : ez;
        const bool out = k >= k0;
        wHx.store(at(qHx | ownBit, sHx, k, out && k < Nz), hx);
        wHy.store(at(qHy | ownBit, sHy, k, out && k < Nz), hy);
        wHz.store(at(qHz | ownBit, sHz, k, out && k <= Nz), hz);
        wEx.store(at(qEx | ownBit, sEx, k, out && k <= Nz), vx);
        wEy.store(at(qEy | ownBit, sEy, k, out && k <= Nz), vy);
        wEz.store(at(qEz | ownBit, sEz, k, out && k < Nz), vz);
        hxm = hx;
        hym = hy;
    };
#if PTK_OVERLAP_AHEAD == 2
    for (int k = ks; k < k1; k += 4) {
        plane(k, S0, S1, S3);
        if (k + 1 < k1) plane(k + 1, S1, S2, S0);
        if (k + 2 < k1) plane(k + 2, S2, S3, S1);
        if (k + 3 < k1) plane(k + 3, S3, S0, S2);
    }
#else
    (void)S3;
    for (int k = ks; k < k1; k += 3) {
        plane(k, S0, S1, S2);
        if (k + 1 < k1) plane(k + 1, S1, S2, S0);
        if (k + 2 < k1) plane(k + 2, S2, S0, S1);
    }
#endif
}

// ---- several time steps per pass on overlapped tiles -------------------------------------------
//
// A block of 64 x R threads (R = blockDim.y, 2T+1..MAXR) advances T time steps in one pass.  It
// covers columns i0-T .. i0+63-T (lane l -> i = i0-T+l) and rows j0-T .. j0+R-1-T (wave r ->
// j = j0-T+r) and owns the inner (64-2T) x (R-2T) cells, for which it writes H and E after the T
// steps.  Each half step loses one cell of valid data on one side (new H needs E at i+1 / j+1,
// new E needs H at i-1 / j-1), so after T steps the block minus T cells on each side is exact;
// the lost cells are recomputed by the neighbouring tiles, bit for bit.  HBM sees each input read
// and each output written once per T steps (48/T B per cell-step plus the overlap).
//
// Planes stream upwards; step s (1..T) runs 2(s-1) planes behind the first, on plane
// p_s = m - 2(s-1) in iteration m:
//   A  for each s: H_s(p_s) from E_{s-1}(p_s), E_{s-1}(p_s+1), H_{s-1}(p_s) and the E_{s-1}(p_s)
//      plane; write H_s(p_s) and E_0(m+1) to LDS
//   barrier
//   B  for each s: E_s(p_s) from E_{s-1}(p_s), H_s(p_s), H_s(p_s-1) and the H_s(p_s) plane; write
//      E_s(p_s) to LDS (s < T); store H_T, E_T of plane p_T if owned
//   barrier
// Step 0 is the input: E_0(m), E_0(m+1) and H_0(m) are loaded two planes ahead.  Step s-1's
// values two and one planes behind its own (those of planes p_s and p_s+1) are carried in
// registers (for T >= 3, the E values are read back from the own slots of the LDS planes).  Ez
// and Ey at i + 1 come from the next lane, so no Ey plane of E_0 is stored, nor, for T < 3, of
// any step (an Ey slot is only read by its own lane).  E_s
// planes are double-buffered by iteration parity (E_s(p_s) is written in B of iteration m and
// read as a plane in A of iteration m+2); H_s planes are written in A and read in B of the same
// iteration (HB = 1, two barriers per plane), or by parity (HB = 2, one barrier per plane).  A
// slab [k0, k1) starts T planes early and runs 2(T-1) planes late for the lag.  Every expression
// is the reference's, in its order (graphfdtd.cpp:185-312), so the result is bitwise that of T
// sequential steps.
template <int T, int MAXR, int HB>
struct OverlapNLds {
    float e[T][2][3][MAXR + 2][66];  // E_0 .. E_{T-1} planes by iteration parity
    float h[HB][T][3][MAXR + 2][66]; // H_1 .. H_T planes of the iteration (by parity if HB = 2)
};

// One field array for the multi-step tiles: the column's byte offset travels in a VGPR and the
// plane's in an SGPR, so a plane costs no vector address arithmetic.  A lane outside the field's
// columns carries bit 31 in its column offset, so its loads read 0 and its stores are dropped.
// Plane offsets are always those of planes inside the array, so a valid cell's column plus plane
// offset is below the array's size and no sum exceeds 2^32: the range check drops exactly the
// invalid lanes whether or not it counts the plane offset.
struct PlaneBuf {
    __amdgpu_buffer_rsrc_t rs;
    __device__ float load(unsigned col, unsigned plane) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)col, (int)plane, 0));
    }
    __device__ void store(unsigned col, unsigned plane, float v) const {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, (int)col, (int)plane,
                                              PTK_OVERLAP_STORE_POLICY);
    }
};

__device__ inline PlaneBuf plane_buf(const float *p, unsigned bytes) {
    return PlaneBuf{__builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)bytes, 0x00020000)};
}

struct F3 {
    float x, y, z;
};

template <int T, int MAXR, int HB>
__device__ inline void overlapn_tile(const Fields &F, const FDTD_PARAMS &p, int i0, int j0, int k0, int k1,
                                     OverlapNLds<T, MAXR, HB> &L) {
    static_assert(T >= 1 && 2 * T < 64, "steps per pass");
    const Ix X{p.Nx, p.Ny, p.Nz};
    const Coef c = make_coef(p);
    const int R = (int)blockDim.y;
    const int l = (int)threadIdx.x, r = (int)threadIdx.y;
    const int i = i0 - T + l, j = j0 - T + r;
    const int Nx = p.Nx, Ny = p.Ny, Nz = p.Nz;
    const bool dom = i >= 0 && i <= Nx && j >= 0 && j <= Ny;
    const bool own = dom && l >= T && l <= 63 - T && r >= T && r <= R - 1 - T;
    auto col = [](bool ok, int idx) { return ok ? 4u * (unsigned)idx : kNoCell; };
    const unsigned qHx = col(dom && j < Ny, X.hx(i, j, 0)), qHy = col(dom && i < Nx, X.hy(i, j, 0));
    const unsigned qHz = col(dom && i < Nx && j < Ny, X.hz(i, j, 0)), qEx = col(dom && i < Nx, X.ex(i, j, 0));
    const unsigned qEy = col(dom && j < Ny, X.ey(i, j, 0)), qEz = col(dom, X.ez(i, j, 0));
    const unsigned ownBit = own ? 0u : kNoCell;  // stores also carry bit 31 where not owned
    const unsigned sHx = 4u * (Nx + 1) * Ny, sHy = 4u * Nx * (Ny + 1), sHz = 4u * Nx * Ny;
    const unsigned sEx = 4u * Nx * (Ny + 1), sEy = 4u * (Nx + 1) * Ny, sEz = 4u * (Nx + 1) * (Ny + 1);
    const PlaneBuf rHx = plane_buf(F.hx, sHx * Nz), rHy = plane_buf(F.hy, sHy * Nz), rHz = plane_buf(F.hz, sHz * (Nz + 1)),
                   rEx = plane_buf(F.ex, sEx * (Nz + 1)), rEy = plane_buf(F.ey, sEy * (Nz + 1)), rEz = plane_buf(F.ez, sEz * Nz);
    const PlaneBuf wHx = plane_buf(F.ohx, sHx * Nz), wHy = plane_buf(F.ohy, sHy * Nz), wHz = plane_buf(F.ohz, sHz * (Nz + 1)),
                   wEx = plane_buf(F.oex, sEx * (Nz + 1)), wEy = plane_buf(F.oey, sEy * (Nz + 1)), wEz = plane_buf(F.oez, sEz * Nz);
    const bool jIn = j >= 1 && j <= Ny - 1, iIn = i >= 1 && i <= Nx - 1;

    struct Set {
        F3 e, h;
    };
    // S_m = {E_0(m+1), H_0(m)}.  The owned planes below k1 depend on input planes up to T above
    // them (each step reaches one plane up), so only m <= k1 + T - 2 feed owned cells; a later
    // set reloads that set's planes (cached) and a plane past a field's last is read as its
    // last: those values reach no stored cell, as the planes formed from them do not.
    auto load_set = [&](Set &S, int m) {
        const int k = m < k1 + T - 2 ? m : k1 + T - 2;
        const int ke = k + 1 <= Nz ? k + 1 : Nz, kez = k + 1 <= Nz - 1 ? k + 1 : Nz - 1;
        const int kh = k <= Nz - 1 ? k : Nz - 1, khz = k <= Nz ? k : Nz;
        S.e.x = rEx.load(qEx, (unsigned)ke * sEx);
        S.e.y = rEy.load(qEy, (unsigned)ke * sEy);
        S.e.z = rEz.load(qEz, (unsigned)kez * sEz);
        S.h.x = rHx.load(qHx, (unsigned)kh * sHx);
        S.h.y = rHy.load(qHy, (unsigned)kh * sHy);
        S.h.z = rHz.load(qHz, (unsigned)khz * sHz);
    };
    // six dropped stores: the prologue then leaves the memory counter as a loop iteration does,
    // so the waits the compiler places in the loop stay two planes behind the loads
    auto pad_stores = [&]() {
        wHx.store(kNoCell, 0u, 0.f);
        wHy.store(kNoCell, 0u, 0.f);
        wHz.store(kNoCell, 0u, 0.f);
        wEx.store(kNoCell, 0u, 0.f);
        wEy.store(kNoCell, 0u, 0.f);
        wEz.store(kNoCell, 0u, 0.f);
    };
    constexpr int kLag = 2 * (T - 1);
    constexpr bool kEFromLds = T >= 3;  // registers: 128 per lane at 16 waves per CU
    // Owned planes from k0 need step s from plane k0 - (T - s) (E) or one below (H), i.e. the
    // first step from k0 - T; the last owned plane k1 - 1 leaves step T at iteration k1 - 1 +
    // 2(T-1).  Iterations m in [ms, me).
    const int ms = k0 >= T ? k0 - T : 0, me = k1 + kLag;
    Set S0, S1, S2, S3;
    {
        const int ke = ms, kez = ms <= Nz - 1 ? ms : Nz - 1;  // ms <= k0 < k1 <= Nz + 1
        S0.e.x = rEx.load(qEx, (unsigned)ke * sEx);  // E_0(ms)
        S0.e.y = rEy.load(qEy, (unsigned)ke * sEy);
        S0.e.z = rEz.load(qEz, (unsigned)kez * sEz);
        S0.h = F3{0.f, 0.f, 0.f};
    }
    load_set(S1, ms);
    pad_stores();
    load_set(S2, ms + 1);
    pad_stores();
    const int y = r + 1, x = l + 1;
    L.e[0][ms & 1][0][y][x] = S0.e.x;
    L.e[0][ms & 1][2][y][x] = S0.e.z;
    // carried own values of steps 1..T: planes one and two behind the step's own (index 0 unused)
    F3 h1[T + 1], h2[T + 1], e1[T + 1], e2[T + 1];
#pragma unroll
    for (int s = 0; s <= T; ++s) h1[s] = h2[s] = e1[s] = e2[s] = F3{0.f, 0.f, 0.f};

    lds_barrier();
    auto plane = [&](int m, const Set &P, const Set &S, Set &N) {
        const int b = m & 1, hb = HB == 2 ? b : 0;
        load_set(N, m + 2);
        // issue the loads of the plane two ahead before this plane's LDS traffic and its waits
        __builtin_amdgcn_sched_barrier(0);
        // ---- A: H_s(p_s) for every step
        F3 hn[T + 1], eo[T + 1];
#pragma unroll
        for (int s = 1; s <= T; ++s) {
            // E_{s-1}(p_s) and E_{s-1}(p_s + 1): with three or more steps, the own slots of the
            // E_{s-1} planes in LDS rather than registers carried across planes
            const auto &E = L.e[s - 1][b];
            const auto &Eu = L.e[s - 1][b ^ 1];
            const F3 ep = s == 1 ? P.e : kEFromLds ? F3{E[0][y][x], E[1][y][x], E[2][y][x]} : e2[s - 1];
            const F3 eu = s == 1 ? S.e : kEFromLds ? F3{Eu[0][y][x], Eu[1][y][x], Eu[2][y][x]} : e1[s - 1];
            const F3 ho = s == 1 ? S.h : h2[s - 1];  // H_{s-1}(p_s)
            eo[s] = ep;
            hn[s].x = ho.x + c.cH * ((eu.y - ep.y) * c.Cz - (E[2][y + 1][x] - ep.z) * c.Cy);
            // Ez and Ey at i + 1 from the next lane (the same values its LDS slots hold)
            hn[s].y = ho.y + c.cH * ((lane_next(ep.z) - ep.z) * c.Cx - (eu.x - ep.x) * c.Cz);
            hn[s].z = ho.z + c.cH * ((E[0][y + 1][x] - ep.x) * c.Cy - (lane_next(ep.y) - ep.y) * c.Cx);
            L.h[hb][s - 1][0][y][x] = hn[s].x;
            L.h[hb][s - 1][1][y][x] = hn[s].y;
            L.h[hb][s - 1][2][y][x] = hn[s].z;
        }
        L.e[0][b ^ 1][0][y][x] = S.e.x;
        L.e[0][b ^ 1][2][y][x] = S.e.z;
        lds_barrier();
        // ---- B: E_s(p_s) for every step (graphfdtd.cpp:243-312: interior cells update, faces
        // copy through)
        F3 en[T + 1];
#pragma unroll
        for (int s = 1; s <= T; ++s) {
            const int ps = m - 2 * (s - 1);
            const bool kIn = ps >= 1 && ps <= Nz - 1;
            const F3 e = eo[s];    // E_{s-1}(p_s)
            const F3 hp = h1[s];  // H_s(p_s - 1)
            const auto &H = L.h[hb][s - 1];
            const float wx = e.x + c.cE * ((hn[s].z - H[2][y - 1][x]) * c.Cy - (hn[s].y - hp.y) * c.Cz);
            const float wy = e.y + c.cE * ((hn[s].x - hp.x) * c.Cz - (hn[s].z - H[2][y][x - 1]) * c.Cx);
            const float wz = e.z + c.cE * ((hn[s].y - H[1][y][x - 1]) * c.Cx - (hn[s].x - H[0][y - 1][x]) * c.Cy);
            en[s].x = (jIn && kIn) ? wx : e.x;
            en[s].y = (iIn && kIn) ? wy : e.y;
            en[s].z = (iIn && jIn) ? wz : e.z;
            if (s < T) {  // E_s(p_s) in this parity's buffer was last read in A
                L.e[s][b][0][y][x] = en[s].x;
                if (kEFromLds) L.e[s][b][1][y][x] = en[s].y;  // read only at its own slot
                L.e[s][b][2][y][x] = en[s].z;
            }
        }
        // plane q of each output if it is in the slab and the field, else bit 31 and plane 0
        const int q = m - kLag;
        const bool out = q >= k0 && q < k1;
        const bool o1 = out && q < Nz, o2 = out && q <= Nz;
        const unsigned m1 = ownBit | (o1 ? 0u : kNoCell), m2 = ownBit | (o2 ? 0u : kNoCell);
        const unsigned p1 = o1 ? (unsigned)q : 0u, p2 = o2 ? (unsigned)q : 0u;
        wHx.store(qHx | m1, p1 * sHx, hn[T].x);
        wHy.store(qHy | m1, p1 * sHy, hn[T].y);
        wHz.store(qHz | m2, p2 * sHz, hn[T].z);
        wEx.store(qEx | m2, p2 * sEx, en[T].x);
        wEy.store(qEy | m2, p2 * sEy, en[T].y);
        wEz.store(qEz | m1, p1 * sEz, en[T].z);
#pragma unroll
        for (int s = 1; s <= T; ++s) {
            h2[s] = h1[s];
            h1[s] = hn[s];
            e2[s] = e1[s];
            e1[s] = en[s];
        }
        // With one H buffer, A of the next plane must not overwrite it before every wave has
        // read it here.  With two, the next A writes the other buffer, and every plane B writes
        // here is read two planes on, after the next barrier; the E_0 plane A writes next (the
        // other parity of e[0]) was last read in this plane's A, before the barrier above.
        if (HB == 1) lds_barrier();
    };
    // The sets rotate through four planes, and the loop runs whole groups of four with no branch
    // inside: up to three planes past me - 1 are formed and discarded (q >= k1: nothing stored).
    for (int m = ms; m < me; m += 4) {
        plane(m, S0, S1, S3);
        plane(m + 1, S1, S2, S0);
        plane(m + 2, S2, S3, S1);
        plane(m + 3, S3, S0, S2);
    }
}

// ---- the same tiles with every lane's column in registers ------------------------------------------
//
// column_tile computes what overlapn_tile computes, over the same tiles and with the same pipeline
// of steps, with less work per plane for problems whose time is a plane's latency rather than HBM:
// a lane keeps its own column of every step in registers (of each step the two planes that step s + 1
// still needs, in two slots by iteration parity; within an iteration the steps go from T down to 1, so
// a slot is overwritten just after its last use and nothing is copied), i - 1 and i + 1 are the
// neighbouring lanes (a DPP operand), and only the row neighbours cross waves, through LDS planes by
// iteration parity: Ex and Ez of row j + 1 for A, Hx and Hz of row j - 1 for B.
//   h[s]  written in A of iteration m, read in B of m, written again in A of m + 2;
//   e[s]  written in B of m (the inputs' in A of m - 1), read in A of m + 2 (m), written again in B
//         of m + 2 (A of m + 1): each pair has a barrier between, so the one barrier between A and
//         B orders every access.
// A step is formed only in the iterations that need it: with T = 3, owned planes [k0, k1) need H_s
// from iteration 3(s - 1) on (counted from plane k0 - T) and E_s up to T - s iterations before the
// last, so a slab of n planes takes 8 + 4 ceil((n - 1) / 4) iterations (the inner ones run in groups of
// four) and 3n + 9 step planes or up to 9 more, instead of 3n + 21: most of the work of the short slabs that
// a small problem is cut into.
// Measured, us per three-step launch on 256 blocks, against overlapn_tile on the same slabs and on equal
// runs of planes:
//   48^3 14.6, 21.2, 20.1;  64^3 21.4, 28.8, 41.3;  96^3 25.2, 33.8, 46.6;  128^3 45.9, 58.6, 66.2;
//   160^3 56.1, 72.4, 84.6;  192^3 129, 125, 135;  224^3 212, 219, 219;  248^3 234, 224, 284;
//   256^3 317, 319, 320;  288^3 572, 573, 574;  320^3 917, 920, 921;  344^3 1128, 1135, 1135;
//   200 x 200 x 800 537, 476, 701;  320 x 320 x 32 60.6, 74.1, 73.2.
// So it is the faster while the fields of a launch lie in cache, and once they do not the two stay within
// 5% of each other, either way, but for a few shapes (80 to 126 tiles of 340 to 730 MB, and 200 x 200 x 800)
// that no line through tiles, planes or bytes separates.  With more tiles than blocks it is the slower,
// 890 us against 755 at 384^3: it computes a launch in 460 us when nothing is read or written, so the blocks
// run at the pace of memory and drift apart, and neighbouring tiles then fetch the three cells they share
// twice (FETCH_SIZE 2.12 GB against 1.67).  overlapn_tile's two barriers and fuller planes keep the blocks
// in step.  So this body serves the launches with fewer tiles than blocks, overlapn_tile the others.
template <int T, int MAXR>
struct ColumnLds {
    float e[T][2][2][MAXR + 1][64]; // Ex, Ez of E_0 .. E_{T-1}: row r's at [r]
    float h[T][2][2][MAXR + 1][64]; // Hx, Hz of H_1 .. H_T: row r's at [r + 1]
};

// A field of `bytes` bytes from the row at byte offset `row` of its first plane on; a plane is then
// addressed by its byte offset in a scalar register and a 32-bit lane part.  Loads are clamped into
// the field (what is read outside it reaches no stored cell).  A lane that stores nothing carries
// bit 31 in its part, which the buffer unit's range check drops whether or not it counts the scalar
// part (their sum stays below 2^32); the scalar part is that of a plane inside the field.
__device__ inline PlaneBuf row_buf(const float *p, unsigned bytes, unsigned row) {
    return plane_buf((const float *)((const char *)p + row), bytes - row);
}

// A value that is the same in every lane, in a scalar register.
__device__ inline unsigned uni(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }

template <int T, int MAXR>
__device__ inline void column_tile(const Fields &F, const FDTD_PARAMS &p, int i0, int j0, int k0, int k1,
                                   ColumnLds<T, MAXR> &L) {
    static_assert(T == 3, "the iterations below are those of three steps");
    const Coef c = make_coef(p);
    i0 = (int)uni((unsigned)i0), j0 = (int)uni((unsigned)j0), k0 = (int)uni((unsigned)k0), k1 = (int)uni((unsigned)k1);
    const int R = (int)blockDim.y;
    const int l = (int)threadIdx.x, r = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int i = i0 - T + l, j = j0 - T + r;
    const int Nx = p.Nx, Ny = p.Ny, Nz = p.Nz;
    auto clamp = [](int v, int hi) { return v < 0 ? 0 : v < hi ? v : hi; };
    // lane offsets of the fields with Nx + 1 and with Nx cells per row; bit 31 where nothing is stored
    const unsigned c1 = 4u * (unsigned)clamp(i, Nx), c0 = 4u * (unsigned)clamp(i, Nx - 1);
    const bool ownL = l >= T && l <= 63 - T, ownR = r >= T && r <= R - 1 - T;
    const unsigned n1 = uni(ownR && j <= Ny ? 0u : kNoCell), n0 = uni(ownR && j < Ny ? 0u : kNoCell);
    // lane parts of the stores to the four extents (see below)
    const unsigned l1 = ownL && i <= Nx ? c1 : kNoCell, l0 = ownL && i < Nx ? c0 : kNoCell;
    const unsigned lA = l1 | n0, lB = l0 | n1, lC = l0 | n0, lD = l1 | n1;
    // row offsets and plane strides of the four extents: (Nx+1, Ny) Hx Ey, (Nx, Ny+1) Hy Ex, (Nx, Ny) Hz,
    // (Nx+1, Ny+1) Ez
    const int j1 = clamp(j, Ny), j0r = clamp(j, Ny - 1);
    const unsigned rA = uni(4u * (Nx + 1) * j0r), rB = uni(4u * Nx * j1), rC = uni(4u * Nx * j0r), rD = uni(4u * (Nx + 1) * j1);
    const unsigned sA = 4u * (Nx + 1) * Ny, sB = 4u * Nx * (Ny + 1), sC = 4u * Nx * Ny, sD = 4u * (Nx + 1) * (Ny + 1);
    const PlaneBuf rHx = row_buf(F.hx, sA * Nz, rA), rHy = row_buf(F.hy, sB * Nz, rB), rHz = row_buf(F.hz, sC * (Nz + 1), rC),
                   rEx = row_buf(F.ex, sB * (Nz + 1), rB), rEy = row_buf(F.ey, sA * (Nz + 1), rA), rEz = row_buf(F.ez, sD * Nz, rD);
    const PlaneBuf wHx = row_buf(F.ohx, sA * Nz, rA), wHy = row_buf(F.ohy, sB * Nz, rB), wHz = row_buf(F.ohz, sC * (Nz + 1), rC),
                   wEx = row_buf(F.oex, sB * (Nz + 1), rB), wEy = row_buf(F.oey, sA * (Nz + 1), rA), wEz = row_buf(F.oez, sD * Nz, rD);
    const bool jIn = j >= 1 && j <= Ny - 1, iIn = i >= 1 && i <= Nx - 1;

    struct Set {
        F3 e, h;
    };
    // S_m = {E_0(m+1), H_0(m)}.  The owned planes below k1 depend on input planes up to T above
    // them (each step reaches one plane up), so only m <= k1 + T - 2 feed owned cells; a later
    // set reloads that set's planes (cached) and a plane outside a field is read as its first or
    // last: those values reach no stored cell, as the planes formed from them do not (E of plane 0
    // and of plane Nz is copied through, whatever the planes beyond).
    auto load_set = [&](Set &S, int m) {
        const int k = m < k1 + T - 2 ? m : k1 + T - 2;
        const unsigned ke = clamp(k + 1, Nz), kez = clamp(k + 1, Nz - 1), kh = clamp(k, Nz - 1), khz = clamp(k, Nz);
        S.e.x = rEx.load(c0, ke * sB);
        S.e.y = rEy.load(c1, ke * sA);
        S.e.z = rEz.load(c1, kez * sD);
        S.h.x = rHx.load(c1, kh * sA);
        S.h.y = rHy.load(c0, kh * sB);
        S.h.z = rHz.load(c0, khz * sC);
    };
    // six dropped stores: the prologue then leaves the memory counter as a loop iteration does,
    // so the waits the compiler places in the loop stay two planes behind the loads
    auto pad_stores = [&]() {
        wHx.store(kNoCell, 0u, 0.f);
        wHy.store(kNoCell, 0u, 0.f);
        wHz.store(kNoCell, 0u, 0.f);
        wEx.store(kNoCell, 0u, 0.f);
        wEy.store(kNoCell, 0u, 0.f);
        wEz.store(kNoCell, 0u, 0.f);
    };
    constexpr int kLag = 2 * (T - 1);
    const int ms = k0 - T;  // the first iteration's plane (see above); the last is k1 - 1 + kLag
    Set S0, S1, S2, S3;
    {
        const unsigned ke = clamp(ms, Nz), kez = clamp(ms, Nz - 1);
        S0.e.x = rEx.load(c0, ke * sB);  // E_0(ms)
        S0.e.y = rEy.load(c1, ke * sA);
        S0.e.z = rEz.load(c1, kez * sD);
        S0.h = F3{0.f, 0.f, 0.f};
    }
    load_set(S1, ms);
    pad_stores();
    load_set(S2, ms + 1);
    pad_stores();
    // this lane's row of an LDS plane; the other planes and rows are constant offsets from it (the
    // empty asm keeps the two bases in registers instead of a sum per access)
    typedef __attribute__((address_space(3))) float Lds;
    Lds *eb = (Lds *)&L.e[0][0][0][r][l], *hb = (Lds *)&L.h[0][0][0][r][l];
    asm("" : "+v"(eb), "+v"(hb));
    constexpr int kRow = 64, kPlane = (MAXR + 1) * kRow;
    auto ls = [](Lds *q, int s, int par, int comp, int row) -> Lds & { return q[((s * 2 + par) * 2 + comp) * kPlane + row * kRow]; };
    ls(eb, 0, 0, 0, 0) = S0.e.x;  // iteration ms has parity 0
    ls(eb, 0, 0, 1, 0) = S0.e.z;
    // own columns of steps 1 .. T by iteration parity (index 0 unused)
    F3 E[T + 1][2], H[T + 1][2];
#pragma unroll
    for (int s = 0; s <= T; ++s) E[s][0] = E[s][1] = H[s][0] = H[s][1] = F3{0.f, 0.f, 0.f};

    lds_barrier();
    // iteration m, forming steps lo .. hi; P, S, N: sets m - 1, m, m + 2
    auto plane = [&](int m, auto parity, auto lo_, auto hi_, const Set &P, const Set &S, Set &N) {
        constexpr int b = decltype(parity)::value, lo = decltype(lo_)::value, hi = decltype(hi_)::value;
        if (lo == 1) {
            load_set(N, m + 2);
            // issue the loads of the plane two ahead before this plane's LDS traffic and its waits
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- A: H_s(p_s) for every step
        float xj[T], zj[T];  // Ex, Ez of E_{s-1}(p_s) in row j + 1: read before anything is written
#pragma unroll
        for (int s = hi; s >= lo; --s) {
            xj[s - 1] = ls(eb, s - 1, b, 0, 1);
            zj[s - 1] = ls(eb, s - 1, b, 1, 1);
        }
#pragma unroll
        for (int s = hi; s >= lo; --s) {
            const F3 ep = s == 1 ? P.e : E[s - 1][b], eu = s == 1 ? S.e : E[s - 1][b ^ 1];
            const F3 ho = s == 1 ? S.h : H[s - 1][b];
            const float exj = xj[s - 1], ezj = zj[s - 1];
            F3 &hn = H[s][b];
            hn.x = ho.x + c.cH * ((eu.y - ep.y) * c.Cz - (ezj - ep.z) * c.Cy);
            hn.y = ho.y + c.cH * ((lane_next(ep.z) - ep.z) * c.Cx - (eu.x - ep.x) * c.Cz);
            hn.z = ho.z + c.cH * ((exj - ep.x) * c.Cy - (lane_next(ep.y) - ep.y) * c.Cx);
            ls(hb, s - 1, b, 0, 1) = hn.x;
            ls(hb, s - 1, b, 1, 1) = hn.z;
        }
        if (lo == 1) {
            ls(eb, 0, b ^ 1, 0, 0) = S.e.x;
            ls(eb, 0, b ^ 1, 1, 0) = S.e.z;
        }
        lds_barrier();
        // ---- B: E_s(p_s) for every step (graphfdtd.cpp:243-312: interior cells update, faces
        // copy through)
        F3 out;
#pragma unroll
        for (int s = hi; s >= lo; --s) {  // Hx, Hz of H_s(p_s) in row j - 1
            xj[s - 1] = ls(hb, s - 1, b, 0, 0);
            zj[s - 1] = ls(hb, s - 1, b, 1, 0);
        }
#pragma unroll
        for (int s = hi; s >= lo; --s) {
            const int ps = m - 2 * (s - 1);
            const bool kIn = ps >= 1 && ps <= Nz - 1;
            const F3 e = s == 1 ? P.e : E[s - 1][b];
            const F3 hn = H[s][b], hp = H[s][b ^ 1];
            const float hxj = xj[s - 1], hzj = zj[s - 1];
            const float wx = e.x + c.cE * ((hn.z - hzj) * c.Cy - (hn.y - hp.y) * c.Cz);
            const float wy = e.y + c.cE * ((hn.x - hp.x) * c.Cz - (hn.z - lane_prev(hn.z)) * c.Cx);
            const float wz = e.z + c.cE * ((hn.y - lane_prev(hn.y)) * c.Cx - (hn.x - hxj) * c.Cy);
            F3 &en = s == T ? out : E[s][b];
            en.x = (jIn && kIn) ? wx : e.x;
            en.y = (iIn && kIn) ? wy : e.y;
            en.z = (iIn && jIn) ? wz : e.z;
            if (s < T) {
                ls(eb, s, b, 0, 0) = en.x;
                ls(eb, s, b, 1, 0) = en.z;
            }
        }
        if (hi < T) {
            pad_stores();
            return;
        }
        // plane q of each output if it is in the slab and the field
        const int q = m - kLag;
        const bool in = q >= k0 && q < k1;
        const unsigned q0 = uni(in && q < Nz ? 0u : kNoCell), q1 = uni(in ? 0u : kNoCell);
        const unsigned k1q = (unsigned)clamp(q, Nz), k0q = (unsigned)clamp(q, Nz - 1);
        wHx.store(lA | q0, k0q * sA, H[T][b].x);
        wHy.store(lB | q0, k0q * sB, H[T][b].y);
        wHz.store(lC | q1, k1q * sC, H[T][b].z);
        wEx.store(lB | q1, k1q * sB, out.x);
        wEy.store(lA | q1, k1q * sA, out.y);
        wEz.store(lD | q0, k0q * sD, out.z);
    };
    // The sets rotate through four iterations.  The loop runs whole groups of four with no branch
    // inside: up to three planes past the slab are formed and discarded (q >= k1: nothing stored).
    typedef std::integral_constant<int, 0> Even;
    typedef std::integral_constant<int, 1> Odd, One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, 3> Three;
    int m = ms;
    plane(m, Even{}, One{}, One{}, S0, S1, S3);
    plane(m + 1, Odd{}, One{}, One{}, S1, S2, S0);
    plane(m + 2, Even{}, One{}, One{}, S2, S3, S1);
    plane(m + 3, Odd{}, One{}, Two{}, S3, S0, S2);
    plane(m + 4, Even{}, One{}, Two{}, S0, S1, S3);
    plane(m + 5, Odd{}, One{}, Two{}, S1, S2, S0);
    for (m += 6; m < k1 + 2; m += 4) {  // iterations 6 .. n + 4
        plane(m, Even{}, One{}, Three{}, S2, S3, S1);
        plane(m + 1, Odd{}, One{}, Three{}, S3, S0, S2);
        plane(m + 2, Even{}, One{}, Three{}, S0, S1, S3);
        plane(m + 3, Odd{}, One{}, Three{}, S1, S2, S0);
    }
    plane(m, Even{}, Two{}, Three{}, S2, S3, S1);
    plane(m + 1, Odd{}, Three{}, Three{}, S3, S0, S2);
}

}  // namespace ptk_fdtd
