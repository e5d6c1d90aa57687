// Device code of the fused stream-collide step (templates), included by the per-storage translation
// units oal_step_<storage>.hip so that the four storage forms compile in parallel.
//
// Work decomposition of the step kernels: one work-item per cell, one workgroup per 16 x 16 plane of
// a 16^3 block (256 lanes = 4 wavefronts of 16 x 4 cells).  Populations are block-major: each block holds its 27 direction arrays of 4096 cells
// contiguously (pop_index), so the 64 lanes of a wavefront touch 4 consecutive 64-byte rows of each
// of the block's direction arrays.  A workgroup's block, plane, domain and neighbour-block indices are
// uniform, which keeps them in scalar registers.
//
// Reference: src/collision/kernel_cumulant.jl:29-912 (stream_collide_cumulant!).
#pragma once

#include <hip/hip_runtime.h>

#include "oal_kernels.h"

namespace oal {

// Workgroups are dispatched round-robin over the 8 XCDs of the MI355X.  Remap the workgroup index so
// that each XCD receives a contiguous range of items: neighbouring planes and blocks, which share
// halo cache lines, then meet in the same L2.
__device__ __forceinline__ uint32_t xcd_item(uint32_t i, uint32_t n) {
    const uint32_t q = n >> 3, r = n & 7u, x = i & 7u, j = i >> 3;
    return x < r ? x * (q + 1u) + j : r * (q + 1u) + (x - r) * q + j;
}

// how the population arriving in one direction is obtained
enum : int {
    SRC_REG = 0,     // pulled from the source cell
    SRC_INLET = 1,   // equilibrium at (1, u_inlet)                       kernel_cumulant.jl:235-239
    SRC_OWN = 2,     // the cell's own population, same direction (outlet) kernel_cumulant.jl:240-245
    SRC_OPP = 3,     // own opposite population: no-slip wall            kernel_cumulant.jl:270-271, 340-341
    SRC_MIRY = 4,    // own y-mirrored population: free slip             kernel_cumulant.jl:342-343
    SRC_MIRZ = 5,    // own z-mirrored population: free slip             kernel_cumulant.jl:344-345
    SRC_REST = 6,    // rest weight (no neighbour block on level 1)      kernel_cumulant.jl:389-390
    SRC_SOLID = 7,   // halfway bounce-back from a solid source cell
    SRC_ZIMG = 8,    // exact specular z wall: the image cell's mirror_z population  kernel_cumulant.jl:272-321
    SRC_TFS = 9      // transverse freestream: own population blended toward feq(1, u_inlet)  :323-339
};

// what a level needs beside the plain step in the two-cells-per-lane kernel
// (or which half-step of the AA pattern, or the plain form of blocks with a base per layer)
enum : int { TWO_PLAIN = 0, TWO_SPONGE = 1, TWO_BFL = 2, TWO_AA_EVEN = 3, TWO_AA_ODD = 4, TWO_WIDE = 5, TWO_AA_ODD_WIDE = 6 };

enum : int { PAT_AB = 0, PAT_AA_EVEN = 1, PAT_AA_ODD = 2 };

// Uniform (per-workgroup) and per-lane state of one cell
struct CellCtx {
    uint32_t b, flags, own;
    uint32_t lmask;   // bit k: the source of direction k is solid; bit 27: the cell is solid
    int lx, ly, z, gx, gy, gz;
    int ext0, ext1, ext2, per0, per1, per2;
    int zwall, ymin_wall;
};

// The source of direction K for this cell: classification and, for SRC_REG / SRC_SOLID, the cell index.
// GEN = false is the interior path (block flags all clear): every source is a regular cell of this
// block or of one of its 26 neighbours, which all exist.
// FX: the exact specular z wall and the transverse freestream are compiled in (levels that use neither
// run a form without them)
template <int K, bool GEN, bool REG = false, bool FX = true>
__device__ __forceinline__ int classify(const StepArgs& a, const CellCtx& c, uint32_t& src) {
    constexpr int cx = dcx(K), cy = dcy(K), cz = dcz(K);
    if constexpr (GEN) {
        if (c.flags & BF_EDGE) {
            const int sgx = c.gx - cx, sgy = c.gy - cy, sgz = c.gz - cz;
            const bool xl = cx > 0 && !c.per0 && sgx < 0;
            const bool xh = cx < 0 && !c.per0 && sgx >= c.ext0;
            const bool yl = cy > 0 && !c.per1 && sgy < 0;
            const bool yh = cy < 0 && !c.per1 && sgy >= c.ext1;
            const bool zl = cz > 0 && !c.per2 && sgz < 0;
            const bool zh = cz < 0 && !c.per2 && sgz >= c.ext2;
            if (xl) return SRC_INLET;
            if (xh) return SRC_OWN;
            if (FX && c.zwall == 1 && (zl || zh)) {
                // the source beyond the wall mirrors the wall-row cell (x - cx, y - cy, z): that cell's
                // population mirror_z(K) arrives; with no such cell on the level (beyond a non-periodic
                // y face, or an absent block) the cell's own mirror_z(K)
                const int ix = c.lx - cx, iy = c.ly - cy, igy = c.gy - cy;
                const int ox = ix < 0 ? -1 : (ix >= BS ? 1 : 0), oy = iy < 0 ? -1 : (iy >= BS ? 1 : 0);
                int32_t nbk = (int32_t)c.b;
                if (ox | oy) nbk = a.nbr_bm[(size_t)c.b * 32 + (ox + 1) + 3 * (oy + 1) + 9];
                if ((!c.per1 && (igy < 0 || igy >= c.ext1)) || nbk < 0) return SRC_MIRZ;
                src = (uint32_t)nbk * BS3 + ((uint32_t)c.z << 8) + ((uint32_t)(iy & (BS - 1)) << 4) + (uint32_t)(ix & (BS - 1));
                return SRC_ZIMG;
            }
            if (c.zwall != 0 && (zl || zh)) return SRC_OPP;
            if (FX && a.cp.tfs && (yl || yh || zl || zh)) return SRC_TFS;
            if (yl && c.ymin_wall == 1) return SRC_OPP;
            if (yl || yh) return SRC_MIRY;
            if (zl || zh) return SRC_MIRZ;
        }
    }
    if constexpr (REG) {
        // regular addressing: the caller forms the address; only the solid test remains
        if constexpr (GEN) {
            if ((c.flags & BF_SOLID) && a.cp.bb_mode == 1 && ((c.lmask >> K) & 1u)) return SRC_SOLID;
        }
        return SRC_REG;
    }
    const int sx = c.lx - cx, sy = c.ly - cy, sz = c.z - cz;
    int32_t nbk = (int32_t)c.b;
    if constexpr (cx != 0 || cy != 0 || cz != 0) {
        // candidate neighbour blocks are uniform (scalar) values; the lane picks one by its crossing
        const int oz = cz == 0 ? 0 : (sz < 0 ? -1 : (sz >= BS ? 1 : 0));
        const int dz = 9 * (oz + 1);
        const int32_t* nt = a.nbr_bm + (size_t)c.b * 32;
        int32_t n_c = oz == 0 ? (int32_t)c.b : nt[4 + dz];
        if constexpr (!GEN) n_c = max(n_c, 0);
        int32_t pick = n_c;
        if constexpr (cx != 0 && cy != 0) {
            int32_t n_x = nt[(1 - cx) + 3 + dz], n_y = nt[1 + 3 * (1 - cy) + dz], n_xy = nt[(1 - cx) + 3 * (1 - cy) + dz];
            if constexpr (!GEN) { n_x = max(n_x, 0); n_y = max(n_y, 0); n_xy = max(n_xy, 0); }
            const bool crx = (unsigned)sx >= (unsigned)BS, cry = (unsigned)sy >= (unsigned)BS;
            pick = crx ? (cry ? n_xy : n_x) : (cry ? n_y : n_c);
        } else if constexpr (cx != 0) {
            int32_t n_x = nt[(1 - cx) + 3 + dz];
            if constexpr (!GEN) n_x = max(n_x, 0);
            pick = ((unsigned)sx >= (unsigned)BS) ? n_x : n_c;
        } else if constexpr (cy != 0) {
            int32_t n_y = nt[1 + 3 * (1 - cy) + dz];
            if constexpr (!GEN) n_y = max(n_y, 0);
            pick = ((unsigned)sy >= (unsigned)BS) ? n_y : n_c;
        }
        nbk = pick;
    }
    if constexpr (GEN) {
        if (nbk < 0) return SRC_REST;   // absent block inside the extent (BF_MISSING); never an address
    }
    src = (uint32_t)nbk * BS3 + ((uint32_t)(sz & (BS - 1)) << 8) + ((uint32_t)(sy & (BS - 1)) << 4) + (uint32_t)(sx & (BS - 1));
    if constexpr (GEN) {
        if ((c.flags & BF_SOLID) && a.cp.bb_mode == 1 && ((c.lmask >> K) & 1u)) return SRC_SOLID;
    }
    return SRC_REG;
}

// Regular interior blocks: the block's neighbours sit at lexicographic offsets (b +- 1, +- nbx,
// +- nbx*nby), so a source cell's address is arithmetic.  Each lane forms, once, the byte offsets of
// its nine in-plane source classes (cx, cy) - own cell shifted by -c in x and y, into the neighbour
// block where it crosses - relative to the start of its own block; every direction's access adds a
// uniform part (the block, the direction slot, the z plane) to its scalar base pointer.
template <class SP>
struct RegAddr {
    int32_t v[3][3];           // [cx+1][cy+1]: byte offset of cell (x - cx, y - cy, zref) from the own block
    int64_t blk0;              // element offset of the own block: b * 27 * BS3
    int64_t plane_elems;       // elements between consecutive block layers (nbx * nby * 27 * BS3)
    int zref;                  // the plane the offsets were formed for (other planes: uniform shift)
    __device__ __forceinline__ void init(const CellCtx& c, int nbx, int nby) {
        blk0 = (int64_t)c.b * (27 * BS3);
        plane_elems = (int64_t)nbx * nby * (27 * BS3);
        zref = c.z;
        const int32_t local = (int32_t)(c.own - c.b * BS3);   // zref * BS2 + ly * BS + lx
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int cx = i - 1, cy = j - 1;
                const int sx = c.lx - cx, sy = c.ly - cy;
                const int dx = sx < 0 ? -1 : (sx >= BS ? 1 : 0);
                const int dy = sy < 0 ? -1 : (sy >= BS ? 1 : 0);
                const int32_t idx = (dx + dy * nbx) * (27 * BS3) + local + (sx - BS * dx - c.lx) + BS * (sy - BS * dy - c.ly);
                v[i][j] = idx * (int32_t)sizeof(typename SP::st);
            }
    }
    // uniform base of direction-slot `slot` for plane z of the block and a source shifted by -cz in z
    __device__ __forceinline__ const char* base(const void* f, int slot, int z, int cz) const {
        const int sz = z - cz;
        const int dz = sz < 0 ? -1 : (sz >= BS ? 1 : 0);
        const int64_t e = blk0 + (int64_t)slot * BS3 + dz * plane_elems + (int64_t)(sz - BS * dz - zref) * BS2;
        return (const char*)f + e * (int64_t)sizeof(typename SP::st);
    }
};

// Population J of this cell's own post-collision state of the previous step: slot (x, J) after an
// AB step, slot (x, opp J) after an AA even step.
template <class SP, int PAT, int J>
__device__ __forceinline__ typename SP::T own_prev(const StepArgs& a, const CellCtx& c) {
    constexpr int slot = PAT == PAT_AB ? J : dopp(J);
    return SP::ld((const typename SP::st*)a.fin + pop_index(c.own, slot), wgt<typename SP::T>(J));
}

template <int J>
using dir_c = std::integral_constant<int, J>;

// transverse freestream: (1 - b) f_K + b feq_K(1, u_inlet) (kernel_cumulant.jl:333-339)
template <int K, class T>
__device__ __forceinline__ T tfs_value(const StepArgs& a, T donor, float u_in) {
    const T b = T(a.cp.tfs_blend);
    const T feq = feq_auto(T(1), T(u_in), T(0), T(0), wgt<T>(K), T(dcx(K)), T(dcy(K)), T(dcz(K)), a.cp.compressible);
    return (T(1) - b) * donor + b * feq;
}

// The value of a boundary rule for direction K.  `own(dir_c<j>)` yields population j of the cell's
// own post-collision state of the step the rule refers to.
template <int K, class T, class OWN>
__device__ __forceinline__ T boundary_value(int kind, const StepArgs& a, const CellCtx& c, float u_in, int32_t step,
                                            OWN&& own) {
    switch (kind) {
        case SRC_INLET: {
            // the noise amplitude in the working precision (FP32 for the FP32-arithmetic forms, as the reference)
            const float turb = a.cp.inlet_turb;
            const T noise = turb > 0.0f ? T(inlet_noise(c.gy + 1, c.gz + 1, step, 1234)) * T(turb) * T(u_in) : T(0);
            const T u_inst = T(u_in) + noise;
            return feq_auto(T(1), u_inst, T(0), T(0), wgt<T>(K), T(dcx(K)), T(dcy(K)), T(dcz(K)), a.cp.compressible);
        }
        case SRC_OWN: return own(dir_c<K>{});
        case SRC_OPP:
        case SRC_SOLID: return own(dir_c<dopp(K)>{});
        case SRC_MIRY: return own(dir_c<dmir_y(K)>{});
        case SRC_MIRZ:
        case SRC_ZIMG: return own(dir_c<dmir_z(K)>{});   // (the pull gather reads the image cell itself)
        case SRC_TFS: return tfs_value<K, T>(a, own(dir_c<K>{}), u_in);
        default: return wgt<T>(K);
    }
}

// The population of the cell's own post-collision state that a boundary rule for direction K returns
// (the rest weight, SRC_REST, does not depend on it)
template <int K>
__device__ __forceinline__ int rule_dir(int kind) {
    switch (kind) {
        case SRC_OPP:
        case SRC_SOLID: return dopp(K);
        case SRC_MIRY: return dmir_y(K);
        case SRC_MIRZ:
        case SRC_ZIMG: return dmir_z(K);
        default: return K;
    }
}

// workgroup sum of 3 doubles into part[item*4 + 0..2]; every lane of the workgroup must call it
__device__ __forceinline__ void wg_sum3(double v0, double v1, double v2, double* part, uint32_t item) {
    __shared__ double red[3][WG / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v0 += __shfl_xor(v0, off, 64);
        v1 += __shfl_xor(v1, off, 64);
        v2 += __shfl_xor(v2, off, 64);
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { red[0][wave] = v0; red[1][wave] = v1; red[2][wave] = v2; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) { s0 += red[0][w]; s1 += red[1][w]; s2 += red[2][w]; }
        part[(size_t)item * 4 + 0] = s0;
        part[(size_t)item * 4 + 1] = s1;
        part[(size_t)item * 4 + 2] = s2;
    }
}

// WALE: central differences of the previous step's velocity over the six face neighbours; a solid or
// absent neighbour contributes the cell's own velocity (physics_utils.jl:1981-2035, 2217-2233)
template <class T>
__device__ __forceinline__ T wale_of(const StepArgs& a, const CellCtx& c) {
    const T* v = (const T*)a.vel_in;
    const uint32_t n = a.ncell;
    T un[6][3];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const int ddx = q == 0 ? 1 : (q == 1 ? -1 : 0);
        const int ddy = q == 2 ? 1 : (q == 3 ? -1 : 0);
        const int ddz = q == 4 ? 1 : (q == 5 ? -1 : 0);
        bool ok = true;
        if (c.flags & BF_EDGE) {
            const int ngx = c.gx + ddx, ngy = c.gy + ddy, ngz = c.gz + ddz;
            if (!c.per0 && (ngx < 0 || ngx >= c.ext0)) ok = false;
            if (!c.per1 && (ngy < 0 || ngy >= c.ext1)) ok = false;
            if (!c.per2 && (ngz < 0 || ngz >= c.ext2)) ok = false;
        }
        const int sx = c.lx + ddx, sy = c.ly + ddy, sz = c.z + ddz;
        const int ox = sx < 0 ? -1 : (sx >= BS ? 1 : 0);
        const int oy = sy < 0 ? -1 : (sy >= BS ? 1 : 0);
        const int oz = sz < 0 ? -1 : (sz >= BS ? 1 : 0);
        int32_t nbk = (int32_t)c.b;
        if (ok && (ox | oy | oz)) nbk = a.nbr_bm[(size_t)c.b * 32 + (ox + 1) + 3 * (oy + 1) + 9 * (oz + 1)];
        if (nbk < 0) ok = false;
        // the face neighbour x + e is the source of the direction -e: its solid bit in the link mask
        constexpr int kq[6] = {12, 14, 10, 16, 4, 22};
        uint32_t idx = c.own;
        if (ok) {
            idx = (uint32_t)nbk * BS3 + ((uint32_t)(sz & (BS - 1)) << 8) + ((uint32_t)(sy & (BS - 1)) << 4) + (uint32_t)(sx & (BS - 1));
            if ((c.lmask >> kq[q]) & 1u) idx = c.own;
        }
        un[q][0] = v[idx]; un[q][1] = v[n + idx]; un[q][2] = v[2 * (size_t)n + idx];
    }
    const T h = T(0.5);
    return wale_nu(h * (un[0][0] - un[1][0]), h * (un[2][0] - un[3][0]), h * (un[4][0] - un[5][0]),
                   h * (un[0][1] - un[1][1]), h * (un[2][1] - un[3][1]), h * (un[4][1] - un[5][1]),
                   h * (un[0][2] - un[1][2]), h * (un[2][2] - un[3][2]), h * (un[4][2] - un[5][2]), T(a.cp.c_wale));
}

// The fused stream-collide step of one cell.  PAT_AB pulls from fin into fout (the reference's
// scheme); PAT_AA_EVEN / PAT_AA_ODD are the two half-steps of the in-place AA pattern on one buffer:
//   even: read f_k(x) from slot (x, k), write f*_k(x) to slot (x, opp k);
//   odd:  read f_k(x) from slot (x - c_k, opp k), write f*_k(x) to slot (x + c_k, k).
// Boundary rules of the odd step's writes: where x + c_k is not a cell that steps, the rule of the
// opposite direction is evaluated from the fresh post-collision state and stored in (x, opp k), the
// slot the following even step reads, so the even step needs no boundary logic.
//
// Momentum exchange (OAL_STEP_FORCE): summed over the links whose populations this step's collision
// produced, i.e. the exchange of the streaming that follows it: 2 (f_i* - w_i) c_i for halfway
// bounce-back, (f_i*(t) + f_i*(t-1) - 2 w_i) c_i for the reference's solid reflection (the solid cell
// returns last step's population), i toward a solid cell (src/octree_q19/src/stream.jl:248-256).
// Interpolated bounce-back (the linear BFL rule of Bouzidi, Firdaouss and Lallemand 2001;
// bouzidi_kernel.jl:204-370 with its D3Q27 settings) in pull form, on the populations of one cell whose
// sources are solid (bits of solid_links).  For such a direction K the link toward the wall is
// I = opp(K), f[K] holds its halfway value f*_I(x) and q is the wall distance of link I:
//   q < 1/2:  2q f*_I(x) + (1 - 2q) f*_I(x - c_I)      (x - c_I: the pull source of direction I,
//             used when it is a fluid cell of the level; otherwise the fallback of a.bfl_fallback)
//   q >= 1/2: f*_I(x) / (2q) + (2q - 1) / (2q) f*_K(x)
// so the reflected population arrives at x itself.  q outside (q_min, 1] keeps halfway bounce-back.
// The link's momentum exchange (f*_I(x) + arriving value) c_I is summed here, at the gather.
template <class SP>
__device__ __forceinline__ void bfl_links(const StepArgs& a, const CellCtx& c, typename SP::T (&f)[27],
                                          uint32_t solid_links, uint32_t reg_links, bool want_force,
                                          double& F0, double& F1, double& F2) {
    using T = typename SP::T;
    using st = typename SP::st;
    const st* fi = (const st*)a.fin;
    const uint16_t* qb = a.qmap + (size_t)a.lslot[c.b] * (27 * BS3) + (c.own - c.b * BS3);
    T rho_f = T(0);
    if (a.bfl_fallback == 1) {
        // density of the cell's own post-collision populations (the wall-equilibrium fallback)
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            rho_f += SP::ld(fi + pop_index(c.own, K), wgt<T>(K));
        });
    }
    // by nine directions: the wall distances and the own populations of a wave's links are requested together
    // (one link after the other, each wave near a wall waits for some 20 pairs of dependent loads: the blocks
    // around a sphere, 160 x 128 x 128 FP32, 34.5 -> 27.6 us, the step 127.5 -> 121.9 us; FP64 has no registers
    // to spare)
    constexpr int BATCH = sizeof(T) == 4 ? 9 : 1;
    for_dirs([&](auto cc) {
        constexpr int C = decltype(cc)::value;
        if constexpr (C * BATCH < 27) {
            if (((solid_links >> (C * BATCH)) & ((1u << BATCH) - 1u)) == 0) return;
            uint16_t qr[BATCH];
            typename SP::raw own[BATCH];
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if constexpr (K / BATCH == C) {
                    qr[K % BATCH] = 0;
                    own[K % BATCH] = typename SP::raw(0);
                    if ((solid_links >> K) & 1u) {
                        qr[K % BATCH] = qb[(size_t)dopp(K) * BS3];
                        own[K % BATCH] = SP::ld_raw(fi + pop_index(c.own, K));
                    }
                }
            });
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if constexpr (K / BATCH == C) {
                    constexpr int I = dopp(K);
                    constexpr T w = wgt<T>(K);
                    if ((solid_links >> K) & 1u) {
                        const T fk = f[K];
                        T val = fk;
                        const float q = (float)__builtin_bit_cast(_Float16, qr[K % BATCH]);
                        if (q > a.q_min && q <= 1.0f) {
                            const T tq = T(q), fo = SP::from_raw(own[K % BATCH], w);
                            if (q < 0.5f) {
                                T fff = fk;
                                if ((reg_links >> I) & 1u) fff = f[I];
                                else if (a.bfl_fallback == 1) fff = rho_f * w;
                                else if (a.bfl_fallback == 2) fff = fo;
                                const T c1 = T(2) * tq;
                                val = c1 * fk + (T(1) - c1) * fff;
                            } else {
                                const T inv = T(1) / (T(2) * tq);
                                const T c2 = (T(2) * tq - T(1)) * inv;
                                val = inv * fk + c2 * fo;
                            }
                        }
                        if (want_force) {
                            const double m = ((double)fk - (double)w) + ((double)val - (double)w);
                            F0 += m * dcx(I); F1 += m * dcy(I); F2 += m * dcz(I);
                        }
                        f[K] = val;
                    }
                }
            });
        }
    });
}

// BFL: the level has a q-map (interpolated bounce-back); a separate instantiation, so that the boundary
// kernels of levels without one keep their register budget.
template <class SP, int PAT, bool WALE, bool GEN, bool REG = false, bool BFL = false, bool SPONGE = false, bool FX = true>
__device__ __forceinline__ void step_cell(const StepArgs& a, const CellCtx& c, const DevDomain* dm, bool active,
                                          bool solid_own, double& F0, double& F1, double& F2) {
    using T = typename SP::T;
    using st = typename SP::st;
    if (!active) return;
    const uint32_t b = c.b;
    const float u_in = dm->u_in;
    st* fo = (st*)a.fout;
    const st* fi = (const st*)a.fin;
    const uint32_t n = a.ncell;
    RegAddr<SP> ra;
    if constexpr (REG) ra.init(c, dm->nbx, dm->nby);

    T f[27];
    typename SP::raw raw[27];     // the loaded populations, decoded after all loads
    uint32_t inlet_links = 0, rest_links = 0, solid_links = 0, reg_links = 0, tfs_links = 0;
    // AA odd half-step: the even step's copy of the populations with cx = -1 of the cell's row on the
    // outlet face (they sit in slots that the west neighbour overwrites during this half-step)
    const st* ocopy = nullptr;
    if constexpr (PAT == PAT_AA_ODD && GEN) {
        if (c.flags & BF_EDGE) {
            const int32_t s = a.oslot[b];
            if (s >= 0) ocopy = (const st*)a.obuf + (size_t)s * 9 * BS2 + c.ly * BS + c.z;
        }
    }
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        constexpr T w = wgt<T>(K);
        T val;
        if constexpr (REG && !GEN && PAT == PAT_AA_EVEN) {
            val = SP::ld((const st*)(ra.base(fi, K, c.z, 0) + ra.v[1][1]), w);
        } else if constexpr (REG && !GEN) {
            static_assert(PAT == PAT_AA_ODD, "the AB pattern's regular blocks without a rule are the one-launch kernels'");
            val = SP::ld((const st*)(ra.base(fi, dopp(K), c.z, dcz(K)) + ra.v[dcx(K) + 1][dcy(K) + 1]), w);
        } else if constexpr (PAT == PAT_AA_EVEN) {
            // every direction loads the own slot K, so the 27 loads are in flight together; an inlet
            // link's value replaces it afterwards, evaluated in full precision as the pull step does
            // rather than read back from a slot that went through the storage rounding
            raw[K] = SP::ld_raw(fi + pop_index(c.own, K));
            if constexpr (GEN && dcx(K) > 0)
                inlet_links |= ((c.flags & BF_EDGE) && !c.per0 && c.gx == 0 ? 1u : 0u) << K;
            val = T(0);   // set below
        } else if constexpr (PAT == PAT_AB) {
            // branch-free gather: each direction reads one population - its source, or the own-cell
            // population its boundary rule returns (an inlet or rest link reads its own slot, unused) -
            // so the 27 loads are all in flight together; the inlet and rest rules replace the value
            // afterwards.  The rules' directions (opposite, mirrors) have the weight of K.
            uint32_t src = 0;
            const int kind = classify<K, GEN, REG, FX>(a, c, src);
            const int jd = kind == SRC_REG ? K : rule_dir<K>(kind);
            const st* p;
            if constexpr (REG)
                p = kind == SRC_REG ? (const st*)(ra.base(fi, K, c.z, dcz(K)) + ra.v[dcx(K) + 1][dcy(K) + 1])
                                    : fi + pop_index(FX && kind == SRC_ZIMG ? src : c.own, jd);
            else
                p = fi + pop_index(kind == SRC_REG || (FX && kind == SRC_ZIMG) ? src : c.own, jd);
            raw[K] = SP::ld_raw(p);
            inlet_links |= (kind == SRC_INLET ? 1u : 0u) << K;
            rest_links |= (kind == SRC_REST ? 1u : 0u) << K;
            if constexpr (FX) tfs_links |= (kind == SRC_TFS ? 1u : 0u) << K;
            solid_links |= (kind == SRC_SOLID ? 1u : 0u) << K;
            reg_links |= (kind == SRC_REG ? 1u : 0u) << K;
            val = T(0);   // set below
        } else {
            // AA odd half-step, branch-free as the AB gather: each direction loads one slot - the
            // source cell's slot opp K, the outlet copy (the own population of direction K, cx = -1),
            // or the own slot opp j of the population j its boundary rule returns; an inlet or rest
            // link reads the own slot K, unused, which no other cell writes in this half-step (its
            // writer would be the absent cell x - c_K) - and the inlet, rest and freestream rules
            // replace the value afterwards
            static_assert(PAT == PAT_AA_ODD, "the AA odd half-step");
            uint32_t src = 0;
            const int kind = classify<K, GEN, REG, FX>(a, c, src);
            const st* p = fi + pop_index(c.own, kind == SRC_INLET || kind == SRC_REST ? K : dopp(rule_dir<K>(kind)));
            if (kind == SRC_REG) {
                if constexpr (REG) p = (const st*)(ra.base(fi, dopp(K), c.z, dcz(K)) + ra.v[dcx(K) + 1][dcy(K) + 1]);
                else p = fi + pop_index(src, dopp(K));
            }
            if constexpr (GEN && dcx(K) < 0)
                if (kind == SRC_OWN) p = ocopy + (K / 3) * BS2;
            raw[K] = SP::ld_raw(p);
            inlet_links |= (kind == SRC_INLET ? 1u : 0u) << K;
            rest_links |= (kind == SRC_REST ? 1u : 0u) << K;
            if constexpr (FX) tfs_links |= (kind == SRC_TFS ? 1u : 0u) << K;
            val = T(0);   // set below
        }
        f[K] = val;
    });
    if constexpr (!(REG && !GEN)) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr T w = wgt<T>(K);
            T val = SP::from_raw(raw[K], w);
            if constexpr (GEN) {
                if ((rest_links >> K) & 1u) val = w;
                if constexpr (dcx(K) > 0)
                    if ((inlet_links >> K) & 1u)
                        val = boundary_value<K, T>(SRC_INLET, a, c, u_in, a.step(), [&](auto) { return T(0); });
                if constexpr (FX && (dcy(K) != 0 || dcz(K) != 0))
                    if ((tfs_links >> K) & 1u) val = tfs_value<K, T>(a, val, u_in);
            }
            f[K] = val;
        });
    }
    if constexpr (PAT == PAT_AB && GEN && BFL) {
        if ((c.flags & BF_SOLID) && solid_links)
            bfl_links<SP>(a, c, f, solid_links, reg_links, a.fpart != nullptr, F0, F1, F2);
    }

    T rho_o, ux_o, uy_o, uz_o;
    if (GEN && solid_own) {
        // reference solid cell: full-way reflection of the gathered populations (kernel_cumulant.jl:405-417)
        T g[27];
#pragma unroll
        for (int k = 0; k < 27; ++k) g[k] = f[26 - k];
#pragma unroll
        for (int k = 0; k < 27; ++k) f[k] = g[k];
        rho_o = T(1); ux_o = uy_o = uz_o = T(0);
    } else {
        CellRates<T> q;
        if constexpr (WALE) {
            const T nu_eddy = wale_of<T>(a, c);
            cell_rates<T>(nu_eddy, T(dm->tau), T(dm->amr_scale), T(a.cp.nu_sgs_bg), a.cp.adaptive_omega4,
                          T(a.cp.lambda), T(a.cp.omega_4), q.omega1, q.omega4_diag);
        } else if constexpr (sizeof(T) == 8) {
            q.omega1 = dm->omega1_d; q.omega4_diag = dm->omega4d_d;
        } else {
            q.omega1 = dm->omega1; q.omega4_diag = dm->omega4d;
        }
        q.forced = dm->forced != 0;
        q.Fx = T(dm->F[0]); q.Fy = T(dm->F[1]); q.Fz = T(dm->F[2]);
        if constexpr (SPONGE) {
            q.sponge = (c.flags & BF_SPONGE) ? T(a.sponge[(size_t)a.sslot[b] * BS3 + (c.own - b * BS3)]) : T(0);
            q.sponge_u = T(u_in);
            q.sponge_blend = a.sponge_blend;
        }
        collide_cell<T, false, SPONGE>(f, q, a.cp, rho_o, ux_o, uy_o, uz_o);
    }
    if (a.vel_out) {
        T* vo = (T*)a.vel_out;
        vo[c.own] = ux_o; vo[n + c.own] = uy_o; vo[2 * (size_t)n + c.own] = uz_o;
    }
    if (a.rho_out) ((T*)a.rho_out)[c.own] = rho_o;

    const bool want_force = a.fpart != nullptr;
    // (with a q-map the links' momentum exchange was taken at the gather)
    const bool link_force = GEN && !BFL && want_force && (c.flags & BF_SOLID) && !solid_own;
    const bool outlet_cell = GEN && PAT == PAT_AA_EVEN && (c.flags & BF_EDGE) && !c.per0 && c.gx == c.ext0 - 1;
    // rounding of the stored post-collision populations: population j of this cell takes the random
    // bits of (cell, j, step) whichever slot it goes to, so every pattern stores the same values
    const bool dith = SP::dithered && a.cp.dither;
    const uint32_t hc = SP::dithered ? round_cell(round_key(a.step()), c.own - dm->cell0) : 0u;
    auto rb = [&](int j) { return round_bits(hc, j); };
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        constexpr int J = dopp(K);   // the source of direction J is x + c_K, where f*_K goes
        constexpr T wK = wgt<T>(K);
        if constexpr (REG && PAT == PAT_AB) {
            SP::sto_r((st*)(ra.base(fo, K, c.z, 0) + ra.v[1][1]), f[K], wK, rb(K), dith);
        } else if constexpr (REG && PAT == PAT_AA_EVEN) {
            SP::sto_r((st*)(ra.base(fo, J, c.z, 0) + ra.v[1][1]), f[K], wK, rb(K), dith);
            if constexpr (GEN && dcx(K) < 0) {
                if (outlet_cell)
                    SP::sto_r((st*)a.obuf + ((size_t)a.oslot[b] * 9 + K / 3) * BS2 + c.ly * BS + c.z, f[K], wK, rb(K), dith);
            }
        } else if constexpr (REG && !GEN) {
            SP::sto_r((st*)(ra.base(fo, K, c.z, -dcz(K)) + ra.v[1 - dcx(K)][1 - dcy(K)]), f[K], wK, rb(K), dith);
        } else if constexpr (REG) {
            uint32_t dst = 0;
            const int kind = classify<J, GEN, REG, FX>(a, c, dst);
            if (kind == SRC_REG) {
                SP::sto_r((st*)(ra.base(fo, K, c.z, -dcz(K)) + ra.v[1 - dcx(K)][1 - dcy(K)]), f[K], wK, rb(K), dith);
            } else if (kind != SRC_INLET) {
                const T v = boundary_value<J, T>(kind, a, c, u_in, a.step() + 1,
                                                 [&](auto jc) { return f[decltype(jc)::value]; });
                SP::sto_r(fo + pop_index(c.own, J), v, wgt<T>(J), rb(rule_dir<J>(kind)), dith);
            }
        } else if constexpr (PAT == PAT_AB) {
            SP::sto_r(fo + pop_index(c.own, K), f[K], wK, rb(K), dith);
        } else if constexpr (PAT == PAT_AA_EVEN) {
            SP::sto_r(fo + pop_index(c.own, J), f[K], wK, rb(K), dith);
            if constexpr (GEN && dcx(K) < 0) {
                if (outlet_cell)
                    SP::sto_r((st*)a.obuf + ((size_t)a.oslot[b] * 9 + K / 3) * BS2 + c.ly * BS + c.z, f[K], wK, rb(K), dith);
            }
        } else {
            uint32_t dst = 0;
            const int kind = classify<J, GEN, false, FX>(a, c, dst);
            if (kind == SRC_REG) {
                SP::sto_r(fo + pop_index(dst, K), f[K], wK, rb(K), dith);
            } else if (kind != SRC_INLET) {   // inlet links are evaluated by the even step itself
                const T v = boundary_value<J, T>(kind, a, c, u_in, a.step() + 1,
                                                 [&](auto jc) { return f[decltype(jc)::value]; });
                SP::sto_r(fo + pop_index(c.own, J), v, wgt<T>(J), rb(rule_dir<J>(kind)), dith);
            }
        }
        if constexpr (GEN) {
            if (link_force) {
                uint32_t dst = 0;
                const int kind = classify<J, GEN, REG, FX>(a, c, dst);
                double m = 0.0;
                if (kind == SRC_SOLID) {
                    m = 2.0 * ((double)SP::rt_r(f[K], wK, rb(K), dith) - (double)wK);
                } else if (PAT == PAT_AB && a.cp.bb_mode == 0 && kind == SRC_REG && ((c.lmask >> J) & 1u)) {
                    m = ((double)SP::rt_r(f[K], wK, rb(K), dith) - (double)wK) +
                        ((double)own_prev<SP, PAT, K>(a, c) - (double)wK);
                }
                F0 += m * dcx(K); F1 += m * dcy(K); F2 += m * dcz(K);
            }
        }
    });
}

// SEL: which block list a launch covers: blocks without a rule or boundary blocks, each also with lexicographic
// neighbours (regular), on a kernel of its own register budget.
enum : int { SEL_INTERIOR = 1, SEL_BOUNDARY = 2, SEL_REGULAR = 3, SEL_BOUNDARY_REGULAR = 4 };

#ifndef OAL_STEP_WAVES
#define OAL_STEP_WAVES 3
#endif
// register budget of the one-plane kernels: 3 waves per SIMD, 2 for the forms that do not fit 168 VGPRs
// without spilling (FP64 arithmetic, the AA pattern's two-sided slots, WALE's velocity gather), 1 for the
// FP64 AA forms
template <class SP, int PAT, bool WALE>
constexpr int step_waves() {
    return sizeof(typename SP::T) == 8 && PAT != PAT_AB ? 1 : sizeof(typename SP::T) == 8 || PAT != PAT_AB || WALE ? 2 : OAL_STEP_WAVES;
}

template <class SP, int PAT, bool WALE, int SEL, bool BFL = false, bool SPONGE = false, bool FX = true>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(step_waves<SP, PAT, WALE>()))) k_step(const StepArgs a) {
    const uint32_t litem = xcd_item(blockIdx.x, gridDim.x);
    const uint32_t lb = litem / PLANES;
    const uint32_t b = (uint32_t)a.blist[lb];
    const uint32_t item = b * PLANES + litem % PLANES;
    CellCtx c;
    c.b = b;
    c.z = (int)(item % PLANES);
    c.lx = threadIdx.x & (BS - 1);
    c.ly = threadIdx.x >> 4;
    c.flags = a.bflags[b];
    const DevDomain* dm = a.doms + a.bdom[b];
    c.ext0 = dm->ext[0]; c.ext1 = dm->ext[1]; c.ext2 = dm->ext[2];
    c.per0 = dm->per[0]; c.per1 = dm->per[1]; c.per2 = dm->per[2];
    c.zwall = dm->zwall; c.ymin_wall = dm->ymin_wall;
    c.gx = a.borg[3 * b] + c.lx;
    c.gy = a.borg[3 * b + 1] + c.ly;
    c.gz = a.borg[3 * b + 2] + c.z;
    c.own = b * BS3 + (uint32_t)c.z * BS2 + (uint32_t)c.ly * BS + (uint32_t)c.lx;
    double F0 = 0.0, F1 = 0.0, F2 = 0.0;
    c.lmask = 0;
    if constexpr (SEL == SEL_REGULAR) {
        step_cell<SP, PAT, WALE, false, true>(a, c, dm, true, false, F0, F1, F2);
    } else if constexpr (SEL == SEL_INTERIOR) {
        step_cell<SP, PAT, WALE, false>(a, c, dm, true, false, F0, F1, F2);
    } else {
        const bool inside = !(c.flags & BF_PARTIAL) || (c.gx < c.ext0 && c.gy < c.ext1 && c.gz < c.ext2);
        if (c.flags & BF_SOLID) c.lmask = a.lmask[(size_t)a.lslot[b] * BS3 + (c.own - b * BS3)];
        const bool solid_own = (c.lmask >> 27) & 1u;
        const bool active = inside && !(solid_own && a.cp.bb_mode == 1);
        if constexpr (SEL == SEL_BOUNDARY_REGULAR)
            step_cell<SP, PAT, WALE, true, true, BFL, SPONGE, FX>(a, c, dm, active, solid_own, F0, F1, F2);
        else
            step_cell<SP, PAT, WALE, true, false, BFL, SPONGE, FX>(a, c, dm, active, solid_own, F0, F1, F2);
    }
    if (a.fpart) wg_sum3(F0 * dm->force_scale, F1 * dm->force_scale, F2 * dm->force_scale, a.fpart, item);
}

// the boundary lists on the one-plane kernel
template <class SP, int PAT, bool WALE>
static void launch_boundary(const StepArgs& a, hipStream_t bs) {
    StepArgs r = a;
    const bool bfl = PAT == PAT_AB && a.qmap != nullptr;
    if constexpr (sizeof(typename SP::T) == 4 || PAT == PAT_AB) {   // blocks without a rule that the one-launch kernels
        if (a.n_interior) {                                         // do not span
            r.blist = a.blist_interior;
            hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_INTERIOR>), dim3(a.n_interior * PLANES), dim3(WG), 0, bs, r);
        }
    }
    if (a.n_boundary_regular) {
        r.blist = a.blist_boundary_regular;
        const dim3 g(a.n_boundary_regular * PLANES);
        if constexpr (PAT == PAT_AB) {
            if (bfl && a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, true>), g, dim3(WG), 0, bs, r);
            else if (bfl) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, true, false, false>), g, dim3(WG), 0, bs, r);
            else if (a.sponge && a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, false, true>), g, dim3(WG), 0, bs, r);
            else if (a.sponge) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, false, true, false>), g, dim3(WG), 0, bs, r);
            else if (a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR>), g, dim3(WG), 0, bs, r);
            else hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, false, false, false>), g, dim3(WG), 0, bs, r);
        } else {
            if (a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR>), g, dim3(WG), 0, bs, r);
            else hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY_REGULAR, false, false, false>), g, dim3(WG), 0, bs, r);
        }
    }
    if (a.n_boundary) {
        r.blist = a.blist_boundary;
        const dim3 g(a.n_boundary * PLANES);
        if constexpr (PAT == PAT_AB) {
            if (bfl && a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, true>), g, dim3(WG), 0, bs, r);
            else if (bfl) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, true, false, false>), g, dim3(WG), 0, bs, r);
            else if (a.sponge && a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, false, true>), g, dim3(WG), 0, bs, r);
            else if (a.sponge) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, false, true, false>), g, dim3(WG), 0, bs, r);
            else if (a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY>), g, dim3(WG), 0, bs, r);
            else hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, false, false, false>), g, dim3(WG), 0, bs, r);
        } else {
            if (a.face_x) hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY>), g, dim3(WG), 0, bs, r);
            else hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_BOUNDARY, false, false, false>), g, dim3(WG), 0, bs, r);
        }
    }
}

// One step of a level: launches over disjoint block lists.
//   FP32 arithmetic: the two-cells-per-lane kernel for every block but a few kinds, those on the one-plane
//     interior and boundary kernels; on small levels in the AB pattern the one-cell-per-lane kernel in its place.
//   FP64, AB pattern: likewise the one-cell-per-lane kernel.
//   FP64, AA pattern: regular, other interior, regular boundary and boundary blocks, each on a kernel
//     compiled for its own register budget.
// The boundary launches go to `side` (when given) so that they overlap the bulk launch; the
// caller joins the two streams.
template <class SP, int PAT, bool WALE>
static hipError_t launch_pat(const StepArgs& a, hipStream_t stream, hipStream_t side, hipEvent_t bulk0, hipEvent_t bulk1) {
    hipStream_t bs = side ? side : stream;
    launch_boundary<SP, PAT, WALE>(a, bs);
    constexpr bool two = sizeof(typename SP::T) == 4;
    if (bulk0) {
        const hipError_t e = hipEventRecord(bulk0, stream);
        if (e != hipSuccess) return e;
    }
    if constexpr (two) {
        if constexpr (PAT != PAT_AB) {
            // (the even half-step stays in the block's own slots: its records serve both forms)
            launch_two(SP::code, WALE, PAT == PAT_AA_EVEN ? TWO_AA_EVEN : TWO_AA_ODD, a.two,
                       a.n_two + (PAT == PAT_AA_EVEN ? a.n_two_wide : 0), stream, a);
            if (PAT == PAT_AA_ODD) launch_two(SP::code, WALE, TWO_AA_ODD_WIDE, a.two + a.n_two, a.n_two_wide, stream, a);
        } else if (a.qmap) {   // interpolated bounce-back: its form of the kernel where there are solid links
            launch_two(SP::code, WALE, TWO_BFL, a.two_links, a.n_two_links, stream, a);
            launch_two(SP::code, WALE, TWO_PLAIN, a.two_free, a.n_two_free, stream, a);
            launch_two(SP::code, WALE, TWO_WIDE, a.two_free + a.n_two_free, a.n_two_wide_free, stream, a);
        } else {
            if (a.n_two <= (WALE ? ONE_BLOCKS / 2 : ONE_BLOCKS)) launch_one(SP::code, WALE, false, a.two, a.n_two, stream, a);
            else launch_two(SP::code, WALE, TWO_PLAIN, a.two, a.n_two, stream, a);
            launch_two(SP::code, WALE, TWO_WIDE, a.two + a.n_two, a.n_two_wide, stream, a);
            launch_two(SP::code, WALE, TWO_SPONGE, a.two_sponge, a.n_two_sponge, stream, a);
        }
    } else if constexpr (PAT == PAT_AB) {   // (with interpolated bounce-back the boundary lists hold the links)
        const TwoRec* rec = a.qmap ? a.two_free : a.two;
        const uint32_t n = a.qmap ? a.n_two_free : a.n_two;
        launch_one(SP::code, WALE, false, rec, n, stream, a);
        launch_one(SP::code, WALE, true, rec + n, a.qmap ? a.n_two_wide_free : a.n_two_wide, stream, a);
    } else {
        StepArgs r = a;
        if (a.n_regular) {
            r.blist = a.blist_regular;
            hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_REGULAR>), dim3(a.n_regular * PLANES), dim3(WG), 0, stream, r);
        }
        if (a.n_interior) {
            r.blist = a.blist_interior;
            hipLaunchKernelGGL((k_step<SP, PAT, WALE, SEL_INTERIOR>), dim3(a.n_interior * PLANES), dim3(WG), 0, stream, r);
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !bulk1) return e;
    return hipEventRecord(bulk1, stream);
}

template <class SP>
static hipError_t launch_sp(int stream_mode, bool wale, const StepArgs& a, hipStream_t s, hipStream_t side, hipEvent_t e0,
                            hipEvent_t e1) {
    if (stream_mode == 0)
        return wale ? launch_pat<SP, PAT_AB, true>(a, s, side, e0, e1) : launch_pat<SP, PAT_AB, false>(a, s, side, e0, e1);
    if (a.parity == 0)
        return wale ? launch_pat<SP, PAT_AA_EVEN, true>(a, s, side, e0, e1)
                    : launch_pat<SP, PAT_AA_EVEN, false>(a, s, side, e0, e1);
    return wale ? launch_pat<SP, PAT_AA_ODD, true>(a, s, side, e0, e1) : launch_pat<SP, PAT_AA_ODD, false>(a, s, side, e0, e1);
}

}  // namespace oal
