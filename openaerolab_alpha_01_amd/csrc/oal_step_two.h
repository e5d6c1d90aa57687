// The step kernel of the FP32-arithmetic forms in the AB pattern, two cells per lane; a
// translation unit per storage form (oal_two_<storage>.hip).
//
// One workgroup of 128 lanes steps one 16 x 16 plane of a block; a lane steps the cells (2j, 2j + 1) of
// a row, A and B below, and every population moves as one word holding both (8 bytes in FP32, 4 bytes in
// the 16-bit forms), aligned.  One launch covers the stepped blocks of every kind: neighbour blocks come
// from the level's table (domain interiors, periodic wraps, octree levels alike), and the domain faces,
// the cells beyond the extent and the solid links are told apart by uniform branches on the block's
// flags.
//
// Gather (pull), first pass: the word of direction k is the aligned pair of the source row
// (y - cy, z - cz).  For cx = 0 that is the pair of sources itself.  For cx = +1 the sources are
// (2j - 1, 2j): B's is the lower cell of the lane's own word, A's the upper cell of the left lane's (DPP
// row_shr:1); the lane at j = 0 takes it from the x-neighbour block (one cell).  cx = -1 mirrors this.
// The end lanes' cells share nine registers: j = 0 needs the directions with cx = +1 only, j = 7 those
// with cx = -1.  On a y or z face the rule replaces the source of both cells by the same population of
// the cell itself (kernel_cumulant.jl:233-345 in the order of classify), read from the own row.
// Second pass, in waves that hold such a cell: solid links (the own population opp k) and the outlet
// (the own population k) replace one cell of a pair; the inlet equilibrium replaces A's value at x = 0
// after decoding.
//
// Bound and shape.  The plane's 27 words are all in flight together and nothing is kept for a next plane,
// so a lane needs 97 to 126 registers and four waves share a SIMD; their loads overlap other waves'
// collisions.  That needs the rare limiter out of the registers (collide_cell's LDS form): with it inline
// the kernel takes 168 and spills.  Bound: HBM in FP32, VALU issue in the 16-bit forms.  Measured against
// walking four planes of a block per workgroup with the next plane's words in flight (two waves per SIMD,
// a launch per kind of block, the default shape before): 256^3 sphere box FP32 667 -> 644 us per step, FP16
// 467 -> 453 us; WALE 192 x 160 x 160 FP32 295 -> 243 us, WALE 200 x 120 x 104 FP16 200 -> 114 us; WALE
// 100 x 60 x 44 75 -> 26 us (that shape left 48 workgroups per launch); 12 ragged boxes with solids and
// sponges FP16 813 -> 542 us.  Blocks run fastest: x-neighbour blocks share the lines of the row ends.
#pragma once

#include "oal_step.h"

namespace oal {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int TWG = 128;   // lanes of a workgroup: 8 pairs x 16 rows

// a pair of cells in storage form
template <class SP>
struct Two {   // 16-bit forms: A in the low half
    using word = uint32_t;
    static constexpr uint32_t es = 2;
    __device__ static __forceinline__ word ld2(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0);
    }
    __device__ static __forceinline__ uint32_t ld1(__amdgpu_buffer_rsrc_t r, uint32_t v) {
        return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)v, 0, 0);
    }
    template <int AUX>
    __device__ static __forceinline__ void st2(word w, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b32(w, r, (int)v, (int)s, AUX);
    }
    template <int AUX>
    __device__ static __forceinline__ void st1(uint32_t c, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)c, r, (int)v, (int)s, AUX);
    }
    __device__ static __forceinline__ uint32_t a(word w) { return w & 0xffffu; }
    __device__ static __forceinline__ uint32_t b(word w) { return w >> 16; }
    __device__ static __forceinline__ word set_a(word w, uint32_t c) { return (w & 0xffff0000u) | c; }
    __device__ static __forceinline__ word set_b(word w, uint32_t c) { return (w & 0xffffu) | (c << 16); }
    // (left lane's B, own A); end: the x-neighbour block's cell of the lane at j = 0
    __device__ static __forceinline__ word from_left(word w, bool first, uint32_t end) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x111, 0xf, 0xf, false);
        return __builtin_amdgcn_alignbyte(w, first ? end << 16 : l, 2);
    }
    // (own B, right lane's A)
    __device__ static __forceinline__ word from_right(word w, bool last, uint32_t end) {
        const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x101, 0xf, 0xf, false);
        return __builtin_amdgcn_alignbyte(last ? end : r, w, 2);
    }
    __device__ static __forceinline__ float dec_a(word w, float wk) { return SP::dec_lo(w, wk); }
    __device__ static __forceinline__ float dec_b(word w, float wk) { return SP::dec_hi(w, wk); }
};
template <>
struct Two<StF32> {
    using word = u32x2;
    static constexpr uint32_t es = 4;
    __device__ static __forceinline__ word ld2(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        return __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0);
    }
    __device__ static __forceinline__ uint32_t ld1(__amdgpu_buffer_rsrc_t r, uint32_t v) {
        return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, 0, 0);
    }
    template <int AUX>
    __device__ static __forceinline__ void st2(word w, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b64(w, r, (int)v, (int)s, AUX);
    }
    template <int AUX>
    __device__ static __forceinline__ void st1(uint32_t c, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b32(c, r, (int)v, (int)s, AUX);
    }
    __device__ static __forceinline__ uint32_t a(word w) { return w.x; }
    __device__ static __forceinline__ uint32_t b(word w) { return w.y; }
    __device__ static __forceinline__ word set_a(word w, uint32_t c) { w.x = c; return w; }
    __device__ static __forceinline__ word set_b(word w, uint32_t c) { w.y = c; return w; }
    __device__ static __forceinline__ word from_left(word w, bool first, uint32_t end) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w.y, 0x111, 0xf, 0xf, false);
        return word{first ? end : l, w.x};
    }
    __device__ static __forceinline__ word from_right(word w, bool last, uint32_t end) {
        const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w.x, 0x101, 0xf, 0xf, false);
        return word{w.y, last ? end : r};
    }
    __device__ static __forceinline__ float dec_a(word w, float) { return __uint_as_float(w.x); }
    __device__ static __forceinline__ float dec_b(word w, float) { return __uint_as_float(w.y); }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_at(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc((char*)p, (short)0, (int)0xffffffff, 0x00020000);
}

// the rules of a lane's row (both cells share y and z) and of its cells
struct TwoFaces {
    bool yl, yh;            // per lane: the row lies on the y-min / y-max face
    bool zl, zh;            // uniform: the plane lies on the z-min / z-max face
    bool zwall, ymin_wall;  // no-slip variants of the z faces and of the y-min face
};
// is the source of direction K beyond a y or z face, and which own population does the rule take
// (precedence: no-slip z wall, no-slip y-min wall, y mirror, z mirror)?
template <int K>
__device__ __forceinline__ bool two_row_rule(const TwoFaces& fc, int& j) {
    constexpr int cy = dcy(K), cz = dcz(K);
    const bool zf = (cz > 0 && fc.zl) || (cz < 0 && fc.zh);
    const bool yf = (cy > 0 && fc.yl) || (cy < 0 && fc.yh);
    j = (fc.zwall && zf) ? dopp(K) : (fc.ymin_wall && cy > 0 && fc.yl) ? dopp(K) : yf ? dmir_y(K) : dmir_z(K);
    return zf || yf;
}

// sum of 3 doubles over the workgroup's two waves into part[item * 4 + 0..2]
__device__ __forceinline__ void two_sum3(double v0, double v1, double v2, double* part, uint32_t item) {
    __shared__ double red[3];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v0 += __shfl_xor(v0, off, 64);
        v1 += __shfl_xor(v1, off, 64);
        v2 += __shfl_xor(v2, off, 64);
    }
    if (threadIdx.x == 64) { red[0] = v0; red[1] = v1; red[2] = v2; }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[(size_t)item * 4 + 0] = v0 + red[0];
        part[(size_t)item * 4 + 1] = v1 + red[1];
        part[(size_t)item * 4 + 2] = v2 + red[2];
    }
}

#ifndef OAL_TWO_STORE_AUX
#define OAL_TWO_STORE_AUX 2   // the non-temporal hint
#endif

template <class SP, bool UNIT, bool WALE, int EXTRA>
__global__ void __launch_bounds__(TWG) __attribute__((amdgpu_waves_per_eu(4)))
k_step_two(const StepArgs a) {
    using W = Two<SP>;
    using word = typename W::word;
    constexpr uint32_t es = W::es;
    constexpr uint32_t slot = BS3 * es;          // bytes of one direction of a block
    constexpr uint32_t blk = 27u * slot;
    const uint32_t litem = xcd_item(blockIdx.x, gridDim.x);
    const uint32_t nblk = gridDim.x / PLANES;
    const uint32_t zi = litem / nblk;
    const uint32_t b = (uint32_t)a.blist[litem - zi * nblk];
    const int z = (int)zi;
    const uint32_t flags = a.bflags[b];
    const DevDomain* dm = a.doms + a.bdom[b];
    const int ox = a.borg[3 * b], oy = a.borg[3 * b + 1], gz = a.borg[3 * b + 2] + z;
    if (gz >= dm->ext[2]) return;                // a plane beyond the extent
    const int jx = (int)(threadIdx.x & 7u), ly = (int)(threadIdx.x >> 3);
    const int32_t* nt = a.nbr_bm + (size_t)b * 32;
    const uint32_t nb0 = (uint32_t)nt[27];       // lowest block index among the neighbours and the block
    // byte offset of a neighbour block (an absent one, never a source: the block itself)
    auto boff = [&](int dx, int dy, int dz) -> uint32_t {
        const int32_t n = nt[(dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)];
        return ((n < 0 ? b : (uint32_t)n) - nb0) * blk;
    };
    const __amdgpu_buffer_rsrc_t fin = buf_at((const char*)a.fin + (size_t)nb0 * blk);
    const uint32_t row = (uint32_t)ly * (BS * es) + (uint32_t)jx * (2 * es);
    const uint32_t zown = (uint32_t)z * (BS2 * es);
    const uint32_t own0 = (b - nb0) * blk;       // uniform
    const bool first = jx == 0, last = jx == 7;

    const bool edge = (flags & BF_EDGE) != 0;
    TwoFaces fc{};
    bool xl = false, xha = false, xhb = false, lva = true, lvb = true;
    if (edge) {
        const int gy = oy + ly, ga = ox + 2 * jx;
        fc.yl = !dm->per[1] && gy == 0;
        fc.yh = !dm->per[1] && gy == dm->ext[1] - 1;
        fc.zl = !dm->per[2] && gz == 0;
        fc.zh = !dm->per[2] && gz == dm->ext[2] - 1;
        fc.zwall = dm->zwall != 0;
        fc.ymin_wall = dm->ymin_wall == 1;
        xl = !dm->per[0] && ga == 0;
        xha = !dm->per[0] && ga == dm->ext[0] - 1;
        xhb = !dm->per[0] && ga + 1 == dm->ext[0] - 1;
        lva = gy < dm->ext[1] && ga < dm->ext[0];
        lvb = gy < dm->ext[1] && ga + 1 < dm->ext[0];
    }
    // solid links of the two cells (bit k: the source of direction k is solid; bit 27: the cell is)
    uint32_t lma = 0, lmb = 0;
    if (flags & BF_SOLID) {
        const u32x2 m = *(const u32x2*)(a.lmask + (size_t)a.lslot[b] * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + 2u * (uint32_t)jx);
        lma = m.x;
        lmb = m.y;
        lva = lva && !((lma >> 27) & 1u);
        lvb = lvb && !((lmb >> 27) & 1u);
    }

    // WALE: the previous step's velocity of the pair and of its neighbour pairs, requested first
    u32x2 vo[3], vyp[3], vym[3], vzp[3], vzm[3];
    uint32_t vend[3];
    bool no_end = false;                         // no x-neighbour block behind the row's end
    if constexpr (WALE) {
        const __amdgpu_buffer_rsrc_t vr = buf_at(a.vel_in);
        const uint32_t comp = a.ncell * 4u;
        auto cell0 = [&](int32_t n) { return (uint32_t)n * (BS3 * 4u); };
        const uint32_t loc = (uint32_t)(ly * BS + 2 * jx) * 4u, zc = (uint32_t)z * (BS2 * 4u);
        const uint32_t own = cell0((int32_t)b) + zc + loc;
        const int32_t nyp = nt[13 + 3], nym = nt[13 - 3], nzp = nt[13 + 9], nzm = nt[13 - 9];
        const bool cp = ly == BS - 1, cm = ly == 0;
        uint32_t oyp = cp ? (nyp < 0 ? own : cell0(nyp) + zc + loc - (BS - 1) * BS * 4u) : own + BS * 4u;
        uint32_t oym = cm ? (nym < 0 ? own : cell0(nym) + zc + loc + (BS - 1) * BS * 4u) : own - BS * 4u;
        uint32_t ozp = z == BS - 1 ? (nzp < 0 ? own : cell0(nzp) + loc) : own + BS2 * 4u;
        uint32_t ozm = z == 0 ? (nzm < 0 ? own : cell0(nzm) + (BS - 1) * BS2 * 4u + loc) : own - BS2 * 4u;
        if (edge) {
            oyp = fc.yh ? own : oyp;
            oym = fc.yl ? own : oym;
            ozp = fc.zh ? own : ozp;
            ozm = fc.zl ? own : ozm;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int so = (int)(q * comp);
            vo[q] = __builtin_amdgcn_raw_buffer_load_b64(vr, (int)own, so, 0);
            vyp[q] = __builtin_amdgcn_raw_buffer_load_b64(vr, (int)oyp, so, 0);
            vym[q] = __builtin_amdgcn_raw_buffer_load_b64(vr, (int)oym, so, 0);
            vzp[q] = __builtin_amdgcn_raw_buffer_load_b64(vr, (int)ozp, so, 0);
            vzm[q] = __builtin_amdgcn_raw_buffer_load_b64(vr, (int)ozm, so, 0);
            vend[q] = 0;
        }
        if (first || last) {
            const int32_t nx = first ? nt[12] : nt[14];
            no_end = nx < 0;
            // (-x block's cell 15 of the row, +x block's cell 0)
            const uint32_t oe = no_end ? own : cell0(nx) + zc + (uint32_t)(ly * BS + (first ? BS - 1 : 0)) * 4u;
#pragma unroll
            for (int q = 0; q < 3; ++q) vend[q] = __builtin_amdgcn_raw_buffer_load_b32(vr, (int)oe, (int)(q * comp), 0);
        }
    }
    float spa = 0.0f, spb = 0.0f;
    if constexpr (EXTRA == TWO_SPONGE) {
        if (flags & BF_SPONGE) {
            const float* sp = a.sponge + (size_t)a.sslot[b] * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + 2u * (uint32_t)jx;
            spa = sp[0];
            spb = sp[1];
        }
    }

    // first pass: per-lane offsets of the source rows by (cy, cz); the plane's uniform part apart
    uint32_t v[3][3], ve[3][3], zs[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int sz = z - (k - 1);
        const int dz = sz < 0 ? -1 : (sz >= BS ? 1 : 0);
        zs[k] = (uint32_t)(sz & (BS - 1)) * (BS2 * es);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int cy = i - 1;
            const uint32_t r = (uint32_t)((ly - cy) & (BS - 1)) * (BS * es);
            const uint32_t c0 = boff(0, 0, dz), m0 = boff(-1, 0, dz), p0 = boff(1, 0, dz);
            uint32_t c = c0, m = m0, p = p0;
            if (cy != 0) {
                const bool cross = cy > 0 ? ly == 0 : ly == BS - 1;
                const uint32_t c1 = boff(0, -cy, dz), m1 = boff(-1, -cy, dz), p1 = boff(1, -cy, dz);
                c = cross ? c1 : c0;
                m = cross ? m1 : m0;
                p = cross ? p1 : p0;
            }
            v[k][i] = c + r + (uint32_t)jx * (2 * es);
            // row ends: direction (+1, cy, cz) from the -x block's cell 15 at j = 0, (-1, cy, cz) from the
            // +x block's cell 0 at j = 7 (slots 2 apart)
            ve[k][i] = (first ? m + (BS - 1) * es + 2 * slot : p) + r;
        }
    }
    word s[27];
    uint32_t e9[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) e9[q] = 0;
    if (edge) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            uint32_t o = v[cz + 1][cy + 1] + (uint32_t)K * slot + zs[cz + 1];
            if constexpr (cy != 0 || cz != 0) {
                int j;
                const bool face = two_row_rule<K>(fc, j);
                o = face ? own0 + row + (uint32_t)j * slot + zown : o;
            }
            s[K] = W::ld2(fin, o, 0);
        });
    } else {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            s[K] = W::ld2(fin, v[cz + 1][cy + 1], (uint32_t)K * slot + zs[cz + 1]);
        });
    }
    if (first || last) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            if constexpr (dcx(K) < 0) e9[K / 3] = W::ld1(fin, ve[cz + 1][cy + 1] + (uint32_t)K * slot + zs[cz + 1]);
        });
    }

    // WALE: the eddy viscosity of both cells, while the populations are in flight
    CellRates<float> qa;
    qa.forced = dm->forced != 0;
    qa.Fx = dm->F[0]; qa.Fy = dm->F[1]; qa.Fz = dm->F[2];
    qa.omega1 = dm->omega1;
    qa.omega4_diag = dm->omega4d;
    if constexpr (EXTRA == TWO_SPONGE) {
        qa.sponge_u = dm->u_in;
        qa.sponge_blend = a.sponge_blend;
    }
    float om1b = qa.omega1, om4b = qa.omega4_diag;
    const uint32_t cell0 = dm->cell0;
    const float u_in = dm->u_in, force_scale = dm->force_scale;
    if constexpr (WALE) {
        const float tau = dm->tau, amr = dm->amr_scale;
        auto f32 = [](uint32_t u) { return __uint_as_float(u); };
        float ga[3][3], gb[3][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const float A = f32(vo[q].x), B = f32(vo[q].y);
            const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vo[q].y, 0x111, 0xf, 0xf, false);
            const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vo[q].x, 0x101, 0xf, 0xf, false);
            float axm = first ? f32(vend[q]) : f32(l), bxp = last ? f32(vend[q]) : f32(r);
            float axp = B, bxm = A;
            float ayp = f32(vyp[q].x), aym = f32(vym[q].x), azp = f32(vzp[q].x), azm = f32(vzm[q].x);
            float byp = f32(vyp[q].y), bym = f32(vym[q].y), bzp = f32(vzp[q].y), bzm = f32(vzm[q].y);
            // across a face, beside an absent block or a solid cell: the cell itself
            axm = (xl || (first && no_end)) ? A : axm;
            axp = xha ? A : axp;
            bxp = (xhb || (last && no_end)) ? B : bxp;
            if (flags & BF_SOLID) {
                axp = (lma >> 12) & 1u ? A : axp; axm = (lma >> 14) & 1u ? A : axm;
                ayp = (lma >> 10) & 1u ? A : ayp; aym = (lma >> 16) & 1u ? A : aym;
                azp = (lma >> 4) & 1u ? A : azp;  azm = (lma >> 22) & 1u ? A : azm;
                bxp = (lmb >> 12) & 1u ? B : bxp; bxm = (lmb >> 14) & 1u ? B : bxm;
                byp = (lmb >> 10) & 1u ? B : byp; bym = (lmb >> 16) & 1u ? B : bym;
                bzp = (lmb >> 4) & 1u ? B : bzp;  bzm = (lmb >> 22) & 1u ? B : bzm;
            }
            ga[q][0] = 0.5f * (axp - axm); ga[q][1] = 0.5f * (ayp - aym); ga[q][2] = 0.5f * (azp - azm);
            gb[q][0] = 0.5f * (bxp - bxm); gb[q][1] = 0.5f * (byp - bym); gb[q][2] = 0.5f * (bzp - bzm);
        }
        const float na = wale_nu(ga[0][0], ga[0][1], ga[0][2], ga[1][0], ga[1][1], ga[1][2], ga[2][0], ga[2][1], ga[2][2], a.cp.c_wale);
        const float nb = wale_nu(gb[0][0], gb[0][1], gb[0][2], gb[1][0], gb[1][1], gb[1][2], gb[2][0], gb[2][1], gb[2][2], a.cp.c_wale);
        cell_rates<float>(na, tau, amr, a.cp.nu_sgs_bg, a.cp.adaptive_omega4, a.cp.lambda, a.cp.omega_4, qa.omega1, qa.omega4_diag);
        cell_rates<float>(nb, tau, amr, a.cp.nu_sgs_bg, a.cp.adaptive_omega4, a.cp.lambda, a.cp.omega_4, om1b, om4b);
    }

    // the sources of the pair
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        constexpr int cx = dcx(K), cy = dcy(K), cz = dcz(K);
        if constexpr (cx != 0) {
            word w;
            if constexpr (cx > 0) w = W::from_left(s[K], first, e9[K / 3]);
            else w = W::from_right(s[K], last, e9[K / 3]);
            if constexpr (cy != 0 || cz != 0) {
                int j;
                const bool face = two_row_rule<K>(fc, j);
                if constexpr (es == 4) { w.x = face ? s[K].x : w.x; w.y = face ? s[K].y : w.y; }
                else w = face ? s[K] : w;
            }
            s[K] = w;
        }
    });
    // second pass: solid links and the outlet, in waves that hold one
    const uint32_t links = lma | lmb;
    if (__builtin_amdgcn_ballot_w64((links & 0x7ffffffu) != 0 || xha || xhb) != 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            uint32_t ra[9], rb[9];
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if (K / 9 == c) {
                    const bool oa = dcx(K) < 0 && xha, ob = dcx(K) < 0 && xhb;
                    ra[K % 9] = 0;
                    rb[K % 9] = 0;
                    if (((lma >> K) & 1u) || oa) ra[K % 9] = W::ld1(fin, own0 + row + zown + (oa ? (uint32_t)K : (uint32_t)dopp(K)) * slot);
                    if (((lmb >> K) & 1u) || ob) rb[K % 9] = W::ld1(fin, own0 + row + es + zown + (ob ? (uint32_t)K : (uint32_t)dopp(K)) * slot);
                }
            });
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if (K / 9 == c) {
                    if (((lma >> K) & 1u) || (dcx(K) < 0 && xha)) s[K] = W::set_a(s[K], ra[K % 9]);
                    if (((lmb >> K) & 1u) || (dcx(K) < 0 && xhb)) s[K] = W::set_b(s[K], rb[K % 9]);
                }
            });
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // collide A, then B; each cell's result takes its half of the words
    const uint32_t ca = b * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + 2u * (uint32_t)jx;
    const bool dith = SP::dithered && a.cp.dither;
    const uint32_t key = SP::dithered ? round_key(a.step()) : 0u;
    double F0 = 0.0, F1 = 0.0, F2 = 0.0;
    const bool want_force = a.fpart != nullptr && (flags & BF_SOLID);
    float va[3], vb[3];
    CellCtx cc{};
    cc.b = b;
    cc.gy = oy + ly;
    cc.gz = gz;
    // populations of the pair's cell K / the interpolated wall's links of one cell
    auto bfl = [&](float (&f)[27], uint32_t cell, uint32_t lm, bool xh, bool in) {
        uint32_t beyond = 0;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            int j;
            const bool f0 = two_row_rule<K>(fc, j) || (dcx(K) > 0 && in) || (dcx(K) < 0 && xh);
            beyond |= (f0 ? 1u : 0u) << K;
        });
        cc.own = cell;
        bfl_links<SP>(a, cc, f, lm & 0x7ffffffu, ~(lm | beyond), a.fpart != nullptr, F0, F1, F2);
    };
    auto link_force = [&](auto half, uint32_t lm) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if ((lm >> dopp(K)) & 1u) {
                const float fs = decltype(half)::value ? W::dec_b(s[K], wgt<float>(K)) : W::dec_a(s[K], wgt<float>(K));
                const double m = 2.0 * ((double)fs - (double)wgt<float>(K));
                F0 += m * dcx(K); F1 += m * dcy(K); F2 += m * dcz(K);
            }
        });
    };
    float rho_o;
    float f[27];
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        f[K] = W::dec_a(s[K], wgt<float>(K));
    });
    if (xl) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (dcx(K) > 0)
                f[K] = boundary_value<K, float>(SRC_INLET, a, cc, u_in, a.step(), [&](auto) { return 0.0f; });
        });
    }
    if constexpr (EXTRA == TWO_BFL) {
        if (lva && (lma & 0x7ffffffu)) bfl(f, ca, lma, xha, xl);
    }
    if constexpr (EXTRA == TWO_SPONGE) qa.sponge = spa;
    collide_cell<float, UNIT, EXTRA == TWO_SPONGE, true>(f, qa, a.cp, rho_o, va[0], va[1], va[2]);
    {
        const uint32_t hc = SP::dithered ? round_cell(key, ca - cell0) : 0u;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (es == 4) s[K].x = __float_as_uint(f[K]);
        });
        if constexpr (es == 2) {
            if (dith) {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    s[K] = SP::template put<false>(s[K], f[K], wgt<float>(K), round_bits(hc, K), true);
                });
            } else {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    s[K] = SP::template put<false>(s[K], f[K], wgt<float>(K), 0u, false);
                });
            }
        }
    }
    if constexpr (EXTRA != TWO_BFL)
        if (want_force && lva) link_force(std::integral_constant<int, 0>{}, lma);
    __builtin_amdgcn_sched_barrier(0);
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        f[K] = W::dec_b(s[K], wgt<float>(K));
    });
    if constexpr (EXTRA == TWO_BFL) {
        if (lvb && (lmb & 0x7ffffffu)) bfl(f, ca + 1u, lmb, xhb, false);
    }
    CellRates<float> qb = qa;
    qb.omega1 = om1b;
    qb.omega4_diag = om4b;
    if constexpr (EXTRA == TWO_SPONGE) qb.sponge = spb;
    collide_cell<float, UNIT, EXTRA == TWO_SPONGE, true>(f, qb, a.cp, rho_o, vb[0], vb[1], vb[2]);
    {
        const uint32_t hc = SP::dithered ? round_cell(key, ca + 1u - cell0) : 0u;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (es == 4) s[K].y = __float_as_uint(f[K]);
        });
        if constexpr (es == 2) {
            if (dith) {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    s[K] = SP::template put<true>(s[K], f[K], wgt<float>(K), round_bits(hc, K), true);
                });
            } else {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    s[K] = SP::template put<true>(s[K], f[K], wgt<float>(K), 0u, false);
                });
            }
        }
    }
    if constexpr (EXTRA != TWO_BFL)
        if (want_force && lvb) link_force(std::integral_constant<int, 1>{}, lmb);

    // store: the whole words where both cells of every lane of the wave step
    const __amdgpu_buffer_rsrc_t fo = buf_at((char*)a.fout + (size_t)nb0 * blk);
    const uint32_t vown = own0 + row;
    const bool both = lva && lvb;
    if (__builtin_amdgcn_ballot_w64(!both) == 0) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            W::template st2<OAL_TWO_STORE_AUX>(s[K], fo, vown, (uint32_t)K * slot + zown);
        });
    } else {
        if (both) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                W::template st2<OAL_TWO_STORE_AUX>(s[K], fo, vown, (uint32_t)K * slot + zown);
            });
        } else if (lva || lvb) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                W::template st1<OAL_TWO_STORE_AUX>(lva ? W::a(s[K]) : W::b(s[K]), fo, vown + (lva ? 0u : es), (uint32_t)K * slot + zown);
            });
        }
    }
    if constexpr (WALE) {
        float* vout = (float*)a.vel_out;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            float* p = vout + (size_t)q * a.ncell + ca;
            if (both) *(float2*)p = make_float2(va[q], vb[q]);
            else if (lva) p[0] = va[q];
            else if (lvb) p[1] = vb[q];
        }
    }
    if (want_force) two_sum3(F0 * force_scale, F1 * force_scale, F2 * force_scale, a.fpart, b * PLANES + (uint32_t)z);
}

// the blocks of one list, one plane per workgroup
template <class SP, bool UNIT>
static void launch_two_u(bool wale, int extra, dim3 g, hipStream_t s, const StepArgs& r) {
    if (wale) {
        if (extra == TWO_SPONGE) hipLaunchKernelGGL((k_step_two<SP, UNIT, true, TWO_SPONGE>), g, dim3(TWG), 0, s, r);
        else if (extra == TWO_BFL) hipLaunchKernelGGL((k_step_two<SP, UNIT, true, TWO_BFL>), g, dim3(TWG), 0, s, r);
        else hipLaunchKernelGGL((k_step_two<SP, UNIT, true, TWO_PLAIN>), g, dim3(TWG), 0, s, r);
    } else {
        if (extra == TWO_SPONGE) hipLaunchKernelGGL((k_step_two<SP, UNIT, false, TWO_SPONGE>), g, dim3(TWG), 0, s, r);
        else if (extra == TWO_BFL) hipLaunchKernelGGL((k_step_two<SP, UNIT, false, TWO_BFL>), g, dim3(TWG), 0, s, r);
        else hipLaunchKernelGGL((k_step_two<SP, UNIT, false, TWO_PLAIN>), g, dim3(TWG), 0, s, r);
    }
}
template <class SP>
static void launch_two_sp(bool wale, int extra, const StepArgs& r, hipStream_t s) {
    const dim3 g(r.n_items);
    if (r.cp.unit) launch_two_u<SP, true>(wale, extra, g, s, r);
    else launch_two_u<SP, false>(wale, extra, g, s, r);
}

}  // namespace oal
