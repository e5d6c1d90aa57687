// The step kernel of the FP32-arithmetic forms, two cells per lane; a
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
// AA pattern (one population buffer, two half-steps): the even one reads population k of a cell from its own
// slot k and writes it to the own slot opp k; the odd one gathers from slot opp k of x - c_k and scatters to
// slot k of x + c_k (two_scatter).  Both are one launch over every block.
//
// Bound and shape.  The plane's 27 words are all in flight together and nothing is kept for a next plane,
// so a lane needs 97 to 125 registers and four waves share a SIMD; their loads overlap other waves'
// collisions.  That needs the rare limiter out of the registers (collide_cell's LDS form): with it inline
// the kernel takes 168 and spills.  Bound: HBM in FP32 (256^3: 5.97 TB/s
// counting 216 bytes per cell, of 6.04 that a copy reaches), in the 16-bit forms VALU and HBM alike (256^3 FP16: about 720
// instructions per cell, half of them issued every second cycle, the others every fourth or eighth, some
// 70 % of the time; 4.9 TB/s).  Measured against walking four planes of a block per workgroup with the
// next plane's words in flight (two waves per SIMD, a launch per kind of block, the default shape
// before): 256^3 sphere box FP32 667 -> 606 us per step, FP16 467 -> 370 us; WALE 192 x 160 x 160 FP32
// 295 -> 229 us, WALE 200 x 120 x 104 FP16 200 -> 93 us; WALE 100 x 60 x 44 75 -> 20 us (that shape left
// 48 workgroups per launch); 12 ragged boxes with solids and sponges FP16 813 -> 460 us.  Blocks run
// fastest: x-neighbour blocks share the lines of the row ends.  One record per block (TwoRec) in place of
// a chain of table reads: FP16 256^3 453 -> 372 us, 48 x 32 x 32 13.5 -> 10.8 us.  Stores written through
// at device scope: 48 x 32 x 32 10.8 -> 10.2 us, WALE 100 x 60 x 44 25.3 -> 20.9 us without the non-
// temporal hint (which 256^3 needs: 635 against 681 us). (Small levels in the AB pattern take the one-
// cell-per-lane form since: 48 x 32 x 32 7.0 us, ONE_BLOCKS.) AA 192 x 160 x 160 FP32, sphere: 340 -> 204
// us per step against a pipelined kernel for the blocks off the faces and a one-plane kernel for the rest
// (a third of the blocks); 5.2 TB/s of the pair's 216 bytes per cell.
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
    // the x-neighbour block's cell of the lane at j = 0 (its last pair, the cell in the high half), at j = 7
    // (its first pair, the cell in the low half)
    static constexpr uint32_t end_first = (BS - 2) * es, end_last = 0;
    __device__ static __forceinline__ uint32_t lde(__amdgpu_buffer_rsrc_t r, uint32_t v) { return ld2(r, v, 0); }
    // (left lane's B, own A); end: the x-neighbour block's cell of the lane at j = 0
    __device__ static __forceinline__ word from_left(word w, bool first, uint32_t end) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x111, 0xf, 0xf, true);
        return __builtin_amdgcn_alignbyte(w, first ? end : l, 2);
    }
    // (own B, right lane's A)
    __device__ static __forceinline__ word from_right(word w, bool last, uint32_t end) {
        const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x101, 0xf, 0xf, true);
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
    static constexpr uint32_t end_first = (BS - 1) * es, end_last = 0;
    __device__ static __forceinline__ uint32_t lde(__amdgpu_buffer_rsrc_t r, uint32_t v) { return ld1(r, v); }
    __device__ static __forceinline__ word from_left(word w, bool first, uint32_t end) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_mov_dpp((int)w.y, 0x111, 0xf, 0xf, true);
        return word{first ? end : l, w.x};
    }
    __device__ static __forceinline__ word from_right(word w, bool last, uint32_t end) {
        const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)w.x, 0x101, 0xf, 0xf, true);
        return word{w.y, last ? end : r};
    }
    __device__ static __forceinline__ float dec_a(word w, float) { return __uint_as_float(w.x); }
    __device__ static __forceinline__ float dec_b(word w, float) { return __uint_as_float(w.y); }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_at(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc((char*)p, (short)0, (int)0xffffffff, 0x00020000);
}
// the populations that a record's offsets of layer dz (uniform) are counted from
template <bool WIDE, class REC>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_layer(const void* p, const REC& R, int dz, uint32_t blk) {
    const uint32_t base = !WIDE || dz == 0 ? R.base : R.base_z[dz < 0 ? 0 : 1];
    return buf_at((const char*)p + (size_t)base * blk);
}

// the rules of a lane's row (both cells share y and z) and of its cells
struct TwoFaces {
    bool yl, yh;            // per lane: the row lies on the y-min / y-max face
    bool zl, zh;            // uniform: the plane lies on the z-min / z-max face
    bool zwall, ymin_wall;  // no-slip variants of the z faces and of the y-min face
};
template <class REC>
__device__ __forceinline__ TwoFaces two_faces(const REC& R, uint32_t flags, int gy, int gz) {
    const bool py = (flags & TR_PER_Y) != 0, pz = (flags & TR_PER_Z) != 0;
    TwoFaces fc;
    fc.yl = !py && gy == 0;
    fc.yh = !py && gy == R.ext[1] - 1;
    fc.zl = !pz && gz == 0;
    fc.zh = !pz && gz == R.ext[2] - 1;
    fc.zwall = (flags & TR_ZWALL) != 0;
    fc.ymin_wall = (flags & TR_YMIN) != 0;
    return fc;
}
// a lane's cells: on the inlet (A), on the outlet, stepped (inside the extent and not solid)
enum : uint32_t { LF_INLET = 1, LF_OUTLET_A = 2, LF_OUTLET_B = 4, LF_LIVE_A = 8, LF_LIVE_B = 16 };
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

// Cache policy of the stores (gfx950's sc and nt bits): written through at device scope, so that the
// kernel's end has no dirty lines to write back; non-temporal too where the level's two population buffers
// exceed TWO_KEEP_BYTES (below that the next step reads them from the 256 MB memory-side cache).
// The AA odd half-step's stores are ordinary ones: the words at the row ends are completed in the cache by
// two workgroups (192 x 160 x 160 FP32: 204 us per step, 213 non-temporal, 271 written through).
enum : int { TWO_ST_KEEP = 16, TWO_ST_STREAM = 18, TWO_ST_SCATTER = 0 };

// The writes of the AA pattern's odd half-step: population K of a cell goes to slot K of x + c_K.  The word
// a lane stores for direction K is the aligned pair of the row (y + cy, z + cz), whose two cells come from
// its own pair and, for cx != 0, the neighbouring lane's; at the row ends one cell goes to the x-neighbour
// block alone.  Where x + c_K does not step (beyond a face, solid), the rule of direction J = opp K is
// evaluated from the fresh state and stored in the own slot J, which the even half-step reads; an inlet
// link is left to the even half-step.  A lane's rows are its own in both passes, and of the words at the
// row ends each workgroup reads and writes its own cells only, so no access meets another's.
template <class SP, bool WIDE, class REC, class WORD>
__device__ __forceinline__ void two_scatter(const REC& R, void* fout, __amdgpu_buffer_rsrc_t fown, int z, int jx, int ly, bool edge,
                                            const TwoFaces& fc, uint32_t lf, uint32_t lma, uint32_t lmb, const WORD (&s)[27]) {
    using W = Two<SP>;
    constexpr uint32_t es = W::es, slot = BS3 * es;
    constexpr int AUX = TWO_ST_SCATTER;
    asm("" : "+v"(ly), "+v"(jx));   // the offsets are formed again here: kept from the gather they would cost 18 registers
    const bool first = jx == 0, last = jx == 7;
    const uint32_t own = R.off[13] + (uint32_t)ly * (BS * es) + (uint32_t)jx * (2 * es) + (uint32_t)z * (BS2 * es);
    // the pair's offset in the row (y + cy, z + cz), and the x-neighbour block's cell next to the row's end
    auto row_of = [&](int cy, int cz, uint32_t& v, uint32_t& e) {
        const REC* p = &R;
        asm("" : "+s"(p));   // (six offsets at a time: all 27 would spill the scalar registers)
        auto boff = [&](int dx, int dy, int dz) -> uint32_t { return p->off[(dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)]; };
        const int tz = z + cz;
        const int dz = tz < 0 ? -1 : (tz >= BS ? 1 : 0);
        const bool cross = cy > 0 ? ly == BS - 1 : (cy < 0 ? ly == 0 : false);
        const uint32_t r = (uint32_t)((ly + cy) & (BS - 1)) * (BS * es) + (uint32_t)(tz & (BS - 1)) * (BS2 * es);
        const uint32_t c0 = boff(0, 0, dz), c1 = boff(0, cy, dz), m0 = boff(-1, 0, dz), m1 = boff(-1, cy, dz), p0 = boff(1, 0, dz),
                       p1 = boff(1, cy, dz);
        v = (cross ? c1 : c0) + r + (uint32_t)jx * (2 * es);
        e = (first ? (cross ? m1 : m0) + (BS - 1) * es : (cross ? p1 : p0)) + r;
    };
    // K: the cells whose x + c_K steps
    uint32_t ra = (lf & LF_LIVE_A) ? 0x7ffffffu : 0u, rb = (lf & LF_LIVE_B) ? 0x7ffffffu : 0u;
    const uint32_t la = ra, lb = rb;
    const bool special = edge || (R.flags & BF_SOLID);
    if (special) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value, J = dopp(K);
            int j;
            const bool row = two_row_rule<J>(fc, j);
            const bool xa = (dcx(K) < 0 && (lf & LF_INLET)) || (dcx(K) > 0 && (lf & LF_OUTLET_A));
            const bool xb = dcx(K) > 0 && (lf & LF_OUTLET_B);
            if (row || xa || ((lma >> J) & 1u)) ra &= ~(1u << K);
            if (row || xb || ((lmb >> J) & 1u)) rb &= ~(1u << K);
        });
    }
    // of the pair left and right of this one in the row
    const uint32_t rl0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)rb, 0x111, 0xf, 0xf, true);
    const uint32_t rr0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)ra, 0x101, 0xf, 0xf, true);
    const uint32_t rl = first ? 0u : rl0, rr = last ? 0u : rr0;
    for_dirs([&](auto cc) {
        constexpr int C = decltype(cc)::value;
        if constexpr (C < 9) {
            constexpr int cy = C % 3 - 1, cz = C / 3 - 1, K0 = 3 * C;   // directions (cx, cy, cz) = K0 + cx + 1
            __builtin_amdgcn_sched_barrier(0);   // (the offsets of one row at a time)
            uint32_t v, e;
            row_of(cy, cz, v, e);
            __amdgpu_buffer_rsrc_t fo = fown;
            if constexpr (WIDE && cz != 0) fo = buf_layer<WIDE>(fout, R, z + cz < 0 ? -1 : (z + cz >= BS ? 1 : 0), 27u * slot);
            auto put = [&](const WORD& w, uint32_t lo, uint32_t hi, int k) {
                if (lo & hi & 1u) W::template st2<AUX>(w, fo, v, (uint32_t)k * slot);
                else if (lo & 1u) W::template st1<AUX>(W::a(w), fo, v, (uint32_t)k * slot);
                else if (hi & 1u) W::template st1<AUX>(W::b(w), fo, v + es, (uint32_t)k * slot);
            };
            put(s[K0 + 1], ra >> (K0 + 1), rb >> (K0 + 1), K0 + 1);
            put(W::from_left(s[K0 + 2], first, 0u), rl >> (K0 + 2), ra >> (K0 + 2), K0 + 2);
            put(W::from_right(s[K0], last, 0u), rb >> K0, rr >> K0, K0);
            // B to the +x block's cell 0, A to the -x block's cell 15
            if (first ? (ra >> K0) & 1u : (last ? (rb >> (K0 + 2)) & 1u : 0u))
                W::template st1<AUX>(first ? W::a(s[K0]) : W::b(s[K0 + 2]), fo, e + (first ? (uint32_t)K0 : (uint32_t)K0 + 2) * slot, 0);
        }
    });
    // the rules' writes, one cell of the pairs after the other: its codes through LDS, a rolled loop over the
    // directions that some lane needs (unrolled, the choices among the 27 words spill)
    uint32_t wa = la & ~ra, wb = lb & ~rb;
    if (lf & LF_INLET) wa &= ~0x1249249u;         // (directions with cx < 0: bits 0, 3, 6, ...)
    if (special && __builtin_amdgcn_ballot_w64((wa | wb) != 0) != 0) {
        uint32_t* lds = two_lds() + threadIdx.x;
        for (int half = 0; half < 2; ++half) {
            const uint32_t w = half ? wb : wa;
            const bool outlet = (lf & (half ? LF_OUTLET_B : LF_OUTLET_A)) != 0;
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                lds[K * TWG] = half ? W::b(s[K]) : W::a(s[K]);
            });
#pragma unroll 1
            for (int k = 0; k < 27; ++k) {
                const bool mine = (w >> k) & 1u;
                if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
                const int j = 26 - k, cx = k % 3 - 1, cyj = 1 - (k / 3) % 3, czj = 1 - k / 9;
                const bool zf = (czj > 0 && fc.zl) || (czj < 0 && fc.zh), yf = (cyj > 0 && fc.yl) || (cyj < 0 && fc.yh);
                const bool wall = (fc.zwall && zf) || (fc.ymin_wall && cyj > 0 && fc.yl);
                // the rule of direction j: its own population, the opposite one (walls and solid links), the mirrors
                const int src = outlet && cx > 0 ? j : (wall || !(zf || yf)) ? k : yf ? j - 6 * cyj : j - 18 * czj;
                if (mine) W::template st1<AUX>(lds[src * TWG], fown, own + (uint32_t)half * es, (uint32_t)j * slot);
            }
        }
    }
}

// DITH: stochastic rounding (the 16-bit forms).  WIDE: each layer of neighbours from its own base.  Only planes 0
// and 15 of a block have sources (or targets) in another layer, of one cz each, so a plane's buffer is uniform per
// cz; where a rule takes the own population of a row's lanes instead, those lanes load it apart.
template <class SP, bool UNIT, bool WALE, int EXTRA, bool DITH, int PAT, bool WIDE = false>
__global__ void __launch_bounds__(TWG) __attribute__((amdgpu_waves_per_eu(PAT == PAT_AA_ODD && SP::dithered ? 2 : EXTRA == TWO_BFL || PAT == PAT_AA_ODD || (EXTRA == TWO_SPONGE && !(UNIT && !WALE)) ? 3 : 4)))
k_step_two(const StepArgs a) {
    using W = Two<SP>;
    using word = typename W::word;
    constexpr uint32_t es = W::es;
    constexpr uint32_t slot = BS3 * es;          // bytes of one direction of a block
    constexpr uint32_t blk = 27u * slot;
    const uint32_t litem = xcd_item(blockIdx.x, gridDim.x);
    const uint32_t nblk = gridDim.x / PLANES;
    const uint32_t zi = litem / nblk;
    // (constant address space: read by scalar loads wherever a field is used)
    const auto& R = ((const __attribute__((address_space(4))) TwoRec*)a.rec)[litem - zi * nblk];
    const uint32_t b = R.block;
    const int z = (int)zi;
    const uint32_t flags = R.flags;
    const int ox = R.org[0], oy = R.org[1], gz = R.org[2] + z;
    if (gz >= R.ext[2]) return;                  // a plane beyond the extent
    const int jx = (int)(threadIdx.x & 7u), ly = (int)(threadIdx.x >> 3);
    auto boff = [&](int dx, int dy, int dz) -> uint32_t { return R.off[(dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)]; };
    const __amdgpu_buffer_rsrc_t fin = buf_at((const char*)a.fin + (size_t)R.base * blk);
    // (of the sources of direction cz)
    auto fin_z = [&](auto czc) {
        constexpr int cz = decltype(czc)::value;
        if constexpr (!WIDE || cz == 0) return fin;
        else return buf_layer<WIDE>(a.fin, R, z - cz < 0 ? -1 : (z - cz >= BS ? 1 : 0), blk);
    };
    const uint32_t row = (uint32_t)ly * (BS * es) + (uint32_t)jx * (2 * es);
    const uint32_t zown = (uint32_t)z * (BS2 * es);
    const uint32_t own0 = R.off[13];             // uniform
    const bool first = jx == 0, last = jx == 7;

    const bool edge = (flags & BF_EDGE) != 0;
    TwoFaces fc{};
    // what the lane's cells are, in a vector register: as booleans each would hold a scalar register pair
    // through the kernel, and the scalar registers spill
    uint32_t lf = LF_LIVE_A | LF_LIVE_B;
    if (edge) {
        const int gy = oy + ly, ga = ox + 2 * jx;
        const bool px = (flags & TR_PER_X) != 0;
        fc = two_faces(R, flags, gy, gz);
        lf = !px && ga == 0 ? LF_INLET : 0u;
        lf |= !px && ga == R.ext[0] - 1 ? LF_OUTLET_A : 0u;
        lf |= !px && ga + 1 == R.ext[0] - 1 ? LF_OUTLET_B : 0u;
        lf |= gy < R.ext[1] && ga < R.ext[0] ? LF_LIVE_A : 0u;
        lf |= gy < R.ext[1] && ga + 1 < R.ext[0] ? LF_LIVE_B : 0u;
    }
    asm("" : "+v"(lf));
    auto is = [&](uint32_t f) { return (lf & f) != 0; };
    // solid links of the two cells (bit k: the source of direction k is solid; bit 27: the cell is)
    uint32_t lma = 0, lmb = 0;
    if (flags & BF_SOLID) {
        const u32x2 m = *(const u32x2*)(a.lmask + (size_t)R.lslot * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + 2u * (uint32_t)jx);
        lma = m.x;
        lmb = m.y;
        if ((lma >> 27) & 1u) lf &= ~LF_LIVE_A;
        if ((lmb >> 27) & 1u) lf &= ~LF_LIVE_B;
    }

    // a wave with nothing to step (rows beyond the extent, the inside of a solid) ends here, unless the
    // workgroup sums the force
    const bool want_force = a.fpart != nullptr && (flags & BF_SOLID);
    if (!want_force && __builtin_amdgcn_ballot_w64(is(LF_LIVE_A | LF_LIVE_B)) == 0) return;

    // WALE: the previous step's velocity of the pair and of its neighbour pairs, requested first
    u32x2 vo[3], vyp[3], vym[3], vzp[3], vzm[3];
    uint32_t vend[3];
    bool no_end = false;                         // no x-neighbour block behind the row's end
    if constexpr (WALE) {
        const __amdgpu_buffer_rsrc_t vr = buf_at(a.vel_in);
        const uint32_t comp = a.ncell * 4u;
        auto at = [&](uint32_t n) { return n * (BS3 * 4u); };
        const uint32_t loc = (uint32_t)(ly * BS + 2 * jx) * 4u, zc = (uint32_t)z * (BS2 * 4u);
        const uint32_t own = at(b) + zc + loc;
        auto absent = [&](int f) { return ((flags >> f) & TR_ABSENT) != 0; };   // (uniform)
        const bool cp = ly == BS - 1, cm = ly == 0;
        uint32_t oyp = cp ? (absent(2) ? own : at(R.face[2]) + zc + loc - (BS - 1) * BS * 4u) : own + BS * 4u;
        uint32_t oym = cm ? (absent(3) ? own : at(R.face[3]) + zc + loc + (BS - 1) * BS * 4u) : own - BS * 4u;
        uint32_t ozp = z == BS - 1 ? (absent(4) ? own : at(R.face[4]) + loc) : own + BS2 * 4u;
        uint32_t ozm = z == 0 ? (absent(5) ? own : at(R.face[5]) + (BS - 1) * BS2 * 4u + loc) : own - BS2 * 4u;
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
            no_end = first ? absent(1) : absent(0);
            // (-x block's cell 15 of the row, +x block's cell 0)
            const uint32_t oe = no_end ? own : at(first ? R.face[1] : R.face[0]) + zc + (uint32_t)(ly * BS + (first ? BS - 1 : 0)) * 4u;
#pragma unroll
            for (int q = 0; q < 3; ++q) vend[q] = __builtin_amdgcn_raw_buffer_load_b32(vr, (int)oe, (int)(q * comp), 0);
        }
    }
    float spa = 0.0f, spb = 0.0f;
    if constexpr (EXTRA == TWO_SPONGE) {
        if (flags & BF_SPONGE) {
            const float* sp = a.sponge + (size_t)R.sslot * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + 2u * (uint32_t)jx;
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
            ve[k][i] = (first ? m + W::end_first + (PAT == PAT_AA_ODD ? -2u * slot : 2 * slot) : p + W::end_last) + r;
        }
    }
    // the slot direction K is read from: in the odd half-step of the AA pattern opp K of the source cell
    constexpr auto rd = [](int k) { return (uint32_t)(PAT == PAT_AA_ODD ? dopp(k) : k); };
    word s[27];
    uint32_t e9[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) e9[q] = 0;
    if constexpr (PAT == PAT_AA_EVEN) {   // every population in the cell's own slot
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            s[K] = W::ld2(fin, own0 + row, (uint32_t)K * slot + zown);
        });
    } else if (edge) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            uint32_t o = v[cz + 1][cy + 1] + rd(K) * slot + zs[cz + 1];
            if constexpr (cy != 0 || cz != 0) {
                int j;
                const bool face = two_row_rule<K>(fc, j);
                if constexpr (WIDE && cz != 0) {
                    if (face) s[K] = W::ld2(fin, own0 + row + rd(j) * slot + zown, 0);
                    else s[K] = W::ld2(fin_z(dir_c<cz>{}), o, 0);
                    return;
                }
                o = face ? own0 + row + rd(j) * slot + zown : o;
            }
            s[K] = W::ld2(fin, o, 0);
        });
    } else {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            s[K] = W::ld2(fin_z(dir_c<cz>{}), v[cz + 1][cy + 1], rd(K) * slot + zs[cz + 1]);
        });
    }
    if (PAT != PAT_AA_EVEN && (first || last)) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cy = dcy(K), cz = dcz(K);
            if constexpr (dcx(K) < 0) e9[K / 3] = W::lde(fin_z(dir_c<cz>{}), ve[cz + 1][cy + 1] + rd(K) * slot + zs[cz + 1]);
        });
    }

    // WALE: the eddy viscosity of both cells, while the populations are in flight
    CellRates<float> qa;
    qa.forced = (flags & TR_FORCED) != 0;
    qa.Fx = R.F[0]; qa.Fy = R.F[1]; qa.Fz = R.F[2];
    qa.omega1 = R.omega1;
    qa.omega4_diag = R.omega4d;
    if constexpr (EXTRA == TWO_SPONGE) {
        qa.sponge_u = R.u_in;
        qa.sponge_blend = a.sponge_blend;
    }
    float om1b = qa.omega1, om4b = qa.omega4_diag;
    const uint32_t cell0 = R.cell0;
    const float u_in = R.u_in, force_scale = R.force_scale;
    if constexpr (WALE) {
        const float tau = R.tau, amr = R.amr_scale;
        auto f32 = [](uint32_t u) { return __uint_as_float(u); };
        float ga[3][3], gb[3][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const float A = f32(vo[q].x), B = f32(vo[q].y);
            const uint32_t l = (uint32_t)__builtin_amdgcn_mov_dpp((int)vo[q].y, 0x111, 0xf, 0xf, true);
            const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)vo[q].x, 0x101, 0xf, 0xf, true);
            float axm = first ? f32(vend[q]) : f32(l), bxp = last ? f32(vend[q]) : f32(r);
            float axp = B, bxm = A;
            float ayp = f32(vyp[q].x), aym = f32(vym[q].x), azp = f32(vzp[q].x), azm = f32(vzm[q].x);
            float byp = f32(vyp[q].y), bym = f32(vym[q].y), bzp = f32(vzp[q].y), bzm = f32(vzm[q].y);
            // across a face, beside an absent block or a solid cell: the cell itself
            axm = (is(LF_INLET) || (first && no_end)) ? A : axm;
            axp = is(LF_OUTLET_A) ? A : axp;
            bxp = (is(LF_OUTLET_B) || (last && no_end)) ? B : bxp;
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
    auto sources = [&](auto rules) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int cx = dcx(K), cy = dcy(K), cz = dcz(K);
            if constexpr (cx != 0) {
                word w;
                if constexpr (cx > 0) w = W::from_left(s[K], first, e9[K / 3]);
                else w = W::from_right(s[K], last, e9[K / 3]);
                if constexpr (decltype(rules)::value && (cy != 0 || cz != 0)) {
                    int j;
                    const bool face = two_row_rule<K>(fc, j);
                    if constexpr (es == 4) { w.x = face ? s[K].x : w.x; w.y = face ? s[K].y : w.y; }
                    else w = face ? s[K] : w;
                }
                s[K] = w;
            }
        });
    };
    if constexpr (PAT != PAT_AA_EVEN) {
        if (edge) sources(std::true_type{});
        else sources(std::false_type{});
    }
    // AA pattern: the lane's row in the outlet copies (9 populations with cx = -1 per row, by (y, z))
    const uint32_t ocopy = PAT == PAT_AB ? 0u : (uint32_t)R.oslot * (9 * BS2 * es) + (uint32_t)(ly * BS + z) * es;
    // second pass: solid links and the outlet, in waves that hold one
    const uint32_t links = lma | lmb;
    if (PAT != PAT_AA_EVEN && __builtin_amdgcn_ballot_w64((links & 0x7ffffffu) != 0 || is(LF_OUTLET_A | LF_OUTLET_B)) != 0) {
        const bool xha = is(LF_OUTLET_A), xhb = is(LF_OUTLET_B);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            uint32_t ra[9], rb[9];
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if (K / 9 == c) {
                    const bool oa = dcx(K) < 0 && xha, ob = dcx(K) < 0 && xhb;
                    ra[K % 9] = 0;
                    rb[K % 9] = 0;
                    if constexpr (PAT == PAT_AB) {
                        if (((lma >> K) & 1u) || oa) ra[K % 9] = W::ld1(fin, own0 + row + zown + (oa ? (uint32_t)K : (uint32_t)dopp(K)) * slot);
                        if (((lmb >> K) & 1u) || ob) rb[K % 9] = W::ld1(fin, own0 + row + es + zown + (ob ? (uint32_t)K : (uint32_t)dopp(K)) * slot);
                    } else {   // the outlet from the even half-step's copy
                        if ((lma >> K) & 1u) ra[K % 9] = W::ld1(fin, own0 + row + zown + (uint32_t)K * slot);
                        if ((lmb >> K) & 1u) rb[K % 9] = W::ld1(fin, own0 + row + es + zown + (uint32_t)K * slot);
                        if (oa) ra[K % 9] = W::ld1(buf_at(a.obuf), ocopy + (uint32_t)(K / 3) * (BS2 * es));
                        if (ob) rb[K % 9] = W::ld1(buf_at(a.obuf), ocopy + (uint32_t)(K / 3) * (BS2 * es));
                    }
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
    const uint32_t key = DITH ? round_key(a.step()) : 0u;
    double F0 = 0.0, F1 = 0.0, F2 = 0.0;
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
    if (is(LF_INLET)) {
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (dcx(K) > 0)
                f[K] = boundary_value<K, float>(SRC_INLET, a, cc, u_in, a.step(), [&](auto) { return 0.0f; });
        });
    }
    if constexpr (EXTRA == TWO_BFL) {
        if (is(LF_LIVE_A) && (lma & 0x7ffffffu)) bfl(f, ca, lma, is(LF_OUTLET_A), is(LF_INLET));
    }
    if constexpr (EXTRA == TWO_SPONGE) qa.sponge = spa;
    collide_cell<float, UNIT, EXTRA == TWO_SPONGE, true, es == 2>(f, qa, a.cp, rho_o, va[0], va[1], va[2]);
    {
        const uint32_t hc = DITH ? round_cell(key, ca - cell0) : 0u;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (es == 4) s[K].x = __float_as_uint(f[K]);
        });
        if constexpr (es == 2) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                s[K] = SP::template put<false, K>(s[K], f[K], DITH ? round_bits(hc, K) : 0u, DITH);
            });
        }
    }
    if constexpr (EXTRA != TWO_BFL)
        if (want_force && is(LF_LIVE_A)) link_force(std::integral_constant<int, 0>{}, lma);
    __builtin_amdgcn_sched_barrier(0);
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        f[K] = W::dec_b(s[K], wgt<float>(K));
    });
    if constexpr (EXTRA == TWO_BFL) {
        if (is(LF_LIVE_B) && (lmb & 0x7ffffffu)) bfl(f, ca + 1u, lmb, is(LF_OUTLET_B), false);
    }
    CellRates<float> qb = qa;
    qb.omega1 = om1b;
    qb.omega4_diag = om4b;
    if constexpr (EXTRA == TWO_SPONGE) qb.sponge = spb;
    collide_cell<float, UNIT, EXTRA == TWO_SPONGE, true, es == 2>(f, qb, a.cp, rho_o, vb[0], vb[1], vb[2]);
    {
        const uint32_t hc = DITH ? round_cell(key, ca + 1u - cell0) : 0u;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (es == 4) s[K].y = __float_as_uint(f[K]);
        });
        if constexpr (es == 2) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                s[K] = SP::template put<true, K>(s[K], f[K], DITH ? round_bits(hc, K) : 0u, DITH);
            });
        }
    }
    if constexpr (EXTRA != TWO_BFL)
        if (want_force && is(LF_LIVE_B)) link_force(std::integral_constant<int, 1>{}, lmb);

    // store
    const __amdgpu_buffer_rsrc_t fo = buf_at((char*)a.fout + (size_t)R.base * blk);
    const uint32_t vown = own0 + row;
    const bool lva = is(LF_LIVE_A), lvb = is(LF_LIVE_B), both = lva && lvb;
    if constexpr (PAT == PAT_AA_ODD) {
        two_scatter<SP, WIDE>(R, a.fout, fo, z, jx, ly, edge, fc, lf, lma, lmb, s);
    } else {
        // (the even half-step writes population K to the own slot opp K)
        constexpr auto wr = [](int k) { return (uint32_t)(PAT == PAT_AA_EVEN ? dopp(k) : k); };
        auto store = [&](auto aux) {
            constexpr int AUX = decltype(aux)::value;
            if (both) {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    W::template st2<AUX>(s[K], fo, vown, wr(K) * slot + zown);
                });
            } else if (lva || lvb) {
                for_dirs([&](auto kc) {
                    constexpr int K = decltype(kc)::value;
                    W::template st1<AUX>(lva ? W::a(s[K]) : W::b(s[K]), fo, vown + (lva ? 0u : es), wr(K) * slot + zown);
                });
            }
        };
        if (a.two_keep) store(std::integral_constant<int, TWO_ST_KEEP>{});
        else store(std::integral_constant<int, TWO_ST_STREAM>{});
    }
    if constexpr (PAT == PAT_AA_EVEN) {
        // the outlet row's populations with cx = -1, which the odd half-step's neighbours overwrite
        if (is(LF_OUTLET_A | LF_OUTLET_B) && (is(LF_OUTLET_A) ? lva : lvb)) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                if constexpr (dcx(K) < 0)
                    W::template st1<0>(is(LF_OUTLET_A) ? W::a(s[K]) : W::b(s[K]), buf_at(a.obuf), ocopy + (uint32_t)(K / 3) * (BS2 * es), 0);
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

// Dynamic LDS that no kernel uses: it leaves five workgroups (ten waves) on a CU instead of eight where an FP32
// level streams through the caches.  The number is measured.  The loads in flight on an XCD (27 KB a workgroup, 32
// CUs) are 7.1 MB with eight against its 4 MB L2, so that lines at the row ends and of half rows leave it before
// the neighbouring workgroup reads them; with five they are 4.4 MB, and reads fall from 1.076 to 1.039 of
// algorithmic; with four too few are in flight.  256^3 FP32: 629.9 us per step, 612 with six workgroups, 605 with
// five, 615 with four; WALE 192 x 160 x 160: 232, 227.7 and 228.2 (no difference), 237; interpolated wall 160 x 128 x
// 128 121.9, with five 119.3.  The AA pattern (204, 209, 215 us), the 16-bit forms (256^3 FP16 376, with six 436
// us) and levels that stay in the memory-side cache keep all.
constexpr uint32_t TWO_HOLD_LDS = 18000;

// the blocks of one list, one plane per workgroup
template <class SP, bool UNIT, bool DITH, bool WALE>
static void launch_two_w(int extra, dim3 g, hipStream_t s, const StepArgs& r) {
    const uint32_t hold = SP::dithered || r.two_keep ? 0u : TWO_HOLD_LDS;
    if (extra == TWO_SPONGE) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_SPONGE, DITH, PAT_AB>), g, dim3(TWG), hold, s, r);
    else if (extra == TWO_BFL) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_BFL, DITH, PAT_AB>), g, dim3(TWG), hold, s, r);
    else if (extra == TWO_AA_EVEN) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_PLAIN, DITH, PAT_AA_EVEN>), g, dim3(TWG), 0, s, r);
    else if (extra == TWO_AA_ODD) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_PLAIN, DITH, PAT_AA_ODD>), g, dim3(TWG), 0, s, r);
    else if (extra == TWO_AA_ODD_WIDE) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_PLAIN, DITH, PAT_AA_ODD, true>), g, dim3(TWG), 0, s, r);
    else if (extra == TWO_WIDE) hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_PLAIN, DITH, PAT_AB, true>), g, dim3(TWG), hold, s, r);
    else hipLaunchKernelGGL((k_step_two<SP, UNIT, WALE, TWO_PLAIN, DITH, PAT_AB>), g, dim3(TWG), hold, s, r);
}
template <class SP>
static void launch_two_sp(bool wale, int extra, const StepArgs& r, hipStream_t s) {
    const dim3 g(r.n_items);
    auto go = [&](auto unit, auto dith) {
        if (wale) launch_two_w<SP, decltype(unit)::value, decltype(dith)::value, true>(extra, g, s, r);
        else launch_two_w<SP, decltype(unit)::value, decltype(dith)::value, false>(extra, g, s, r);
    };
    auto rates = [&](auto dith) {
        if (r.cp.unit) go(std::true_type{}, dith);
        else go(std::false_type{}, dith);
    };
    if constexpr (SP::dithered) {
        if (r.cp.dither) rates(std::true_type{});
        else rates(std::false_type{});
    } else {
        rates(std::false_type{});
    }
}

}  // namespace oal
