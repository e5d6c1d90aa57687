// The block records of the one-launch step kernels and the offsets in them (host and device; no HIP).
#pragma once

#include <stdint.h>

#include <algorithm>

namespace oal {

constexpr int BS = 16;            // cells per block edge
constexpr int BS2 = BS * BS;
constexpr int BS3 = BS * BS * BS;

// All a workgroup of a one-launch step kernel (k_step_two, k_step_one) reads about its block, one record per entry of a block
// list: one round of scalar loads in place of a chain (list entry, block tables, domain).  Neighbour
// offsets are in bytes of populations from the lowest block among the neighbours and the block (absent:
// the block's own), so that 32 bits reach every one.  Where they do not (two_fit), each of the three layers of
// neighbours has a base of its own, base_z[0], base, base_z[1] (absent: that layer's base), and the kernel's
// WIDE form reads a source plane from the buffer of its layer.
struct TwoRec {
    uint32_t off[27];          // by (dx + 1) + 3 (dy + 1) + 9 (dz + 1); [13]: the block itself
    uint32_t base;             // the lowest block (WIDE: of the block's own layer)
    uint32_t block;
    uint32_t flags;            // BF_* and TR_*
    int32_t org[3];
    int32_t lslot, sslot, oslot;   // link-mask, sponge and outlet-copy slots
    int32_t ext[3];
    float u_in, omega1, omega4d, F[3], tau, amr_scale, force_scale;
    uint32_t cell0;
    uint32_t face[6];          // neighbour blocks x+, x-, y+, y-, z+, z- (WALE; absent: the block itself)
    uint32_t pad0;
    double omega1_d, omega4d_d;   // FP64 form
    uint32_t base_z[2];           // WIDE: the lowest block of the layer below (dz = -1) and above (dz = +1)
    uint32_t pad[2];
};
static_assert(sizeof(TwoRec) == 256, "a record is four cache lines of the scalar cache");
enum : uint32_t {
    TR_PER_X = 1u << 8, TR_PER_Y = 1u << 9, TR_PER_Z = 1u << 10,   // periodic axes
    TR_ZWALL = 1u << 11, TR_YMIN = 1u << 12,                       // no-slip z faces, no-slip y-min face
    TR_FORCED = 1u << 13,
    TR_ABSENT = 1u << 16       // shifted by 0..5: the face neighbour is absent
};

// How the one-launch kernels' 32-bit byte offsets span a block's neighbours (populations of `esize` bytes): all 27
// from one base, or else (their WIDE form) those of each layer from its own.  A block inside a domain spans two
// layers of the domain's blocks, which cease to fit beyond 1114 x 1114 cells per layer in FP32 (FP64 788 x 788,
// 16 bits 1576 x 1576), and the wraps of a z-periodic level span the whole of it; by layers it spans two rows.
// Against the general kernel, which steps whatever no 32 bits span (ms per step): 1136 x 1120 x 96 FP32 5.64 ->
// 4.42, with WALE 7.60 -> 5.30, AA 7.74 -> 5.50; 800 x 800 x 112 FP64 5.85 -> 5.50; 1600 x 1600 x 48 FP16 3.97 ->
// 2.54; 400 x 416 x 416 FP32 periodic 2.62 -> 2.52.  A form of its own, so that the narrow one keeps its
// scalar registers.
enum : char { FIT_NONE = 0, FIT_ALL = 1, FIT_LAYERS = 2 };

// Byte offset, from a block's start, of the cell `local` of its neighbour (dx, dy) in a row of nbx blocks: k_step's
// regular forms keep it in signed 32 bits per lane (RegAddr) ...
inline int64_t row_offset(int dx, int dy, int64_t nbx, int64_t local, uint64_t esize) {
    return ((dx + dy * nbx) * (27 * BS3) + local) * (int64_t)esize;
}
// ... which hold the blocks of the rows before and after where a row spans less than 2 GiB (4853 blocks in FP32, 77 648
// cells; FP64 2426); blocks of longer rows are not regular: the general forms' addresses have 64 bits
inline bool row_fits(int64_t nbx, uint64_t esize) {
    return row_offset(1, 1, nbx, BS3, esize) < (1ll << 31) && row_offset(-1, -1, nbx, 0, esize) >= -(1ll << 31);
}

// The block that a record counts the offsets of each layer of neighbours from (nt: the block's row of neighbours,
// -1 = absent): the lowest of all of them, or (by layers) of the layer, which the block itself stands for where it
// has none
inline void two_bases(const int32_t* nt, uint32_t b, bool layers, uint32_t (&lo)[3]) {
    for (int z = 0; z < 3; ++z) {
        bool any = z == 1;
        lo[z] = b;
        for (int k = 9 * z; k < 9 * z + 9; ++k)
            if (nt[k] >= 0) {
                lo[z] = any ? std::min(lo[z], (uint32_t)nt[k]) : (uint32_t)nt[k];
                any = true;
            }
    }
    if (!layers) lo[0] = lo[1] = lo[2] = std::min({b, lo[0], lo[1], lo[2]});
}

inline char two_fit(const int32_t* nt, uint32_t b, uint64_t esize) {
    for (const bool layers : {false, true}) {
        uint32_t lo[3];
        two_bases(nt, b, layers, lo);
        bool fits = true;
        for (int z = 0; z < 3; ++z) {
            uint32_t hi = z == 1 || !layers ? std::max(lo[z], b) : lo[z];
            for (int k = 9 * z; k < 9 * z + 9; ++k)
                if (nt[k] >= 0) hi = std::max(hi, (uint32_t)nt[k]);
            fits = fits && (uint64_t)(hi - lo[z] + 1u) * 27u * BS3 * esize < (1ull << 32);
        }
        if (fits) return layers ? FIT_LAYERS : FIT_ALL;
    }
    return FIT_NONE;
}

// A record's bases and offsets.  Absent neighbours are never read for a value, only by lanes whose rule or place
// beyond the extent discards it: any block in reach stands for them.
inline void two_offsets(const int32_t* nt, uint32_t b, bool layers, uint32_t esize, TwoRec& r) {
    uint32_t lo[3];
    two_bases(nt, b, layers, lo);
    for (int k = 0; k < 27; ++k)
        r.off[k] = nt[k] < 0 && layers ? 0u : ((nt[k] < 0 ? b : (uint32_t)nt[k]) - lo[k / 9]) * (27u * BS3 * esize);
    r.base = lo[1];
    r.base_z[0] = lo[0];
    r.base_z[1] = lo[2];
}

}  // namespace oal
