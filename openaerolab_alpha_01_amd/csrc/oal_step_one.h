// The step kernel of the AB pattern with one cell per lane: every FP64 level, and small levels of the other
// storage forms (launch_pat); a translation unit per form (oal_one_<storage>.hip).
//
// One workgroup of 256 lanes steps one 16 x 16 plane of a block; one launch covers the blocks of every kind
// but a few (build_lists), from the records and with the rules of the two-cells-per-lane kernel: the 27
// sources of a cell are loaded together, each from its source cell or, across a face, at a solid link or on
// the outlet, from the own cell's population that the rule names; the inlet replaces values afterwards.
//
// Bound and shape.  FP64: 27 doubles are 54 registers; with the unit-rate collision and without the positivity
// limiter's branch a lane needs 118 (124 with WALE), so four waves share a SIMD and 64^3 cells are all resident
// at once.  Bound: HBM (192 x 160 x 160: 5.5 TB/s of 432 bytes per cell), at 64^3 the memory-side cache and one
// wave's latency.  Measured against a kernel per kind of block, two waves per SIMD, on two streams: 64^3
// periodic 30.5 -> 18.5 us per step; sphere boxes 192 x 160 x 160 472 -> 384 us, with WALE 568 -> 479 us,
// 100 x 60 x 44 with WALE 94 -> 28.5 us, 48 x 32 x 32 13.1 -> 7.3 us.
// FP32 and the 16-bit forms: 58 to 62 registers, eight waves per SIMD.  A small level's step is one wave's
// latency, and here a wave collides one cell per lane instead of two in turn: 48 x 32 x 32 FP32 10.0 -> 7.0 us
// per step, WALE 100 x 60 x 44 20.2 -> 17.6 us, octrees around a sphere 1562 -> 1525 us (FP16, 4 levels) and
// 594 -> 575 us (FP32 WALE, 3 levels) per coarse step.  On large levels pairs win: half the addresses and half
// the memory instructions (256^3 FP32 634 against 653 us, FP16 371 against 385 us).
#pragma once

#include "oal_step_two.h"

namespace oal {

// a cell in storage form
template <class SP>
struct One {   // 16-bit forms
    using word = uint32_t;
    static constexpr uint32_t es = 2;
    __device__ static __forceinline__ word ld(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)v, (int)s, 0);
    }
    template <int AUX>
    __device__ static __forceinline__ void st(word w, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)w, r, (int)v, (int)s, AUX);
    }
    __device__ static __forceinline__ float dec(word w, float wk) { return SP::dec_lo(w, wk); }
    // (2^(|cx| + |cy| + |cz|) f, collide_cell's SCALED form; the upper half is not stored: what it holds needs
    // no register of its own)
    template <int K, bool DITH>
    __device__ static __forceinline__ word enc(float f, uint32_t r) {
        return SP::template put<false, K>(__float_as_uint(SP::template unscaled<K>(f)), f, r, DITH);
    }
};
template <>
struct One<StF32> {
    using word = uint32_t;
    static constexpr uint32_t es = 4;
    __device__ static __forceinline__ word ld(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0);
    }
    template <int AUX>
    __device__ static __forceinline__ void st(word w, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b32(w, r, (int)v, (int)s, AUX);
    }
    __device__ static __forceinline__ float dec(word w, float) { return __uint_as_float(w); }
    template <int, bool>
    __device__ static __forceinline__ word enc(float f, uint32_t) { return __float_as_uint(f); }
};
template <>
struct One<StF64> {
    using word = u32x2;
    static constexpr uint32_t es = 8;
    __device__ static __forceinline__ word ld(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        return __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0);
    }
    template <int AUX>
    __device__ static __forceinline__ void st(word w, __amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
        __builtin_amdgcn_raw_buffer_store_b64(w, r, (int)v, (int)s, AUX);
    }
    __device__ static __forceinline__ double dec(word w, double) { return __builtin_bit_cast(double, w); }
    template <int, bool>
    __device__ static __forceinline__ word enc(double f, uint32_t) { return __builtin_bit_cast(u32x2, f); }
};

// POS: with the positivity limiter, whose 54 equilibria cost the other form half its occupancy
template <class SP>
constexpr int one_waves(bool unit, bool wale, bool pos) {
    if (sizeof(typename SP::T) == 8) return pos ? 2 : unit ? 4 : 3;
    return pos ? 3 : unit ? 8 : wale ? 5 : 6;
}
// WIDE: as in k_step_two (a lane whose rule takes its own population loads it apart)
template <class SP, bool UNIT, bool WALE, bool POS, bool DITH, bool WIDE = false>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(one_waves<SP>(UNIT, WALE, POS))))
k_step_one(const StepArgs a) {
    using T = typename SP::T;
    using W = One<SP>;
    constexpr uint32_t es = W::es, slot = BS3 * es, blk = 27u * slot;
    const uint32_t litem = xcd_item(blockIdx.x, gridDim.x);
    const uint32_t nblk = gridDim.x / PLANES;
    const uint32_t zi = litem / nblk;
    const auto& R = ((const __attribute__((address_space(4))) TwoRec*)a.rec)[litem - zi * nblk];
    const int z = (int)zi;
    if (R.org[2] + z >= R.ext[2]) return;        // a plane beyond the extent
    const uint32_t b = R.block, flags = R.flags;
    const int lx = (int)(threadIdx.x & 15u), ly = (int)(threadIdx.x >> 4);
    const uint32_t plane = (uint32_t)z * BS2 + (uint32_t)ly * BS + (uint32_t)lx;
    const __amdgpu_buffer_rsrc_t fin = buf_at((const char*)a.fin + (size_t)R.base * blk);
    const uint32_t own = R.off[13] + plane * es;

    CellCtx c{};
    c.b = b;
    c.z = z;
    c.lx = lx;
    c.ly = ly;
    c.flags = flags;
    c.gx = R.org[0] + lx;
    c.gy = R.org[1] + ly;
    c.gz = R.org[2] + z;
    c.own = b * BS3 + plane;
    TwoFaces fc{};
    bool inlet = false, outlet = false, live = true;
    if (flags & BF_EDGE) {
        const bool px = (flags & TR_PER_X) != 0;
        fc = two_faces(R, flags, c.gy, c.gz);
        inlet = !px && c.gx == 0;
        outlet = !px && c.gx == R.ext[0] - 1;
        live = c.gx < R.ext[0] && c.gy < R.ext[1];
    }
    if (flags & BF_SOLID) {
        c.lmask = a.lmask[(size_t)R.lslot * BS3 + plane];
        live = live && !((c.lmask >> 27) & 1u);
    }
    const bool want_force = a.fpart != nullptr && (flags & BF_SOLID);
    if (!want_force && __builtin_amdgcn_ballot_w64(live) == 0) return;

    // the source of direction (cx, cy, cz): row (ly - cy, z - cz), whose cells lie in the block itself or a
    // y or z neighbour, but for the one beyond the row's end.  What a lane adds for crossing a block's side is
    // the uniform difference of two offsets under the lane's mask (first, last cell of the row; first, last
    // row): masks stay in vector registers, and no choice between scalars needs moves into them.
    typename W::word s[27];
    auto mask = [](bool m) { uint32_t v = m ? ~0u : 0u; asm("" : "+v"(v)); return v; };
    const bool r0 = ly == 0, r15 = ly == BS - 1, x0 = lx == 0, x15 = lx == BS - 1;
    const uint32_t mrow[3] = {mask(r15), 0u, mask(r0)};                             // by cy + 1: the row crosses
    const uint32_t mxl[3][2] = {{mask(x0 && !r15), mask(x0 && r15)}, {mask(x0), 0u}, {mask(x0 && !r0), mask(x0 && r0)}};
    const uint32_t mxr[3][2] = {{mask(x15 && !r15), mask(x15 && r15)}, {mask(x15), 0u}, {mask(x15 && !r0), mask(x15 && r0)}};
    auto gather = [&](auto rules) {
        for_dirs([&](auto rc) {
            constexpr int C = decltype(rc)::value;
            if constexpr (C < 9) {
                constexpr int cy = C % 3 - 1, cz = C / 3 - 1;
                const int sz = z - cz;
                const int dz = sz < 0 ? -1 : (sz >= BS ? 1 : 0);
                auto boff = [&](int dx, int dy) -> uint32_t { return R.off[(dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)]; };
                const uint32_t zs = (uint32_t)(sz & (BS - 1)) * (BS2 * es);
                [[maybe_unused]] const __amdgpu_buffer_rsrc_t fz = buf_layer<WIDE>(a.fin, R, dz, blk);   // (WIDE, cz != 0)
                const uint32_t in_row = (uint32_t)((ly - cy) & (BS - 1)) * (BS * es) + (uint32_t)lx * es;
                const uint32_t c0 = boff(0, 0);
                // (a row's end is 16 cells from its start: - es becomes + 15 es, and the other way round)
                const uint32_t l0 = boff(-1, 0) - c0 + BS * es, h0 = boff(1, 0) - c0 - BS * es;
                uint32_t here = in_row + c0, left, right;
                if constexpr (cy == 0) {
                    left = here + (mxl[1][0] & l0) - es;
                    right = here + (mxr[1][0] & h0) + es;
                } else {
                    const uint32_t c1 = boff(0, -cy), l1 = boff(-1, -cy) - c1 + BS * es, h1 = boff(1, -cy) - c1 - BS * es;
                    here += mrow[cy + 1] & (c1 - c0);
                    left = here + ((mxl[cy + 1][0] & l0) | (mxl[cy + 1][1] & l1)) - es;
                    right = here + ((mxr[cy + 1][0] & h0) | (mxr[cy + 1][1] & h1)) + es;
                }
                for_dirs([&](auto xc) {
                    constexpr int cx = decltype(xc)::value - 1;
                    if constexpr (cx < 2) {
                        constexpr int K = 3 * C + cx + 1;
                        const uint32_t o = cx == 0 ? here : cx > 0 ? left : right;
                        if constexpr (decltype(rules)::value) {
                            // (whole offsets: a difference of slots would wrap below zero)
                            uint32_t w = o + ((uint32_t)K * slot + zs);
                            if constexpr (cy != 0 || cz != 0) {
                                int j;
                                const bool face = two_row_rule<K>(fc, j);
                                w = face ? own + (uint32_t)j * slot : w;
                            }
                            w = (c.lmask >> K) & 1u ? own + (uint32_t)dopp(K) * slot : w;
                            if constexpr (cx < 0) w = outlet ? own + (uint32_t)K * slot : w;
                            if constexpr (WIDE && cz != 0) {
                                int j;
                                const bool ownp = two_row_rule<K>(fc, j) || ((c.lmask >> K) & 1u) || (cx < 0 && outlet);
                                if (ownp) s[K] = W::ld(fin, w, 0);
                                else s[K] = W::ld(fz, w, 0);
                            } else {
                                s[K] = W::ld(fin, w, 0);
                            }
                        } else {
                            if constexpr (WIDE && cz != 0) s[K] = W::ld(fz, o, (uint32_t)K * slot + zs);
                            else s[K] = W::ld(fin, o, (uint32_t)K * slot + zs);
                        }
                    }
                });
            }
        });
    };
    if (flags & (BF_EDGE | BF_SOLID)) gather(std::true_type{});
    else gather(std::false_type{});

    CellRates<T> q{};
    q.forced = (flags & TR_FORCED) != 0;
    q.Fx = T(R.F[0]); q.Fy = T(R.F[1]); q.Fz = T(R.F[2]);
    q.omega1 = es == 8 ? T(R.omega1_d) : T(R.omega1);
    q.omega4_diag = es == 8 ? T(R.omega4d_d) : T(R.omega4d);
    if constexpr (WALE) {
        c.per0 = (flags & TR_PER_X) != 0; c.per1 = (flags & TR_PER_Y) != 0; c.per2 = (flags & TR_PER_Z) != 0;
        c.ext0 = R.ext[0]; c.ext1 = R.ext[1]; c.ext2 = R.ext[2];
        cell_rates<T>(wale_of<T>(a, c), T(R.tau), T(R.amr_scale), T(a.cp.nu_sgs_bg), a.cp.adaptive_omega4, T(a.cp.lambda),
                      T(a.cp.omega_4), q.omega1, q.omega4_diag);
    }
    T f[27];
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        f[K] = W::dec(s[K], wgt<T>(K));
    });
    if (inlet) {
        const float u_in = R.u_in;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if constexpr (dcx(K) > 0) f[K] = boundary_value<K, T>(SRC_INLET, a, c, u_in, a.step(), [&](auto) { return T(0); });
        });
    }
    CollParams cp = a.cp;
    if (!POS && cp.limiter == 2) cp.limiter = 0;   // (never: the launch's choice; leaves its branch out)
    T rho_o, ux, uy, uz;
    collide_cell<T, UNIT, false, false, es == 2>(f, q, cp, rho_o, ux, uy, uz);

    const uint32_t hc = DITH ? round_cell(round_key(a.step()), c.own - R.cell0) : 0u;
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        s[K] = W::template enc<K, DITH>(f[K], DITH ? round_bits(hc, K) : 0u);
    });
    const __amdgpu_buffer_rsrc_t fo = buf_at((char*)a.fout + (size_t)R.base * blk);
    if (live) {
        auto store = [&](auto aux) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                W::template st<decltype(aux)::value>(s[K], fo, own, (uint32_t)K * slot);
            });
        };
        if (a.two_keep) store(std::integral_constant<int, TWO_ST_KEEP>{});
        else store(std::integral_constant<int, TWO_ST_STREAM>{});
        if constexpr (WALE) {
            T* vo = (T*)a.vel_out;
            vo[c.own] = ux; vo[(size_t)a.ncell + c.own] = uy; vo[2 * (size_t)a.ncell + c.own] = uz;
        }
    }
    if (want_force) {
        // momentum exchange of the links toward solid cells (halfway bounce-back), of the stored populations
        double F0 = 0.0, F1 = 0.0, F2 = 0.0;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if (live && ((c.lmask >> dopp(K)) & 1u)) {
                const double m = 2.0 * ((double)W::dec(s[K], wgt<T>(K)) - (double)wgt<T>(K));
                F0 += m * dcx(K); F1 += m * dcy(K); F2 += m * dcz(K);
            }
        });
        const float fs = R.force_scale;
        wg_sum3(F0 * fs, F1 * fs, F2 * fs, a.fpart, b * PLANES + (uint32_t)z);
    }
}

// Dynamic LDS that no kernel uses, as TWO_HOLD_LDS: two workgroups (eight waves) on a CU where an FP64 level streams
// through the caches.  Sphere boxes 192 x 160 x 160 418 us per step, 404 with three workgroups, 384 with two;
// 160 x 128 x 128 with the interpolated wall 250, 228, 225 us.  With WALE it costs (480, 488, 515 us).
constexpr uint32_t ONE_HOLD_LDS = 70000;

template <class SP>
static void launch_one_sp(bool wale, const StepArgs& r, hipStream_t stream, bool wide = false) {
    const dim3 g(r.n_items);
    auto go = [&](auto unit, auto w, auto dith) {
        constexpr bool U = decltype(unit)::value, W = decltype(w)::value, D = decltype(dith)::value;
        const uint32_t hold = sizeof(typename SP::T) == 8 && !W && !r.two_keep ? ONE_HOLD_LDS : 0u;
        if constexpr (sizeof(typename SP::T) == 8) {
            if (wide && r.cp.limiter == 2) {
                hipLaunchKernelGGL((k_step_one<SP, U, W, true, D, true>), g, dim3(WG), hold, stream, r);
                return;
            }
            if (wide) {
                hipLaunchKernelGGL((k_step_one<SP, U, W, false, D, true>), g, dim3(WG), hold, stream, r);
                return;
            }
        }
        if (r.cp.limiter == 2) hipLaunchKernelGGL((k_step_one<SP, U, W, true, D>), g, dim3(WG), hold, stream, r);
        else hipLaunchKernelGGL((k_step_one<SP, U, W, false, D>), g, dim3(WG), hold, stream, r);
    };
    auto walef = [&](auto unit, auto dith) {
        if (wale) go(unit, std::true_type{}, dith);
        else go(unit, std::false_type{}, dith);
    };
    auto rates = [&](auto dith) {
        if (r.cp.unit) walef(std::true_type{}, dith);
        else walef(std::false_type{}, dith);
    };
    if constexpr (SP::dithered) {
        if (r.cp.dither) rates(std::true_type{});
        else rates(std::false_type{});
    } else {
        rates(std::false_type{});
    }
}

}  // namespace oal
