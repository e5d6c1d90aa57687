// The FP64 step kernel of the AB pattern, one cell per lane (oal_one_f64.hip).
//
// One workgroup of 256 lanes steps one 16 x 16 plane of a block; one launch covers the blocks of every kind
// but a few (build_lists), from the records and with the rules of the two-cells-per-lane kernel: the 27
// sources of a cell are loaded together, each from its source cell or, across a face, at a solid link or on
// the outlet, from the own cell's population that the rule names; the inlet replaces values afterwards.
//
// Bound and shape.  27 doubles are 54 registers: with the unit-rate collision and without the positivity
// limiter's branch a lane needs 118 (124 with WALE), so four waves share a SIMD and 64^3 cells are all resident
// at once.  Bound: HBM (192 x 160 x 160: 5.1 TB/s of 432 bytes per cell), at 64^3 the memory-side cache and one
// wave's latency.  Measured against a kernel per kind of block, two waves per SIMD, on two streams: 64^3
// periodic 30.5 -> 18.5 us per step; sphere boxes 192 x 160 x 160 472 -> 416 us, with WALE 568 -> 479 us,
// 100 x 60 x 44 with WALE 94 -> 28.5 us, 48 x 32 x 32 13.1 -> 7.3 us.
#pragma once

#include "oal_step_two.h"

namespace oal {

// POS: with the positivity limiter, whose 54 equilibria cost the other form half its occupancy
template <bool UNIT, bool WALE, bool POS>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(POS ? 2 : UNIT ? 4 : 3)))
k_step_one(const StepArgs a) {
    using T = double;
    constexpr uint32_t es = sizeof(T), slot = BS3 * es, blk = 27u * slot;
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
    // y or z neighbour, but for the one beyond the row's end
    T f[27];
    auto load = [&](uint32_t o, uint32_t s) -> T {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(fin, (int)o, (int)s, 0));
    };
    auto gather = [&](auto rules) {
        for_dirs([&](auto rc) {
            constexpr int C = decltype(rc)::value;
            if constexpr (C < 9) {
                constexpr int cy = C % 3 - 1, cz = C / 3 - 1;
                const int sz = z - cz;
                const int dz = sz < 0 ? -1 : (sz >= BS ? 1 : 0);
                auto boff = [&](int dx, int dy) -> uint32_t { return R.off[(dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)]; };
                const uint32_t zs = (uint32_t)(sz & (BS - 1)) * (BS2 * es), r = (uint32_t)((ly - cy) & (BS - 1)) * (BS * es);
                const uint32_t c0 = boff(0, 0), m0 = boff(-1, 0), p0 = boff(1, 0);
                uint32_t oc = c0, om = m0, op = p0;
                if constexpr (cy != 0) {
                    const bool cross = cy > 0 ? ly == 0 : ly == BS - 1;
                    const uint32_t c1 = boff(0, -cy), m1 = boff(-1, -cy), p1 = boff(1, -cy);
                    oc = cross ? c1 : c0;
                    om = cross ? m1 : m0;
                    op = cross ? p1 : p0;
                }
                const uint32_t here = oc + r + (uint32_t)lx * es;
                const uint32_t left = lx == 0 ? om + r + (BS - 1) * es : here - es;
                const uint32_t right = lx == BS - 1 ? op + r : here + es;
                for_dirs([&](auto xc) {
                    constexpr int cx = decltype(xc)::value - 1;
                    if constexpr (cx < 2) {
                        constexpr int K = 3 * C + cx + 1;
                        const uint32_t o = (cx == 0 ? here : cx > 0 ? left : right) + zs;
                        if constexpr (decltype(rules)::value) {
                            // (whole offsets: a difference of slots would wrap below zero)
                            uint32_t w = o + (uint32_t)K * slot;
                            if constexpr (cy != 0 || cz != 0) {
                                int j;
                                const bool face = two_row_rule<K>(fc, j);
                                w = face ? own + (uint32_t)j * slot : w;
                            }
                            w = (c.lmask >> K) & 1u ? own + (uint32_t)dopp(K) * slot : w;
                            if constexpr (cx < 0) w = outlet ? own + (uint32_t)K * slot : w;
                            f[K] = load(w, 0);
                        } else {
                            f[K] = load(o, (uint32_t)K * slot);
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
    q.omega1 = R.omega1_d;
    q.omega4_diag = R.omega4d_d;
    if constexpr (WALE) {
        c.per0 = (flags & TR_PER_X) != 0; c.per1 = (flags & TR_PER_Y) != 0; c.per2 = (flags & TR_PER_Z) != 0;
        c.ext0 = R.ext[0]; c.ext1 = R.ext[1]; c.ext2 = R.ext[2];
        cell_rates<T>(wale_of<T>(a, c), T(R.tau), T(R.amr_scale), T(a.cp.nu_sgs_bg), a.cp.adaptive_omega4, T(a.cp.lambda),
                      T(a.cp.omega_4), q.omega1, q.omega4_diag);
    }
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
    collide_cell<T, UNIT>(f, q, cp, rho_o, ux, uy, uz);

    const __amdgpu_buffer_rsrc_t fo = buf_at((char*)a.fout + (size_t)R.base * blk);
    if (live) {
        auto store = [&](auto aux) {
            for_dirs([&](auto kc) {
                constexpr int K = decltype(kc)::value;
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f[K]), fo, (int)own, (int)((uint32_t)K * slot),
                                                      decltype(aux)::value);
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
        // momentum exchange of the links toward solid cells (halfway bounce-back)
        T F0 = 0.0, F1 = 0.0, F2 = 0.0;
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if (live && ((c.lmask >> dopp(K)) & 1u)) {
                const T m = 2.0 * (f[K] - wgt<T>(K));
                F0 += m * dcx(K); F1 += m * dcy(K); F2 += m * dcz(K);
            }
        });
        const float fs = R.force_scale;
        wg_sum3(F0 * fs, F1 * fs, F2 * fs, a.fpart, b * PLANES + (uint32_t)z);
    }
}

}  // namespace oal
