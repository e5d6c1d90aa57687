// Kernels of liboal for gfx950 other than the stream-collide step (oal_step.h): initialisation,
// layout conversion, macroscopic output, FP64 reductions, the stability guard and the bandwidth probe,
// and the storage dispatch of the step launches.
#include <hip/hip_runtime.h>

#include "oal_kernels.h"

namespace oal {

hipError_t launch_step(int storage, int stream_mode, bool wale, const StepArgs& a, hipStream_t stream, hipStream_t side,
                       hipEvent_t bulk0, hipEvent_t bulk1) {
    switch (storage) {
        case 0: return launch_step_f32(stream_mode, wale, a, stream, side, bulk0, bulk1);
        case 1: return launch_step_f64(stream_mode, wale, a, stream, side, bulk0, bulk1);
        case 2: return launch_step_f16s(stream_mode, wale, a, stream, side, bulk0, bulk1);
        case 3: return launch_step_bf16s(stream_mode, wale, a, stream, side, bulk0, bulk1);
        default: return hipErrorInvalidValue;
    }
}

void launch_two(int storage, bool wale, int extra, const TwoRec* rec, uint32_t n, hipStream_t stream, const StepArgs& a) {
    if (!n) return;
    StepArgs r = a;
    r.rec = rec;
    r.n_items = n * PLANES;
    switch (storage) {
        case 0: launch_two_f32(wale, extra, r, stream); break;
        case 2: launch_two_f16s(wale, extra, r, stream); break;
        default: launch_two_bf16s(wale, extra, r, stream); break;
    }
}

void launch_one(int storage, bool wale, bool wide, const TwoRec* rec, uint32_t n, hipStream_t stream, const StepArgs& a) {
    if (!n) return;
    StepArgs r = a;
    r.rec = rec;
    r.n_items = n * PLANES;
    switch (storage) {
        case 0: launch_one_f32(wale, r, stream); break;
        case 1: launch_one_f64(wale, wide, r, stream); break;
        case 2: launch_one_f16s(wale, r, stream); break;
        default: launch_one_bf16s(wale, r, stream); break;
    }
}

// ------------------------------------------------------------------------------------------------
// Bandwidth probe: a streaming 16-byte copy, the measured HBM ceiling of the roofline
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(WG) k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * WG;
    for (size_t i = (size_t)blockIdx.x * WG + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy16(const void* src, void* dst, size_t bytes, hipStream_t s) {
    const size_t n = bytes / 16;
    const unsigned grid = (unsigned)((n + WG - 1) / WG < 65536 * 8 ? (n + WG - 1) / WG : 65536 * 8);
    hipLaunchKernelGGL(k_copy16, dim3(grid), dim3(WG), 0, s, (const uint4*)src, (uint4*)dst, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// Initialisation: init_eq! (src/main.jl:546-572), per-cell or uniform (rho, u)
// ------------------------------------------------------------------------------------------------
template <class SP>
__global__ void __launch_bounds__(WG) k_init_eq(typename SP::st* f, uint32_t ncell, uint32_t nhost, const double* rho,
                                                const double* u, double rho0, double ux0, double uy0, double uz0,
                                                int permute, typename SP::T* vel) {
    using T = typename SP::T;
    const uint32_t cidx = blockIdx.x * WG + threadIdx.x;
    if (cidx >= ncell) return;
    // host fields cover the first nhost cells; the rest (ghost blocks of a refined level) take (rho0, u0)
    const bool h = cidx < nhost;
    const T r = rho && h ? T(rho[cidx]) : T(rho0);
    const T ux = u && h ? T(u[cidx]) : T(ux0);
    const T uy = u && h ? T(u[nhost + cidx]) : T(uy0);
    const T uz = u && h ? T(u[2 * (size_t)nhost + cidx]) : T(uz0);
    const T cs2 = T(1) / T(3);
    const T cs4 = cs2 * cs2;
    const T usq = ux * ux + uy * uy + uz * uz;
    const T inv_cs2 = T(1) / cs2, inv_2cs4 = T(0.5) / cs4, inv_2cs2 = T(0.5) / cs2;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const T cu = T(dcx(k)) * ux + T(dcy(k)) * uy + T(dcz(k)) * uz;
        const T feq = r * wgt<T>(k) * (T(1) + inv_cs2 * cu + inv_2cs4 * cu * cu - inv_2cs2 * usq);
        SP::sto(f + pop_index(cidx, permute ? 26 - k : k), feq, wgt<T>(k));
    }
    if (vel) { vel[cidx] = ux; vel[ncell + cidx] = uy; vel[2 * (size_t)ncell + cidx] = uz; }
}

template <class SP>
static hipError_t init_sp(void* f, uint32_t ncell, uint32_t nhost, const double* rho, const double* u, double rho0,
                          double ux0, double uy0, double uz0, int permute, void* vel, hipStream_t s) {
    hipLaunchKernelGGL((k_init_eq<SP>), dim3((ncell + WG - 1) / WG), dim3(WG), 0, s, (typename SP::st*)f, ncell, nhost, rho,
                       u, rho0, ux0, uy0, uz0, permute, (typename SP::T*)vel);
    return hipGetLastError();
}

hipError_t launch_init_eq(int storage, void* f, uint32_t ncell, uint32_t nhost, const double* rho, const double* u,
                          double rho0, double ux0, double uy0, double uz0, int permute, void* vel, hipStream_t s) {
    switch (storage) {
        case 0: return init_sp<StF32>(f, ncell, nhost, rho, u, rho0, ux0, uy0, uz0, permute, vel, s);
        case 1: return init_sp<StF64>(f, ncell, nhost, rho, u, rho0, ux0, uy0, uz0, permute, vel, s);
        case 2: return init_sp<StF16S>(f, ncell, nhost, rho, u, rho0, ux0, uy0, uz0, permute, vel, s);
        case 3: return init_sp<StBF16S>(f, ncell, nhost, rho, u, rho0, ux0, uy0, uz0, permute, vel, s);
        default: return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------------------------------------------------
// Layout conversion between host populations (unshifted f32/f64) and the storage form
// ------------------------------------------------------------------------------------------------
template <class SP, class H>
__global__ void __launch_bounds__(WG) k_convert_in(typename SP::st* f, const H* src, uint32_t ncell, uint32_t nhost,
                                                   int permute) {
    using T = typename SP::T;
    const uint32_t cidx = blockIdx.x * WG + threadIdx.x;
    const int k = blockIdx.y;
    if (cidx >= nhost) return;
    SP::sto(f + pop_index(cidx, permute ? 26 - k : k), T(src[(size_t)k * nhost + cidx]), wgt<T>(k));
}

template <class SP, class H>
__global__ void __launch_bounds__(WG) k_convert_out(const typename SP::st* f, H* dst, uint32_t ncell, uint32_t nhost,
                                                    int permute) {
    using T = typename SP::T;
    const uint32_t cidx = blockIdx.x * WG + threadIdx.x;
    const int k = blockIdx.y;
    if (cidx >= nhost) return;
    dst[(size_t)k * nhost + cidx] = H(SP::ld(f + pop_index(cidx, permute ? 26 - k : k), wgt<T>(k)));
}

template <class SP>
static hipError_t conv_in_sp(void* f, const void* src, int dt, uint32_t ncell, uint32_t nhost, int permute, hipStream_t s) {
    dim3 grid((nhost + WG - 1) / WG, 27);
    if (dt == 0) hipLaunchKernelGGL((k_convert_in<SP, float>), grid, dim3(WG), 0, s, (typename SP::st*)f, (const float*)src, ncell, nhost, permute);
    else hipLaunchKernelGGL((k_convert_in<SP, double>), grid, dim3(WG), 0, s, (typename SP::st*)f, (const double*)src, ncell, nhost, permute);
    return hipGetLastError();
}
template <class SP>
static hipError_t conv_out_sp(const void* f, void* dst, int dt, uint32_t ncell, uint32_t nhost, int permute, hipStream_t s) {
    dim3 grid((nhost + WG - 1) / WG, 27);
    if (dt == 0) hipLaunchKernelGGL((k_convert_out<SP, float>), grid, dim3(WG), 0, s, (const typename SP::st*)f, (float*)dst, ncell, nhost, permute);
    else hipLaunchKernelGGL((k_convert_out<SP, double>), grid, dim3(WG), 0, s, (const typename SP::st*)f, (double*)dst, ncell, nhost, permute);
    return hipGetLastError();
}

hipError_t launch_convert_in(int storage, void* f, const void* src, int dt, uint32_t ncell, uint32_t nhost, int permute,
                             hipStream_t s) {
    switch (storage) {
        case 0: return conv_in_sp<StF32>(f, src, dt, ncell, nhost, permute, s);
        case 1: return conv_in_sp<StF64>(f, src, dt, ncell, nhost, permute, s);
        case 2: return conv_in_sp<StF16S>(f, src, dt, ncell, nhost, permute, s);
        case 3: return conv_in_sp<StBF16S>(f, src, dt, ncell, nhost, permute, s);
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_convert_out(int storage, const void* f, void* dst, int dt, uint32_t ncell, uint32_t nhost, int permute,
                             hipStream_t s) {
    switch (storage) {
        case 0: return conv_out_sp<StF32>(f, dst, dt, ncell, nhost, permute, s);
        case 1: return conv_out_sp<StF64>(f, dst, dt, ncell, nhost, permute, s);
        case 2: return conv_out_sp<StF16S>(f, dst, dt, ncell, nhost, permute, s);
        case 3: return conv_out_sp<StBF16S>(f, dst, dt, ncell, nhost, permute, s);
        default: return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------------------------------------------------
// Macroscopic output in FP64: rho = 1 + sum (f_k - w_k), u = sum c_k (f_k - w_k) / rho
// ------------------------------------------------------------------------------------------------
template <class SP>
__global__ void __launch_bounds__(WG) k_macro(const typename SP::st* f, double* rho, double* u, uint32_t ncell,
                                              uint32_t nhost, int permute, typename SP::T* vel) {
    using T = typename SP::T;
    const uint32_t cidx = blockIdx.x * WG + threadIdx.x;
    if (cidx >= nhost) return;
    double dr = 0.0, jx = 0.0, jy = 0.0, jz = 0.0;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const double s = (double)SP::ld(f + pop_index(cidx, permute ? 26 - k : k), wgt<T>(k)) - (double)wgt<T>(k);
        dr += s; jx += s * dcx(k); jy += s * dcy(k); jz += s * dcz(k);
    }
    const double r = 1.0 + dr;
    if (rho) rho[cidx] = r;
    if (u) { u[cidx] = jx / r; u[nhost + cidx] = jy / r; u[2 * (size_t)nhost + cidx] = jz / r; }
    if (vel) { vel[cidx] = T(jx / r); vel[ncell + cidx] = T(jy / r); vel[2 * (size_t)ncell + cidx] = T(jz / r); }
}

template <class SP>
static hipError_t macro_sp(const void* f, double* rho, double* u, uint32_t ncell, uint32_t nhost, int permute, void* vel,
                          hipStream_t s) {
    hipLaunchKernelGGL((k_macro<SP>), dim3((nhost + WG - 1) / WG), dim3(WG), 0, s, (const typename SP::st*)f, rho, u, ncell,
                       nhost, permute, (typename SP::T*)vel);
    return hipGetLastError();
}

hipError_t launch_macro(int storage, const void* f, double* rho, double* u, uint32_t ncell, uint32_t nhost, int permute,
                        void* vel, hipStream_t s) {
    switch (storage) {
        case 0: return macro_sp<StF32>(f, rho, u, ncell, nhost, permute, vel, s);
        case 1: return macro_sp<StF64>(f, rho, u, ncell, nhost, permute, vel, s);
        case 2: return macro_sp<StF16S>(f, rho, u, ncell, nhost, permute, vel, s);
        case 3: return macro_sp<StBF16S>(f, rho, u, ncell, nhost, permute, vel, s);
        default: return hipErrorInvalidValue;
    }
}

// The same for a range of the caller's cells [c0, c0 + n), written as [4][n] (rho, ux, uy, uz) into pinned
// host memory over the link; map: the library cell of each caller cell (levels in 8^3 blocks), or null.
template <class SP>
__global__ void __launch_bounds__(WG) k_macro_out(const typename SP::st* f, const uint32_t* map, uint32_t c0, uint32_t n,
                                                  int permute, double* out) {
    using T = typename SP::T;
    const uint32_t i = blockIdx.x * WG + threadIdx.x;
    if (i >= n) return;
    const uint32_t cell = map ? map[c0 + i] : c0 + i;
    double dr = 0.0, jx = 0.0, jy = 0.0, jz = 0.0;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const double s = (double)SP::ld(f + pop_index(cell, permute ? 26 - k : k), wgt<T>(k)) - (double)wgt<T>(k);
        dr += s; jx += s * dcx(k); jy += s * dcy(k); jz += s * dcz(k);
    }
    const double r = 1.0 + dr;
    out[i] = r;
    out[n + i] = jx / r;
    out[2 * (size_t)n + i] = jy / r;
    out[3 * (size_t)n + i] = jz / r;
}

hipError_t launch_macro_out(int storage, const void* f, const uint32_t* map, uint32_t c0, uint32_t n, int permute, double* out,
                            hipStream_t s) {
    const dim3 g((n + WG - 1) / WG);
    switch (storage) {
        case 0: hipLaunchKernelGGL((k_macro_out<StF32>), g, dim3(WG), 0, s, (const float*)f, map, c0, n, permute, out); break;
        case 1: hipLaunchKernelGGL((k_macro_out<StF64>), g, dim3(WG), 0, s, (const double*)f, map, c0, n, permute, out); break;
        case 2: hipLaunchKernelGGL((k_macro_out<StF16S>), g, dim3(WG), 0, s, (const _Float16*)f, map, c0, n, permute, out); break;
        case 3: hipLaunchKernelGGL((k_macro_out<StBF16S>), g, dim3(WG), 0, s, (const uint16_t*)f, map, c0, n, permute, out); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// AA pattern: outlet side buffer from a state in stored form (after upload / initialisation), the
// copy the even step makes of every outlet-face population with cx = -1
// ------------------------------------------------------------------------------------------------
template <class SP>
__global__ void __launch_bounds__(WG) k_aa_outlet_prep(const StepArgs a) {
    using st = typename SP::st;
    const uint32_t b = blockIdx.x;
    const int32_t os = a.oslot[b];
    if (os < 0) return;
    const DevDomain* dm = a.doms + a.bdom[b];
    const int lx = dm->ext[0] - 1 - a.borg[3 * b];   // the outlet plane of this block
    const int ly = threadIdx.x & (BS - 1), z = threadIdx.x >> 4;
    const uint32_t own = b * BS3 + (uint32_t)z * BS2 + (uint32_t)ly * BS + (uint32_t)lx;
    const st* f = (const st*)a.fin;
    st* o = (st*)a.obuf;
#pragma unroll
    for (int q = 0; q < 9; ++q) o[((size_t)os * 9 + q) * BS2 + ly * BS + z] = f[pop_index(own, 26 - 3 * q)];
}

hipError_t launch_aa_outlet_prep(int storage, const StepArgs& a, hipStream_t s) {
    switch (storage) {
        case 0: hipLaunchKernelGGL((k_aa_outlet_prep<StF32>), dim3(a.nb), dim3(WG), 0, s, a); break;
        case 1: hipLaunchKernelGGL((k_aa_outlet_prep<StF64>), dim3(a.nb), dim3(WG), 0, s, a); break;
        case 2: hipLaunchKernelGGL((k_aa_outlet_prep<StF16S>), dim3(a.nb), dim3(WG), 0, s, a); break;
        case 3: hipLaunchKernelGGL((k_aa_outlet_prep<StBF16S>), dim3(a.nb), dim3(WG), 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// FP64 mass and momentum partials, one workgroup per block (16 cells per lane); then a per-domain
// reduction over contiguous item ranges in a fixed order, so results are bit-reproducible.
// ------------------------------------------------------------------------------------------------
template <class SP>
__global__ void __launch_bounds__(WG) k_mass(const typename SP::st* f, const uint8_t* solid, const int32_t* borg,
                                             const int32_t* bdom, const uint32_t* bflags, const DevDomain* doms,
                                             int permute, double* part) {
    using T = typename SP::T;
    const uint32_t b = blockIdx.x;
    if (bflags[b] & BF_INACTIVE) {   // covered or ghost block of a refined level: counted on another level
        if (threadIdx.x < 4) part[(size_t)b * 4 + threadIdx.x] = 0.0;
        return;
    }
    const DevDomain* dm = doms + bdom[b];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int z = 0; z < BS; ++z) {
        const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
        const uint32_t cidx = b * BS3 + z * BS2 + ly * BS + lx;
        const bool inside = borg[3 * b] + lx < dm->ext[0] && borg[3 * b + 1] + ly < dm->ext[1] && borg[3 * b + 2] + z < dm->ext[2];
        if (!inside || (solid && solid[cidx])) continue;
        double dr = 0.0, jx = 0.0, jy = 0.0, jz = 0.0;
#pragma unroll
        for (int k = 0; k < 27; ++k) {
            const double s = (double)SP::ld(f + pop_index(cidx, permute ? 26 - k : k), wgt<T>(k)) - (double)wgt<T>(k);
            dr += s; jx += s * dcx(k); jy += s * dcy(k); jz += s * dcz(k);
        }
        acc[0] += 1.0 + dr; acc[1] += jx; acc[2] += jy; acc[3] += jz;
    }
    __shared__ double red[4][WG / 64];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        double v = acc[q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) s += red[threadIdx.x][w];
        part[(size_t)b * 4 + threadIdx.x] = s;
    }
}

hipError_t launch_mass(int storage, const void* f, const uint8_t* solid, const int32_t* borg, const int32_t* bdom,
                       const uint32_t* bflags, const DevDomain* doms, uint32_t nb, int permute, double* part, hipStream_t s) {
    switch (storage) {
        case 0: hipLaunchKernelGGL((k_mass<StF32>), dim3(nb), dim3(WG), 0, s, (const float*)f, solid, borg, bdom, bflags, doms, permute, part); break;
        case 1: hipLaunchKernelGGL((k_mass<StF64>), dim3(nb), dim3(WG), 0, s, (const double*)f, solid, borg, bdom, bflags, doms, permute, part); break;
        case 2: hipLaunchKernelGGL((k_mass<StF16S>), dim3(nb), dim3(WG), 0, s, (const _Float16*)f, solid, borg, bdom, bflags, doms, permute, part); break;
        case 3: hipLaunchKernelGGL((k_mass<StBF16S>), dim3(nb), dim3(WG), 0, s, (const uint16_t*)f, solid, borg, bdom, bflags, doms, permute, part); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// one workgroup per domain: lanes stride over the domain's items, then a fixed-order tree
__global__ void __launch_bounds__(WG) k_reduce(const ReduceArgs r) {
    const int d = blockIdx.x;
    const int i0 = r.dom_item0[d], i1 = r.dom_item0[d + 1];
    __shared__ double sh[4][WG];
    for (int q = 0; q < 4; ++q) {
        double s = 0.0;
        if (q < r.width)
            for (int i = i0 + (int)threadIdx.x; i < i1; i += WG) s += r.part[(size_t)i * 4 + q];
        sh[q][threadIdx.x] = s;
    }
    __syncthreads();
    for (int w = WG / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int q = 0; q < 4; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 4) r.out[(size_t)d * 4 + threadIdx.x] = sh[threadIdx.x][0];
}

hipError_t launch_reduce(const ReduceArgs& r, hipStream_t s) {
    hipLaunchKernelGGL(k_reduce, dim3(r.n_domains), dim3(WG), 0, s, r);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// Stability guard: rho <= rho_min, |u| >= u_max or a non-finite population in a fluid cell
// (src/octree_q19/src/io_run.jl:31-65)
// ------------------------------------------------------------------------------------------------
template <class SP>
__global__ void __launch_bounds__(WG) k_guard(const typename SP::st* f, const uint8_t* solid, const int32_t* borg,
                                              const int32_t* bdom, const uint32_t* bflags, const DevDomain* doms,
                                              float rho_min, float u_max, unsigned long long* count) {
    using T = typename SP::T;
    const uint32_t b = blockIdx.x;
    if (bflags[b] & BF_INACTIVE) return;
    const DevDomain* dm = doms + bdom[b];
    unsigned bad = 0;
    for (int z = 0; z < BS; ++z) {
        const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
        const uint32_t cidx = b * BS3 + z * BS2 + ly * BS + lx;
        const bool inside = borg[3 * b] + lx < dm->ext[0] && borg[3 * b + 1] + ly < dm->ext[1] && borg[3 * b + 2] + z < dm->ext[2];
        if (!inside || (solid && solid[cidx])) continue;
        float r = 0.0f, jx = 0.0f, jy = 0.0f, jz = 0.0f;
        bool finite = true;
#pragma unroll
        for (int k = 0; k < 27; ++k) {
            const float v = (float)SP::ld(f + pop_index(cidx, k), wgt<T>(k));
            finite = finite && isfinite(v);
            r += v; jx += v * dcx(k); jy += v * dcy(k); jz += v * dcz(k);
        }
        const float u2 = (jx * jx + jy * jy + jz * jz) / (r * r);
        if (!finite || !(r > rho_min) || !(u2 < u_max * u_max)) ++bad;
    }
    for (int off = 32; off > 0; off >>= 1) bad += __shfl_xor(bad, off, 64);
    if ((threadIdx.x & 63) == 0 && bad) atomicAdd(count, (unsigned long long)bad);
}

hipError_t launch_guard(int storage, const void* f, const uint8_t* solid, const int32_t* borg, const int32_t* bdom,
                        const uint32_t* bflags, const DevDomain* doms, uint32_t nb, float rho_min, float u_max,
                        unsigned long long* count, hipStream_t s) {
    switch (storage) {
        case 0: hipLaunchKernelGGL((k_guard<StF32>), dim3(nb), dim3(WG), 0, s, (const float*)f, solid, borg, bdom, bflags, doms, rho_min, u_max, count); break;
        case 1: hipLaunchKernelGGL((k_guard<StF64>), dim3(nb), dim3(WG), 0, s, (const double*)f, solid, borg, bdom, bflags, doms, rho_min, u_max, count); break;
        case 2: hipLaunchKernelGGL((k_guard<StF16S>), dim3(nb), dim3(WG), 0, s, (const _Float16*)f, solid, borg, bdom, bflags, doms, rho_min, u_max, count); break;
        case 3: hipLaunchKernelGGL((k_guard<StBF16S>), dim3(nb), dim3(WG), 0, s, (const uint16_t*)f, solid, borg, bdom, bflags, doms, rho_min, u_max, count); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// Level transfers of a refined plan (the role of the octree's coupling, src/octree_q19/src/coupling.jl:
// 86-233): a written cell receives the stencil-weighted sum of its donors' post-collision populations,
// whose second-order non-equilibrium moments are then set to those of the receiving level: the donors'
// Pi_neq times `scale` (1/(1 - omega) of the sending level and the ratio of the levels' relaxation
// times) times `keep` (1 - omega of the receiving level), through the second-order Hermite term.  All
// other moments of the interpolated state are kept: the cumulant collision's higher-order state
// crosses the interface unchanged (a rebuild from rho, u and Pi_neq alone, as the octree's D3Q19
// regularised collision allows, would impose the polynomial equilibrium's higher moments and make a
// uniform flow change at the interfaces).  A cell whose corrected state has a population below 1e-6
// of its weight takes the equilibrium of its rho and u (kernel.jl:94-100).  Every operation is written
// out in a fixed order: the CPU oracle restates the same sequence and must agree bit for bit.
// ------------------------------------------------------------------------------------------------
// 16-byte vectors of the working type (records of the level transfers)
template <class T> struct Vec16;
template <> struct Vec16<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int n = 4;
};
template <> struct Vec16<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    static constexpr int n = 2;
};

// RAW (16-bit storage, no blend): records of the 27 stored codes padded to 32 (64 bytes), decoded by
// the rebuild; the decoded values are the ones a float record would hold.
constexpr int XFER_RAW_STRIDE = 32;

// gather: one lane per donor, so that a direction's loads run over consecutive cells (donors ascend), all
// 27 in flight; the records leave through LDS as 16-byte pieces in order.  RAW: the stored codes.
template <class SP, bool RAW>
__global__ void __launch_bounds__(WG) k_xfer_gather(const typename SP::st* fnew, const typename SP::st* fold,
                                                    const uint32_t* cells, uint32_t n, typename SP::T w1, typename SP::T* out) {
    using T = typename SP::T;
    constexpr int RW = RAW ? XFER_RAW_STRIDE / 2 : xfer_stride<T>() * (int)sizeof(T) / 4;   // 32-bit words of a record
    constexpr int P = RW / 4;                                                             // its 16-byte pieces
    __shared__ uint4 sh[WG / 64][64][P + 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t i0 = blockIdx.x * WG + (uint32_t)wave * 64u;
    if (i0 >= n) return;
    const uint32_t i = i0 + (uint32_t)lane < n ? i0 + (uint32_t)lane : n - 1;
    const uint32_t e = cells[i];
    const uint32_t c = e & 0x7fffffffu;
    uint32_t w[RW];
#pragma unroll
    for (int k = 0; k < RW; ++k) w[k] = 0;
    if constexpr (RAW) {
        uint32_t h[27];
        for_dirs([&](auto kc) { constexpr int K = decltype(kc)::value; h[K] = SP::ld_raw(fnew + pop_index(c, K)); });
        for_dirs([&](auto kc) { constexpr int K = decltype(kc)::value; w[K / 2] |= h[K] << (16 * (K % 2)); });
    } else {
        const bool blend = fold && !(e >> 31);
        typename SP::raw a[27], b[27];
        for_dirs([&](auto kc) { constexpr int K = decltype(kc)::value; a[K] = SP::ld_raw(fnew + pop_index(c, K)); });
        if (fold) for_dirs([&](auto kc) { constexpr int K = decltype(kc)::value; b[K] = SP::ld_raw(fold + pop_index(c, K)); });
        for_dirs([&](auto kc) {
            constexpr int K = decltype(kc)::value;
            T x = SP::from_raw(a[K], wgt<T>(K));
            if (blend) x = SP::from_raw(b[K], wgt<T>(K)) * (T(1) - w1) + x * w1;
            if constexpr (sizeof(T) == 4) {
                w[K] = __float_as_uint((float)x);
            } else {
                const uint64_t u = (uint64_t)__double_as_longlong((double)x);
                w[2 * K] = (uint32_t)u;
                w[2 * K + 1] = (uint32_t)(u >> 32);
            }
        });
    }
#pragma unroll
    for (int p = 0; p < P; ++p) sh[wave][lane][p] = make_uint4(w[4 * p], w[4 * p + 1], w[4 * p + 2], w[4 * p + 3]);
    wave_sync();
    const uint32_t pieces = (n - i0 < 64u ? n - i0 : 64u) * P;
    uint4* o = reinterpret_cast<uint4*>(out) + (size_t)i0 * P;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const uint32_t t = (uint32_t)(q * 64 + lane);
        if (t < pieces) o[t] = sh[wave][t / P][t % P];
    }
}

// sum of a value over the 16 lanes of a DPP row, as a fixed pairwise tree: lanes l and l xor 1, then
// l xor 2 (quad permutations), then the two quads of each half-row (row_half_mirror: every lane of a
// quad holds its quad's sum, so the mirror pairs the quad sums) and the two half-rows (row_mirror).
// Every lane ends with ((p0 + p1) + (p2 + p3)) + ((p4 + p5) + (p6 + p7)) + ((p8 + ...)) in the same
// bits (addition commutes).
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_get(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <class T>
__device__ __forceinline__ T row_sum(T v) {
    v = v + dpp_get<0xb1>(v);    // quad_perm [1, 0, 3, 2]
    v = v + dpp_get<0x4e>(v);    // quad_perm [2, 3, 0, 1]
    v = v + dpp_get<0x141>(v);   // row_half_mirror
    v = v + dpp_get<0x140>(v);   // row_mirror
    return v;
}
// any lane of the lane's DPP row
__device__ __forceinline__ bool row_any(bool b) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(b);
    return ((m >> (threadIdx.x & 48u)) & 0xffffull) != 0;
}

// moments of an interpolated state: density, velocity and the change of its second-order non-equilibrium
// moments
template <class T>
struct XferMoments {
    T rho, ux, uy, uz, dxx, dyy, dzz, dxy, dxz, dyz, tr, usq;
};
template <class T>
__device__ __forceinline__ XferMoments<T> xfer_moments(const T (&acc)[27], T scale, T keep) {
    T rho = T(0), jx = T(0), jy = T(0), jz = T(0), pxx = T(0), pyy = T(0), pzz = T(0), pxy = T(0), pxz = T(0), pyz = T(0);
    for_dirs([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        constexpr int cx = dcx(K), cy = dcy(K), cz = dcz(K);
        const T v = acc[K];
        rho = rho + v;
        if constexpr (cx > 0) jx = jx + v;
        if constexpr (cx < 0) jx = jx - v;
        if constexpr (cy > 0) jy = jy + v;
        if constexpr (cy < 0) jy = jy - v;
        if constexpr (cz > 0) jz = jz + v;
        if constexpr (cz < 0) jz = jz - v;
        if constexpr (cx != 0) pxx = pxx + v;
        if constexpr (cy != 0) pyy = pyy + v;
        if constexpr (cz != 0) pzz = pzz + v;
        if constexpr (cx * cy > 0) pxy = pxy + v;
        if constexpr (cx * cy < 0) pxy = pxy - v;
        if constexpr (cx * cz > 0) pxz = pxz + v;
        if constexpr (cx * cz < 0) pxz = pxz - v;
        if constexpr (cy * cz > 0) pyz = pyz + v;
        if constexpr (cy * cz < 0) pyz = pyz - v;
    });
    const T ux = jx / rho, uy = jy / rho, uz = jz / rho;
    const T third = T(1.0 / 3.0);
    const T rx = rho * ux, ry = rho * uy;
    const T qxx = (pxx - rho * third) - rx * ux, qyy = (pyy - rho * third) - ry * uy, qzz = (pzz - rho * third) - (rho * uz) * uz;
    const T qxy = pxy - rx * uy, qxz = pxz - rx * uz, qyz = pyz - ry * uz;
    // change of the second-order non-equilibrium moments
    const T sk = scale * keep;
    const T dxx = sk * qxx - qxx, dyy = sk * qyy - qyy, dzz = sk * qzz - qzz;
    const T dxy = sk * qxy - qxy, dxz = sk * qxz - qxz, dyz = sk * qyz - qyz;
    const T tr = (dxx + dyy) + dzz;
    const T usq = (ux * ux + uy * uy) + uz * uz;
    return XferMoments<T>{rho, ux, uy, uz, dxx, dyy, dzz, dxy, dxz, dyz, tr, usq};
}
// one population of the rebuilt cell (a: the interpolated one) and of its equilibrium
template <class T>
__device__ __forceinline__ void xfer_value(const XferMoments<T>& q, T a, T w, T cx, T cy, T cz, T& out, T& eq) {
    const T third = T(1.0 / 3.0);
    const T cac = ((cx * cx * q.dxx + cy * cy * q.dyy) + cz * cz * q.dzz) + T(2) * ((cx * cy * q.dxy + cx * cz * q.dxz) + cy * cz * q.dyz);
    out = a + (w * T(4.5)) * (cac - q.tr * third);
    const T cu = (cx * q.ux + cy * q.uy) + cz * q.uz;
    eq = (w * q.rho) * (((T(1) + T(3) * cu) + T(4.5) * cu * cu) - T(1.5) * q.usq);
}

// rebuild, FP64: 16 lanes (one DPP row) per written cell, lane j summing stencil nodes 4j .. 4j + 3 in node
// order from zero, the 16 partial sums then added as a pairwise tree (row_sum); every lane forms the
// moments, lane j rebuilds and stores directions j and j + 16.  Stencils are cell-major: slot[i][64],
// wt[i][64].
template <class SP>
__global__ void __launch_bounds__(WG) k_xfer_rebuild_row(typename SP::st* f, uint32_t ncell, const uint32_t* tcells, uint32_t n,
                                                     const int32_t* slot, const float* wt, const typename SP::T* m,
                                                     typename SP::T scale, typename SP::T keep, typename SP::T* vel) {
    using T = typename SP::T;
    const uint32_t i = blockIdx.x * (WG / 16) + (threadIdx.x >> 4);
    const int j = (int)(threadIdx.x & 15);
    if (i >= n) return;   // whole rows: the lanes of a live cell stay together
    const int4 s4 = *reinterpret_cast<const int4*>(slot + (size_t)i * 64 + 4 * j);
    const float4 w4 = *reinterpret_cast<const float4*>(wt + (size_t)i * 64 + 4 * j);
    const int32_t sr[4] = {s4.x, s4.y, s4.z, s4.w};
    const T wn[4] = {T(w4.x), T(w4.y), T(w4.z), T(w4.w)};
    T acc[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) acc[k] = T(0);
    {
        using V = typename Vec16<T>::type;
        constexpr int VN = Vec16<T>::n;
        constexpr int ST = xfer_stride<T>();
        V rec[4][ST / VN];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const V* row = reinterpret_cast<const V*>(m + (size_t)(sr[g] >= 0 ? sr[g] : 0) * ST);
#pragma unroll
            for (int q = 0; q < ST / VN; ++q) rec[g][q] = row[q];
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const bool use = sr[g] >= 0;
#pragma unroll
            for (int q = 0; q < ST / VN; ++q)
#pragma unroll
                for (int e = 0; e < VN; ++e)
                    if (q * VN + e < 27) {
                        const T add = acc[q * VN + e] + wn[g] * rec[g][q][e];
                        acc[q * VN + e] = use ? add : acc[q * VN + e];
                    }
        }
    }
#pragma unroll
    for (int k = 0; k < 27; ++k) acc[k] = row_sum(acc[k]);
    const XferMoments<T> m0 = xfer_moments<T>(acc, scale, keep);
    // lane j: directions j and j + 16
    T out[2], eq[2];
    bool bad = false;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = j + 16 * h;
        if (k < 27) {
            const T cx = T(k % 3 - 1), cy = T((k / 3) % 3 - 1), cz = T(k / 9 - 1);
            const T w = wgt_rt<T>(k);
            T a = acc[0];
#pragma unroll
            for (int kk = 1; kk < 27; ++kk) a = kk == k ? acc[kk] : a;
            xfer_value(m0, a, w, cx, cy, cz, out[h], eq[h]);
            bad = bad || out[h] < T(1e-6) * w;
        }
    }
    bad = row_any(bad);
    const uint32_t c = tcells[i];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = j + 16 * h;
        if (k < 27) SP::sto(f + pop_index(c, k), bad ? eq[h] : out[h], wgt_rt<T>(k));
    }
    // WALE: the written cell's velocity (that of the interpolated state, which the rescale and the
    // equilibrium fallback keep) for the receiving level's gradient gather
    if (vel && j == 0) {
        vel[c] = m0.ux;
        vel[ncell + c] = m0.uy;
        vel[2 * (size_t)ncell + c] = m0.uz;
    }
}

// rebuild, FP32 arithmetic: a wave sums one written cell at a time with all lanes, and rebuilds up to
// XFER_CELLS of them together.
//   Sums: the lanes of a record are neighbours (8 of 16 bytes for float records, 4 for stored codes), so
//   that a load instruction reads whole lines; the lanes of a group sum its stencil nodes 4j .. 4j + 3 in
//   node order from zero (float records: two such partial sums per group), and the 16 partial sums add as
//   a pairwise tree: the low bits of j within a DPP row (rotations by 8 and by 4 lanes, the second on
//   values alike in the first's lanes), the high bits over the wave's four rows through LDS.
//   Cells: two lanes per cell read its 27 sums, form the moments and write half the directions each.
//   Groups: neighbouring entries with the same nodes (a fill's cells between the same coarse centres, four in
//   a layer on a face) share the records read and decoded once.
// Bound: VALU issue, some 70 % of the time (64 x 27 multiplies and adds per cell, unfused, in a fixed order: 165
// to 195 instructions per cell and lane in all, a third of them the moments and the directions).  Against 16
// lanes per cell with one record per lane, all of them forming the moments: a 4-level octree step 1668 -> 1571
// us; the groups then 1528 -> 1472 us, a 3-level step with WALE 575 -> 545 us.
constexpr int XFER_CELLS = 16;   // written cells per wave, at most
constexpr int XWG = 256;         // lanes of a workgroup
template <class SP, bool RAW>
__global__ void __launch_bounds__(XWG) k_xfer_rebuild(typename SP::st* f, uint32_t ncell, const uint32_t* tcells, uint32_t n,
                                                     uint32_t per, const int32_t* slot, const float* wt, const uint8_t* same,
                                                     const float* m, float scale, float keep, float* vel) {
    constexpr int V = RAW ? 8 : 4;            // directions per lane
    constexpr int NODES = RAW ? 4 : 8;        // nodes per lane
    constexpr int H = NODES / 4;              // partial sums per lane
    __shared__ float sums[XWG / 64][XFER_CELLS][4 * 32 + 4];   // [cell][row][direction], padded off the banks
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t i0 = (blockIdx.x * (XWG / 64) + (uint32_t)wave) * per;
    if (i0 >= n) return;
    const int cnt = (int)(n - i0 < per ? n - i0 : per);
    const int q = RAW ? lane & 3 : lane & 7;
    // group of nodes: its low bits in lane bit 3 (then 2), the high ones in the row
    const int g = RAW ? ((lane >> 3) & 1) | (((lane >> 2) & 1) << 1) | ((lane >> 4) << 2) : lane >> 3;
    float wk[V];
#pragma unroll
    for (int e = 0; e < V; ++e) wk[e] = wgt_rt<float>(V * q + e < 27 ? V * q + e : 13);
    // a quad's lanes read the nodes of its group, one (RAW) or two (lane and lane + 4) each, and pass them on
    // by quad broadcasts
    const uint32_t mine = (uint32_t)(g * NODES + (lane & 3));
    struct Stencil {          // of a group's first cell
        uint32_t r[H];        // record in 16-byte units (0xffffffff: an unused node)
        float w[H];
    };
    auto weights = [&](int d, float (&w)[H]) {
        const size_t o = (size_t)(i0 + (uint32_t)(d < cnt ? d : cnt - 1)) * 64 + mine;
#pragma unroll
        for (int h = 0; h < H; ++h) w[h] = wt[o + 4 * h];
    };
    auto stencil = [&](int d, Stencil& t) {
        const size_t o = (size_t)(i0 + (uint32_t)(d < cnt ? d : cnt - 1)) * 64 + mine;
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int32_t sv = slot[o + 4 * h];
            t.r[h] = sv < 0 ? 0xffffffffu : (uint32_t)sv * (RAW ? 4u : 8u);
        }
        weights(d, t.w);
    };
    // groups of cells on the same records: bit d of starts = cell d begins one
    const uint32_t starts = 1u | (uint32_t)__builtin_amdgcn_ballot_w64(lane < cnt && !(same && same[i0 + (uint32_t)lane]));
    auto next = [&](int d) {
        const uint32_t later = d < cnt ? (starts >> d) & ~1u : 0u;
        return later ? d + __builtin_ctz(later) : cnt;
    };
    const uint4* mq = reinterpret_cast<const uint4*>(m) + q;
    auto records = [&](const Stencil& t, uint4 (&rec)[NODES]) {
        for_each_dir(std::make_integer_sequence<int, NODES>{}, [&](auto ec) {
            constexpr int E = decltype(ec)::value;
            const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)t.r[E / 4], (E & 3) * 0x55, 0xf, 0xf, false);
            rec[E] = mq[r == 0xffffffffu ? 0u : r];
        });
    };
    auto one = [&](int d, const Stencil& t, const float (&tw)[H], const float (&x)[NODES][V]) {
        float acc[H][V];
        bool some = false;
#pragma unroll
        for (int h = 0; h < H; ++h) some = some || t.r[h] == 0xffffffffu;
        auto add = [&](auto check) {
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int e = 0; e < V; ++e) acc[h][e] = 0.0f;
            for_each_dir(std::make_integer_sequence<int, NODES>{}, [&](auto ec) {
                constexpr int E = decltype(ec)::value;
                const float w = dpp_get<(E & 3) * 0x55>(tw[E / 4]);
                bool use = true;
                if constexpr (decltype(check)::value)
                    use = (uint32_t)__builtin_amdgcn_mov_dpp((int)t.r[E / 4], (E & 3) * 0x55, 0xf, 0xf, false) != 0xffffffffu;
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float v = acc[E / 4][k] + w * x[E][k];
                    if constexpr (decltype(check)::value) acc[E / 4][k] = use ? v : acc[E / 4][k];
                    else acc[E / 4][k] = v;
                }
            });
        };
        if (__builtin_amdgcn_ballot_w64(some) == 0) add(std::false_type{});
        else add(std::true_type{});
#pragma unroll
        for (int k = 0; k < V; ++k) {
            float t;
            if constexpr (RAW) {
                t = acc[0][k];
                t = t + dpp_get<0x128>(t);    // row_ror:8
                t = t + dpp_get<0x124>(t);    // row_ror:4
            } else {
                t = acc[0][k] + acc[1][k];
                t = t + dpp_get<0x128>(t);
            }
            acc[0][k] = t;
        }
        if ((lane & 15) < (RAW ? 4 : 8)) {
            float4* o = reinterpret_cast<float4*>(&sums[wave][d][(lane >> 4) * 32 + V * q]);
#pragma unroll
            for (int k = 0; k < V / 4; ++k) o[k] = make_float4(acc[0][4 * k], acc[0][4 * k + 1], acc[0][4 * k + 2], acc[0][4 * k + 3]);
        }
    };
    // the cells d0 .. d1 - 1 of a group, the weights of the next one in flight during a cell's sums
    auto group = [&](int d0, int d1, const Stencil& t, const uint4 (&rec)[NODES]) {
        float x[NODES][V];
#pragma unroll
        for (int e = 0; e < NODES; ++e) {
            const uint32_t wd[4] = {rec[e].x, rec[e].y, rec[e].z, rec[e].w};
#pragma unroll
            for (int k = 0; k < V; ++k) {
                if constexpr (RAW) x[e][k] = SP::from_raw((wd[k >> 1] >> (16 * (k & 1))) & 0xffffu, wk[k]);
                else x[e][k] = __uint_as_float(wd[k]);
            }
        }
        float tw[H], tn[H];
#pragma unroll
        for (int h = 0; h < H; ++h) tw[h] = t.w[h];
#pragma unroll 1
        for (int d = d0; d < d1; ++d) {
            weights(d + 1, tn);
            one(d, t, tw, x);
#pragma unroll
            for (int h = 0; h < H; ++h) tw[h] = tn[h];
        }
    };
    // the next group's records and the stencil after it are in flight during a group's sums
    Stencil sa, sb, sc{};
    uint4 ra[NODES], rb[NODES];
    int d0 = 0, d1 = next(0), d2 = next(d1);
    stencil(d0, sa);
    stencil(d1, sb);
    records(sa, ra);
    while (true) {
        stencil(d2, sc);
        records(sb, rb);
        group(d0, d1, sa, ra);
        if (d1 >= cnt) break;
        const int d3 = next(d2);
        sa = sc;
        stencil(d3, sc);
        records(sa, ra);
        group(d1, d2, sb, rb);
        if (d2 >= cnt) break;
        sb = sc;
        d0 = d2;
        d1 = d3;
        d2 = next(d3);
    }
    wave_sync();
    // two lanes per cell, for a direction and its opposite: c c is the same and c u changes its sign
    const int d = lane >> 1;
    const bool opp = lane & 1;
    if (d >= cnt) return;
    float acc[27];
    {
        const float* b = &sums[wave][d][0];
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const float4 r0 = *reinterpret_cast<const float4*>(b + 4 * k), r1 = *reinterpret_cast<const float4*>(b + 32 + 4 * k);
            const float4 r2 = *reinterpret_cast<const float4*>(b + 64 + 4 * k), r3 = *reinterpret_cast<const float4*>(b + 96 + 4 * k);
            acc[4 * k] = (r0.x + r1.x) + (r2.x + r3.x);
            acc[4 * k + 1] = (r0.y + r1.y) + (r2.y + r3.y);
            acc[4 * k + 2] = (r0.z + r1.z) + (r2.z + r3.z);
            if (k < 6) acc[4 * k + 3] = (r0.w + r1.w) + (r2.w + r3.w);
        }
    }
    const XferMoments<float> m0 = xfer_moments<float>(acc, scale, keep);
    float out[14], eq[14];
    bool bad = false;
    for_each_dir(std::make_integer_sequence<int, 14>{}, [&](auto kc) {
        constexpr int K = decltype(kc)::value;
        constexpr float w = wgt<float>(K);
        XferMoments<float> q0 = m0;
        // (c -> -c: the signs of c u only)
        q0.ux = opp ? -m0.ux : m0.ux;
        q0.uy = opp ? -m0.uy : m0.uy;
        q0.uz = opp ? -m0.uz : m0.uz;
        xfer_value(q0, opp ? acc[26 - K] : acc[K], w, (float)dcx(K), (float)dcy(K), (float)dcz(K), out[K], eq[K]);
        bad = bad || out[K] < 1e-6f * w;
    });
    bad = ((__builtin_amdgcn_ballot_w64(bad) >> (lane & 62)) & 3ull) != 0;
    const uint32_t c = tcells[i0 + (uint32_t)d];
    for_each_dir(std::make_integer_sequence<int, 14>{}, [&](auto kc) {
        constexpr int K = decltype(kc)::value;
        if (K < 13 || !opp) SP::sto(f + pop_index(c, opp ? 26 - K : K), bad ? eq[K] : out[K], wgt<float>(K));
    });
    // WALE: the written cell's velocity (that of the interpolated state, which the rescale and the
    // equilibrium fallback keep) for the receiving level's gradient gather
    if (vel && !opp) {
        vel[c] = m0.ux;
        vel[ncell + c] = m0.uy;
        vel[2 * (size_t)ncell + c] = m0.uz;
    }
}

__global__ void k_set_i32(int32_t* p, int32_t v) {
    if (threadIdx.x == 0) p[0] = v;
}

hipError_t launch_set_i32(int32_t* p, int32_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_set_i32, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}


template <class SP, bool RAW>
static hipError_t xfer_sp(const void* fnew, const void* fold, const uint32_t* cells, uint32_t n, double w1, void* out,
                          hipStream_t s) {
    using T = typename SP::T;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL((k_xfer_gather<SP, RAW>), dim3((n + WG - 1) / WG), dim3(WG), 0, s, (const typename SP::st*)fnew,
                       (const typename SP::st*)fold, cells, n, T(w1), (T*)out);
    return hipGetLastError();
}
template <class SP, bool RAW>
static hipError_t rebuild_sp(void* f, uint32_t ncell, const uint32_t* tcells, uint32_t n, const int32_t* slot, const float* w,
                             const uint8_t* same, const void* m, double scale, double keep, void* vel, hipStream_t s) {
    using T = typename SP::T;
    using st = typename SP::st;
    if (!n) return hipSuccess;
    if constexpr (sizeof(T) == 8) {
        hipLaunchKernelGGL((k_xfer_rebuild_row<SP>), dim3((n + WG / 16 - 1) / (WG / 16)), dim3(WG), 0, s, (st*)f, ncell, tcells, n,
                           slot, w, (const T*)m, T(scale), T(keep), (T*)vel);
    } else {
        // written cells per wave, so that every CU gets the same number k of workgroups (k waves per SIMD): the
        // cost is k (cells + 7), the rebuild of a wave's cells together counting as 7 more; at least two waves
        // per SIMD.  Against 16 cells per wave wherever two waves per SIMD are left: a 4-level octree step 1472
        // -> 1423 us, a 3-level one with WALE 545 -> 513 us (33 800 cells: 11 per wave on three workgroups per
        // CU, not 16 on two, with a third on a few); from three waves per SIMD on: 1421 and 522 us.
        uint32_t per = XFER_CELLS, best = 0xffffffffu;
        for (uint32_t k = 2; k <= 8 || best == 0xffffffffu; ++k) {
            const uint32_t c = (n + 1024u * k - 1u) / (1024u * k);
            if (c > (uint32_t)XFER_CELLS || k * (c + 7u) >= best) continue;
            best = k * (c + 7u);
            per = c;
        }
        const uint32_t waves = (n + per - 1) / per;
        hipLaunchKernelGGL((k_xfer_rebuild<SP, RAW>), dim3((waves + XWG / 64 - 1) / (XWG / 64)), dim3(XWG), 0, s, (st*)f, ncell, tcells,
                           n, per, slot, w, same, (const float*)m, (float)scale, (float)keep, (float*)vel);
    }
    return hipGetLastError();
}

// raw records when the storage is 16-bit and no time blend is asked for
hipError_t launch_xfer_gather(int storage, const void* fnew, const void* fold, const uint32_t* cells, uint32_t n,
                               uint32_t ncell, double w1, void* out, hipStream_t s) {
    const bool raw = fold == nullptr;
    switch (storage) {
        case 0: return xfer_sp<StF32, false>(fnew, fold, cells, n, w1, out, s);
        case 1: return xfer_sp<StF64, false>(fnew, fold, cells, n, w1, out, s);
        case 2: return raw ? xfer_sp<StF16S, true>(fnew, fold, cells, n, w1, out, s)
                           : xfer_sp<StF16S, false>(fnew, fold, cells, n, w1, out, s);
        case 3: return raw ? xfer_sp<StBF16S, true>(fnew, fold, cells, n, w1, out, s)
                           : xfer_sp<StBF16S, false>(fnew, fold, cells, n, w1, out, s);
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_xfer_rebuild(int storage, bool raw, void* f, uint32_t ncell, const uint32_t* tcells, uint32_t n,
                               const int32_t* slot, const float* w, const uint8_t* same, const void* m, double scale,
                               double keep, void* vel, hipStream_t s) {
    switch (storage) {
        case 0: return rebuild_sp<StF32, false>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s);
        case 1: return rebuild_sp<StF64, false>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s);
        case 2: return raw ? rebuild_sp<StF16S, true>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s)
                           : rebuild_sp<StF16S, false>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s);
        case 3: return raw ? rebuild_sp<StBF16S, true>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s)
                           : rebuild_sp<StBF16S, false>(f, ncell, tcells, n, slot, w, same, m, scale, keep, vel, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace oal
