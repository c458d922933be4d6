// kernels.hip -- the E and H half-step kernels, one cell per thread (gfx950).
//
#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>

#include "cell_sweep.h"
#include "device_common.h"
#include "internal.h"
#include "sweep_common.h"

// Occupancy floors of the two sweep kernels (waves per SIMD).
#ifdef FDTD_E_WAVES
#define E_OCC __attribute__((amdgpu_waves_per_eu(FDTD_E_WAVES, FDTD_E_WAVES)))
#else
#define E_OCC
#endif
#ifdef FDTD_H_WAVES
#define H_OCC __attribute__((amdgpu_waves_per_eu(FDTD_H_WAVES, FDTD_H_WAVES)))
#else
#define H_OCC
#endif

namespace fdtd {

// A half-step in one launch: ng workgroups of the general variant first (they
// take longest), nx of the x-edge one, the rest the interior's.  In a launch
// each, the variants of a medium grid leave most of the chip idle at their
// ends, and the next does not start before the last workgroup is done.  The
// registers are the general variant's (FP32, E: 91 against 58 of the
// interior's alone, five waves per SIMD for eight), which costs less: us per
// step, a launch each / one launch: 150x131x118 70 / 52, 203x149x97 with
// magnetic classes 86 / 65, 400x130x70 82 / 67, 320x320x130 magnetic 234 /
// 226, 512x512x64 322 / 310.
// GEN: the general variant alone (no interior box, light-cone steps), in a
// kernel without the others: block-scaled H with one class needs 89 registers
// for 97, five waves per SIMD for four.  us per step, block-scaled int16, as one of
// the variants / alone (and a launch for each variant): 140x134x84 51.1 / 48.6
// (50.1), 264x47x53 27.9 / 26.7 (27.8), 83x62x88 32.3 / 31.2 (32.2).
template <class T, int CM, int ST, bool GEN>
__global__ void __launch_bounds__(TX * BY) E_OCC e_kernel(const KArgs a, const int m, const int ng, const int nx)
{
    const int b = blockIdx.x;
    int tx, ty, tz;
    if (GEN || b < ng) {
        tile_of_region<V_GEN>(a, tx, ty, tz, b);
        e_tile<T, CM, V_GEN | ST>(a, m, tx, ty, tz);
    } else if (b < ng + nx) {
        tile_of_region<V_X>(a, tx, ty, tz, b - ng);
        e_tile<T, CM, V_X | ST>(a, m, tx, ty, tz);
    } else {
        tile_of_region<V_IN>(a, tx, ty, tz, b - ng - nx);
        e_tile<T, CM, V_IN | ST>(a, m, tx, ty, tz);
    }
}
template <class T, int CM, int ST, bool GEN>
__global__ void __launch_bounds__(TX * BY) H_OCC h_kernel(const KArgs a, const int m, const int ng, const int nx)
{
    const int b = blockIdx.x;
    int tx, ty, tz;
    if (GEN || b < ng) {
        tile_of_region<V_GEN>(a, tx, ty, tz, b);
        h_tile<T, CM, V_GEN | ST>(a, m, tx, ty, tz);
    } else if (b < ng + nx) {
        tile_of_region<V_X>(a, tx, ty, tz, b - ng);
        h_tile<T, CM, V_X | ST>(a, m, tx, ty, tz);
    } else {
        tile_of_region<V_IN>(a, tx, ty, tz, b - ng - nx);
        h_tile<T, CM, V_IN | ST>(a, m, tx, ty, tz);
    }
}

// ---- launchers --------------------------------------------------------------
template <class T, int ST, bool GEN>
static void launch_g(bool efield, int mode, const KArgs &a, int m, int ng, int nx, int nb, hipStream_t s)
{
    dim3 grid(ng + nx + nb), block(TX * BY);
    if (efield) {
        if (mode == CLS_UNIFORM) hipLaunchKernelGGL((e_kernel<T, CLS_UNIFORM, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
        else if (mode == CLS_U16) hipLaunchKernelGGL((e_kernel<T, CLS_U16, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
        else hipLaunchKernelGGL((e_kernel<T, CLS_U32, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
    } else {
        if (mode == CLS_UNIFORM) hipLaunchKernelGGL((h_kernel<T, CLS_UNIFORM, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
        else if (mode == CLS_U16) hipLaunchKernelGGL((h_kernel<T, CLS_U16, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
        else hipLaunchKernelGGL((h_kernel<T, CLS_U32, ST, GEN>), grid, block, 0, s, a, m, ng, nx);
    }
}
template <class T, int ST>
static hipError_t launch_t(bool efield, int mode, const KArgs &a, int m, hipStream_t s)
{
    int nb, nx, nzt, ng;   // nzt = 0: the forward sweeps run without zsplit
    region_tiles(a, nb, nx, nzt, ng);
    if (nb + nx == 0) launch_g<T, ST, true>(efield, mode, a, m, ng, nx, nb, s);
    else launch_g<T, ST, false>(efield, mode, a, m, ng, nx, nb, s);
    return hipGetLastError();
}

// storage: 0 FP32, 1 FP16, 2 BF16, 3 block-scaled int16 (fields; psi FP16).  e_mode/h_mode: ClassMode of each sweep.
hipError_t launch_half_step(bool efield, int storage, int mode, const KArgs &a, int m, hipStream_t s)
{
    switch (storage) {
    case 0: return a.stream ? launch_t<float, V_STREAM>(efield, mode, a, m, s) : launch_t<float, 0>(efield, mode, a, m, s);
    case 1: return a.stream ? launch_t<_Float16, V_STREAM>(efield, mode, a, m, s) : launch_t<_Float16, 0>(efield, mode, a, m, s);
    case 2: return a.stream ? launch_t<bf16_t, V_STREAM>(efield, mode, a, m, s) : launch_t<bf16_t, 0>(efield, mode, a, m, s);
    case 3: return a.stream ? launch_t<bq16_t, V_STREAM>(efield, mode, a, m, s) : launch_t<bq16_t, 0>(efield, mode, a, m, s);
    default: return hipErrorInvalidValue;
    }
}

// Values g0 .. g0 + n - 1 of a component ([nz][ny][nx], SI) to `out`, pinned
// host memory: rows packed, converted and scaled on the way, one 4-byte store
// a lane.  f, q: the component and (block-scaled) its exponents at plane 0.
// Bound by the link to the host: 2^20 values in 57 us (74 GB/s); pieces of 2^17,
// 11 us each, half of that the launch.
template <class T>
__global__ void __launch_bounds__(256)
    unpack_kernel(const T *f, const std::uint8_t *q, float *out, std::uint32_t g0, std::uint32_t n, std::uint32_t nx,
                  std::uint32_t px, float scale)
{
    const std::uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const std::uint32_t r = (g0 + e) / nx, i = (g0 + e) % nx;
    const i64 c = (i64)r * px + i;
    float v;
    if constexpr (is_bq<T>::value) v = ldexpf((float)f[c].v, (int)q[c / BQ_BLOCK * BQ_STRIDE] - BQ_BIAS);
    else v = ld(f + c);
    out[e] = v * scale;
}

hipError_t launch_unpack(int storage, const void *f, const std::uint8_t *q, float *out, std::uint32_t g0, std::uint32_t n,
                         int nx, int px, float scale, hipStream_t s)
{
    dim3 grid((n + 255) / 256), block(256);
    switch (storage) {
    case 0: hipLaunchKernelGGL((unpack_kernel<float>), grid, block, 0, s, (const float *)f, q, out, g0, n, nx, px, scale); break;
    case 1:
        hipLaunchKernelGGL((unpack_kernel<_Float16>), grid, block, 0, s, (const _Float16 *)f, q, out, g0, n, nx, px, scale);
        break;
    case 2: hipLaunchKernelGGL((unpack_kernel<bf16_t>), grid, block, 0, s, (const bf16_t *)f, q, out, g0, n, nx, px, scale); break;
    case 3: hipLaunchKernelGGL((unpack_kernel<bq16_t>), grid, block, 0, s, (const bq16_t *)f, q, out, g0, n, nx, px, scale); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

int tile_rows() { return BY; }
int tile_cols() { return TX; }

}  // namespace fdtd
