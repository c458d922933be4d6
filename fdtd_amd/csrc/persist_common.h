// persist_common.h -- what the kernels that run many steps in one launch share
// (persist.hip: forward steps; adj_persist.hip: reverse steps): the exchange
// of rows between tiles, and the units' descriptions.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "internal.h"

namespace fdtd {

typedef std::uint32_t u32;
typedef std::uint64_t u64;

constexpr int PW = 16;   // waves per workgroup
constexpr int COOP_LDS_MAX = 160 * 1024;   // bytes of a workgroup

__device__ __forceinline__ void ll_put(u64 *p, float v, u32 tag)
{
    __hip_atomic_store(p, (u64)__float_as_uint(v) | ((u64)tag << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 ll_get(const u64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ll_val(u64 w) { return __uint_as_float((u32)w); }
__device__ __forceinline__ bool ll_is(u64 w, u32 tag) { return (u32)(w >> 32) == tag; }

// The words at pa, pa + n (when ga) and pb, pb + n (when gb), once all of
// them carry `tag` on every lane of the wave (ga and gb are wave-uniform).
template <class Args>
__device__ __forceinline__ void ll_wait(const Args &p, bool ga, const u64 *pa, bool gb, const u64 *pb, int n, u32 tag,
                                        bool &dead, float &a0, float &a1, float &b0, float &b1)
{
    u64 w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    for (int t = 0;; ++t) {
        if (ga) {
            w0 = ll_get(pa);
            w1 = ll_get(pa + n);
        }
        if (gb) {
            w2 = ll_get(pb);
            w3 = ll_get(pb + n);
        }
        const bool ok = (!ga || (ll_is(w0, tag) && ll_is(w1, tag))) && (!gb || (ll_is(w2, tag) && ll_is(w3, tag)));
        if (dead || __all(ok)) break;
        if (t >= p.max_polls) {   // a neighbour that never answers: give up, and tell everyone
            __hip_atomic_store(p.failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            dead = true;
        } else if ((t & 1023) == 1023) {
            dead = __hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        }
    }
    a0 = ll_val(w0);
    a1 = ll_val(w1);
    b0 = ll_val(w2);
    b1 = ll_val(w3);
}

// The 16-word descriptions of a wave's units (the same on every lane and
// step), four units in the lanes of one register: a word is one lane read,
// where scalar loads would each wait for the cache.
template <int NU>
struct PDesc {
    int v[(NU + 3) / 4];
    template <class UnitT>
    __device__ __forceinline__ void load(const UnitT *u, int w, int nu, int lane)
    {
        static_assert(sizeof(UnitT) == 64, "16 words");
        for (int q = 0; q < (NU + 3) / 4; ++q) {
            const int n = w + (4 * q + lane / 16) * PW;
            v[q] = n < nu ? ((const int *)(u + n))[lane % 16] : 0;
        }
    }
    // word f of unit n
    __device__ __forceinline__ int at(int n, int f) const { return __builtin_amdgcn_readlane(v[n / 4], (n % 4) * 16 + f); }
};

// Whether `tiles` workgroups of PW waves with `lds` bytes each can be
// resident at once (and the kernel is set up to use them: its limit of dynamic
// LDS is one of the process, so it is set to the most that any context asks for).
inline bool coop_fits(const void *fn, int tiles, size_t lds, int device)
{
    int coop = 0, cus = 0, per = 0;
    bool ok = fn && lds <= (size_t)COOP_LDS_MAX &&
              hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) == hipSuccess && coop &&
              hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
              hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, COOP_LDS_MAX) == hipSuccess &&
              hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, 64 * PW, lds) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    return ok && per >= 1 && tiles <= cus * per;
}

}  // namespace fdtd
