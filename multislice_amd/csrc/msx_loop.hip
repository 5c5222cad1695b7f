// msx_loop.hip -- instantiations and launcher of the persistent slice loop for
// rows of MSX_N elements and every column length it is built for.
#include <atomic>

#include "msx_internal.h"
#include "msx_loop.hpp"

#ifndef MSX_N
#error "compile with -DMSX_N=<row length>"
#endif
#define MSX_CAT2(a, b) a##b
#define MSX_CAT(a, b) MSX_CAT2(a, b)

namespace msx {
namespace {

template <typename C, int NX> hipError_t prepare(int* units, int* resident) {
    using S = LoopShape<C, NX, MSX_N>;
    const void* k = reinterpret_cast<const void*>(&slice_loop_kernel<C, NX, MSX_N>);
    *units = S::row_units;
    // work-groups resident on the device at once, kept per device (0: not asked yet)
    static std::atomic<int> cache[16];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (S::lds > 64 * 1024) {
        e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::lds);
        if (e != hipSuccess) return e;
    }
    const int slot = dev < 16 ? dev : 15;
    *resident = dev < 16 ? cache[slot].load(std::memory_order_relaxed) : 0;
    if (*resident > 0) return hipSuccess;
    int per = 0, cus = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, S::BT, S::lds);
    if (e != hipSuccess) return e;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    *resident = per * cus;
    if (dev < 16) cache[slot].store(*resident, std::memory_order_relaxed);
    return hipSuccess;
}

template <typename C, int NX> hipError_t go(const LoopArgs<C>& a, int teams, hipStream_t s) {
    using S = LoopShape<C, NX, MSX_N>;
    LoopArgs<C> arg = a;
    void* args[] = {&arg};
    return hipLaunchCooperativeKernel(reinterpret_cast<void*>(&slice_loop_kernel<C, NX, MSX_N>),
                                      dim3((unsigned)(teams * a.team)), dim3(S::BT), args, S::lds, s);
}

}  // namespace

#define MSX_LOOP_EACH(X) X(128) X(256) X(384) X(512)
template <typename C> hipError_t MSX_CAT(loop_prepare_, MSX_N)(int nx, int* units, int* resident) {
#define MSX_CASE(NX) \
    if (nx == NX) return prepare<C, NX>(units, resident);
    MSX_LOOP_EACH(MSX_CASE)
#undef MSX_CASE
    return hipErrorInvalidValue;
}
template <typename C> hipError_t MSX_CAT(launch_loop_, MSX_N)(int nx, const LoopArgs<C>& a, int teams, hipStream_t s) {
#define MSX_CASE(NX) \
    if (nx == NX) return go<C, NX>(a, teams, s);
    MSX_LOOP_EACH(MSX_CASE)
#undef MSX_CASE
    return hipErrorInvalidValue;
}
template hipError_t MSX_CAT(loop_prepare_, MSX_N)<float2>(int, int*, int*);
template hipError_t MSX_CAT(loop_prepare_, MSX_N)<double2>(int, int*, int*);
template hipError_t MSX_CAT(launch_loop_, MSX_N)<float2>(int, const LoopArgs<float2>&, int, hipStream_t);
template hipError_t MSX_CAT(launch_loop_, MSX_N)<double2>(int, const LoopArgs<double2>&, int, hipStream_t);

}  // namespace msx
