// Launcher of the kernel on 128 x 128 tiles with a ring of 64-deep slabs.
#include <atomic>
#include "gemm_mid_kernel.hip.h"

namespace ck {

template <typename DT, bool KTAIL>
static hipError_t mid_allow_lds() {
    static std::atomic<bool> opted[64] = {};   // (threads may launch at once; setting the attribute twice is harmless)
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || (dev >= 0 && dev < 64 && opted[dev].load(std::memory_order_acquire))) return e;
    e = hipFuncSetAttribute((const void*)gemm_mid_kernel<DT, KTAIL>, hipFuncAttributeMaxDynamicSharedMemorySize, MID_LDS_BYTES);
    if (e == hipSuccess && dev >= 0 && dev < 64) opted[dev].store(true, std::memory_order_release);
    return e;
}
template <typename DT>
static hipError_t mid_prepare() {
    const hipError_t e = mid_allow_lds<DT, false>();
    return e == hipSuccess ? mid_allow_lds<DT, true>() : e;
}
hipError_t prepare_gemm_mid(bool bf16) { return bf16 ? mid_prepare<bf16_tag>() : mid_prepare<f16_tag>(); }

template <typename DT, bool KTAIL>
static hipError_t mid_launch(hipStream_t stream, const GemmArgs& a) {
    const hipError_t e = mid_allow_lds<DT, KTAIL>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_mid_kernel<DT, KTAIL>), dim3((unsigned)(a.tiles_m * a.tiles_n * a.split_k)), dim3(512), MID_LDS_BYTES, stream, a);
    return hipGetLastError();
}
template <typename DT>
static hipError_t mid_dispatch(hipStream_t stream, const GemmArgs& a) {
    return a.K % MID_SLAB_K ? mid_launch<DT, true>(stream, a) : mid_launch<DT, false>(stream, a);
}
hipError_t launch_gemm_mid(bool bf16, hipStream_t stream, const GemmArgs& a) { return bf16 ? mid_dispatch<bf16_tag>(stream, a) : mid_dispatch<f16_tag>(stream, a); }

}  // namespace ck
