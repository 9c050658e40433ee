// Launcher of the kernel on 128 x 128 tiles with a ring of 64-deep slabs.
#include <atomic>
#include "gemm_mid_kernel.hip.h"

namespace ck {

template <typename DT, bool KTAIL>
static hipError_t mid_launch(hipStream_t stream, const GemmArgs& a) {
    auto kern = gemm_mid_kernel<DT, KTAIL>;
    static std::atomic<bool> opted[64] = {};   // (threads may launch at once; setting the attribute twice is harmless)
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64 || !opted[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, MID_LDS_BYTES);
        if (e != hipSuccess) return e;
        if (dev >= 0 && dev < 64) opted[dev].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n * a.split_k)), dim3(512), MID_LDS_BYTES, stream, a);
    return hipGetLastError();
}
template <typename DT>
static hipError_t mid_dispatch(hipStream_t stream, const GemmArgs& a) {
    return a.K % MID_SLAB_K ? mid_launch<DT, true>(stream, a) : mid_launch<DT, false>(stream, a);
}
hipError_t launch_gemm_mid(bool bf16, hipStream_t stream, const GemmArgs& a) { return bf16 ? mid_dispatch<bf16_tag>(stream, a) : mid_dispatch<f16_tag>(stream, a); }

}  // namespace ck
