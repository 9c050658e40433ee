// Launcher of the small-product kernel (one instance per element type, tile, operand alignment, and with K slices or without).
#include <atomic>
#include "gemm_direct_kernel.hip.h"

namespace ck {

template <typename DT, int WT, int DEPTH, bool EVEN, bool SLICED>
static hipError_t direct_launch_as(hipStream_t stream, const GemmArgs& a) {
    auto kern = gemm_direct_kernel<DT, WT, DEPTH, EVEN, SLICED>;
    constexpr int lds = direct_lds_bytes(WT * 16);
    if (lds > 64 * 1024) {
        static std::atomic<bool> opted[64] = {};   // (threads may launch at once; setting the attribute twice is harmless)
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= 64 || !opted[dev].load(std::memory_order_acquire)) {
            e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return e;
            if (dev >= 0 && dev < 64) opted[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n * a.split_k)), dim3(DIRECT_WAVES * WAVE), lds, stream, a);
    return hipGetLastError();
}
template <typename DT, int WT, int DEPTH, bool EVEN>
static hipError_t direct_launch_one(hipStream_t stream, const GemmArgs& a) {
    return a.split_k > 1 ? direct_launch_as<DT, WT, DEPTH, EVEN, true>(stream, a) : direct_launch_as<DT, WT, DEPTH, EVEN, false>(stream, a);
}
template <typename DT>
static hipError_t direct_launch(int tile, bool even, hipStream_t stream, const GemmArgs& a) {
    // the depths are what the 256 registers of a wave hold
    if (tile == 32) return even ? direct_launch_one<DT, 2, 4, true>(stream, a) : direct_launch_one<DT, 2, 2, false>(stream, a);
    if (tile == 64) return even ? direct_launch_one<DT, 4, 1, true>(stream, a) : direct_launch_one<DT, 4, 1, false>(stream, a);
    return hipErrorInvalidValue;
}

// tile: 32 or 64 (a.tiles_m and a.tiles_n count tiles of that size); even: rows start on 4-byte boundaries
hipError_t launch_gemm_direct(bool bf16, int tile, bool even, hipStream_t stream, const GemmArgs& a) {
    return bf16 ? direct_launch<bf16_tag>(tile, even, stream, a) : direct_launch<f16_tag>(tile, even, stream, a);
}

}  // namespace ck
