// Launcher of the small-product kernel (one instance per element type, tile, operand alignment, and with K slices or without).
#include <atomic>
#include "gemm_direct_kernel.hip.h"

namespace ck {

// The instances on 64 tiles take more than 64 KiB of LDS, which has to be allowed per device. All at once: the first call may run any of them, and a later one, which may
// be recorded into a graph, another.
template <typename DT>
static hipError_t direct_allow_lds() {
    static std::atomic<bool> opted[64] = {};   // (threads may launch at once; setting the attributes twice is harmless)
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || (dev >= 0 && dev < 64 && opted[dev].load(std::memory_order_acquire))) return e;
    for (const void* kern : {(const void*)gemm_direct_kernel<DT, 4, 1, true, true>, (const void*)gemm_direct_kernel<DT, 4, 1, true, false>,
                             (const void*)gemm_direct_kernel<DT, 4, 1, false, true>, (const void*)gemm_direct_kernel<DT, 4, 1, false, false>}) {
        e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, direct_lds_bytes(64));
        if (e != hipSuccess) return e;
    }
    if (dev >= 0 && dev < 64) opted[dev].store(true, std::memory_order_release);
    return hipSuccess;
}
hipError_t prepare_gemm_direct(bool bf16) { return bf16 ? direct_allow_lds<bf16_tag>() : direct_allow_lds<f16_tag>(); }

template <typename DT, int WT, int DEPTH, bool EVEN, bool SLICED>
static hipError_t direct_launch_as(hipStream_t stream, const GemmArgs& a) {
    static_assert(direct_lds_bytes(WT * 16) <= 64 * 1024 || (WT == 4 && DEPTH == 1), "one of direct_allow_lds's instances");
    if (direct_lds_bytes(WT * 16) > 64 * 1024) {
        const hipError_t e = direct_allow_lds<DT>();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((gemm_direct_kernel<DT, WT, DEPTH, EVEN, SLICED>), dim3((unsigned)(a.tiles_m * a.tiles_n * a.split_k)), dim3(DIRECT_WAVES * WAVE), direct_lds_bytes(WT * 16), stream, a);
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
