// matmul_shmem on few outputs per CU, on the vector ALUs only: the sums of simt_kernel.hip.h (one accumulator per output, ascending k, one
// fused multiply-add per k), bit for bit, from operand slices that lie in LDS as rows of 32 k.
//
// What bounds such a product is a wave's own chain of LDS reads, multiply-adds and barriers, with one wave or two on a SIMD: the other kernel's k-major slices
// of 16 k give a thread two 8-byte reads per k for four multiply-adds, and a row-major operand goes into them one value at a time. Rows of k give it 16-byte
// reads for four k at a time and 16-byte writes, a slice of 32 k halves the barriers, and the chunks are fetched two slices ahead. Tiles of 16 x 16 give
// the smallest grids four times the workgroups.
#ifndef CK_SIMT_SMALL_KERNEL_HIP_H
#define CK_SIMT_SMALL_KERNEL_HIP_H

#include "simt_kernel.hip.h"

namespace ck {

constexpr int SIMT_SMALL_KT = 32;                 // k of a slice; K is a multiple of half of it
constexpr int SIMT_SMALL_LD = SIMT_SMALL_KT + 4;  // pitch of a row in LDS: 16 rows of a 16-byte read start in 16 different groups of four banks
constexpr int simt_small_lds_bytes(int tile) { return 2 * 2 * tile * SIMT_SMALL_LD * 4; }

// BT: B is given transposed (N x K row-major); otherwise K x N. A thread has the rows ty, ty + TY, ... and the columns tx, tx + TX, ... of its tile.
template <typename DT, int TILE, int RM, int RN, bool BT>
__global__ __launch_bounds__(TILE * TILE / (RM * RN)) void matmul_shmem_small_kernel(const SimtArgs g) {
    typedef SimtIo<DT> Io;
    typedef typename Io::acc_t ACC;
    typedef typename Io::elem_t ELEM;
    typedef ELEM elem4 __attribute__((ext_vector_type(4)));
    constexpr int KT = SIMT_SMALL_KT, LD = SIMT_SMALL_LD, VEC = Io::VEC;
    constexpr int NT = TILE * TILE / (RM * RN), TX = TILE / RN, TY = TILE / RM;
    constexpr int CH = TILE * KT / VEC;            // 16-byte chunks of an operand's slice
    constexpr int ITS = (2 * CH + NT - 1) / NT;    // chunks of both operands per thread
    constexpr int CPR = KT / VEC, CPN = TILE / VEC;
    static_assert(CH % 64 == 0, "a wave's chunks belong to one operand");
    extern __shared__ __attribute__((aligned(16))) char ck_simt_smem[];
    ELEM* const lds = reinterpret_cast<ELEM*>(ck_simt_smem);
    auto slice_of = [&](int buf, int operand) { return lds + (buf * 2 + operand) * TILE * LD; };

    const DT* A = static_cast<const DT*>(g.A);
    const DT* B = static_cast<const DT*>(g.B);
    DT* C = static_cast<DT*>(g.C);
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int64_t m0 = (int64_t)blockIdx.x * TILE, n0 = (int64_t)blockIdx.y * TILE;
    const int K = g.K, N = g.N;

    struct Fetched { simt_raw_t x[ITS]; };
    // (a chunk past the end of K: the last slice's first half once more, which is not multiplied)
    auto fetch = [&](int k0, Fetched& f) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
            const int at = it * NT + tid, ch = at % CH;
            if ((2 * CH) % NT != 0 && at >= 2 * CH) continue;
            if (at < CH || BT) {
                const int r = ch / CPR, k = k0 + ch % CPR * VEC;
                const DT* row = at < CH ? A + (m0 + r) * K : B + (n0 + r) * K;
                f.x[it] = *reinterpret_cast<const simt_raw_t*>(row + (k < K ? k : K - VEC));
            } else {
                const int k = k0 + ch / CPN;
                f.x[it] = *reinterpret_cast<const simt_raw_t*>(B + (int64_t)(k < K ? k : K - 1) * N + n0 + ch % CPN * VEC);
            }
        }
    };
    auto stash = [&](int buf, const Fetched& f) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
            const int at = it * NT + tid, ch = at % CH;
            if ((2 * CH) % NT != 0 && at >= 2 * CH) continue;
            ELEM v[VEC];
            Io::spread(f.x[it], v);
            if (at < CH || BT) {
                ELEM* to = slice_of(buf, at < CH ? 0 : 1) + ch / CPR * LD + ch % CPR * VEC;
#pragma unroll
                for (int e = 0; e < VEC; e += 4) *reinterpret_cast<elem4*>(to + e) = elem4{v[e], v[e + 1], v[e + 2], v[e + 3]};
            } else {
                ELEM* to = slice_of(buf, 1) + ch % CPN * VEC * LD + ch / CPN;
#pragma unroll
                for (int e = 0; e < VEC; ++e) to[e * LD] = v[e];
            }
        }
    };
    ACC acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = (ACC)0;
    auto multiply = [&](int buf, int half) __attribute__((always_inline)) {
        const ELEM* as = slice_of(buf, 0) + ty * LD + half * (KT / 2);
        const ELEM* bs = slice_of(buf, 1) + tx * LD + half * (KT / 2);
#pragma unroll
        for (int k = 0; k < KT / 2; k += 4) {
            elem4 a[RM], b[RN];
#pragma unroll
            for (int i = 0; i < RM; ++i) a[i] = *reinterpret_cast<const elem4*>(as + i * TY * LD + k);
#pragma unroll
            for (int j = 0; j < RN; ++j) b[j] = *reinterpret_cast<const elem4*>(bs + j * TX * LD + k);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < RM; ++i)
#pragma unroll
                    for (int j = 0; j < RN; ++j) acc[i][j] = Io::mad(a[i][e], b[j][e], acc[i][j]);
        }
    };

    const int slices = (K + KT - 1) / KT;
    // Slice s lies in LDS, s + 1 in f, s + 2 on its way behind it.
    auto slice = [&](int s, Fetched& f) __attribute__((always_inline)) {
        multiply(s & 1, 0);
        if (s * KT + KT / 2 < K) multiply(s & 1, 1);
        stash(~s & 1, f);
        fetch((s + 3) * KT, f);
        __syncthreads();
    };
    Fetched even, odd;
    fetch(0, even);
    fetch(KT, odd);
    stash(0, even);
    fetch(2 * KT, even);
    __syncthreads();
    int s = 0;
    for (; s + 1 < slices; s += 2) {
        slice(s, odd);
        slice(s + 1, even);
    }
    if (s < slices) slice(s, odd);

#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) C[(m0 + ty + i * TY) * N + n0 + tx + j * TX] = Io::out(acc[i][j]);
}

}  // namespace ck
#endif  // CK_SIMT_SMALL_KERNEL_HIP_H
