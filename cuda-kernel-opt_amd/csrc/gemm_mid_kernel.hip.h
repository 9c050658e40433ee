// 128 x 128 tiles on a ring of five 64-deep slabs: one workgroup of eight waves per tile of D (and K slice), all of the CU's LDS.
//
// What bounds it: on a full device the L2s, which give 26 TB/s to loads of whole lines (5.2 ns per k of 256 tiles; the loads of this
// kernel alone reach that), and on random operands the power limit (2048^2 x 8192: 64 us at 1.85 GHz, 53 us at 2.4 GHz on constant
// ones). On few tiles the loads of one CU take 4.0 ns per k, the MFMAs 3.5 and MFMAs with fragment reads 4.2; all together 5.4.
//
// A slab is one 128-byte line of every row. A wave brings 16 rows of each operand straight into LDS, four loads of 1 KiB, four to
// five slabs ahead of the MFMAs. The waves form two groups of four; each covers the tile with wave tiles of 64 x 64 and takes one of a
// slab's two k-steps: 16 MFMAs on 8 fragments per slab and wave, a third less LDS traffic than eight tiles of 32 x 64. The fragments
// of slab s + 1 are read under the MFMAs of slab s, and the barrier of body s stands for slab s + 2, so that no read waits behind it.
// The partial tiles of the two groups meet in LDS at the end, in rows: first + second, and whole lines of D.
//
// The eight XCDs begin at eight different slabs. With rows of a power of two in bytes all tiles would otherwise ask the same few
// memory channels at a time: bf16 256 x 16384 x 4096 from memory 52.0 -> 46.4 us, loads alone on 4096^2 x 8192 228 -> 192.
//
// Against the kernel before (two 128-deep stages written through registers; a wave's reads, MFMAs and writes added up): fp16 2048^3
// 25.5 -> 21.8 us, bf16 256 x 16384 x 4096 with 16-bit results 53.5 -> 45.0.
#ifndef CK_GEMM_MID_KERNEL_HIP_H
#define CK_GEMM_MID_KERNEL_HIP_H

#include "gemm_fused_kernel.hip.h"

namespace ck {

constexpr int MID_TILE = 128;
constexpr int MID_SLAB_K = 64;                                 // one 128-byte line of an operand row
constexpr int MID_OPERAND = MID_TILE * MID_SLAB_K * 2;
constexpr int MID_STAGE = 2 * MID_OPERAND;
constexpr int MID_STAGES = 5;
constexpr int MID_OUT_ROW = 64 * 4 + 16;                       // a row of a wave's partial tile: 64 sums, and 16 bytes against bank conflicts
constexpr int MID_OUT_WAVE = 64 * MID_OUT_ROW;
constexpr int MID_LDS_BYTES = MID_STAGES * MID_STAGE;
static_assert(8 * MID_OUT_WAVE <= MID_LDS_BYTES && MID_LDS_BYTES <= LDS_BYTES_PER_CU, "the partial tiles take the ring's place");

// Four neighbouring results of a row, the first in column n: D = alpha * sum + beta * C. C is what row_c() fetched.
template <typename DT>
__device__ __forceinline__ f32x4 row_c(const GemmArgs& g, int m, int n) {
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    if (g.beta == 0.f || m >= g.M || n >= g.N) return c;
    const int64_t off = (int64_t)m * g.N + n;
    const unsigned short* c16 = (const unsigned short*)g.C;
    if (n + 4 <= g.N) {
        if (!g.out16) return *(const f32x4_u*)(g.C + off);
        const u32x2_a2 x = *(const u32x2_a2*)(c16 + off);
        return f32x4{Out16<DT>::load((unsigned short)(x[0] & 0xffffu)), Out16<DT>::load((unsigned short)(x[0] >> 16)),
                     Out16<DT>::load((unsigned short)(x[1] & 0xffffu)), Out16<DT>::load((unsigned short)(x[1] >> 16))};
    }
#pragma unroll
    for (int e = 0; e < 3; ++e)
        if (n + e < g.N) c[e] = g.out16 ? Out16<DT>::load(c16[off + e]) : g.C[off + e];
    return c;
}
template <typename DT>
__device__ __forceinline__ void store_row(const GemmArgs& g, float* D, int m, int n, f32x4 sum, f32x4 c) {
    if (m >= g.M || n >= g.N) return;
    const int64_t off = (int64_t)m * g.N + n;
    f32x4 v = sum * g.alpha;
    if (g.beta != 0.f) v += c * g.beta;
    unsigned short* d16 = (unsigned short*)D;
    if (n + 4 <= g.N) {
        if (!g.out16) {
            if (g.nt_store) store_b128_nt(D + off, __builtin_bit_cast(u32x4, v));
            else *(f32x4_u*)(D + off) = v;
        } else {
            const u32x2 o = {(uint32_t)Out16<DT>::store(v[0]) | (uint32_t)Out16<DT>::store(v[1]) << 16, (uint32_t)Out16<DT>::store(v[2]) | (uint32_t)Out16<DT>::store(v[3]) << 16};
            if (g.nt_store) store_b64_nt(d16 + off, o);
            else *(u32x2_a2*)(d16 + off) = o;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 3; ++e)
        if (n + e < g.N) {
            if (g.out16) d16[off + e] = Out16<DT>::store(v[e]);
            else D[off + e] = v[e];
        }
}

// Rows start on 16-byte boundaries and K % 8 == 0 (a 16-byte chunk of a row is inside it or past it), or with KTAIL (K % 64 != 0) on 4-byte
// boundaries and K is even: direct-to-LDS loads take such rows as they are, and the last K % 8 values of the rows, which no whole chunk holds, are one
// more k-step on fragments straight from memory (no zero-padded copies: bf16 384 x 10310 x 2692 60.4 -> 33.5 us, 914 x 3264 x 916 with 16-bit results 31.0 -> 16.9).
template <typename DT, bool KTAIL>
__global__ __launch_bounds__(512) void gemm_mid_kernel(const GemmArgs g) {
    constexpr int WT = 4;   // 16 x 16 blocks per edge of a wave tile
    extern __shared__ __attribute__((aligned(1024))) char ck_smem[];
    const uint32_t ring = (uint32_t)(uintptr_t)(CK_LDS char*)ck_smem;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned long long clk0 = clock64(), wall0 = wall_clock64();

    // work items: the tiles of the first K slice, then those of the second ...; an XCD's run of items shares operand panels
    const int item = xcd_tile(blockIdx.x, gridDim.x, g.num_xcd), tiles = g.tiles_m * g.tiles_n, slice = g.split_k > 1 ? __builtin_amdgcn_readfirstlane(item / tiles) : 0;
    const TileRC rc = tile_order(g.tiles_m, g.tiles_n, g.tile_group_m, item - slice * tiles);
    const int row_a = __builtin_amdgcn_readfirstlane(rc.row * MID_TILE), row_b = __builtin_amdgcn_readfirstlane(rc.col * MID_TILE);
    const uint32_t pitch = (uint32_t)g.K * 2u;
    const int rows_a = g.M - row_a < MID_TILE ? g.M - row_a : MID_TILE, rows_b = g.N - row_b < MID_TILE ? g.N - row_b : MID_TILE;
    i32x4 rsrc_a = make_rsrc((const char*)g.A + (int64_t)row_a * pitch, (uint32_t)rows_a * pitch);
    i32x4 rsrc_b = make_rsrc((const char*)g.Bt + (int64_t)row_b * pitch, (uint32_t)rows_b * pitch);

    // Loader: wave w brings rows 16w .. 16w + 15 of both operands, a load is 8 rows of one line. The offset inside the tile is range
    // checked: rows past the edge of a ragged tile, chunks past the end of K and slabs past the last one are zeros in LDS.
    uint32_t off[2];
    int chunk_k[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = wave * 16 + j * 8 + lane / 8, chunk = swizzle_slot(row, lane % 8, 8, 1);
        off[j] = (uint32_t)row * pitch + (uint32_t)chunk * CHUNK_BYTES;
        chunk_k[j] = chunk * CHUNK_ELEMS;
    }
    const int whole_k = KTAIL ? g.K & ~7 : g.K, all = (whole_k + MID_SLAB_K - 1) / MID_SLAB_K;
    int begin = 0, end = all;
    if (g.split_k > 1) {
        begin = __builtin_amdgcn_readfirstlane(slice_begin(all, slice, g.split_k));
        end = __builtin_amdgcn_readfirstlane(slice_begin(all, slice + 1, g.split_k));
    }
    const int slabs = end - begin;
    int ld_slab = begin + (int)(blockIdx.x % (unsigned)g.num_xcd) % slabs, ld_left = slabs, ld_stage = 0;
    auto load = [&](int i) __attribute__((always_inline)) {   // 0, 1: A; 2, 3: Bt
        uint32_t voff = off[i % 2];
        // (beyond every descriptor's range, which is below 2^31)
        if (KTAIL && ld_slab * MID_SLAB_K + chunk_k[i % 2] >= whole_k) voff = 0x80000000u;
        dma_load_b128(i < 2 ? rsrc_a : rsrc_b, ring + (uint32_t)(ld_stage * MID_STAGE + (i < 2 ? 0 : MID_OPERAND) + wave * 2048 + i % 2 * 1024), voff,
                      (uint32_t)ld_slab * (MID_SLAB_K * 2));
    };
    // (behind the last slab the loads go on, for the count of those in flight, with descriptors of no bytes)
    auto next_slab = [&]() __attribute__((always_inline)) {
        ld_slab = ld_slab + 1 == end ? begin : ld_slab + 1;
        if (--ld_left <= 0) { rsrc_a[2] = rsrc_b[2] = 0; ld_slab = 0; }
        ld_stage = ld_stage + 1 == MID_STAGES ? 0 : ld_stage + 1;
    };

    const int group = wave / 4, R = wave % 4 / 2, Cc = wave % 2;
    const int lr = lane & 15, lg = lane >> 4;
    const uint32_t slot = (uint32_t)(swizzle_slot(lr, group * 4 + lg, 8, 1) * CHUNK_BYTES);
    const uint32_t get_a = ring + (uint32_t)(R * 64 + lr) * (MID_SLAB_K * 2) + slot, get_b = ring + MID_OPERAND + (uint32_t)(Cc * 64 + lr) * (MID_SLAB_K * 2) + slot;
    u32x4 fa[2][WT], fb[2][WT];   // fragments of the slab being multiplied and of the next one
    f32x4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the values behind the last whole chunk: k 0 .. 7 of one k-step, lanes of chunk 0 (rows past the edge: the last row, never stored)
    const bool has_rest = KTAIL && whole_k != g.K && end == all && group == 0;
    uint32_t ta[WT][3] = {}, tb[WT][3] = {};
    if (KTAIL && has_rest && lg == 0) {
        const int row0_a = R * 64 + lr, row0_b = Cc * 64 + lr;
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            const int ra = row0_a + i * 16 < rows_a ? row0_a + i * 16 : rows_a - 1, rb = row0_b + i * 16 < rows_b ? row0_b + i * 16 : rows_b - 1;
            const uint32_t* at_a = (const uint32_t*)((const char*)g.A + (int64_t)(row_a + ra) * pitch + whole_k * 2);
            const uint32_t* at_b = (const uint32_t*)((const char*)g.Bt + (int64_t)(row_b + rb) * pitch + whole_k * 2);
#pragma unroll
            for (int d = 0; d < 3; ++d)
                if (whole_k + 2 * d < g.K) { ta[i][d] = at_a[d]; tb[i][d] = at_b[d]; }
        }
    }

#pragma unroll 1
    for (int p = 0; p < MID_STAGES; ++p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load(i);
        next_slab();
    }
    if (KTAIL && has_rest) {
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j)
                acc[i][j] = MfmaOp<DT>::run(u32x4{tb[j][0], tb[j][1], tb[j][2], 0}, u32x4{ta[i][0], ta[i][1], ta[i][2], 0}, acc[i][j]);
    }
    wait_vmcnt_imm<12>();   // slabs 0 and 1
    wg_barrier();
#pragma unroll
    for (int i = 0; i < WT; ++i) {
        fa[0][i] = *(const CK_LDS u32x4*)(uintptr_t)(get_a + i * 16 * MID_SLAB_K * 2);
        fb[0][i] = *(const CK_LDS u32x4*)(uintptr_t)(get_b + i * 16 * MID_SLAB_K * 2);
    }
    uint32_t stage = 0;
    // Body s: its fragments are in f[P]. Behind its barrier slab s + 2 is complete (this wave's loads of s + 3 and s + 4 may fly), and every
    // wave holds the fragments of s: slab s + 5 takes their stage. (After the last slab the fragments of a stage that nothing needs are read.)
    auto body = [&](auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value;
        stage = stage + 1 == MID_STAGES ? 0 : stage + 1;
        const uint32_t at_a = get_a + stage * MID_STAGE, at_b = get_b + stage * MID_STAGE;
        use_fragments(fa[P], fb[P]);
        wait_vmcnt_imm<8>();
        wg_barrier();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            load(j);
            if (j == WT - 1) next_slab();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int f = j * 2 + i;
                if (f < WT) fa[1 - P][f] = *(const CK_LDS u32x4*)(uintptr_t)(at_a + f * 16 * MID_SLAB_K * 2);
                else fb[1 - P][f - WT] = *(const CK_LDS u32x4*)(uintptr_t)(at_b + (f - WT) * 16 * MID_SLAB_K * 2);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < WT; ++i) acc[i][j] = MfmaOp<DT>::run(fb[P][j], fa[P][i], acc[i][j]);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
#pragma unroll 1
    for (; s + 1 < slabs; s += 2) {
        body(std::integral_constant<int, 0>{});
        body(std::integral_constant<int, 1>{});
    }
    if (s < slabs) body(std::integral_constant<int, 0>{});

    // The partial sums in rows: every wave writes its wave tile, and of the two waves of one place each finishes 32 rows, 16 lanes to
    // a row. (No load, of nothing, is on its way into LDS any more.)
    wait_vmcnt_imm<0>();
    wait_lgkmcnt0();
    wg_barrier();
    CK_LDS char* const out = (CK_LDS char*)ck_smem;
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
            *(CK_LDS f32x4*)(out + wave * MID_OUT_WAVE + (i * 16 + lr) * MID_OUT_ROW + (j * 16 + lg * 4) * 4) = acc[i][j];
    const int m0 = row_a + R * 64 + group * 32 + lg, n0 = row_b + Cc * 64 + lr * 4;
    f32x4 c[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) c[t] = row_c<DT>(g, m0 + t * 4, n0);
    wait_lgkmcnt0();
    wg_barrier();
    float* const plane = g.D + (int64_t)slice * g.M * g.N;   // (more than one slice: fp32 planes of a workspace)
    const CK_LDS char* first = out + wave % 4 * MID_OUT_WAVE + (group * 32 + lg) * MID_OUT_ROW + lr * 16;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const CK_LDS char* at = first + t * 4 * MID_OUT_ROW;
        store_row<DT>(g, plane, m0 + t * 4, n0, *(const CK_LDS f32x4*)at + *(const CK_LDS f32x4*)(at + 4 * MID_OUT_WAVE), c[t]);
    }

    if (blockIdx.x == 0 && threadIdx.x == blockDim.x - 1) {
        const unsigned long long dc = clock64() - clk0, dw = wall_clock64() - wall0;
        g.status[2] = (unsigned)dc; g.status[3] = (unsigned)(dc >> 32);
        g.status[4] = (unsigned)dw; g.status[5] = (unsigned)(dw >> 32);
    }
}

}  // namespace ck
#endif  // CK_GEMM_MID_KERNEL_HIP_H
