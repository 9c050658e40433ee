// 128 x 128 tiles with the operands staged through registers: one workgroup of eight waves per tile of D, two LDS stages of 128 k.
//
// What bounds it: a segment (64 KiB of operands) takes about 1.2 us, on one CU as on all of them, where its MFMAs take 0.43: the
// phases of a wave - fragment reads, MFMAs, writes of the next segment - add up instead of covering each other. The compiled loop
// shows where: the wait in front of the barrier orders memory accesses only, so the compiler moves the MFMAs of the second k-step
// behind it, and the eight writes drain with no MFMA of their own wave beside them; at the head of every other segment all 16
// fragment reads are waited for before the first MFMA; the test for the end of K splits the loop into blocks that the scheduler
// does not cross. The kernel takes all 256 registers of a wave. (The ring kernels on the same tile take 1.3 us with two stages as with five, with direct-to-LDS loads
// and fragments read one k-step ahead; neither the rate of the loads nor L2 is the limit.) A wave fetches its share of a segment
// into registers two segments ahead, whole 128-byte lines, and writes it to LDS behind the MFMAs of the first k-step.
//
// The waves form two groups of four; each covers the tile with wave tiles of 64 x 64 and takes two of a segment's four k-steps
// (16 MFMAs on 8 fragments: a third less LDS traffic than eight tiles of 32 x 64). The partial tiles of the two
// groups meet in LDS at the end, first + second.
// Against the ring kernel: bf16 256 x 16384 x 4096 with 16-bit results 59.3 -> 53.5 us (642 TFLOP/s; 49.9 -> 44.8 where
// the operands stay in the last-level cache from call to call), fp16 1024^2 x 4096 41.8 -> 39.0, 2048^3 25.8 -> 25.5. One workgroup
// per tile and CU: the launcher takes it where a deep K or fewer tiles than CUs make up for the prologue and epilogue of every tile.
#ifndef CK_GEMM_MID_KERNEL_HIP_H
#define CK_GEMM_MID_KERNEL_HIP_H

#include "gemm_fused_kernel.hip.h"

namespace ck {

constexpr int MID_TILE = 128;
constexpr int MID_SEGK = 128;
constexpr int MID_ROW_BYTES = MID_SEGK * 2;
constexpr int MID_OPERAND = MID_TILE * MID_ROW_BYTES;
constexpr int MID_LDS_BYTES = 2 * 2 * MID_OPERAND;

// Rows start on 16-byte boundaries and K % 8 == 0 (a 16-byte chunk of a row is inside it or past it).
template <typename DT>
__global__ __launch_bounds__(512) void gemm_mid_kernel(const GemmArgs g) {
    constexpr int WT = 4;   // 16 x 16 blocks per edge of a wave tile
    extern __shared__ __attribute__((aligned(1024))) char ck_smem[];
    CK_LDS char* const lds = (CK_LDS char*)ck_smem;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned long long clk0 = clock64(), wall0 = wall_clock64();

    const TileRC rc = tile_order(g.tiles_m, g.tiles_n, g.tile_group_m, xcd_tile(blockIdx.x, gridDim.x, g.num_xcd));
    const int row_a = rc.row * MID_TILE, row_b = rc.col * MID_TILE;
    const int64_t pitch = (int64_t)g.K * 2;
    const char* base_a = (const char*)g.A + row_a * pitch;
    const char* base_b = (const char*)g.Bt + row_b * pitch;

    // Loader: wave w brings rows 16w .. 16w + 15 of both operands, a load is 8 rows of one 128-byte line. Rows past the edge
    // of a ragged tile read the last row instead: what they give is never stored.
    const int lane_row = lane / 8, lane_chunk = lane % 8;
    uint32_t off_a[2], off_b[2];
    CK_LDS char* put[2][2];   // [rows 0 .. 7, 8 .. 15][first, second line of the segment]
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = wave * 16 + j * 8 + lane_row, ra = g.M - 1 - row_a, rb = g.N - 1 - row_b;
        off_a[j] = (uint32_t)(row < ra ? row : ra) * (uint32_t)pitch;
        off_b[j] = (uint32_t)(row < rb ? row : rb) * (uint32_t)pitch;
#pragma unroll
        for (int h = 0; h < 2; ++h) put[j][h] = lds + row * MID_ROW_BYTES + swizzle_slot(row, h * 8 + lane_chunk, 16, 1) * CHUNK_BYTES;
    }
    struct Part { u32x4 a[2][2], b[2][2]; };
    // (a segment past the end of K reads the row's last chunks over again: its part is never multiplied, and a fetch under no
    // condition lets the compiler count the loads in flight)
    auto fetch = [&](Part& p, int seg) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = seg * MID_SEGK + h * 64 + lane_chunk * 8;
            const uint32_t at = (uint32_t)(k < g.K - 8 ? k : g.K - 8) * 2;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                p.a[j][h] = *(const u32x4*)(base_a + (off_a[j] + at));
                p.b[j][h] = *(const u32x4*)(base_b + (off_b[j] + at));
            }
        }
    };
    auto stash = [&](Part& p, int seg, int stage) __attribute__((always_inline)) {
        if ((seg + 1) * MID_SEGK > g.K) {   // zeros from K on
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (seg * MID_SEGK + h * 64 + lane_chunk * 8 >= g.K)
#pragma unroll
                    for (int j = 0; j < 2; ++j) p.a[j][h] = p.b[j][h] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                *(CK_LDS u32x4*)(put[j][h] + stage * 2 * MID_OPERAND) = p.a[j][h];
                *(CK_LDS u32x4*)(put[j][h] + stage * 2 * MID_OPERAND + MID_OPERAND) = p.b[j][h];
            }
    };
    auto meet = []() __attribute__((always_inline)) {   // every wave's LDS accesses are done
        wait_lgkmcnt0();
        wg_barrier();
    };

    const int group = wave / 4, R = wave % 4 / 2, Cc = wave % 2;
    const int lr = lane & 15, lg = lane >> 4;
    const CK_LDS char* get_a[2];
    const CK_LDS char* get_b[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int chunk = (group * 2 + s) * 4 + lg;
        get_a[s] = lds + (R * 64 + lr) * MID_ROW_BYTES + swizzle_slot(lr, chunk, 16, 1) * CHUNK_BYTES;
        get_b[s] = lds + MID_OPERAND + (Cc * 64 + lr) * MID_ROW_BYTES + swizzle_slot(lr, chunk, 16, 1) * CHUNK_BYTES;
    }
    f32x4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int segs = (g.K + MID_SEGK - 1) / MID_SEGK;
    // Segment s lies in stage STAGE, segment s + 1 in p on its way: the fragments of s first, then p goes to the other stage
    // (whose readers met at the barrier before) and the loads of s + 3 take its registers, then the MFMAs.
    auto segment = [&](int s, auto stage_index, Part& p) __attribute__((always_inline)) {
        constexpr int STAGE = decltype(stage_index)::value;
        u32x4 a[2][WT], b[2][WT];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < WT; ++i) {
                a[t][i] = *(const CK_LDS u32x4*)(get_a[t] + STAGE * 2 * MID_OPERAND + i * 16 * MID_ROW_BYTES);
                b[t][i] = *(const CK_LDS u32x4*)(get_b[t] + STAGE * 2 * MID_OPERAND + i * 16 * MID_ROW_BYTES);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j) acc[i][j] = MfmaOp<DT>::run(b[0][j], a[0][i], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        stash(p, s + 1, 1 - STAGE);
        fetch(p, s + 3);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j) acc[i][j] = MfmaOp<DT>::run(b[1][j], a[1][i], acc[i][j]);
        meet();
    };
    Part odd, even;
    fetch(even, 0);
    fetch(odd, 1);
    stash(even, 0, 0);
    fetch(even, 2);
    meet();
    int s = 0;
    for (; s + 1 < segs; s += 2) {
        segment(s, std::integral_constant<int, 0>{}, odd);
        segment(s + 1, std::integral_constant<int, 1>{}, even);
    }
    if (s < segs) segment(s, std::integral_constant<int, 0>{}, odd);

    // (the lane's number once more: carried through the loop it and what comes of it went to scratch memory)
    const int out_lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), out_lr = out_lane & 15, out_lg = out_lane >> 4;
    // The two partial sums of a wave tile: the first group keeps the upper half of the block rows, the second the lower one, and
    // each hands the other half over.
    const bool lower = group != 0;
    CK_LDS char* mine = lds + wave * (WT / 2 * WT * 1024) + out_lane * 16;
    const CK_LDS char* theirs = lds + (wave ^ 4) * (WT / 2 * WT * 1024) + out_lane * 16;
#pragma unroll
    for (int i = 0; i < WT / 2; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) *(CK_LDS f32x4*)(mine + (i * WT + j) * 1024) = lower ? acc[i][j] : acc[WT / 2 + i][j];
    meet();
    const bool vec_cols = g.vec_store && (rc.col + 1) * MID_TILE <= g.N;
#pragma unroll
    for (int i = 0; i < WT / 2; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            const f32x4 sum = (lower ? acc[WT / 2 + i][j] : acc[i][j]) + *(const CK_LDS f32x4*)(theirs + (i * WT + j) * 1024);
            epilogue_block<DT>(g, row_a + R * 64 + ((lower ? WT / 2 : 0) + i) * 16 + out_lr, row_b + Cc * 64 + j * 16 + out_lg * 4, sum, vec_cols);
        }

    if (blockIdx.x == 0 && wave == 7 && out_lane == 63) {
        const unsigned long long dc = clock64() - clk0, dw = wall_clock64() - wall0;
        g.status[2] = (unsigned)dc; g.status[3] = (unsigned)(dc >> 32);
        g.status[4] = (unsigned)dw; g.status[5] = (unsigned)(dw >> 32);
    }
}

}  // namespace ck
#endif  // CK_GEMM_MID_KERNEL_HIP_H
