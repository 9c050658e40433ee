// Small products: no LDS ring and no barrier in the loop. One workgroup of eight waves computes one tile of D; its waves share
// the tile and split K, each wave fetching its own operand chunks into registers, and the eight partial tiles meet once, in
// LDS, at the end.
//
// What bounds it: a call of a few microseconds is memory latency and the launch. A ring pays that latency in the prologue and
// a barrier per segment behind it, with one workgroup per 64 x 64 tile (512^3: 64 of 256 CUs). Here the loads of DEPTH units
// of 64 k are in flight per wave before the first of them is used, and 32 x 32 tiles give four times the workgroups.
//
// The fragments an MFMA takes have 16 rows in 16 neighbouring lanes. Loaded that way every lane starts a line of its own, and
// the memory path takes one such lane per cycle (18 bytes per cycle and CU; 512 x 512 x 2048: 10.0 us a launch, 6.4 as it is). So a wave loads
// whole 128-byte lines, 8 lanes to a row, and turns them round through an LDS buffer of its own (no barrier: one wave's LDS
// accesses stay in order), with the chunks of a row exchanged as in the ring kernels against bank conflicts.
//
// Rows need not start on 16-byte boundaries: the vector memory path takes a 16-byte load from any 4-byte boundary at the full
// rate (EVEN: K even, operands on 4-byte boundaries), and rows on 2-byte boundaries are put together from such loads. So
// there are no zero-padded operand copies here: one launch instead of two and no scratch memory.
#ifndef CK_GEMM_DIRECT_KERNEL_HIP_H
#define CK_GEMM_DIRECT_KERNEL_HIP_H

#include "gemm_pc_kernel.hip.h"

namespace ck {

constexpr int DIRECT_WAVES = 8;
constexpr int DIRECT_UNIT_K = 64;   // one 128-byte line of an operand row
constexpr int DIRECT_ROW_BYTES = DIRECT_UNIT_K * 2;
// dynamic LDS for tiles of T x T: per wave one unit of both operands; afterwards its partial tile
constexpr int direct_lds_bytes(int T) { return DIRECT_WAVES * 2 * T * DIRECT_ROW_BYTES; }

// WT: 16 x 16 blocks per tile edge (2: 32 x 32 tiles, 4: 64 x 64 tiles); DEPTH: units in flight per wave; SLICED: work items are (tile, K slice), an
// instance of its own because its divisions and bounds cost a call of 6 to 10 us 0.1 to 0.25 us
template <typename DT, int WT, int DEPTH, bool EVEN, bool SLICED>
__global__ __launch_bounds__(DIRECT_WAVES * 64) void gemm_direct_kernel(const GemmArgs g) {
    constexpr int T = WT * 16;
    constexpr int BLOCKS = WT * WT;
    constexpr int LOADS = T / 8;        // wave loads per operand and unit: 8 rows of 128 bytes each
    constexpr int OPERAND = T * DIRECT_ROW_BYTES;
    static_assert(BLOCKS * 1024 <= 2 * OPERAND, "a wave's partial tile takes the place of its unit buffer");
    extern __shared__ __attribute__((aligned(1024))) char ck_smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned long long clk0 = clock64(), wall0 = wall_clock64();

    // work items: the tiles of the first K slice, then those of the second ...
    const int item = xcd_tile(blockIdx.x, gridDim.x, g.num_xcd), tiles = g.tiles_m * g.tiles_n, slice = SLICED ? item / tiles : 0;
    const TileRC rc = tile_order(g.tiles_m, g.tiles_n, g.tile_group_m, item - slice * tiles);
    const int row_a = rc.row * T, row_b = rc.col * T;
    const int64_t pitch = (int64_t)g.K * 2;
    const char* base_a = (const char*)g.A + row_a * pitch;
    const char* base_b = (const char*)g.Bt + row_b * pitch;
    // Load l of an operand: rows 8l .. 8l + 7, lane (row, chunk). Rows past the edge of a ragged tile read the last row
    // instead: what they give is never stored.
    const int lane_row = lane / 8, lane_chunk = lane % 8;
    uint32_t off_a[LOADS], off_b[LOADS];   // the lane's row, in bytes from the tile's first
    // EVEN false: byte selectors (x[i], x[i - 1]) -> elements 2i, 2i + 1 of a chunk, and the same for i = 0 with element 0 in the place of x[-1]
    constexpr uint32_t ON_EVEN = 0x07060504u;
    uint32_t sel_a[LOADS], sel_b[LOADS], sel0_a[LOADS], sel0_b[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const int row = l * 8 + lane_row, ra = g.M - 1 - row_a, rb = g.N - 1 - row_b;
        off_a[l] = (uint32_t)(row < ra ? row : ra) * (uint32_t)pitch;
        off_b[l] = (uint32_t)(row < rb ? row : rb) * (uint32_t)pitch;
        const bool odd_a = ((uint32_t)(uintptr_t)base_a + off_a[l]) & 2, odd_b = ((uint32_t)(uintptr_t)base_b + off_b[l]) & 2;
        sel_a[l] = odd_a ? 0x05040302u : ON_EVEN;
        sel0_a[l] = odd_a ? 0x05040100u : ON_EVEN;
        sel_b[l] = odd_b ? 0x05040302u : ON_EVEN;
        sel0_b[l] = odd_b ? 0x05040100u : ON_EVEN;
    }

    // A fetched unit. EVEN: its chunks. Otherwise a chunk whose first element lies on an odd 2-byte boundary comes as its
    // elements 1 .. 8 from the 4-byte boundary behind it, and element 0 beside them: a 16-byte load from an odd boundary is
    // taken apart into its lanes by the memory path (200 x 136 x 1001: 10.8 us a launch with such loads, 5.1 with K 1002).
    struct Unit {
        u32x4 a[LOADS], b[LOADS];
        uint32_t head_a[LOADS], head_b[LOADS];
    };
    typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
    auto fetch_chunk = [](const char* base, uint32_t off, uint32_t sel, u32x4& x, uint32_t& head) __attribute__((always_inline)) {
        if constexpr (EVEN) x = (u32x4)*(const u32x4_a4*)(base + off);
        else {
            // (elements 1 .. 8 of a chunk are in the row: the unit with the end of K is not fetched here)
            x = (u32x4)*(const u32x4_a4*)(base + (off + (sel == ON_EVEN ? 0u : 2u)));
            head = *(const unsigned short*)(base + off);
        }
    };
    auto fetch = [&](Unit& f, int u) __attribute__((always_inline)) {
        const uint32_t k = (uint32_t)(u * DIRECT_UNIT_K + lane_chunk * 8) * 2;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            fetch_chunk(base_a, off_a[l] + k, sel_a[l], f.a[l], f.head_a[l]);
            fetch_chunk(base_b, off_b[l] + k, sel_b[l], f.b[l], f.head_b[l]);
        }
    };
    // Of a slice's whole units, the w-th, w + 8-th, ... belong to wave w; the one with the end of K comes first in the wave that it falls to. (EVEN
    // false: also a K that is a multiple of 64 ends in such a unit, since the element behind a chunk is read as well.)
    const int whole = EVEN ? g.K / DIRECT_UNIT_K : (g.K - 1) / DIRECT_UNIT_K;
    const int units = whole + (whole * DIRECT_UNIT_K != g.K);
    int begin = 0, end = units;
    if constexpr (SLICED) {
        begin = slice_begin(units, slice, g.split_k);
        end = slice_begin(units, slice + 1, g.split_k);
    }
    const bool has_end = end > whole && (whole - begin) % DIRECT_WAVES == wave;
    // In the unit with the end of K, chunks that reach past a row's end are read so that they end with the row (K >= 8), and
    // mask_end drops what lies in front of them and fills up with zeros. Two steps, so that nothing waits for the loads
    // between them.
    const int k_end = whole * DIRECT_UNIT_K + lane_chunk * 8;
    auto fetch_end = [&](Unit& f) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)(k_end < g.K - 8 ? k_end : g.K - 8) * 2;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            f.a[l] = (u32x4)*(const u32x4_a2*)(base_a + (off_a[l] + at));
            f.b[l] = (u32x4)*(const u32x4_a2*)(base_b + (off_b[l] + at));
        }
    };
    auto mask_end = [&](Unit& f) __attribute__((always_inline)) {
        const int past = k_end - (g.K - 8), drop = past > 0 ? past * 16 : 0;   // bits in front of the chunk's first element
        auto masked = [&](u32x4& x, uint32_t& head, uint32_t sel) __attribute__((always_inline)) {
            uint64_t lo = x[0] | (uint64_t)x[1] << 32, hi = x[2] | (uint64_t)x[3] << 32;
            if (drop >= 64) { lo = drop >= 128 ? 0 : hi >> (drop - 64); hi = 0; }
            else if (drop) { lo = lo >> drop | hi << (64 - drop); hi >>= drop; }
            if constexpr (!EVEN) {   // in the form that fetch_chunk leaves
                head = (uint32_t)lo & 0xffffu;
                if (sel != ON_EVEN) { lo = lo >> 16 | hi << 48; hi >>= 16; }
            }
            x = u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
        };
#pragma unroll
        for (int l = 0; l < LOADS; ++l) { masked(f.a[l], f.head_a[l], sel_a[l]); masked(f.b[l], f.head_b[l], sel_b[l]); }
    };

    // the unit goes through the wave's LDS buffer into fragments
    CK_LDS char* buffer = (CK_LDS char*)ck_smem + wave * 2 * OPERAND;
    CK_LDS char* put_even = buffer + lane_row * DIRECT_ROW_BYTES + swizzle_slot(lane_row, lane_chunk, 8, 1) * CHUNK_BYTES;      // rows 0 .., 16 ..
    CK_LDS char* put_odd = buffer + (8 + lane_row) * DIRECT_ROW_BYTES + swizzle_slot(8 + lane_row, lane_chunk, 8, 1) * CHUNK_BYTES;   // rows 8 .., 24 ..
    const int lr = lane & 15, lg = lane >> 4;
    const CK_LDS char* get[2] = {buffer + lr * DIRECT_ROW_BYTES + swizzle_slot(lr, lg, 8, 1) * CHUNK_BYTES,
                                 buffer + lr * DIRECT_ROW_BYTES + swizzle_slot(lr, 4 + lg, 8, 1) * CHUNK_BYTES};
    auto in_order = [](u32x4 x, uint32_t head, uint32_t sel, uint32_t sel0) __attribute__((always_inline)) {
        if constexpr (EVEN) return x;
        else return u32x4{__builtin_amdgcn_perm(x[0], head, sel0), __builtin_amdgcn_perm(x[1], x[0], sel), __builtin_amdgcn_perm(x[2], x[1], sel),
                          __builtin_amdgcn_perm(x[3], x[2], sel)};
    };
    auto stash = [&](const Unit& f) __attribute__((always_inline)) {
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            CK_LDS char* to = (l % 2 ? put_odd : put_even) + l / 2 * 16 * DIRECT_ROW_BYTES;
            *(CK_LDS u32x4*)to = in_order(f.a[l], f.head_a[l], sel_a[l], sel0_a[l]);
            *(CK_LDS u32x4*)(to + OPERAND) = in_order(f.b[l], f.head_b[l], sel_b[l], sel0_b[l]);
        }
    };
    f32x4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // lanes read what other lanes of the wave wrote: the compiler, which sees one lane, may not exchange the two
    auto wave_order = []() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto multiply = [&]() __attribute__((always_inline)) {
        wave_order();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 a[WT], b[WT];
#pragma unroll
            for (int i = 0; i < WT; ++i) {
                a[i] = *(const CK_LDS u32x4*)(get[h] + i * 16 * DIRECT_ROW_BYTES);
                b[i] = *(const CK_LDS u32x4*)(get[h] + OPERAND + i * 16 * DIRECT_ROW_BYTES);
            }
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j) acc[i][j] = MfmaOp<DT>::run(b[j], a[i], acc[i][j]);
        }
        wave_order();
    };

    const int first = begin + (has_end ? wave - DIRECT_WAVES : wave), stop = end < whole ? end : whole;
    const int mine = first < stop ? (stop - first + DIRECT_WAVES - 1) / DIRECT_WAVES : 0;   // units of this wave
    Unit f[DEPTH];
    auto fetch_first = [&]() __attribute__((always_inline)) {
        if (has_end) fetch_end(f[0]);
        else fetch(f[0], first);
    };
    // (The fetches of the long loop stand under no condition: the compiler counts the loads in flight, and one that may or may
    // not have been issued makes every wait behind it a wait for all of them.)
    if (mine >= DEPTH) {
        fetch_first();
#pragma unroll
        for (int d = 1; d < DEPTH; ++d) fetch(f[d], first + d * DIRECT_WAVES);
        if (has_end) mask_end(f[0]);
        int u = first + DEPTH * DIRECT_WAVES, left = mine - DEPTH;   // the next unit to fetch; units not yet fetched
        for (; left >= DEPTH; left -= DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                stash(f[d]);
                fetch(f[d], u);
                u += DIRECT_WAVES;
                multiply();
            }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            stash(f[d]);
            if (d < left) fetch(f[d], u + d * DIRECT_WAVES);
            multiply();
        }
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d)
            if (d < left) { stash(f[d]); multiply(); }
    } else if (mine > 0) {
        fetch_first();
#pragma unroll
        for (int d = 1; d < DEPTH - 1; ++d)
            if (d < mine) fetch(f[d], first + d * DIRECT_WAVES);
        if (has_end) mask_end(f[0]);
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d)
            if (d < mine) { stash(f[d]); multiply(); }
    }

    // The partial tiles, each in its wave's buffer (a wave writes it behind its own last fragment reads), added in the waves'
    // order by the waves that had a share of K.
    const int waves = end - begin < DIRECT_WAVES ? end - begin : DIRECT_WAVES;
    const bool whole_cols = (rc.col + 1) * T <= g.N;
    GemmArgs go = g;
    if constexpr (SLICED) go.D = g.D + (int64_t)slice * g.M * g.N;   // fp32 planes of a workspace
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) *(CK_LDS f32x4*)(buffer + b * 1024 + lane * 16) = acc[b / WT][b % WT];
    __syncthreads();
    for (int b = wave; b < BLOCKS; b += DIRECT_WAVES) {
        const CK_LDS char* at = (const CK_LDS char*)ck_smem + b * 1024 + lane * 16;
        f32x4 sum = *(const CK_LDS f32x4*)at;
        for (int w = 1; w < waves; ++w) sum += *(const CK_LDS f32x4*)(at + w * 2 * OPERAND);
        const f32x4 block[1][1] = {{sum}};
        epilogue_blocks<DT, 1, 1>(go, row_a + b / WT * 16 + lr, row_b + b % WT * 16 + lg * 4, block, whole_cols);
    }

    if (blockIdx.x == 0 && threadIdx.x == blockDim.x - 1) {
        const unsigned long long dc = clock64() - clk0, dw = wall_clock64() - wall0;
        g.status[2] = (unsigned)dc; g.status[3] = (unsigned)(dc >> 32);
        g.status[4] = (unsigned)dw; g.status[5] = (unsigned)(dw >> 32);
    }
}

}  // namespace ck
#endif  // CK_GEMM_DIRECT_KERNEL_HIP_H
