// The 256x256x128-byte tile of the four-wave NT products and the shapes that take it (the main loop: gemm_walk16.cuh;
// fp8: gemm_wave128_q16.cuh, int8: gemm_wave128_i8.cuh, bf16: mix_gemm.hip).
//
// Why four waves of 128(m) x 128(n). A wave tile reads (128+128) x 128 bytes of operands from LDS per K slab for 2048 MFMA
// cycles: 128 KiB per workgroup and slab against the 192 KiB of eight 128x64 wave tiles. LDS serves both the
// operand reads and the incoming direct-to-LDS loads (64 KiB a slab), so that
// third less read traffic is what lets the MFMA pipe stay busy. The price: the
// 256 accumulator registers of a wave leave room for one wave per SIMD only, so
// nothing can hide one wave's memory phase behind another wave's MFMAs -- each
// wave interleaves its own LDS reads and loads between its own MFMAs instead.
// No L2 prefetch touches: a touch pulls its whole line through the CU's one load path a second
// time, which costs more than the L2 misses it saves.
//
// LDS layout of a stage: 256 rows of 128 bytes, chunk c (16 bytes) of row r at position c ^ (r & 7) ^ ((r >> 3) & 1).
#pragma once
#include "gemm_pingpong.cuh"

namespace w8a8 {

struct Wave128Cfg {
    static constexpr int BM = 256, BN = 256, BK = 128;
    static constexpr int THREADS = 256;
    static constexpr int OPERAND_BYTES = 256 * BK;       // one operand's slab: 32 KiB
    static constexpr int X_STAGES = 3, W_STAGES = 2;
    static constexpr int W_BASE = X_STAGES * OPERAND_BYTES;  // weights after activations
    static constexpr int EPI_ROW_BYTES = 272;            // 128 bf16 + 16 bytes of padding
    static constexpr int EPI_PASS_BYTES = 32 * EPI_ROW_BYTES;  // one 32-row pass of a wave
    static constexpr int LDS_BYTES = (X_STAGES + W_STAGES) * OPERAND_BYTES;  // all 160 KiB
    static_assert(4 * 2 * EPI_PASS_BYTES <= LDS_BYTES, "epilogue staging must fit");
};

// bf16 output with whole 16-byte output pieces only; other outputs keep the
// ping-pong kernel, whose epilogue handles every case
inline bool wave128_shape_ok(const GemmArgs& g) {
    // (a tile's 256 output rows are addressed with 32-bit byte offsets)
    return pingpong_shape_ok(g) && g.out_kind == OUT_BF16 && (g.n & 7) == 0 && g.n <= (1 << 22);
}

// A token count a little above a multiple of 256 (M = 256 q + r, 0 < r <= 128) can cost the
// large-tile kernel a whole extra round of workgroups for r rows (4100 x 4096 x 4096: 272 tiles on
// 256 compute units, 96 us against 69 us at 4096 rows). When it does, and the weight-streaming
// decode kernel takes the shape, those rows are better served by it in a launch of their own
// (70 us for the two). Returns r then, else 0.
inline int ragged_tail_rows(const GemmArgs& g) {
    const int r = g.m & 255;
    if (r == 0 || r > 128 || g.m < 256 || (g.k & 255) != 0) return 0;
    const int64_t tn = (g.n + 255) / 256;
    const int64_t full = (int64_t)((g.m + 255) / 256) * tn, cut = (int64_t)(g.m / 256) * tn;
    return (full + 255) / 256 > (cut + 255) / 256 ? r : 0;
}

// the first m - r rows and the last r rows of a product as calls of their own (bf16 output;
// `rowcol`: sa holds one step per row)
inline void split_rows(const GemmArgs& g, int r, bool rowcol, GemmArgs& head, GemmArgs& tail) {
    head = g;
    head.m = g.m - r;
    tail = g;
    tail.m = r;
    const size_t row0 = (size_t)head.m;
    tail.a = static_cast<const uint8_t*>(g.a) + row0 * (size_t)g.k;
    if (rowcol) tail.sa = g.sa + row0;
    tail.out = static_cast<uint8_t*>(g.out) + row0 * (size_t)g.n * 2;
    if (g.resid) tail.resid = static_cast<const uint8_t*>(g.resid) + row0 * (size_t)g.n * 2;
}

// Plain bf16 products that the large tiles take, behind wide256_shape_ok: where they fill most of the chip, or from 449 tiles of 128 x
// 128 on (those past what tiles of 128 x 256 do in one round: few columns). Two
// workgroups of those share a compute unit and take longer the more units have two, where a round of large tiles costs
// the same however empty (us, 128 x 128 / large, fp8 and int8: 14000 x 640 x 512, 550 tiles, 12.1 / 11.0 and 13.2 / 12.6, x 4096 48 / 36
// and 53 / 39; 12000 x 640 x 11008, 470 tiles, 103 / 89 and 106 / 91). What it costs: up to 512 tiles with K to 4096 (12000 x 640 x 512
// 9.6 / 10.8 and 10.4 / 12.4, x 2048 19.9 / 22.0 and 21.7 / 23.9, x 4096 34.0 / 36.2 and 37.0 / 38.7).
inline bool wave128_takes(const GemmArgs& g) {
    if (wave128_shape_ok(g)) return true;
    if (!tiled_shape_ok(g) || (g.k & 127) != 0 || g.k < 256 || g.out_kind != OUT_BF16 || (g.n & 7) != 0 || g.n > (1 << 22))
        return false;
    return (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128) > 448;
}

// Rows of a product that are better served by smaller tiles in a launch of their own: those past the last
// row of tiles that fits whole rounds of 256 large tiles, where they make up at most kTailTiles tiles of
// 128 x 128. Returns their number, else 0. The last round of large tiles costs nearly as much with few tiles as
// with many. Measured (fp8, one launch -> two; tiles of the tail): 4300 x 4096 x 4096 84 -> 63 us (64), 4300 x 4096 x
// 11008 199 -> 142 (64), 3001 x 11264 x 2048 77 -> 73 (176), 3001 x 11008 x 4096 133 -> 123 (172), 5000 x 4096 x 4096
// 86 -> 77 (256), 5500 x 4096 x 4096 87 -> 84 (352); beyond that nothing is left: 6000 x 4096 x 4096 89 -> 89
// (480), 6500 x 11264 x 2048 134 -> 141 (440).
constexpr int64_t kTailTiles = 384;
inline int tile_tail_rows(const GemmArgs& g, int64_t most = kTailTiles) {
    const int64_t tm = (g.m + 255) / 256, tn = (g.n + 255) / 256, rounds = (tm * tn + 255) / 256;
    const int64_t head = (rounds - 1) * 256 / tn;  // row tiles that stay
    if (rounds < 2 || head < 1 || head >= tm) return 0;
    const int64_t rows = g.m - head * 256;
    return (rows + 127) / 128 * ((g.n + 127) / 128) <= most ? (int)rows : 0;
}

}  // namespace w8a8
