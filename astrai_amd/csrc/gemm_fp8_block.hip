// e4m3fn MFMA GEMM with 128-block scales (1x128 activation groups, 128x128
// weight blocks): the 256x256 ping-pong kernel for large shapes (a K slab is
// exactly one scale block; the promotion runs in place on the accumulators),
// 128x128 tiles of the same instruction for mid-size shapes (a slab's product scaled before it
// joins the accumulator), the generic tiled kernel otherwise (one 16x16x128 MFMA per scale
// block, partial product promoted with sa[m,kb] * sb[n/128,kb]).
#include "gemm_wave128.cuh"
#include "gemm_mid128.cuh"
#include "gemm_small64.cuh"
#include "gemm_wide256.cuh"
#include "gemm_tile.cuh"

namespace w8a8 {

namespace {

// Tiles of 256 x 256, behind those of 128 x 256, where they fill most of the chip, or where 128 x 128 tiles would put a second workgroup
// on compute units (from 257 of them), which takes nearly twice as long as one, where a round of large tiles costs little more
// than the first (us, 128 x 128 / large: 14000 x 640 x 2048, 550 tiles, 42 / 25.5, x 512 14.5 / 11.5; 17000 x 384 x 2048, 399 tiles, 28.5 /
// 24.5, x 11008 152 / 117. Up to 512 tiles with few slabs end sooner: 17000 x 384 x 512 9.9 / 10.7, 12000 x 640 x 256 8.3 / 8.8).
bool large_tiles_take(const GemmArgs& g) {
    if ((g.n & 7) != 0 || g.out_kind != OUT_BF16) return false;
    return pingpong_shape_ok(g) || (g.k >= 256 && (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128) > 256);
}

// Tiles of 128 x 256 where those are one round of the chip and 128 x 128 tiles more than one, ahead of the large tiles, which leave
// half of the chip idle there (us, 256 x 256 / 128 x 256: 2100 x 2048 x 7168 73 / 52, 4000 x 2048 x 7168 77 / 66, 1100 x 4096 x 4096 46 /
// 32, 2000 x 4096 x 4096 49 / 40, 700 x 7168 x 2048 25.6 / 19.9, 2100 x 2048 x 1024 16.5 / 12.8, 1100 x 4096 x 256 9.5 / 8.6, 1700 10.4 / 9.8; not the fullest with the fewest slabs, 2048 10.2 / 10.4).
bool wide_tiles_take(const GemmArgs& g) {
    const int64_t small = (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128);
    return g.k >= (small > 448 ? 384 : 256) && wide256_shape_ok(g);
}

// Tails on smaller tiles as in tile_tail_rows (one launch / two; tiles of the tail): 4300 x 4096 x 4096 102 / 79 us (64), x 256
// 19.8 / 17.5; 4500 x 4096 x 4096 101 / 86 (128); 4700 101 / 98 (192), x 256 19.6 / 19.9; 5000 x 4096 x 256 (256) 19.9 / 21.8, x
// 1024 36.3 / 37.1, x 1536 46.1 / 46.1, x 4096 101 / 100, x 11008 249 / 233: more than 192 only with K from 1536 on.
int64_t block_tail_tiles(const GemmArgs& g) { return g.k >= 1536 ? 256 : 192; }

}  // namespace

bool launch_gemm_fp8_block128_tiled(const GemmArgs& g, hipStream_t stream) {
    if (!tiled_shape_ok(g) || (g.k & 127) != 0) return false;
    if (wide_tiles_take(g)) {
        launch_wide256<Op32F8<0>, SCALE_BLOCK128>(g, stream);
        return true;
    }
    if (large_tiles_take(g)) {
        if (const int r = tile_tail_rows(g, block_tail_tiles(g))) {
            GemmArgs head, tail;
            split_rows(g, r, false, head, tail);
            tail.sa = g.sa + (size_t)head.m * (g.k >> 7);   // a step per row and K block
            if (mid128_shape_ok(tail)) launch_mid128<Op32F8<0>, SCALE_BLOCK128>(tail, stream);
            else launch_small64<Op32F8<0>, SCALE_BLOCK128>(tail, stream);
            launch_pingpong<Op32F8<0>, SCALE_BLOCK128, PingPongCfgBlock>(head, stream);
            return true;
        }
        launch_pingpong<Op32F8<0>, SCALE_BLOCK128, PingPongCfgBlock>(g, stream);
        return true;
    }
    // the 256x256 configuration of the generic tiled kernel runs out of registers
    // with the per-block promotion; 128x128 and 64x64 do not
    const int64_t tiles128 = (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128);
    if (mid128_shape_ok(g))   // blocks of a few hundred to a few thousand tokens: 128 x 128 tiles of the 32x32x64 MFMA
        launch_mid128<Op32F8<0>, SCALE_BLOCK128>(g, stream);
    else if (small64_shape_ok(g))   // fewer tokens: 64 x 64 tiles behind a ring of stages
        launch_small64<Op32F8<0>, SCALE_BLOCK128>(g, stream);
    else if (tiles128 >= 192)
        launch_tiled<OpF8<0>, CfgMid, SCALE_BLOCK128>(g, stream);
    else
        launch_tiled<OpF8<0>, CfgSmall, SCALE_BLOCK128>(g, stream);
    return true;
}

}  // namespace w8a8
