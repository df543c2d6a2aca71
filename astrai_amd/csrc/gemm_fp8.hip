// fp8 (OCP e4m3fn / e5m2) MFMA GEMMs, per-tensor scales (optional bias, bf16 /
// e4m3 / fp32 output) or one scale per activation row and per weight row (bf16 output).
// Large shapes run 256x256 tiles: the four-wave 128x128-register-tile kernel for bf16
// output (v_mfma_f32_16x16x128_f8f6f4), the eight-wave ping-pong kernel (32x32x64) for the other outputs; bf16 shapes with too few of
// those tiles for the chip run 128x256, 128x128 or 64x64 tiles of that instruction; the generic
// tiled kernel takes everything else.
#include "gemm_wave128_q16.cuh"
#include "gemm_mid128.cuh"
#include "gemm_small64.cuh"
#include "gemm_wide256.cuh"
#include "gemm_tile.cuh"

namespace w8a8 {

namespace {
template <int Fmt, int ScaleKind>
void launch_big(const GemmArgs& g, hipStream_t stream) {
    if (!g.bias || !g.round_first) return launch_wave128_q16<Fmt, ScaleKind>(g, stream);
    if constexpr (Fmt == 0 && ScaleKind == SCALE_TENSOR) return launch_wave128_q16<0, SCALE_TENSOR, true>(g, stream);
    // (no instance: nothing asks for the others often)
    GemmArgs plain = g;
    plain.bias = nullptr;
    launch_wave128_q16<Fmt, ScaleKind>(plain, stream);
    launch_add_bias_bf16(g.out, g.bias, g.m, g.n, stream);
}
template <int Fmt, int ScaleKind>
void launch_for(const GemmArgs& g, hipStream_t stream) {
    if (wide256_shape_ok(g)) return launch_wide256<Op32F8<Fmt>, ScaleKind>(g, stream);
#ifndef W8A8_NO_WAVE128
    if (wave128_takes(g)) {
        GemmArgs head, tail;
        if (const int r = ragged_tail_rows(g)) {
            split_rows(g, r, ScaleKind == SCALE_ROWCOL, head, tail);
            if (wave128_shape_ok(head) && launch_gemv_fp8(tail, Fmt, ScaleKind, stream))   // (disjoint rows: either order)
                return launch_big<Fmt, ScaleKind>(head, stream);
        }
        if (const int r = tile_tail_rows(g)) {
            split_rows(g, r, ScaleKind == SCALE_ROWCOL, head, tail);
            if (wide256_shape_ok(tail)) launch_wide256<Op32F8<Fmt>, ScaleKind>(tail, stream);
            else if (mid128_shape_ok(tail)) launch_mid128<Op32F8<Fmt>, ScaleKind>(tail, stream);
            else launch_small64<Op32F8<Fmt>, ScaleKind>(tail, stream);
            return launch_big<Fmt, ScaleKind>(head, stream);
        }
        return launch_big<Fmt, ScaleKind>(g, stream);
    }
#endif
    if (pingpong_shape_ok(g)) return launch_pingpong<Op32F8<Fmt>, ScaleKind>(g, stream);
    if (mid128_shape_ok(g)) return launch_mid128<Op32F8<Fmt>, ScaleKind>(g, stream);
    if (small64_shape_ok(g)) return launch_small64<Op32F8<Fmt>, ScaleKind>(g, stream);
    launch_tiled_auto<OpF8<Fmt>, ScaleKind>(g, stream);
}
}  // namespace

bool launch_gemm_fp8_tiled(const GemmArgs& g, int fmt, hipStream_t stream) {
    if (!tiled_shape_ok(g)) return false;
    if (fmt) launch_for<1, SCALE_TENSOR>(g, stream);
    else launch_for<0, SCALE_TENSOR>(g, stream);
    return true;
}

bool launch_gemm_fp8_rowcol_tiled(const GemmArgs& g, int fmt, hipStream_t stream) {
    if (!tiled_shape_ok(g) || g.out_kind != OUT_BF16) return false;
    if (fmt) launch_for<1, SCALE_ROWCOL>(g, stream);
    else launch_for<0, SCALE_ROWCOL>(g, stream);
    return true;
}

}  // namespace w8a8
