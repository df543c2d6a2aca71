// fp8 products on 256 x 256 tiles, per-tensor or row x column scales, bf16 output: the main loop of gemm_walk16.cuh on
// v_mfma_f32_16x16x128_f8f6f4, scales and bias in the epilogue.
//
// What bounds it: the power cap. Against the 32x32x64 MFMA on the same tile 49.6 for 52.3 us at 4096^3 on normally
// distributed operands; with sums pinned in place, load offsets formed once and operands read in the first half of a
// quadrant then 8000 x 4096 x 11008 321 -> 314 us, 8000 x 2048 x 11264 190 -> 182 (dynamic scaling's passes included).
#pragma once
#include "gemm_walk16.cuh"

namespace w8a8 {

// RoundFirst (per-tensor scales): the product is rounded to bf16 before the bias joins it
template <int Fmt, int ScaleKind, bool RoundFirst = false>
__global__ __launch_bounds__(Wave128Cfg::THREADS) void gemm_wave128_q16_kernel(GemmArgs g) {
    static_assert(ScaleKind == SCALE_TENSOR || ScaleKind == SCALE_ROWCOL, "per-tensor or row x column scales");
    PP_STAMP_INIT();
    using Cfg = Wave128Cfg;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave & 1;
    const int wave_n = wave >> 1;
    const int lrow = lane & 15;
    const int lgrp = lane >> 4;

    const int tiles_m = (g.m + Cfg::BM - 1) / Cfg::BM;
    const int tiles_n = (g.n + Cfg::BN - 1) / Cfg::BN;
    const TileCoord tc = map_tile(tiles_m, tiles_n);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * Cfg::BN;
    const int K = g.k;
    const int ksteps = K >> 7;
    // requested now, used in the epilogue: the latency hides under the main loop
    const EpilogueScalars es = load_epilogue_scalars<ScaleKind>(g);
    [[maybe_unused]] const float s_tensor = es.sa * es.sb;
    float sx[8];  // per-row scales of this lane's eight rows (SCALE_ROWCOL)
#pragma unroll
    for (int mi = 0; mi < 8; ++mi) {
        sx[mi] = 1.0f;
        if constexpr (ScaleKind == SCALE_ROWCOL) {
            const int m = m0 + wave_m * 128 + mi * 16 + lrow;
            sx[mi] = (m < g.m) ? g.sa[m] : 0.0f;
        }
    }

    uint32_t x_off[8], w_off[8];
    walk16_offsets(lane, m0 + wave * 64, 64, (uint32_t)K, x_off);
    walk16_offsets(lane, n0 + wave * 64, 64, (uint32_t)K, w_off);
    f32x4 acc[8][8];  // [n sub-tile][m sub-tile]
    PP_STAMP();
    PP_STAMP();
    walk16<Walk16F8<Fmt>>(lds, g.a, (uint32_t)g.m * (uint32_t)K, x_off, g.b, (uint32_t)g.n * (uint32_t)K, w_off, ksteps, acc);

    PP_STAMP();
    // ---------------- epilogue ----------------
    // bf16, N % 8 == 0. A pass is 32 tokens (two m sub-tiles) x 128 columns, laid down
    // row-major in a wave-private staging buffer (272-byte rows: the 8-byte writes of 32
    // lanes cover all 64 banks once) and streamed out as whole 256-byte row pieces, 16
    // bytes a lane, through a bounds-checked buffer descriptor; two buffers in turn.
    {
        constexpr int ROWB = Cfg::EPI_ROW_BYTES, PASS_BYTES = Cfg::EPI_PASS_BYTES;
        uint8_t* const mine = lds + wave * (2 * PASS_BYTES);
        const uint16_t* bias = static_cast<const uint16_t*>(g.bias);
        const int rows_here = min(Cfg::BM, g.m - m0);
        const uint32_t row_bytes = (uint32_t)g.n * 2u;
        const __amdgpu_buffer_rsrc_t rout =
            make_rsrc(static_cast<uint16_t*>(g.out) + (size_t)m0 * g.n, (uint32_t)rows_here * row_bytes);
        const int nwv = n0 + wave_n * 128;
        f32x4 sw4[8];
        u32x2 braw[8];
#pragma unroll
        for (int ni = 0; ni < 8; ++ni) {
            const int n = nwv + ni * 16 + lgrp * 4;
            sw4[ni] = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
            braw[ni] = u32x2{0u, 0u};
            if (n < g.n) {
                if constexpr (ScaleKind == SCALE_ROWCOL) sw4[ni] = *reinterpret_cast<const f32x4*>(g.sb + n);
                if (bias) braw[ni] = *reinterpret_cast<const u32x2*>(bias + n);
            }
        }
        const int r4 = lane >> 4, c16 = lane & 15;
        const int nst = nwv + c16 * 8;
        const uint32_t lane_off = (nst < g.n)
            ? (uint32_t)(wave_m * 128 + r4) * row_bytes + (uint32_t)nst * 2u
            : kOutOfRange;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint8_t* const buf = mine + (p & 1) * PASS_BYTES;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int mi = 2 * p + h;
#pragma unroll
                for (int ni = 0; ni < 8; ++ni) {
                    const u32x2 raw = braw[ni];
                    const f32x4 b4 = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                                      __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float f = acc[ni][mi][j];
                        if constexpr (ScaleKind == SCALE_TENSOR && RoundFirst) {
                            v[j] = add_bias(f * s_tensor, b4[j], true);
                        } else if constexpr (ScaleKind == SCALE_TENSOR) {
                            v[j] = f * s_tensor + b4[j];
                        } else {
#pragma clang fp contract(off)
                            const float scaled = f * sx[mi] * sw4[ni][j];
                            v[j] = scaled + b4[j];
                        }
                    }
                    u32x2 pk;
                    pk.x = pack_bf16x2(v[0], v[1]);
                    pk.y = pack_bf16x2(v[2], v[3]);
                    *reinterpret_cast<u32x2*>(buf + (h * 16 + lrow) * ROWB + (ni * 16 + lgrp * 4) * 2) = pk;
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(buf + (i * 4 + r4) * ROWB + c16 * 16);
                __builtin_amdgcn_raw_buffer_store_b128(v, rout, lane_off + (uint32_t)(p * 32 + i * 4) * row_bytes, 0, 2);
            }
        }
    }
    PP_STAMP();
}

template <int Fmt, int ScaleKind, bool RoundFirst = false>
inline void launch_wave128_q16(const GemmArgs& g, hipStream_t stream) {
    using Cfg = Wave128Cfg;
    const int tiles = ((g.m + Cfg::BM - 1) / Cfg::BM) * ((g.n + Cfg::BN - 1) / Cfg::BN);
    auto kern = gemm_wave128_q16_kernel<Fmt, ScaleKind, RoundFirst>;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::LDS_BYTES, lds_allowed);
    note_kernel("wave128_q16");
    kern<<<dim3((unsigned)tiles), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream>>>(g);
}

}  // namespace w8a8
