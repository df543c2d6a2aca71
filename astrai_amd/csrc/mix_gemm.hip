// y = x W^T of a prompt's tokens, bf16 operands and output, fp32 sums, on the 256 x 256 tiles of gemm_walk16.cuh.
//
// ACT: the weight holds the rows of gate, then those of up. A wave's 128 weight rows are 64 of gate and the 64 of up
// of the same columns (an address of the loads, not a layout of the weight), so a lane holds each pair, and
// act(gate) * up leaves in place of both, as act_mul (mix_rows.hip) would make it of the rounded product.
//
// What bounds it: the power cap (gemm_walk16.cuh). 8192 x 2048 x 5632 with 32x32x16 MFMAs 132 us, with 16x16x32 124 (the
// vendor library 121), on zeros 100 and 98; 1.38 to 1.57 PFLOP/s where the tiles fill the chip. gate and up of 5632 from
// 16384 x 2048 with silu 517 us, of 4096 rows with gelu 137; the library's product and act_mul 607 and 176.
#include "gemm_walk16.cuh"
#include "mix_common.cuh"
#include "mix_launchers.h"

namespace astrai_mix {

namespace {

using w8a8::kOutOfRange;
using Cfg = w8a8::Wave128Cfg;

constexpr int kSlab = 64;  // values of K per slab

template <int ACT>
__device__ __forceinline__ float act_of(float z) {
    return ACT == kActGelu ? gelu_as<uint16_t>(z) : silu_fast(z);
}

template <int ACT>
__global__ __launch_bounds__(Cfg::THREADS) void prompt_linear_kernel(PromptLinearArgs g) {
    constexpr bool PAIR = ACT >= 0;
    constexpr int BN = PAIR ? Cfg::BN / 2 : Cfg::BN;   // output columns of a workgroup
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave & 1, wave_n = wave >> 1;
    const int lrow = lane & 15, lgrp = lane >> 4;

    const w8a8::TileCoord tc = w8a8::map_tile((g.m + Cfg::BM - 1) / Cfg::BM, (g.n + BN - 1) / BN);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * BN;
    const uint32_t x_row = (uint32_t)g.ldx * 2, w_row = (uint32_t)g.k * 2;

    // ---- loads: wave w fills rows 64w .. 64w + 63 of both operands, 8 rows per instruction. Rows past M read as
    // zeros; so do weight rows past N (PAIR: a wave's 64 rows are of gate or of up, and each half ends for itself)
    const uint32_t x_bytes = (uint32_t)(g.m - 1) * x_row + w_row, w_bytes = (uint32_t)((PAIR ? 2 : 1) * g.n) * w_row;
    uint32_t x_off[8], w_off[8];
    int first = n0 + wave * 64, live = 64;   // weight rows of this wave's loads, and how many of them there are
    if constexpr (PAIR) {
        const int col = n0 + (wave >> 1) * 64;
        live = g.n - col;
        first = (wave & 1) * g.n + col;
    }
    w8a8::walk16_offsets(lane, m0 + wave * 64, 64, x_row, x_off);
    w8a8::walk16_offsets(lane, first, live, w_row, w_off);
    f32x4 acc[8][8];  // [weight sub-tile][token sub-tile]
    w8a8::walk16<w8a8::Walk16Bf16>(lds, g.x, x_bytes, x_off, g.w, w_bytes, w_off, g.k / kSlab, acc);

    // ---- epilogue: 32 tokens at a time row-major through a wave-private buffer, out as whole row pieces, 16 bytes a
    // lane, through a bounds-checked descriptor; two buffers in turn
    constexpr int COLS = PAIR ? 64 : 128;             // output columns of a wave
    constexpr int ROWB = COLS * 2 + 16, PASS = 32 * ROWB;
    constexpr int LPR = COLS / 8, RPI = 64 / LPR;     // lanes per row, rows per store instruction
    uint8_t* const mine = lds + wave * (2 * PASS);
    const uint32_t row_bytes = (uint32_t)g.n * 2u;
    const __amdgpu_buffer_rsrc_t rout = w8a8::make_rsrc(static_cast<uint16_t*>(g.out) + (size_t)m0 * g.n,
                                                        (uint32_t)min(Cfg::BM, g.m - m0) * row_bytes);
    const int nwv = n0 + wave_n * COLS;
    [[maybe_unused]] f32x4 b4[8];
    if constexpr (!PAIR) {
#pragma unroll
        for (int ni = 0; ni < 8; ++ni) {
            const int n = nwv + ni * 16 + lgrp * 4;
            b4[ni] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (g.bias && n < g.n) b4[ni] = Elem<uint16_t>::get4(static_cast<const uint16_t*>(g.bias) + n);
        }
    }
    const int rs = lane / LPR, cs = lane % LPR;
    const uint32_t lane_off = nwv + cs * 8 < g.n ? (uint32_t)(wave_m * 128 + rs) * row_bytes + (uint32_t)(nwv + cs * 8) * 2u
                                                 : kOutOfRange;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint8_t* const buf = mine + (p & 1) * PASS;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int mi = 2 * p + h;
#pragma unroll
            for (int ni = 0; ni < (PAIR ? 4 : 8); ++ni) {
                f32x4 v = acc[ni][mi];
                if constexpr (PAIR) {
                    const f32x4 up = acc[ni + 4][mi];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[j] = act_of<ACT>(w8a8::bf16_to_f32(f32_to_bf16(v[j]))) * w8a8::bf16_to_f32(f32_to_bf16(up[j]));
                } else {
                    v += b4[ni];
                }
                Elem<uint16_t>::put4(reinterpret_cast<uint16_t*>(buf + (h * 16 + lrow) * ROWB) + ni * 16 + lgrp * 4, v);
            }
        }
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(buf + (i * RPI + rs) * ROWB + cs * 16);
            __builtin_amdgcn_raw_buffer_store_b128(v, rout, lane_off + (uint32_t)(p * 32 + i * RPI) * row_bytes, 0, 2);
        }
    }
}

template <int ACT>
void launch_inst(const PromptLinearArgs& a, hipStream_t stream) {
    const int bn = ACT >= 0 ? Cfg::BN / 2 : Cfg::BN;
    const int tiles = ((a.m + Cfg::BM - 1) / Cfg::BM) * ((a.n + bn - 1) / bn);
    static std::atomic<uint64_t> lds_allowed{0};
    w8a8::allow_dynamic_lds(reinterpret_cast<const void*>(prompt_linear_kernel<ACT>), Cfg::LDS_BYTES, lds_allowed);
    prompt_linear_kernel<ACT><<<dim3((unsigned)tiles), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream>>>(a);
}

}  // namespace

bool prompt_linear_supported(int64_t m, int64_t n, int64_t k, int64_t ldx, bool act) {
    constexpr int64_t kMost = (int64_t)1 << 31;   // bytes that the descriptors' offsets reach
    if (m <= 0 || n <= 0 || k <= 0 || m >= kMost || n >= kMost || k >= kMost || ldx >= kMost) return false;
    const int64_t rows = (act ? 2 : 1) * n;       // of the weight
    return n % 8 == 0 && k % kSlab == 0 && ldx >= k && ldx % 8 == 0 && (m + Cfg::BM) * ldx < kMost / 2 &&
           (rows + Cfg::BN) * k < kMost / 2 && n * 2 * Cfg::BM < kMost;
}

bool launch_prompt_linear(const PromptLinearArgs& a, int act, hipStream_t stream) {
    if (!prompt_linear_supported(a.m, a.n, a.k, a.ldx, act >= 0)) return false;
    if (act == kActGelu) launch_inst<kActGelu>(a, stream);
    else if (act == kActSilu) launch_inst<kActSilu>(a, stream);
    else launch_inst<-1>(a, stream);
    return true;
}

}  // namespace astrai_mix
