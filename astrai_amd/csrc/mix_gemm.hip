// y = x W^T of a prompt's tokens, bf16 operands and output, fp32 sums: 256 x 256 weight-row tiles, four waves of
// 128 x 128, one wave to a SIMD, software-pipelined inside each wave (gemm_wave128_q16.cuh tells the walk: a slab is
// 128 bytes of K, here 64 values; quadrants of 64 x 64, the half the next one is missing read from LDS meanwhile,
// direct-to-LDS loads two slabs ahead into three activation and two weight stages, one barrier a slab). A bf16 slab
// is two 16x16x32 MFMAs of 16 cycles where an fp8 one is one of 32, on the same 16-byte pieces of a lane, so bytes,
// registers and cycles of a slab are those of that kernel; all MFMAs of the first pieces of a quadrant come before
// those of the second, sixteen accumulators apart.
//
// ACT: the weight holds the rows of gate, then those of up. A wave's 128 weight rows are 64 of gate and the 64 of up
// of the same columns (an address of the loads, not a layout of the weight), so a lane holds each pair, and
// act(gate) * up leaves in place of both, as act_mul (mix_rows.hip) would make it of the rounded product.
//
// What bounds it: the power cap. Registers-only loops on random operands sustain 1.85 PFLOP/s of 32x32x16 and 2.06 of
// 16x16x32 MFMAs (2.48 and 2.37 on zeros), hence the small ones, although 32 cycles of a large one hide 24 of other
// instructions and 16 of a small one about 4: 8192 x 2048 x 5632 with large ones 132 us, with these 124 (the vendor
// library 121), on zeros 100 and 98; 1.38 to 1.57 PFLOP/s where the tiles fill the chip. gate and up of 5632 from
// 16384 x 2048 with silu 517 us, of 4096 rows with gelu 137; the library's product and act_mul 607 and 176.
#include "gemm_wave128.cuh"
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

// acc += a b^T in the same registers: behind the builtin the compiler gives results other registers than it takes sums
// from and moves them back
__device__ __forceinline__ void mfma_in_place(u32x4 a, u32x4 b, f32x4& acc) {
    __asm__ volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
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
    const int slabs = g.k / kSlab;
    const uint32_t x_row = (uint32_t)g.ldx * 2, w_row = (uint32_t)g.k * 2;

    // ---- loads: wave w fills rows 64w .. 64w + 63 of both operands, 8 rows per instruction. Rows past M read as
    // zeros; so do weight rows past N (PAIR: a wave's 64 rows are of gate or of up, and each half ends for itself)
    const uint32_t x_bytes = (uint32_t)(g.m - 1) * x_row + w_row, w_bytes = (uint32_t)((PAIR ? 2 : 1) * g.n) * w_row;
    uint32_t x_off[8], w_off[8];   // of each instruction: no address arithmetic between the MFMAs
    {
        const uint32_t xr = (uint32_t)(m0 + wave * 64 + (lane >> 3)) * x_row;
        int first = n0 + wave * 64, live = 64;   // weight rows of this wave's part, and how many of them there are
        if constexpr (PAIR) {
            const int col = n0 + (wave >> 1) * 64;
            live = g.n - col;
            first = (wave & 1) * g.n + col;
        }
        const uint32_t wr = (uint32_t)(first + (lane >> 3)) * w_row;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t chunk = (uint32_t)((lane & 7) ^ (lane >> 3) ^ (r & 1)) * 16;
            x_off[r] = xr + (uint32_t)r * (8u * x_row) + chunk;
            w_off[r] = 8 * r < live ? wr + (uint32_t)r * (8u * w_row) + chunk : kOutOfRange;
        }
    }
    uint8_t* const dma_base = lds + wave * (64 * 128);
    auto dma_x = [&](int r, __amdgpu_buffer_rsrc_t rx, int stage, uint32_t k0) __attribute__((always_inline)) {
        w8a8::lds_dma16(rx, dma_base + stage * Cfg::OPERAND_BYTES + r * 1024, x_off[r], k0);
    };
    auto dma_w = [&](int r, __amdgpu_buffer_rsrc_t rw, int stage, uint32_t k0) __attribute__((always_inline)) {
        w8a8::lds_dma16(rw, dma_base + Cfg::W_BASE + stage * Cfg::OPERAND_BYTES + r * 1024, w_off[r], k0);
    };

    // ---- operand reads: the lane's two 16-byte pieces of its row of a 16-row sub-tile
    int frag_off[2];
    {
        const int sw = (lrow & 7) ^ ((lrow >> 3) & 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) frag_off[j] = lrow * 128 + (((2 * lgrp + j) ^ sw) << 4);
    }
    const int x_rd = (wave_m * 128) * 128, w_rd = Cfg::W_BASE + (wave_n * 128) * 128;
    // read r of 8 of half h of an operand: piece r / 4 of sub-tile 4h + r % 4
    auto read_x = [&](int r, int stage, int h, u32x4 (&f)[4][2]) __attribute__((always_inline)) {
        f[r & 3][r >> 2] = *reinterpret_cast<const u32x4*>(
            lds + x_rd + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048 + frag_off[r >> 2]);
    };
    auto read_w = [&](int r, int stage, int h, u32x4 (&f)[4][2]) __attribute__((always_inline)) {
        f[r & 3][r >> 2] = *reinterpret_cast<const u32x4*>(
            lds + w_rd + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048 + frag_off[r >> 2]);
    };

    f32x4 acc[8][8];  // [weight sub-tile][token sub-tile]
#pragma unroll
    for (int ni = 0; ni < 8; ++ni)
#pragma unroll
        for (int mi = 0; mi < 8; ++mi) acc[ni][mi] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 xa[4][2], xb[4][2], wa[4][2], wb[4][2];

    // ---- prologue: slabs 0 and 1 in flight; slab 0 visible; halves 0 of slab 0 in xa, wa
    {
        const __amdgpu_buffer_rsrc_t rx = w8a8::make_rsrc(g.x, x_bytes), rw = w8a8::make_rsrc(g.w, w_bytes);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_x(r, rx, 0, 0u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_w(r, rw, 0, 0u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_x(r, rx, 1, 128u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_w(r, rw, 1, 128u);
        w8a8::wait_vmcnt<16>();  // slab 0
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) read_x(r, 0, 0, xa);
#pragma unroll
        for (int r = 0; r < 8; ++r) read_w(r, 0, 0, wa);
    }

    int xs = 0;  // k % 3
    // One quadrant: 32 MFMAs on (xf, wf); between them the 8 reads of the half the next quadrant is missing and 4 loads
    auto phase = [&](const u32x4 (&xf)[4][2], const u32x4 (&wf)[4][2], int xh, int wh, auto&& rd, auto&& ld) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int c = i >> 4, mi = (i >> 2) & 3, ni = i & 3;
            mfma_in_place(wf[ni][c], xf[mi][c], acc[4 * wh + ni][4 * xh + mi]);
#pragma unroll
            for (int r = 0; r < 8; ++r)
                if (r * 2 == i) rd(r);
#pragma unroll
            for (int d = 0; d < 4; ++d)
                if (d * 8 + 4 == i) ld(d);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // one slab; ODD: its place in the two-slab walk. Past the end of K the loads run on an empty descriptor
    auto slab = [&](auto odd_c, int k) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd_c)::value;
        const int ws = k & 1;
        const int xs1 = (xs == 2) ? 0 : xs + 1;   // (k + 1) % 3
        const int xs2 = (xs == 0) ? 2 : xs - 1;   // (k + 2) % 3
        const uint32_t k2 = (uint32_t)(k + 2) << 7;
        const bool more = k + 2 < slabs;
        const __amdgpu_buffer_rsrc_t rx = w8a8::make_rsrc(g.x, more ? x_bytes : 0u);
        const __amdgpu_buffer_rsrc_t rw = w8a8::make_rsrc(g.w, more ? w_bytes : 0u);
        auto ldx = [&](int base) __attribute__((always_inline)) { return [&, base](int d) __attribute__((always_inline)) { dma_x(base + d, rx, xs2, k2); }; };
        auto ldw = [&](int base) __attribute__((always_inline)) { return [&, base](int d) __attribute__((always_inline)) { dma_w(base + d, rw, ws, k2); }; };
        if constexpr (!ODD) {
            phase(xa, wa, 0, 0, [&](int r) __attribute__((always_inline)) { read_w(r, ws, 1, wb); }, ldx(0));
            phase(xa, wb, 0, 1, [&](int r) __attribute__((always_inline)) { read_x(r, xs, 1, xb); }, ldx(4));
        } else {
            phase(xa, wb, 0, 1, [&](int r) __attribute__((always_inline)) { read_w(r, ws, 0, wa); }, ldx(0));
            phase(xa, wa, 0, 0, [&](int r) __attribute__((always_inline)) { read_x(r, xs, 1, xb); }, ldx(4));
        }
        // Slab k+1 has landed for this wave (all but this half's eight loads are older) and this wave has read slab k;
        // after the barrier both hold for every wave
        w8a8::wait_vmcnt<8>();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        w8a8::phase_barrier();
        // (after the last slab the reads fetch stale bytes that are never used)
        if constexpr (!ODD) {
            phase(xb, wb, 1, 1, [&](int r) __attribute__((always_inline)) { read_x(r, xs1, 0, xa); }, ldw(0));
            phase(xb, wa, 1, 0, [&](int r) __attribute__((always_inline)) { read_w(r, ws ^ 1, 1, wb); }, ldw(4));
        } else {
            phase(xb, wa, 1, 0, [&](int r) __attribute__((always_inline)) { read_x(r, xs1, 0, xa); }, ldw(0));
            phase(xb, wb, 1, 1, [&](int r) __attribute__((always_inline)) { read_w(r, ws ^ 1, 0, wa); }, ldw(4));
        }
        xs = xs1;
    };
    for (int k = 0; k < slabs; k += 2) {
        slab(std::false_type{}, k);
        slab(std::true_type{}, k + 1);
    }
    __asm__ volatile("s_nop 15\n\ts_nop 3");   // the last MFMAs' results, before the epilogue moves them
    // no load outlives the loop; the stages are dead for every wave
    __builtin_amdgcn_s_waitcnt(0x0070);
    w8a8::phase_barrier();

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
    return m > 0 && n > 0 && n % 8 == 0 && k > 0 && k % (2 * kSlab) == 0 && ldx >= k && ldx % 8 == 0 &&
           (m + Cfg::BM) * ldx * 2 < kMost && (n + Cfg::BN) * k * (act ? 4 : 2) < kMost && n * 2 * Cfg::BM < kMost;
}

bool launch_prompt_linear(const PromptLinearArgs& a, int act, hipStream_t stream) {
    if (!prompt_linear_supported(a.m, a.n, a.k, a.ldx, act >= 0)) return false;
    if (act == kActGelu) launch_inst<kActGelu>(a, stream);
    else if (act == kActSilu) launch_inst<kActSilu>(a, stream);
    else launch_inst<-1>(a, stream);
    return true;
}

}  // namespace astrai_mix
