// 8-bit NT GEMM for shapes between the decode kernels and the large-tile kernels: a few
// hundred to a few thousand activation rows, where 256 x 256 tiles leave most of the chip
// idle (2048 x 3072: 96 tiles for 256 compute units) and what counts is having every
// compute unit busy, not the last percent of operand reuse.
//
// 128 x 128 output tiles, eight waves of 64 x 32 (two MFMA 32x32 sub-tiles, 32 accumulator
// registers), K in 128-byte slabs through two LDS stages of 32 KiB filled by direct-to-LDS
// loads: 64 KiB per workgroup and ~95 registers per wave, so two workgroups -- four waves per
// SIMD -- share a compute unit and cover each other's barriers and memory waits; no hand-pinned
// schedule here (four waves of 64 x 64 measured 2-4% slower on the decoder's shapes). LDS
// layout of a slab, fragment reads and accumulator layout are those of the large-tile
// kernels (gemm_pingpong.cuh): 128 activation rows then 128 weight rows of 128 bytes, chunk
// c of row r at position c ^ (r & 7) ^ ((r >> 3) & 1); weight rows are the first MFMA operand.
#pragma once
#include <type_traits>

#include "gemm_pingpong.cuh"

namespace w8a8 {

struct Mid128Cfg {
    static constexpr int BM = 128, BN = 128, BK = 128;
    static constexpr int THREADS = 512;
    static constexpr int MI = 2, NI = 1;                 // 32-row sub-tiles per wave: 64 m x 32 n
    static constexpr int OPERAND_BYTES = 128 * BK;       // one operand's slab: 16 KiB
    static constexpr int STAGE_BYTES = 2 * OPERAND_BYTES;
    static_assert(TileOut<BM, BN, THREADS>::BYTES <= 2 * STAGE_BYTES, "outputs fit the stages");
};

// RoundFirst (per-tensor scales): the product is rounded to bf16 before the bias joins it. An instance of its own: chosen
// in the epilogue, it cost every per-tensor product 0.2 us (354 x 11008 x 4096: 34.3 -> 34.6).
// S: LDS stages. 2: as above. 4: for launches of one workgroup per compute unit at most, where nobody covers its waits (1500
// cycles a slab, against 512 of MFMAs): a ring filled four slabs ahead, one barrier per slab, the fragments of slab k + 1
// read into a second register set beside the MFMAs of slab k; 1050 cycles a slab, bound by LDS (96 KiB of fragments, 32 KiB of
// loads). int8 / fp8, us: 256 x 11264 x 2048 14.7 / 14.2 -> 13.1 / 12.6, 640 x 4096 x 4096 22.8 / 22.5 -> 20.5 / 18.7, 130 x 11008
// x 4096 22.4 / 23.7 -> 18.7 / 18.4, 600 x 4096 x 11008 49.2 / 49.4 -> 43.9 / 39.9; 2048^3 (256 tiles) 16.0 / 15.1 either way.
// 128-block scales (steps four slabs at a time, scaled additions behind the other half's MFMAs): 1454 x 2048 x 7168 57.2 -> 35.6, 600 x
// 4096 x 4096 34.5 -> 21.5, 450 x 7168 x 2048 17.6 -> 14.0, 2600 x 1536 x 7168 59.6 -> 39.2, 600 x 4096 x 640 8.5 -> 8.0; with a step a
// slab and row in this ring 51.5 and 31.3 of the first two: 16 scattered loads a slab held up the load path that the slabs take.
// Up to four slabs the ring is filled once, and its larger prologue is a loss (600 x 4096 x 256 6.9 / 6.4 -> 7.3 / 7.0, x 512
// 7.9 / 7.5 -> 8.1 / 7.75; x 640 the first where it is none): two stages.
template <class Op, int ScaleKind, bool RoundFirst, int S>
__global__ __launch_bounds__(Mid128Cfg::THREADS, S == 2 ? 4 : 2) void gemm_mid128_kernel(GemmArgs g) {
    using Cfg = Mid128Cfg;
    using Acc = typename Op::Acc;
    constexpr int MI = Cfg::MI, NI = Cfg::NI;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave & 1, wave_n = wave >> 1;   // 2 x 4 waves
    const int lrow = lane & 31, lgrp = lane >> 5;

    const int tiles_m = (g.m + Cfg::BM - 1) / Cfg::BM;
    const int tiles_n = (g.n + Cfg::BN - 1) / Cfg::BN;
    const TileCoord tc = map_tile(tiles_m, tiles_n);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * Cfg::BN;
    const int K = g.k;
    const int ksteps = K >> 7;

    // epilogue operands, requested now
    const EpilogueScalars es = load_epilogue_scalars<ScaleKind>(g);
    [[maybe_unused]] const float s_tensor = es.sa * es.sb;
    const int mw = m0 + wave_m * 64, nw = n0 + wave_n * 32;
    float sx[MI];
    f32x4 sw4[NI][4], b4[NI][4];
    const uint16_t* bias = static_cast<const uint16_t*>(g.bias);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
        sx[mi] = 1.0f;
        if constexpr (ScaleKind == SCALE_ROWCOL) {
            const int m = mw + mi * 32 + lrow;
            sx[mi] = (m < g.m) ? g.sa[m] : 0.0f;
        }
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = nw + ni * 32 + q * 8 + lgrp * 4 + j;
                sw4[ni][q][j] = 1.0f;
                b4[ni][q][j] = 0.0f;
                if (n < g.n) {
                    if constexpr (ScaleKind == SCALE_ROWCOL) sw4[ni][q][j] = g.sb[n];
                    // (the block-scaled instance needs its registers in the loop and fetches the bias at the end)
                    if constexpr (ScaleKind != SCALE_BLOCK128)
                        if (bias) b4[ni][q][j] = bf16_to_f32(bias[n]);
                }
            }

    // ---- direct-to-LDS load plan: wave w fills rows 16w .. 16w+15 of both operands, 8 rows per
    // instruction. Lane l lands at row l>>3, position l&7 of its 1 KiB block and fetches logical
    // chunk (l&7) ^ f(row): c0 for even instructions, c0 ^ 1 for odd ones. Rows past M / N are
    // past the buffer's num_records and read as zero.
    const uint32_t x_bytes = (uint32_t)g.m * (uint32_t)K, w_bytes = (uint32_t)g.n * (uint32_t)K;
    const __amdgpu_buffer_rsrc_t rx0 = make_rsrc(g.a, x_bytes), rw0 = make_rsrc(g.b, w_bytes);
    uint32_t x_off[2], w_off[2];
    {
        const int c0 = (lane & 7) ^ (lane >> 3);
        const uint32_t xr = (uint32_t)(m0 + wave * 16 + (lane >> 3)) * (uint32_t)K;
        const uint32_t wr = (uint32_t)(n0 + wave * 16 + (lane >> 3)) * (uint32_t)K;
        x_off[0] = xr + (uint32_t)c0 * 16;
        x_off[1] = xr + (uint32_t)(c0 ^ 1) * 16;
        w_off[0] = wr + (uint32_t)c0 * 16;
        w_off[1] = wr + (uint32_t)(c0 ^ 1) * 16;
    }
    const uint32_t row8 = 8u * (uint32_t)K;
    uint8_t* const dma_base = lds + wave * (16 * 128);
    auto issue = [&](int stage, int slab) __attribute__((always_inline)) {   // past the last slab: zeros, no memory traffic
        __amdgpu_buffer_rsrc_t rx = rx0, rw = rw0;
        if constexpr (S > 2) {
            rx = make_rsrc(g.a, slab < ksteps ? x_bytes : 0u);
            rw = make_rsrc(g.b, slab < ksteps ? w_bytes : 0u);
        }
        const uint32_t k0 = (uint32_t)slab << 7;
        uint8_t* const dst = dma_base + stage * Cfg::STAGE_BYTES;
#pragma unroll
        for (int r = 0; r < 2; ++r) lds_dma16(rx, dst + r * 1024, x_off[r & 1] + (uint32_t)r * row8, k0);
#pragma unroll
        for (int r = 0; r < 2; ++r)
            lds_dma16(rw, dst + Cfg::OPERAND_BYTES + r * 1024, w_off[r & 1] + (uint32_t)r * row8, k0);
    };

    // ---- fragment read plan: lane (row lrow of a 32-row sub-tile, K-group lgrp) owns chunks 4 lgrp .. 4 lgrp + 3
    int frag_off[4];
    {
        const int sw = (lrow & 7) ^ ((lrow >> 3) & 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) frag_off[j] = lrow * 128 + (((4 * lgrp + j) ^ sw) << 4);
    }
    const int x_rd = (wave_m * 64) * 128;
    const int w_rd = Cfg::OPERAND_BYTES + (wave_n * 32) * 128;

    Acc acc[NI][MI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[ni][mi][j] = 0;

    // ---- 128-block scales: a slab is exactly one K-block. The slab's product is formed in a
    // temporary and joins the accumulator scaled by the activation rows' and the weight block's
    // steps (the tile's 128 columns lie in one weight block). With two stages the steps of slab k + 1 are requested
    // while slab k is computed.
    [[maybe_unused]] float blk_step[MI], blk_sa_next[MI];
    [[maybe_unused]] float blk_sb_next = 0.0f;
    [[maybe_unused]] const int kblocks = K >> 7;
    auto request_steps = [&](int kb) {
        if constexpr (ScaleKind == SCALE_BLOCK128) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
                const int m = mw + mi * 32 + lrow;
                blk_sa_next[mi] = (m < g.m && kb < kblocks) ? g.sa[(size_t)m * kblocks + kb] : 0.0f;
            }
            blk_sb_next = kb < kblocks ? g.sb[(size_t)(n0 >> 7) * kblocks + kb] : 0.0f;
        }
    };

    auto read = [&](int stage, u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4]) __attribute__((always_inline)) {
        const uint8_t* const base = lds + stage * Cfg::STAGE_BYTES;
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                wf[ni][j] = *reinterpret_cast<const u32x4*>(base + w_rd + ni * 4096 + frag_off[j]);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                xf[mi][j] = *reinterpret_cast<const u32x4*>(base + x_rd + mi * 4096 + frag_off[j]);
    };
    auto multiply = [&](u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4]) __attribute__((always_inline)) {
        if constexpr (ScaleKind == SCALE_BLOCK128) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    Acc part;
#pragma unroll
                    for (int j = 0; j < 16; ++j) part[j] = 0;
#pragma unroll
                    for (int q = 0; q < Op::STEPS; ++q) part = Op::mma_step(q, wf[ni], xf[mi], part);
                    const float sc = blk_step[mi];
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc[ni][mi][j] += part[j] * sc;
                }
        } else {
#pragma unroll
            for (int q = 0; q < Op::STEPS; ++q)
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                    for (int ni = 0; ni < NI; ++ni) acc[ni][mi] = Op::mma_step(q, wf[ni], xf[mi], acc[ni][mi]);
        }
    };

    // ---- main loop: slab k+1 in flight while slab k is read; a barrier before a stage is
    // read (every wave's part has landed) and one before it is filled again
    if constexpr (S == 2) {
        request_steps(0);
        issue(0, 0);
        for (int k = 0; k < ksteps; ++k) {
            if constexpr (ScaleKind == SCALE_BLOCK128) {
    #pragma unroll
                for (int mi = 0; mi < MI; ++mi) blk_step[mi] = blk_sa_next[mi] * blk_sb_next;
            }
            if (k + 1 < ksteps) {
                issue((k + 1) & 1, k + 1);
                wait_vmcnt<4>();   // the four loads of slab k are older than those just issued
            } else {
                wait_vmcnt<0>();
            }
            phase_barrier();
            // (after the wait: the next slab's steps are then older than the slab loads of the following
            // iteration, whose wait they pass without holding it up -- a compute phase has gone by)
            request_steps(k + 1);
            u32x4 xf[MI][4], wf[NI][4];
            read(k & 1, xf, wf);
            multiply(xf, wf);
            wait_lgkmcnt0();
            phase_barrier();
        }
    } else {
        u32x4 xa[MI][4], wa[NI][4], xb[MI][4], wb[NI][4];
        // 128-block scales: a row's steps of four slabs are one load (16 lines for each row and slab otherwise, and the load path
        // that the slabs come through takes a line a cycle), requested in the first slab of the four before, ahead of its slab
        // loads; past the last slab and past M they are never used. MI + 1 vector loads whatever the compiler makes of the
        // addresses: the waits count them.
        constexpr int STEPS = ScaleKind == SCALE_BLOCK128 ? MI + 1 : 0;
        [[maybe_unused]] u32x4 steps[MI + 1], steps_next[MI + 1];
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsa = make_rsrc(g.sa, STEPS ? (uint32_t)g.m * (uint32_t)kblocks * 4u : 0u);
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsb = make_rsrc(g.sb, STEPS ? (uint32_t)tiles_n * (uint32_t)kblocks * 4u : 0u);
        auto request = [&](int kb, u32x4 (&d)[MI + 1]) __attribute__((always_inline)) {
            if constexpr (STEPS > 0) {
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
                    d[mi] = buf_load16(rsa, (uint32_t)(mw + mi * 32 + lrow) * (uint32_t)kblocks * 4u, (uint32_t)kb * 4u);
                d[MI] = buf_load16(rsb, (uint32_t)(n0 >> 7) * (uint32_t)kblocks * 4u, (uint32_t)kb * 4u);
            }
        };
        // Two waves of a SIMD meet at the barrier of every slab, so that a slab's scaled additions, left to its end, run with the matrix
        // cores idle: each half goes behind the other half's MFMAs instead, the second half's into the next slab.
        [[maybe_unused]] Acc part[MI];
        [[maybe_unused]] float behind = 0.0f;
        if constexpr (STEPS > 0) {
#pragma unroll
            for (int j = 0; j < 16; ++j) part[MI - 1][j] = 0;
        }
        auto multiply_scaled = [&](u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4]) __attribute__((always_inline)) {
            static_assert(MI == 2 && NI == 1, "halves");
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
                const float sc = mi == 0 ? behind : blk_step[0];
#pragma unroll
                for (int q = 0; q < Op::STEPS; ++q) {
                    if (q == 0) part[mi] = Op::mma_step(q, wf[0], xf[mi], Acc{});
                    else part[mi] = Op::mma_step(q, wf[0], xf[mi], part[mi]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 16 / Op::STEPS * q; j < 16 / Op::STEPS * (q + 1); ++j) acc[0][1 - mi][j] += part[1 - mi][j] * sc;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            behind = blk_step[1];
        };
        request(0, steps);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < S; ++t) issue(t, t);
        wait_vmcnt<4 * (S - 1)>();
        phase_barrier();
        read(0, xa, wa);
        // in: this slab's fragments, its reads under way. AT: which of its four slabs; MORE: four more follow them, whose steps
        // the first requests (both with 128-block scales)
        auto slab = [&](auto at, auto more, int k, u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4], u32x4 (&xn)[MI][4], u32x4 (&wn)[NI][4])
                        __attribute__((always_inline)) {
            constexpr int AT = decltype(at)::value;
            constexpr bool MORE = decltype(more)::value;
            wait_lgkmcnt0();
            wait_vmcnt<4 * (S - 2) + (MORE && (AT == 1 || AT == 2) ? STEPS : 0)>();   // slab k + 1 has landed
            phase_barrier();             // for every wave, and every wave has read slab k: its stage is free
            if constexpr (STEPS > 0) {
                if constexpr (MORE && AT == 0) {
                    request(k + 4, steps_next);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) blk_step[mi] = __uint_as_float(steps[mi][AT]) * __uint_as_float(steps[MI][AT]);
            }
            issue(k & (S - 1), k + S);
            read((k + 1) & (S - 1), xn, wn);   // (past the last slab: zeros)
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (STEPS > 0) multiply_scaled(xf, wf);
            else multiply(xf, wf);
        };
        constexpr std::integral_constant<int, 0> at0{};
        int k = 0;
        if constexpr (STEPS > 0) {
            constexpr std::integral_constant<int, 1> at1{};
            constexpr std::integral_constant<int, 2> at2{};
            constexpr std::integral_constant<int, 3> at3{};
            for (; k + 3 < ksteps; k += 4) {
                slab(at0, std::true_type{}, k, xa, wa, xb, wb);
                slab(at1, std::true_type{}, k + 1, xb, wb, xa, wa);
                slab(at2, std::true_type{}, k + 2, xa, wa, xb, wb);
                slab(at3, std::true_type{}, k + 3, xb, wb, xa, wa);
#pragma unroll
                for (int i = 0; i <= MI; ++i) steps[i] = steps_next[i];
            }
            if (k < ksteps) slab(at0, std::false_type{}, k, xa, wa, xb, wb);
            if (k + 1 < ksteps) slab(at1, std::false_type{}, k + 1, xb, wb, xa, wa);
            if (k + 2 < ksteps) slab(at2, std::false_type{}, k + 2, xa, wa, xb, wb);
        } else {
            for (; k + 1 < ksteps; k += 2) {
                slab(at0, std::false_type{}, k, xa, wa, xb, wb);
                slab(at0, std::false_type{}, k + 1, xb, wb, xa, wa);
            }
            if (k < ksteps) slab(at0, std::false_type{}, k, xa, wa, xb, wb);
        }
        wait_vmcnt<0>();
        if constexpr (STEPS > 0) {
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[0][1][j] += part[1][j] * behind;
        }
    }

    // ---- epilogue: a lane holds four consecutive n of one m per (sub-tile, quad)
    if (g.out_kind != OUT_BF16) return;   // (the launcher sends other outputs elsewhere)
    TileOut<Cfg::BM, Cfg::BN, Cfg::THREADS>::store(g, lds, m0, n0, [&](auto put) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int c = wave_n * 32 + ni * 32 + q * 8 + lgrp * 4;
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float f = (float)acc[ni][mi][4 * q + j];
                        if constexpr (ScaleKind == SCALE_BLOCK128) {
                            v[j] = f + ((bias && n0 + c + j < g.n) ? bf16_to_f32(bias[n0 + c + j]) : 0.0f);
                        } else if constexpr (ScaleKind == SCALE_TENSOR) {
                            v[j] = RoundFirst ? add_bias(f * s_tensor, b4[ni][q][j], true) : f * s_tensor + b4[ni][q][j];
                        } else {
#pragma clang fp contract(off)
                            const float scaled = f * sx[mi] * sw4[ni][q][j];
                            v[j] = scaled + b4[ni][q][j];
                        }
                    }
                    put(wave_m * 64 + mi * 32 + lrow, c, v);
                }
    });
}

// bf16 output, K in whole slabs, and a shape this tile size suits: at least 140 tiles of 128 x 128
// (below that the 64 x 64 tiles of the generic kernel spread the work further and win or draw: 512 x
// 3072 x 2048 13.2 against 15.1 us, 1024 x 2048 x 2048 13.3 against 14.9 us, 512 x 4096 x 4096 (128
// tiles) 22.5 against 22.3 us; from there on this kernel wins: 768 x 3072 x 2048 (144 tiles) 14.2
// against 16.4 us, 256 x 11008 x 4096 (172) 23.7 against 28.6 us, 1024 x 3072 x 2048 16.0 against
// 23.6 us, 2048 x 3072 x 2048 22.9 against 30.7 us). With four stages the line stays: 512 x 4096 x 4096 19.9 / 19.0 (int8 / fp8)
// against 20.4 / 17.7 on 64 x 64 tiles, 1024 x 2048 x 2048 12.3 against 10.1, 700 x 2048 x 5632 (96) 22.5 against 19.8
inline bool mid128_shape_ok(const GemmArgs& g) {
    if (!tiled_shape_ok(g) || (g.k & 127) != 0 || g.k < 128 || g.out_kind != OUT_BF16) return false;
    const int64_t tiles = (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128);
    return tiles >= 140;
}

template <class Op, int ScaleKind, bool RoundFirst = false, int S = 2>
inline void launch_mid128(const GemmArgs& g, hipStream_t stream) {
    using Cfg = Mid128Cfg;
    if constexpr (!RoundFirst && ScaleKind == SCALE_TENSOR)
        if (g.round_first) return launch_mid128<Op, ScaleKind, true>(g, stream);
    const int tiles = ((g.m + Cfg::BM - 1) / Cfg::BM) * ((g.n + Cfg::BN - 1) / Cfg::BN);
    if constexpr (S == 2)
        if (tiles <= 256 && g.k > 512) return launch_mid128<Op, ScaleKind, RoundFirst, 4>(g, stream);
    constexpr int lds_bytes = S * Cfg::STAGE_BYTES;
    auto kern = gemm_mid128_kernel<Op, ScaleKind, RoundFirst, S>;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, lds_allowed);
    note_kernel(ScaleKind == SCALE_BLOCK128 ? "mid128_block128" : "mid128");
    kern<<<dim3((unsigned)tiles), dim3(Cfg::THREADS), lds_bytes, stream>>>(g);
}

}  // namespace w8a8
