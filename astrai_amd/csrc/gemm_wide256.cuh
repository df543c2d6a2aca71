// 8-bit NT GEMM on tiles of 128 (m) x 256 (n): products whose tiles of 128 x 128 are one to two rounds of the chip, so
// that a compute unit takes two of those or one of these.
//
// Eight waves of 64 x 64 (two by two MFMA 32x32 sub-tiles, 64 accumulator registers), one workgroup per compute unit. What
// bounds tiles of 128 x 128 is LDS: 96 KiB of fragments and 32 KiB of loads for 512 cycles of MFMAs. Here it is 128 + 48 KiB for 1024.
// K in 128-byte slabs through three LDS stages of 48 KiB, filled three slabs ahead by direct-to-LDS loads: slab k + 1 is read into a
// second register set, and slab k + 3 requested into the stage of slab k (which every wave has read before the one barrier of a slab),
// behind slab k's MFMAs. Four waves of 64 x 128 (96 + 48 KiB, one wave a SIMD) took 0.69 us a slab (fp8, K = 11008, 144 tiles; without the
// loads 0.56, without the MFMAs 0.62, without the reads 0.65) and were 1 to 10% slower, most with few slabs; with all loads of a slab
// behind its first three MFMAs 4 to 8% slower still.
// LDS layout of a slab, load plan, fragment reads and accumulator layout are those of gemm_mid128_kernel.
#pragma once
#include <type_traits>

#include "gemm_pingpong.cuh"

namespace w8a8 {

struct Wide256Cfg {
    static constexpr int BM = 128, BN = 256, BK = 128;
    static constexpr int THREADS = 512, WAVES = 8;
    static constexpr int MI = 2, NI = 2;                    // 32-row sub-tiles per wave: 64 m x 64 n
    static constexpr int STAGES = 3;
    static constexpr int X_BYTES = BM * BK;                 // 16 KiB, then 32 KiB of weights
    static constexpr int STAGE_BYTES = (BM + BN) * BK;
    static constexpr int COLUMNS = STAGES * STAGE_BYTES;    // the columns' steps and biases behind the stages
    static constexpr int LDS_BYTES = COLUMNS + 2 * BN * 4;
    static_assert(TileOut<BM, BN, THREADS>::BYTES <= COLUMNS, "outputs fit ahead of the columns");
    static constexpr int X_LOADS = BM / 8 / WAVES, LOADS = (BM + BN) / 8 / WAVES;   // of a wave and slab: eight rows each
};

template <class Op, int ScaleKind, bool RoundFirst>
__global__ __launch_bounds__(Wide256Cfg::THREADS, 2) void gemm_wide256_kernel(GemmArgs g) {
    using Cfg = Wide256Cfg;
    using Acc = typename Op::Acc;
    constexpr int MI = Cfg::MI, NI = Cfg::NI, S = Cfg::STAGES;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave & 1, wave_n = wave >> 1;   // 2 x 4 waves
    const int lrow = lane & 31, lgrp = lane >> 5;

    const TileCoord tc = map_tile((g.m + Cfg::BM - 1) / Cfg::BM, (g.n + Cfg::BN - 1) / Cfg::BN);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * Cfg::BN;
    const int K = g.k;
    const int ksteps = K >> 7;

    // epilogue operands, requested now: a row's step in a register, a column's step and bias for LDS
    const EpilogueScalars es = load_epilogue_scalars<ScaleKind>(g);
    [[maybe_unused]] const float s_tensor = es.sa * es.sb;
    const int mw = m0 + wave_m * 64, nw = wave_n * 32 * NI;   // (nw: inside the tile)
    float sx[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
        sx[mi] = 1.0f;
        if constexpr (ScaleKind == SCALE_ROWCOL) {
            const int m = mw + mi * 32 + lrow;
            sx[mi] = (m < g.m) ? g.sa[m] : 0.0f;
        }
    }
    const uint16_t* bias = static_cast<const uint16_t*>(g.bias);
    float col_step = 1.0f, col_bias = 0.0f;
    if ((int)threadIdx.x < Cfg::BN && n0 + (int)threadIdx.x < g.n) {
        if constexpr (ScaleKind == SCALE_ROWCOL) col_step = g.sb[n0 + threadIdx.x];
        if (bias) col_bias = bf16_to_f32(bias[n0 + threadIdx.x]);
    }

    // ---- direct-to-LDS load plan: wave w fills rows 16w .. 16w+15 of the activations and 32w .. 32w+31 of the weights, 8
    // rows per instruction. Lane l lands at row l>>3, position l&7 of its 1 KiB block and fetches logical chunk (l&7) ^ f(row): c0
    // for even instructions, c0 ^ 1 for odd ones. Rows past M / N are past the buffer's num_records and read as zero.
    const uint32_t x_bytes = (uint32_t)g.m * (uint32_t)K, w_bytes = (uint32_t)g.n * (uint32_t)K;
    uint32_t x_off[2], w_off[2];
    {
        const int c0 = (lane & 7) ^ (lane >> 3);
        const uint32_t xr = (uint32_t)(m0 + wave * 8 * Cfg::X_LOADS + (lane >> 3)) * (uint32_t)K;
        const uint32_t wr = (uint32_t)(n0 + wave * 16 * Cfg::X_LOADS + (lane >> 3)) * (uint32_t)K;
        x_off[0] = xr + (uint32_t)c0 * 16;
        x_off[1] = xr + (uint32_t)(c0 ^ 1) * 16;
        w_off[0] = wr + (uint32_t)c0 * 16;
        w_off[1] = wr + (uint32_t)(c0 ^ 1) * 16;
    }
    const uint32_t row8 = 8u * (uint32_t)K;
    // load r of a slab (past the last slab: zeros, no memory traffic)
    auto load = [&](int r, uint8_t* stage, int slab) __attribute__((always_inline)) {
        const uint32_t k0 = (uint32_t)slab << 7;
        const bool live = slab < ksteps;
        if (r < Cfg::X_LOADS) {
            lds_dma16(make_rsrc(g.a, live ? x_bytes : 0u), stage + (wave * Cfg::X_LOADS + r) * 1024, x_off[r & 1] + (uint32_t)r * row8, k0);
        } else {
            const int i = r - Cfg::X_LOADS;
            lds_dma16(make_rsrc(g.b, live ? w_bytes : 0u), stage + Cfg::X_BYTES + (wave * 2 * Cfg::X_LOADS + i) * 1024,
                      w_off[i & 1] + (uint32_t)i * row8, k0);
        }
    };

    // ---- fragment read plan: lane (row lrow of a 32-row sub-tile, K-group lgrp) owns chunks 4 lgrp .. 4 lgrp + 3
    int frag_off[4];
    {
        const int sw = (lrow & 7) ^ ((lrow >> 3) & 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) frag_off[j] = lrow * 128 + (((4 * lgrp + j) ^ sw) << 4);
    }
    const int x_rd = wave_m * 64 * 128;
    const int w_rd = Cfg::X_BYTES + nw * 128;
    constexpr int READS = 4 * (MI + NI);
    auto read = [&](int r, const uint8_t* stage, u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4]) __attribute__((always_inline)) {
        const int t = r >> 2, j = r & 3;
        if (t < MI) xf[t][j] = *reinterpret_cast<const u32x4*>(stage + x_rd + t * 4096 + frag_off[j]);
        else wf[t - MI][j] = *reinterpret_cast<const u32x4*>(stage + w_rd + (t - MI) * 4096 + frag_off[j]);
    };

    Acc acc[NI][MI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[ni][mi][j] = 0;

    // ---- 128-block scales: a slab is one K-block, a wave's columns lie in one weight block. A sub-tile's product of a slab is formed
    // apart and joins the accumulator scaled by the row's and the block's steps ahead of the next sub-tile's MFMAs, with the
    // other wave's of the SIMD beside it. A row's steps of four slabs are one load, requested in the last slab before them, ahead of its
    // slab loads; past the last slab and past M they are never used.
    constexpr int STEPS = ScaleKind == SCALE_BLOCK128 ? MI + 1 : 0;
    [[maybe_unused]] u32x4 steps[MI + 1];
    [[maybe_unused]] Acc part;
    [[maybe_unused]] float behind = 0.0f;
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsa = make_rsrc(g.sa, STEPS ? (uint32_t)g.m * (uint32_t)ksteps * 4u : 0u);
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsb = make_rsrc(g.sb, STEPS ? (uint32_t)((g.n + 127) >> 7) * (uint32_t)ksteps * 4u : 0u);
    auto request = [&](int kb, u32x4 (&d)[MI + 1]) __attribute__((always_inline)) {
        if constexpr (STEPS > 0) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) d[mi] = buf_load16(rsa, (uint32_t)(mw + mi * 32 + lrow) * (uint32_t)ksteps * 4u, (uint32_t)kb * 4u);
            d[MI] = buf_load16(rsb, (uint32_t)((n0 + nw) >> 7) * (uint32_t)ksteps * 4u, (uint32_t)kb * 4u);
        }
    };
    if constexpr (STEPS > 0) {
#pragma unroll
        for (int j = 0; j < 16; ++j) part[j] = 0;
        request(0, steps);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int r = 0; r < Cfg::LOADS; ++r) load(r, lds + s * Cfg::STAGE_BYTES, s);
    float* const columns = reinterpret_cast<float*>(lds + Cfg::COLUMNS);
    if ((int)threadIdx.x < Cfg::BN) {
        columns[threadIdx.x] = col_step;
        columns[Cfg::BN + threadIdx.x] = col_bias;
    }
    wait_vmcnt<Cfg::LOADS*(S - 1)>();
    wait_lgkmcnt0();
    phase_barrier();
    u32x4 xa[MI][4], wa[NI][4], xb[MI][4], wb[NI][4];
#pragma unroll
    for (int r = 0; r < READS; ++r) read(r, lds, xa, wa);

    uint8_t* here = lds;                             // stage of slab k
    uint8_t* next = lds + Cfg::STAGE_BYTES;          // of slab k + 1
    uint8_t* const last = lds + (S - 1) * Cfg::STAGE_BYTES;
    // in: this slab's fragments, their reads under way
    auto slab = [&](auto at, auto more, int k, u32x4 (&xf)[MI][4], u32x4 (&wf)[NI][4], u32x4 (&xn)[MI][4], u32x4 (&wn)[NI][4])
                    __attribute__((always_inline)) {
        constexpr int AT = decltype(at)::value;
        constexpr bool MORE = decltype(more)::value;
        [[maybe_unused]] float step[MI];
        auto arrive = [&]() __attribute__((always_inline)) {
            wait_lgkmcnt0();
            wait_vmcnt<Cfg::LOADS*(S - 2)>();   // slab k + 1 has landed
            phase_barrier();                    // for every wave, and every wave has read slab k: its stage is free
        };
        if constexpr (STEPS > 0) {
            // MFMA i of 8; the columns' fragments are overwritten by the next slab's where they have been used last
            static_assert(Op::STEPS == 2 && MI == 2 && NI == 2 && Cfg::LOADS == 6, "places of the reads and loads");
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xc07f | 4 << 8);   // all but the last four reads: those of the second columns
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) step[mi] = __uint_as_float(steps[mi][AT]) * __uint_as_float(steps[MI][AT]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int t = i / 2, q = i % 2;
                if (q == 0) {   // the last sub-tile's product joins its sums, then this one's takes its place
                    const int before = (t + 3) % 4;
                    const float by = t == 0 ? behind : step[before % MI];
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc[before / MI][before % MI][j] += part[j] * by;
                    __builtin_amdgcn_sched_barrier(0);
                    part = Op::mma_step(q, wf[t / MI], xf[t % MI], Acc{});
                } else {
                    part = Op::mma_step(q, wf[t / MI], xf[t % MI], part);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (i == 1) {
                    arrive();
                    if constexpr (MORE && AT == 3) {
                        request(k + 1, steps);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if (i >= 1 && i < 7) load(i - 1, here, k + S);
                if (i >= 1 && i < 5) read(2 * i - 2, next, xn, wf), read(2 * i - 1, next, xn, wf);
                if (i >= 5 && i < 7) read(2 * i - 2, next, xn, wf), read(2 * i - 1, next, xn, wf);
                if (i == 7)
#pragma unroll
                    for (int r = 12; r < 16; ++r) read(r, next, xn, wf);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            arrive();
            constexpr int MFMAS = Op::STEPS * NI * MI, BUSY = MFMAS * 3 / 4;   // reads and loads behind the first three quarters
#pragma unroll
            for (int i = 0; i < MFMAS; ++i) {
                const int q = i / (NI * MI), ni = i / MI % NI, mi = i % MI;
                acc[ni][mi] = Op::mma_step(q, wf[ni], xf[mi], acc[ni][mi]);
                __builtin_amdgcn_sched_barrier(0);
                if (i < BUSY) {
#pragma unroll
                    for (int r = READS * i / BUSY; r < READS * (i + 1) / BUSY; ++r) read(r, next, xn, wn);
#pragma unroll
                    for (int r = Cfg::LOADS * i / BUSY; r < Cfg::LOADS * (i + 1) / BUSY; ++r) load(r, here, k + S);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if constexpr (STEPS > 0) behind = step[MI - 1];
        here = next;
        next = next == last ? lds : next + Cfg::STAGE_BYTES;
    };
    constexpr std::integral_constant<int, 0> at0{};
    int k = 0;
    if constexpr (STEPS > 0) {
        constexpr std::integral_constant<int, 1> at1{};
        constexpr std::integral_constant<int, 2> at2{};
        constexpr std::integral_constant<int, 3> at3{};
        for (; k + 3 < ksteps; k += 4) {
            slab(at0, std::true_type{}, k, xa, wa, xb, wa);
            slab(at1, std::true_type{}, k + 1, xb, wa, xa, wa);
            slab(at2, std::true_type{}, k + 2, xa, wa, xb, wa);
            slab(at3, std::true_type{}, k + 3, xb, wa, xa, wa);
        }
        if (k < ksteps) slab(at0, std::false_type{}, k, xa, wa, xb, wa);
        if (k + 1 < ksteps) slab(at1, std::false_type{}, k + 1, xb, wa, xa, wa);
        if (k + 2 < ksteps) slab(at2, std::false_type{}, k + 2, xa, wa, xb, wa);
    } else {
        for (; k + 1 < ksteps; k += 2) {
            slab(at0, std::false_type{}, k, xa, wa, xb, wb);
            slab(at0, std::false_type{}, k + 1, xb, wb, xa, wa);
        }
        if (k < ksteps) slab(at0, std::false_type{}, k, xa, wa, xb, wb);
    }
    wait_vmcnt<0>();   // (the loads of slabs past the end)
    if constexpr (STEPS > 0) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[NI - 1][MI - 1][j] += part[j] * behind;
    }

    // ---- epilogue: a lane holds four consecutive n of one m per (sub-tile, quad)
    TileOut<Cfg::BM, Cfg::BN, Cfg::THREADS>::store(g, lds, m0, n0, [&](auto put) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int c = nw + ni * 32 + q * 8 + lgrp * 4;
                    const f32x4 b4 = *reinterpret_cast<const f32x4*>(columns + Cfg::BN + c);
                    float v[4];
                    if constexpr (ScaleKind == SCALE_TENSOR) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float f = (float)acc[ni][mi][4 * q + j];
                            v[j] = RoundFirst ? add_bias(f * s_tensor, b4[j], true) : f * s_tensor + b4[j];
                        }
                    } else {
#pragma clang fp contract(off)
                        const f32x4 s4 = *reinterpret_cast<const f32x4*>(columns + c);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float scaled = (float)acc[ni][mi][4 * q + j] * sx[mi] * s4[j];
                            v[j] = scaled + b4[j];
                        }
                    }
                    put(wave_m * 64 + mi * 32 + lrow, c, v);
                }
    });
}

// bf16 output, K in whole slabs, more tiles of 128 x 128 than compute units and no more of these than that. us, int8 / fp8, on tiles
// of 128 x 128 (to 448 of them, else 256 x 256) -> here: 1111 x 4096 x 11008 86 / 84 -> 66 / 61, 2048 x 4096 x 4096 43.9 / 41.7 ->
// 35.8 / 33, 1100 x 4096 x 4096 36.2 / 35.0 -> 27.8 / 25.4, 1954 x 3072 x 2048 25.0 / 23.3 -> 18.6 / 17.5, 4000 x 2048 x 2048 27.4 /
// 25.9 -> 21.9 / 20.3, 500 x 11264 x 2048 24.6 / 22.5 -> 17.8 / 17.0, 1200 x 4096 x 256 12.2 / 11.4 -> 8.8 / 8.4. With half as
// many tiles those of 128 x 128 are one round too, and the faster one (900 x 4096 x 4096, 256 of them, 23.5 of fp8).
inline bool wide256_shape_ok(const GemmArgs& g) {
    if (!tiled_shape_ok(g) || (g.k & 127) != 0 || g.k < 128 || g.out_kind != OUT_BF16) return false;
    const int64_t tm = (g.m + 127) / 128, small = tm * ((g.n + 127) / 128);
    return small > 256 && tm * ((g.n + 255) / 256) <= 256;
}

template <class Op, int ScaleKind, bool RoundFirst = false>
inline void launch_wide256(const GemmArgs& g, hipStream_t stream) {
    using Cfg = Wide256Cfg;
    if constexpr (!RoundFirst && ScaleKind == SCALE_TENSOR)
        if (g.round_first) return launch_wide256<Op, ScaleKind, true>(g, stream);
    const int tiles = ((g.m + Cfg::BM - 1) / Cfg::BM) * ((g.n + Cfg::BN - 1) / Cfg::BN);
    auto kern = gemm_wide256_kernel<Op, ScaleKind, RoundFirst>;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::LDS_BYTES, lds_allowed);
    note_kernel(ScaleKind == SCALE_BLOCK128 ? "mid128x256_block128" : "mid128x256");
    kern<<<dim3((unsigned)tiles), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream>>>(g);
}

}  // namespace w8a8
