// 8-bit NT GEMM for shapes with too few 128 x 128 tiles to occupy the chip: a few hundred
// activation rows against a narrow weight matrix (a short prompt, a large decode batch), or few
// rows with a K the decode kernels do not take.
//
// 64 x 64 output tiles, four waves of 32 x 32 (one MFMA 32x32 sub-tile, 16 accumulator registers),
// K in 128-byte slabs. With one or two workgroups on a compute unit little else hides a slab's
// memory latency, so the slabs come through a ring of S LDS stages of 16 KiB filled by
// direct-to-LDS loads S - 1 slabs ahead, and a wave reads the fragments of slab k + 1 into a second
// register set before it issues the MFMAs of slab k (the generic tiled kernel, which stages a slab
// through registers and waits for it, needs 1.2 k cycles a slab on these shapes; this one ~500,
// which is the L2 bandwidth 256 workgroups pulling 16 KiB a slab get). One workgroup barrier per slab: it publishes
// slab k + 1 (every wave has waited for its own loads) and retires slab k - 1's stage, which the
// load of slab k + S - 1 then overwrites. Past the end of K the loads run on an empty descriptor
// (no traffic), so the wait counts are the same in every iteration.
//
// LDS layout of a slab, load plan per wave (rows 16 w .. 16 w + 15 of both operands), fragment
// reads, accumulator layout and epilogue are those of gemm_mid128_kernel.
#pragma once
#include <type_traits>

#include "gemm_pingpong.cuh"

namespace w8a8 {

template <int S>
struct Small64Cfg {
    static constexpr int BM = 64, BN = 64, BK = 128;
    static constexpr int THREADS = 256;
    static constexpr int STAGES = S;
    static constexpr int OPERAND_BYTES = 64 * BK;        // one operand's slab: 8 KiB
    static constexpr int STAGE_BYTES = 2 * OPERAND_BYTES;
    static constexpr int LDS_BYTES = S * STAGE_BYTES;
    static_assert(S >= 3 && 4 * (S - 2) < 64, "ring depth");
};

// RoundFirst (per-tensor scales): the product is rounded to bf16 before the bias joins it (see gemm_mid128.cuh; 200 x 2048
// x 2048 6.2 us, with the choice in the epilogue 6.3)
// G: groups of four waves. 2: where each tile has a compute unit to itself, two groups form the tile over half of K each, with
// rings of their own, and add their sums at the end; the one covers the other's waits, and a barrier publishes two slabs. us, one
// group -> two, int8 / fp8: 200 x 4096 x 11008 27.3 / 26.6 -> 23.6 / 22.6, 193 x 2048 x 5632 13.9 / 12.9 -> 11.9 / 11.2, 256 x 4096 x
// 4096 12.6 / 11.5 -> 11.2 / 10.7, 300 x 2048 x 2048 8.4 / 7.8 -> 7.6 / 7.3. With few slabs the exchange of the sums costs more than
// the half chain saves, an odd slab more still (500 x 2048 x 128 4.2 / 3.9 -> 4.5 / 4.3, x 640 4.9 / 4.6 -> 5.2 / 5.0; one
// group's time over two's with 8 slabs 1.02 / 0.98, 10 1.04 / 1.00, 11 1.01 / 0.98, 12 1.05 / 1.02): from 10 slabs with a step a row and column, from
// 12 with one step. 128-block scales gain from 40 slabs on, where their longer prologue is made up for: 374 x 1536 x 7168 17.4 -> 15.5, 70 x 2048 x 7168 14.5 -> 13.2, 145 x
// 4096 x 4096 10.3 -> 10.0, 250 x 4096 x 4096 10.7 -> 10.8, 100 x 7168 x 2048 7.1 -> 7.3. (Four waves of the whole tile over a
// quarter of K each, with no barrier and every slab read once: the same with long K, 0.6 to 1.4 us slower with up to 16 slabs.)
template <class Op, int ScaleKind, int S, bool RoundFirst, int G>
__global__ __launch_bounds__(256 * G, G == 2 || ScaleKind == SCALE_BLOCK128 ? 2 : 1) void gemm_small64_kernel(GemmArgs g) {
    using Cfg = Small64Cfg<S>;
    using Acc = typename Op::Acc;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave_m = wave & 1, wave_n = wave >> 1;   // 2 x 2 waves
    const int lrow = lane & 31, lgrp = lane >> 5;

    const int tiles_m = (g.m + Cfg::BM - 1) / Cfg::BM;
    const int tiles_n = (g.n + Cfg::BN - 1) / Cfg::BN;
    const TileCoord tc = map_tile(tiles_m, tiles_n);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * Cfg::BN;
    const int K = g.k;
    const int ksteps = K >> 7;
    // the group's slabs: `count` of them from `first` on, those from `end` on zeros
    const int count = (ksteps + G - 1) / G, first = group * count, end = min(first + count, ksteps);
    constexpr int QUADS = 4 / G;              // of a wave's accumulators, that it finishes: from quad0 on
    const int quad0 = group * QUADS;

    // epilogue operands, requested now
    const EpilogueScalars es = load_epilogue_scalars<ScaleKind>(g);
    [[maybe_unused]] const float s_tensor = es.sa * es.sb;
    const int mw = m0 + wave_m * 32, nw = n0 + wave_n * 32;
    float sx = 1.0f;
    if constexpr (ScaleKind == SCALE_ROWCOL) {
        const int m = mw + lrow;
        sx = (m < g.m) ? g.sa[m] : 0.0f;
    }
    f32x4 sw4[QUADS], b4[QUADS];
    const uint16_t* bias = static_cast<const uint16_t*>(g.bias);
#pragma unroll
    for (int q = 0; q < QUADS; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = nw + (quad0 + q) * 8 + lgrp * 4 + j;
            sw4[q][j] = 1.0f;
            b4[q][j] = 0.0f;
            if (n < g.n) {
                if constexpr (ScaleKind == SCALE_ROWCOL) sw4[q][j] = g.sb[n];
                // (the block-scaled instance fetches the bias at the end: its loop counts its own loads)
                if constexpr (ScaleKind != SCALE_BLOCK128)
                    if (bias) b4[q][j] = bf16_to_f32(bias[n]);
            }
        }

    // ---- direct-to-LDS load plan: wave w fills rows 16w .. 16w+15 of both operands, 8 rows per
    // instruction (two instructions an operand and slab). Rows past M / N are past the buffer's
    // num_records and read as zero.
    const uint32_t x_bytes = (uint32_t)g.m * (uint32_t)K, w_bytes = (uint32_t)g.n * (uint32_t)K;
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
    uint8_t* const ring = lds + group * Cfg::LDS_BYTES;
    uint8_t* const dma_base = ring + wave * (16 * 128);
    auto issue = [&](int stage, int slab) __attribute__((always_inline)) {
        const bool live = slab < end;
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(g.a, live ? x_bytes : 0u);
        const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.b, live ? w_bytes : 0u);
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
    const int x_rd = (wave_m * 32) * 128;
    const int w_rd = Cfg::OPERAND_BYTES + (wave_n * 32) * 128;
    auto read = [&](int stage, u32x4 (&xf)[4], u32x4 (&wf)[4]) __attribute__((always_inline)) {
        const uint8_t* const base = ring + stage * Cfg::STAGE_BYTES;
#pragma unroll
        for (int j = 0; j < 4; ++j) wf[j] = *reinterpret_cast<const u32x4*>(base + w_rd + frag_off[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) xf[j] = *reinterpret_cast<const u32x4*>(base + x_rd + frag_off[j]);
    };

    Acc acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0;
    u32x4 xa[4], wa[4], xb[4], wb[4];

    // ---- 128-block scales: a slab is exactly one K-block and the tile's 64 columns lie in one
    // weight block. The slab's product is formed in a temporary and joins the accumulator scaled by
    // the row's and the block's steps, behind the MFMAs of the next slab. The steps of four slabs are one load of the row's and
    // one of the block's (a load a slab touched a line a row, on the load path that the slabs come through), requested in the
    // first slab of the four before, ahead of its slab loads; past the last slab and past M they are never used. Buffer loads
    // whatever the compiler makes of the addresses: the waits count them. 145 x 4096 x 4096 12.9 -> 9.4 us (9.0 with one scale),
    // 300 x 4096 x 4096 19.6 -> 15.5, 600 x 1536 x 7168 22.4 -> 18.1, 70 x 7168 x 2048 8.1 -> 6.5; the products behind the next slab's
    // MFMAs alone 11.3, 20.4, 19.9, 7.35.
    constexpr int STEPS = ScaleKind == SCALE_BLOCK128 ? 2 : 0;
    [[maybe_unused]] u32x4 steps[2], steps_next[2];
    [[maybe_unused]] float behind = 0.0f;
    [[maybe_unused]] Acc pa, pb;
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsa = make_rsrc(g.sa, STEPS ? (uint32_t)g.m * (uint32_t)ksteps * 4u : 0u);
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsb = make_rsrc(g.sb, STEPS ? (uint32_t)((g.n + 127) >> 7) * (uint32_t)ksteps * 4u : 0u);
    auto request_steps = [&](int kb, u32x4 (&d)[2]) __attribute__((always_inline)) {
        if constexpr (STEPS > 0) {
            d[0] = buf_load16(rsa, (uint32_t)(mw + lrow) * (uint32_t)ksteps * 4u, (uint32_t)kb * 4u);
            d[1] = buf_load16(rsb, (uint32_t)(n0 >> 7) * (uint32_t)ksteps * 4u, (uint32_t)kb * 4u);
        }
    };
    if constexpr (STEPS > 0) {
#pragma unroll
        for (int j = 0; j < 16; ++j) pb[j] = 0;
    }

    // ---- prologue: slabs 0 .. S-2 in flight; slab 0 visible and in the first register set
    request_steps(first, steps);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S - 1; ++s) issue(s, first + s);
    wait_vmcnt<4 * (S - 2)>();
    phase_barrier();
    read(0, xa, wa);

    int rd_stage = 1;        // stage of slab k + 1
    int wr_stage = S - 1;    // stage of slab k + S - 1
    // one slab: MFMAs on (xc, wc) = slab k; slab k + 1 published and read into (xn, wn); slab k + S - 1 requested
    // (128-block scales: AT: which of its four slabs; MORE: four more follow them, whose steps the first requests; part, before:
    // this slab's product and the last one's)
    auto step = [&](auto at, auto more, int k, const u32x4 (&xc)[4], const u32x4 (&wc)[4], u32x4 (&xn)[4], u32x4 (&wn)[4],
                    [[maybe_unused]] Acc& part, [[maybe_unused]] const Acc& before) __attribute__((always_inline)) {
        constexpr int AT = decltype(at)::value;
        constexpr bool MORE = decltype(more)::value;
        wait_vmcnt<4 * (S - 3) + (MORE && AT == 1 ? STEPS : 0)>();   // own loads of slab k + 1 (younger: slabs k + 2 .. k + S - 2)
        wait_lgkmcnt0();             // own reads of slab k
        phase_barrier();
        if constexpr (STEPS > 0 && MORE && AT == 0) {
            static_assert(S == 4, "the waits of the block-scaled loop are written for four stages");
            request_steps(k + 4, steps_next);
            __builtin_amdgcn_sched_barrier(0);
        }
        issue(wr_stage, k + S - 1);
        read(rd_stage, xn, wn);
        if constexpr (ScaleKind == SCALE_BLOCK128) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < Op::STEPS; ++q) {
                if (q == 0) part = Op::mma_step(q, wc, xc, Acc{});
                else part = Op::mma_step(q, wc, xc, part);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 16 / Op::STEPS * q; j < 16 / Op::STEPS * (q + 1); ++j) acc[j] += before[j] * behind;
                __builtin_amdgcn_sched_barrier(0);
            }
            behind = G == 1 || k < end ? __uint_as_float(steps[0][AT]) * __uint_as_float(steps[1][AT]) : 0.0f;
        } else {
#pragma unroll
            for (int q = 0; q < Op::STEPS; ++q) acc = Op::mma_step(q, wc, xc, acc);
        }
        rd_stage = (rd_stage == S - 1) ? 0 : rd_stage + 1;
        wr_stage = (wr_stage == S - 1) ? 0 : wr_stage + 1;
    };
    constexpr std::integral_constant<int, 0> at0{};
    int k = first;
    if constexpr (STEPS > 0) {
        constexpr std::integral_constant<int, 1> at1{};
        constexpr std::integral_constant<int, 2> at2{};
        constexpr std::integral_constant<int, 3> at3{};
        for (; k + 3 < first + count; k += 4) {
            step(at0, std::true_type{}, k, xa, wa, xb, wb, pa, pb);
            step(at1, std::true_type{}, k + 1, xb, wb, xa, wa, pb, pa);
            step(at2, std::true_type{}, k + 2, xa, wa, xb, wb, pa, pb);
            step(at3, std::true_type{}, k + 3, xb, wb, xa, wa, pb, pa);
            steps[0] = steps_next[0];
            steps[1] = steps_next[1];
        }
        if (k < first + count) step(at0, std::false_type{}, k, xa, wa, xb, wb, pa, pb);
        if (k + 1 < first + count) step(at1, std::false_type{}, k + 1, xb, wb, xa, wa, pb, pa);
        if (k + 2 < first + count) step(at2, std::false_type{}, k + 2, xa, wa, xb, wb, pa, pb);
    } else {
        for (; k < first + count; k += 2) {
            step(at0, std::false_type{}, k, xa, wa, xb, wb, pa, pb);
            if (k + 1 < first + count) step(at0, std::false_type{}, k + 1, xb, wb, xa, wa, pb, pa);
        }
    }
    if constexpr (STEPS > 0) {
        const Acc& last = (count & 1) ? pa : pb;
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] += last[j] * behind;
    }
    // no load outlives the kernel's use of LDS: the remaining ones ran on empty descriptors or are waited for here
    wait_vmcnt<0>();

    // ---- two groups: each finishes half of the quads, with the other's sums of them
    [[maybe_unused]] typename Op::AccScalar half[8];
    if constexpr (G == 2) {
        typedef typename Op::AccScalar Four __attribute__((ext_vector_type(4)));
        wait_lgkmcnt0();
        phase_barrier();   // the rings are free: every wave's reads of them, and loads into them, are behind it
        uint8_t* const there = lds + wave * 2048 + lane * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            Four give;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                give[j] = group ? acc[4 * i + j] : acc[8 + 4 * i + j];
                half[4 * i + j] = group ? acc[8 + 4 * i + j] : acc[4 * i + j];
            }
            *reinterpret_cast<Four*>(there + (1 - group) * 8192 + i * 1024) = give;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const Four got = *reinterpret_cast<const Four*>(there + group * 8192 + i * 1024);
#pragma unroll
            for (int j = 0; j < 4; ++j) half[4 * i + j] += got[j];
        }
    }

    // ---- epilogue: a lane holds four consecutive n of one m per quad: 8-byte stores
    uint16_t* const out = static_cast<uint16_t*>(g.out);
    const bool vec_ok = (g.n & 3) == 0;
    const int m = mw + lrow;
    if (m >= g.m) return;
#pragma unroll
    for (int q = 0; q < QUADS; ++q) {
        const int n = nw + (quad0 + q) * 8 + lgrp * 4;
        if (n >= g.n) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float f = G == 2 ? (float)half[4 * q + j] : (float)acc[4 * q + j];
            if constexpr (ScaleKind == SCALE_BLOCK128) {
                v[j] = f + ((bias && n + j < g.n) ? bf16_to_f32(bias[n + j]) : 0.0f);
            } else if constexpr (ScaleKind == SCALE_TENSOR) {
                v[j] = RoundFirst ? add_bias(f * s_tensor, b4[q][j], true) : f * s_tensor + b4[q][j];
            } else {
#pragma clang fp contract(off)
                const float scaled = f * sx * sw4[q][j];
                v[j] = scaled + b4[q][j];
            }
        }
        const size_t o = (size_t)m * g.n + n;
        if (vec_ok) {
            u32x2 pk;
            pk.x = pack_bf16x2(v[0], v[1]);
            pk.y = pack_bf16x2(v[2], v[3]);
            *reinterpret_cast<u32x2*>(out + o) = pk;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (n + j < g.n) out[o + j] = f32_to_bf16(v[j]);
        }
    }
}

// bf16 output, K in whole slabs; the caller decides by tile counts
inline bool small64_shape_ok(const GemmArgs& g) {
    return tiled_shape_ok(g) && (g.k & 127) == 0 && g.k >= 128 && g.out_kind == OUT_BF16;
}

// Four stages (three slabs ahead, 64 KiB: two workgroups share a compute unit). A ring of eight
// stages measured the same or slower (256 x 2048 x 2048: 8.3 against 7.6 us; 384 x 2048 x 5632: 14.4
// against 15.0 us): 128 KiB of LDS leaves one workgroup per compute unit, and what bounds the
// kernel is the 16 KiB a 64 x 64 tile pulls out of L2 per slab, not latency.
constexpr int kSmall64Stages = 4;

template <class Op, int ScaleKind, bool RoundFirst = false, int G = 1>
inline void launch_small64(const GemmArgs& g, hipStream_t stream) {
    using Cfg = Small64Cfg<kSmall64Stages>;
    if constexpr (!RoundFirst && ScaleKind == SCALE_TENSOR)
        if (g.round_first) return launch_small64<Op, ScaleKind, true>(g, stream);
    const int64_t tiles = (int64_t)((g.m + 63) / 64) * ((g.n + 63) / 64);
    constexpr int kTwoGroups = ScaleKind == SCALE_BLOCK128 ? 40 : ScaleKind == SCALE_TENSOR ? 12 : 10;   // slabs from which they gain
    if constexpr (G == 1)
        if (tiles <= 256 && g.k >= kTwoGroups * 128)
            return launch_small64<Op, ScaleKind, RoundFirst, 2>(g, stream);
    auto kern = gemm_small64_kernel<Op, ScaleKind, kSmall64Stages, RoundFirst, G>;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), G * Cfg::LDS_BYTES, lds_allowed);
    note_kernel("small64");
    kern<<<dim3((unsigned)tiles), dim3(G * Cfg::THREADS), G * Cfg::LDS_BYTES, stream>>>(g);
}

}  // namespace w8a8
