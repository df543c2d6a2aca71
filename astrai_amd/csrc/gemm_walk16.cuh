// The main loop of the 256 x 256 NT products on 16x16 MFMAs of 16 cycles (int8, bf16): four waves of 128 x 128, one to a
// SIMD, software-pipelined inside each wave. The walk is that of gemm_wave128_q16.cuh (a slab is 128 bytes of K, its
// quadrants of 64 x 64 in an order in which consecutive ones share an operand half, the half the next one is missing read
// from LDS meanwhile, direct-to-LDS loads two slabs ahead into three activation and two weight stages, one barrier a
// slab); a slab is two MFMAs of a pair of 16-row sub-tiles, on the two 16-byte pieces of a lane, where fp8 has one of 32
// cycles. All MFMAs of the first pieces of a quadrant come before those of the second, sixteen accumulators apart.
//
// Why the small MFMAs: under the power cap loops of nothing else sustain on random operands 1.82 PFLOP/s of bf16
// 32x32x16 and 1.92 of 16x16x32, 3.36 POP/s of int8 32x32x32 and 3.77 of 16x16x64. (On zeros 2.48 and 2.33, 4.96 and 4.71;
// other instructions fit less well beside them: 32 cycles of a large one hide 24 of others, 16 of a small one about 4.)
// The sums stay in one register each, by assembly: behind the builtins the compiler gives results other registers than
// it takes sums from and moves them back, which halves the rate.
#pragma once
#include "gemm_wave128.cuh"

namespace w8a8 {

struct Walk16I8 {
    using Acc = i32x4;
    static __device__ __forceinline__ void mma(u32x4 w, u32x4 x, Acc& acc) {
        __asm__ volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
    }
};

struct Walk16Bf16 {
    using Acc = f32x4;
    static __device__ __forceinline__ void mma(u32x4 w, u32x4 x, Acc& acc) {
        __asm__ volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
    }
};

// This lane's byte offsets of the eight loads of an operand's slab: wave w fills rows 64w .. 64w + 63 of a stage, 8 rows to
// an instruction, which are the rows first .. first + 63 of the operand; those from `live` on read as zeros.
__device__ __forceinline__ void walk16_offsets(int lane, int first, int live, uint32_t row_bytes, uint32_t (&off)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const uint32_t chunk = (uint32_t)((lane & 7) ^ (lane >> 3) ^ (r & 1)) * 16;
        off[r] = 8 * r < live ? (uint32_t)(first + 8 * r + (lane >> 3)) * row_bytes + chunk : kOutOfRange;
    }
}

// acc[weight sub-tile][token sub-tile] of a wave's 128 x 128: lane (lgrp, lrow) = (lane >> 4, lane & 15) holds, for token
// 16 mi + lrow, weight rows 16 ni + 4 lgrp .. + 3. The stages are free for other use when it returns.
template <class Op>
__device__ __forceinline__ void walk16(uint8_t* lds, const void* x, uint32_t x_bytes, const uint32_t (&x_off)[8],
                                       const void* w, uint32_t w_bytes, const uint32_t (&w_off)[8], int slabs,
                                       typename Op::Acc (&acc)[8][8]) {
    using Cfg = Wave128Cfg;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 15, lgrp = lane >> 4;

    uint8_t* const dma_base = lds + wave * (64 * 128);
    auto dma_x = [&](int r, __amdgpu_buffer_rsrc_t rx, int stage, uint32_t k0) __attribute__((always_inline)) {
        lds_dma16(rx, dma_base + stage * Cfg::OPERAND_BYTES + r * 1024, x_off[r], k0);
    };
    auto dma_w = [&](int r, __amdgpu_buffer_rsrc_t rw, int stage, uint32_t k0) __attribute__((always_inline)) {
        lds_dma16(rw, dma_base + Cfg::W_BASE + stage * Cfg::OPERAND_BYTES + r * 1024, w_off[r], k0);
    };

    // the lane's two 16-byte pieces of its row of a 16-row sub-tile
    int frag_off[2];
    {
        const int sw = (lrow & 7) ^ ((lrow >> 3) & 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) frag_off[j] = lrow * 128 + (((2 * lgrp + j) ^ sw) << 4);
    }
    const int x_rd = (wave & 1) * 128 * 128, w_rd = Cfg::W_BASE + (wave >> 1) * 128 * 128;
    // read r of 8 of half h of an operand: piece r / 4 of sub-tile 4h + r % 4
    auto read_x = [&](int r, int stage, int h, u32x4 (&f)[4][2]) __attribute__((always_inline)) {
        f[r & 3][r >> 2] = *reinterpret_cast<const u32x4*>(
            lds + x_rd + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048 + frag_off[r >> 2]);
    };
    auto read_w = [&](int r, int stage, int h, u32x4 (&f)[4][2]) __attribute__((always_inline)) {
        f[r & 3][r >> 2] = *reinterpret_cast<const u32x4*>(
            lds + w_rd + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048 + frag_off[r >> 2]);
    };

#pragma unroll
    for (int ni = 0; ni < 8; ++ni)
#pragma unroll
        for (int mi = 0; mi < 8; ++mi) acc[ni][mi] = typename Op::Acc{0, 0, 0, 0};
    u32x4 xa[4][2], xb[4][2], wa[4][2], wb[4][2];

    // slabs 0 and 1 in flight; slab 0 visible; halves 0 of slab 0 in xa, wa
    {
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, x_bytes), rw = make_rsrc(w, w_bytes);
        const __amdgpu_buffer_rsrc_t rx1 = make_rsrc(x, slabs > 1 ? x_bytes : 0u);
        const __amdgpu_buffer_rsrc_t rw1 = make_rsrc(w, slabs > 1 ? w_bytes : 0u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_x(r, rx, 0, 0u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_w(r, rw, 0, 0u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_x(r, rx1, 1, 128u);
#pragma unroll
        for (int r = 0; r < 8; ++r) dma_w(r, rw1, 1, 128u);
        wait_vmcnt<16>();  // slab 0
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) read_x(r, 0, 0, xa);
#pragma unroll
        for (int r = 0; r < 8; ++r) read_w(r, 0, 0, wa);
    }

    int xs = 0;  // k % 3
    // One quadrant: 32 MFMAs on (xf, wf); between them the 8 reads of the half the next quadrant is missing (in the first
    // half: the last has returned when they are needed) and 4 loads
    auto phase = [&](const u32x4 (&xf)[4][2], const u32x4 (&wf)[4][2], int xh, int wh, auto&& rd, auto&& ld) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int c = i >> 4, mi = (i >> 2) & 3, ni = i & 3;
            Op::mma(wf[ni][c], xf[mi][c], acc[4 * wh + ni][4 * xh + mi]);
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
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, more ? x_bytes : 0u);
        const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, more ? w_bytes : 0u);
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
        wait_vmcnt<8>();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        phase_barrier();
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
    int k = 0;
    for (; k + 1 < slabs; k += 2) {
        slab(std::false_type{}, k);
        slab(std::true_type{}, k + 1);
    }
    if (k < slabs) slab(std::false_type{}, k);
    // the last MFMAs' results, before vector instructions move them (the compiler does not see into the assembly); no load
    // outlives the loop, and every wave is done with the stages
    __asm__ volatile("s_nop 15\n\ts_nop 3");
    __builtin_amdgcn_s_waitcnt(0x0070);
    phase_barrier();
}

}  // namespace w8a8
