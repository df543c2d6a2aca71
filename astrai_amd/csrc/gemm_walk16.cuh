// The main loop of the 256 x 256 NT products on 16x16 MFMAs: four waves of 128 x 128, one to a SIMD, software-pipelined
// inside each wave. Operand bytes only: 8-bit or bf16 values differ in the instruction.
//
// A slab is 128 bytes of K: one fp8 16x16x128 MFMA of 32 cycles for a pair of 16-row sub-tiles, or two of 16 cycles
// (int8 16x16x64, bf16 16x16x32) on the two 16-byte pieces of a lane; all MFMAs of the first pieces of a quadrant come
// before those of the second, sixteen accumulators apart. A slab is cut into quadrants: the 128(m) x 128(n) wave tile =
// 2 x 2 quadrants of 64 x 64 = 4 x 4 pairs of sub-tiles, 512 MFMA cycles. A quadrant needs one half of the wave's
// activation rows (4 sub-tiles of 16 rows: 32 registers) and one half of its weight rows (32 registers). The
// quadrants are walked so that consecutive ones share one of the two halves, and
// during a quadrant the one half the next quadrant is missing is read from LDS into
// the buffer that is idle: four 32-register buffers XA, XB (activation halves 0, 1)
// and WA, WB (weight halves 0, 1).
// The walk has period two slabs (Q<x half><w half>, what is read meanwhile):
//   even slab k:   Q00 | W1(k) -> WB     Q01 | X1(k) -> XB      -- barrier --
//                  Q11 | X0(k+1) -> XA   Q10 | W1(k+1) -> WB
//   odd slab k+1:  Q01 | W0(k+1) -> WA   Q00 | X1(k+1) -> XB    -- barrier --
//                  Q10 | X0(k+2) -> XA   Q11 | W0(k+2) -> WA
// Every quadrant has 8 LDS reads of 1 KiB and 4 direct-to-LDS loads between its MFMAs. The order is written out and pinned,
// so that the MFMA pipe always has the next instruction waiting; the loads are spread evenly, because the CU's one load
// path takes a 1 KiB instruction every 16 cycles: four waves must not issue them faster than one per 64 cycles each, and have
// 128 for each of a slab's sixteen.
// Three activation and two weight stages (all 160 KiB): all of a slab's operands have been read when its second quadrant
// ends, at the slab's one barrier; the activation rows of slab k+2 are fetched before it (into the stage of slab k-1), the
// weight rows behind it.
//
// Operand roles and layouts: weight rows are the first MFMA operand; lane l supplies
// row (l & 15) of a sub-tile and the 32 bytes of K-group (l >> 4) (chunks 2g, 2g+1
// of the row's eight 16-byte chunks; any assignment of K bytes to lanes is a valid
// contraction as long as both operands share it); the accumulator lane holds, for
// token m = l & 15, the four outputs n = 4 (l >> 4) .. + 3 of the sub-tile.
//
// Why not 32x32 MFMAs: under the power cap loops of nothing else sustain on random operands 1.82 PFLOP/s of bf16
// 32x32x16 and 1.92 of 16x16x32, 3.36 POP/s of int8 32x32x32 and 3.77 of 16x16x64, 3.77 PFLOP/s of fp8 32x32x64 and 4.16
// of 16x16x128. (On zeros 2.48 and 2.33, 4.96 and 4.71, 4.99 and 4.98; other instructions fit less well beside them: 32 cycles of a large one hide 24 of others, 16 of a small one about 4.)
// The sums stay in one register each, by assembly: behind the builtins the compiler gives results other registers than
// it takes sums from and moves them back, which halves the rate.
#pragma once
#include "gemm_wave128.cuh"

namespace w8a8 {

typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));

// A lane's 32 bytes of a row, as the MFMAs of a slab take them: one for each 16-byte piece,
struct Walk16Pieces {
    static constexpr int kMfmas = 2;
    struct Frag {
        u32x4 piece[2];
        __device__ __forceinline__ void set(int j, u32x4 v) { piece[j] = v; }
    };
};

struct Walk16I8 : Walk16Pieces {
    using Acc = i32x4;
    static __device__ __forceinline__ void mma(int c, const Frag& w, const Frag& x, Acc& acc) {
        __asm__ volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(acc) : "v"(w.piece[c]), "v"(x.piece[c]));
    }
};

struct Walk16Bf16 : Walk16Pieces {
    using Acc = f32x4;
    static __device__ __forceinline__ void mma(int c, const Frag& w, const Frag& x, Acc& acc) {
        __asm__ volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w.piece[c]), "v"(x.piece[c]));
    }
};

// or one of twice the cycles for both (Fmt 0 e4m3, 1 e5m2)
template <int Fmt>
struct Walk16F8 {
    static constexpr int kMfmas = 1;
    using Acc = f32x4;
    struct Frag {
        u32x8 both;
        __device__ __forceinline__ void set(int j, u32x4 v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) both[4 * j + e] = v[e];
        }
    };
    static __device__ __forceinline__ void mma(int, const Frag& w, const Frag& x, Acc& acc) {
        __asm__ volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:%3 blgp:%3"
                         : "+a"(acc) : "v"(w.both), "v"(x.both), "n"(Fmt));
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
    using Frag = typename Op::Frag;
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

    // the lane's two 16-byte pieces of its row of a 16-row sub-tile. (Whole addresses that the compiler does not take apart
    // again: every weight stage and sub-tile is then a constant offset away, every sub-tile of an activation stage too.)
    int x_rd[2], w_rd[2];
    {
        const int sw = (lrow & 7) ^ ((lrow >> 3) & 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int off = lrow * 128 + (((2 * lgrp + j) ^ sw) << 4);
            x_rd[j] = off + (wave & 1) * 128 * 128;
            w_rd[j] = off + (wave >> 1) * 128 * 128 + Cfg::W_BASE;
            __asm__("" : "+v"(x_rd[j]), "+v"(w_rd[j]));
        }
    }
    // read r of 8 of half h of an operand: piece r / 4 of sub-tile 4h + r % 4
    auto read_x = [&](int r, int stage, int h, Frag (&f)[4]) __attribute__((always_inline)) {
        f[r & 3].set(r >> 2, *reinterpret_cast<const u32x4*>(
            lds + x_rd[r >> 2] + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048));
    };
    auto read_w = [&](int r, int stage, int h, Frag (&f)[4]) __attribute__((always_inline)) {
        f[r & 3].set(r >> 2, *reinterpret_cast<const u32x4*>(
            lds + w_rd[r >> 2] + stage * Cfg::OPERAND_BYTES + (4 * h + (r & 3)) * 2048));
    };

#pragma unroll
    for (int ni = 0; ni < 8; ++ni)
#pragma unroll
        for (int mi = 0; mi < 8; ++mi) acc[ni][mi] = typename Op::Acc{0, 0, 0, 0};
    Frag xa[4], xb[4], wa[4], wb[4];

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
    auto phase = [&](const Frag (&xf)[4], const Frag (&wf)[4], int xh, int wh, auto&& rd, auto&& ld) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16 * Op::kMfmas; ++i) {
            const int c = i >> 4, mi = (i >> 2) & 3, ni = i & 3;
            Op::mma(c, wf[ni], xf[mi], acc[4 * wh + ni][4 * xh + mi]);
#pragma unroll
            for (int r = 0; r < 8; ++r)
                if (r * Op::kMfmas == i) rd(r);
#pragma unroll
            for (int d = 0; d < 4; ++d)
                if ((d * 4 + 2) * Op::kMfmas == i) ld(d);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // one slab; ODD: its place in the two-slab walk. Past the end of K the loads run on an empty descriptor
    auto slab = [&](auto odd_c, int k) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd_c)::value;
        constexpr int ws = ODD ? 1 : 0;           // k % 2
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
