// int8 x int8 products on 256 x 256 tiles, one step per token and one per output channel, bf16 output: the main loop of
// gemm_walk16.cuh and, behind it, one of four epilogues.
//
//   EPI_PLAIN   dequantized, with a bias if there is one
//   EPI_SWIGLU  the pairs of a fused gate|up weight (64 gate rows, then the 64 up rows of the same columns, per block of
//               128) leave as h = up * silu(gate), with the maxima that the quantizer behind it needs
//   EPI_ROPE    the fused q|k|v projection of a prompt, rotated and written to q and the caches
//   EPI_RESID   plus the residual row
//
// What bounds it: the power cap (see gemm_walk16.cuh). On 32x32x32 MFMAs before -> here: 4096 x 11008 x 4096 173 -> 158 us
// (quantizer included), 8000 tokens 333 -> 303, 8000 x 11264 x 2048 190 -> 178; gate|up of a 16384-token prompt with its
// epilogue (11264 x 2048) 369 -> 356, its down and output projections with their residual 159 -> 147 and 82 -> 75.
#pragma once
#include "gemm_walk16.cuh"

namespace w8a8 {

// silu(g) = g / (1 + exp(-g)) on the hardware's exp2 and reciprocal, the arithmetic of the
// SwiGLU producer kernel (quantize.hip)
__device__ __forceinline__ float silu_hw(float g) {
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.44269504088896340736f));
}

enum : int { EPI_PLAIN = 0, EPI_SWIGLU = 1, EPI_ROPE = 2, EPI_RESID = 3 };

template <int Epi>
__global__ __launch_bounds__(Wave128Cfg::THREADS) void gemm_wave128_i8_kernel(GemmArgs g, RopeCacheArgs rc) {
    using Cfg = Wave128Cfg;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave & 1, wave_n = wave >> 1;
    const int lrow = lane & 15, lgrp = lane >> 4;

    const TileCoord tc = map_tile((g.m + Cfg::BM - 1) / Cfg::BM, (g.n + Cfg::BN - 1) / Cfg::BN);
    const int m0 = tc.tm * Cfg::BM, n0 = tc.tn * Cfg::BN;
    const int mw = m0 + wave_m * 128, nwv = n0 + wave_n * 128;   // first token and column of this wave
    // requested now, used in the epilogue: the latency hides under the main loop
    float sx[8];  // steps of this lane's eight tokens
#pragma unroll
    for (int mi = 0; mi < 8; ++mi) {
        const int m = mw + mi * 16 + lrow;
        sx[mi] = (m < g.m) ? g.sa[m] : 0.0f;
    }

    // (rows past M / N lie past the descriptors and read as zeros)
    uint32_t x_off[8], w_off[8];
    walk16_offsets(lane, m0 + wave * 64, 64, (uint32_t)g.k, x_off);
    walk16_offsets(lane, n0 + wave * 64, 64, (uint32_t)g.k, w_off);
    i32x4 acc[8][8];  // [column sub-tile][token sub-tile]
    walk16<Walk16I8>(lds, g.a, (uint32_t)g.m * (uint32_t)g.k, x_off, g.b, (uint32_t)g.n * (uint32_t)g.k, w_off, g.k >> 7, acc);

    // ---------------- epilogue ----------------
    // N % 8 == 0. A pass is 32 tokens (two sub-tiles), laid down row-major in a wave-private staging buffer and streamed out
    // as whole row pieces, 16 bytes a lane; two buffers in turn. Per-column operands are all requested before the first
    // one is used. Output rows go through a buffer descriptor: rows past M and (by the offset chosen below) columns past N
    // are dropped by the bounds check; the row step goes into the checked (vector) offset because the scalar offset of a
    // buffer instruction takes no part in the check. The stores are non-temporal (aux bit 1): the output streams to memory
    // while the epilogue still computes instead of sitting dirty in L2 until the end-of-kernel write-back.
    const int rows_here = min(Cfg::BM, g.m - m0);
    f32x4 sw4[8];
#pragma unroll
    for (int ni = 0; ni < 8; ++ni) {
        const int n = nwv + ni * 16 + lgrp * 4;
        sw4[ni] = (n < g.n) ? *reinterpret_cast<const f32x4*>(g.sb + n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto dequant = [&](int ni, int mi, float (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma clang fp contract(off)
            v[j] = (float)acc[ni][mi][j] * sx[mi] * sw4[ni][j];
        }
    };
    if constexpr (Epi == EPI_ROPE) {
        // The rows are the fused q|k|v projection of a decoder layer, head_dim 128: the 128
        // columns of a wave tile are one head. The epilogue goes on where the separate rotary /
        // cache-write kernel would start: the bf16-rounded value pairs of q and k are rotated
        // (fp32 products and sums rounded one by one, one rounding to bf16 -- the arithmetic of
        // rope_cache.hip on the same rounded inputs), a pass of 32 tokens x 128 dims is staged
        // through LDS and leaves as whole 256-byte head rows: q to [batch, heads, seq, 128], k
        // and v into the cache at the tokens' positions (a position outside the cache: nothing).
        constexpr int ROWB = Cfg::EPI_ROW_BYTES, PASS_BYTES = Cfg::EPI_PASS_BYTES;
        uint8_t* const mine = lds + wave * (2 * PASS_BYTES);
        const int hh = nwv >> 7;                         // head among q heads | k heads | v heads
        const bool live_head = nwv < g.n;
        const bool is_q = hh < rc.n_heads, rotate = hh < rc.n_heads + rc.n_kv_heads;
        const int hk = hh - rc.n_heads - (rotate ? 0 : rc.n_kv_heads);
        void* const dst_base = is_q ? rc.q_out : (rotate ? rc.k_cache : rc.v_cache);
        const uint32_t dst_bytes = is_q ? (uint32_t)g.m * (uint32_t)rc.n_heads * 256u
                                        : (uint32_t)rc.batch * (uint32_t)rc.n_kv_heads * (uint32_t)rc.max_len * 256u;
        const __amdgpu_buffer_rsrc_t rout = make_rsrc(dst_base, live_head ? dst_bytes : 0u);
        const int r4 = lane >> 4, c16 = lane & 15;
        // One wave per SIMD: nothing hides a memory round trip inside the epilogue, so everything
        // it reads is requested ahead of its use -- the destinations of the 8 rows this lane will
        // store (cache slots: one lookup of the token's position each) a pass ahead (those of all four passes at once
        // spilled 22 registers: 32 x 512 x 512 74.9 us, here 71.7), the (cos, sin) pairs of
        // a group of 32 columns x 16 tokens four groups before the group that uses them.
        // token index -> (sequence, token in sequence) without an integer division per row: the
        // float quotient of m < 2^23 is off by at most one, which the remainder shows
        const float inv_seq = 1.0f / (float)rc.seq;
        auto split_token = [&](int m, int& bt, int& sq) {
            bt = (int)((float)m * inv_seq);
            sq = m - bt * rc.seq;
            if (sq < 0) { --bt; sq += rc.seq; }
            else if (sq >= rc.seq) { ++bt; sq -= rc.seq; }
        };
        uint32_t dst_off[2][8];
        auto find_rows = [&](int p) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int m = mw + p * 32 + i * 4 + r4;
                int bt, sq;
                split_token(m, bt, sq);
                uint32_t at = kOutOfRange;
                if (m < g.m) {
                    if (is_q) {
                        at = (uint32_t)((bt * rc.n_heads + hh) * rc.seq + sq) * 256u + (uint32_t)c16 * 16u;
                    } else {
                        const int64_t pos = rc.positions[sq];
                        if (pos >= 0 && pos < rc.max_len)
                            at = (uint32_t)((int64_t)(bt * rc.n_kv_heads + hk) * rc.max_len + pos) * 256u + (uint32_t)c16 * 16u;
                    }
                }
                dst_off[p & 1][i] = at;
            }
        };
        find_rows(0);
        // group gi = mi * 4 + c: the lane's token of sub-tile mi, columns 32 c .. 32 c + 31
        constexpr int kAhead = 4;
        f32x4 cs[kAhead + 1][2];
        const float* cs_row[8];
#pragma unroll
        for (int mi = 0; mi < 8; ++mi) {
            int bt, sq;
            split_token(mw + mi * 16 + lrow, bt, sq);
            cs_row[mi] = rc.freqs + ((int64_t)sq * 64 + (lgrp * 2)) * 2;
        }
        auto request_cs = [&](int gi) {
            if (!rotate || gi >= 32) return;
#pragma unroll
            for (int q = 0; q < 2; ++q)  // d = 16 ni + 4 lgrp: pair index d / 2
                cs[gi % (kAhead + 1)][q] = *reinterpret_cast<const f32x4*>(cs_row[gi >> 2] + ((gi & 3) * 16 + q * 8) * 2);
        };
#pragma unroll
        for (int gi = 0; gi < kAhead; ++gi) request_cs(gi);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint8_t* const buf = mine + (p & 1) * PASS_BYTES;
            if (p + 1 < 4) find_rows(p + 1);
#pragma unroll
            for (int gg = 0; gg < 8; ++gg) {
                const int gi = p * 8 + gg, mi = gi >> 2;
                request_cs(gi + kAhead);
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int ni = (gi & 3) * 2 + q;
                    float v[4];
                    dequant(ni, mi, v);
                    u32x2 pk;
                    pk.x = pack_bf16x2(v[0], v[1]);
                    pk.y = pack_bf16x2(v[2], v[3]);
                    if (rotate) {
                        const f32x4 c4 = cs[gi % (kAhead + 1)][q];
                        const float x[4] = {__uint_as_float(pk.x << 16), __uint_as_float(pk.x & 0xffff0000u),
                                            __uint_as_float(pk.y << 16), __uint_as_float(pk.y & 0xffff0000u)};
                        float y[4];
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
#pragma clang fp contract(off)
                            const float c = c4[2 * t], sn = c4[2 * t + 1];
                            const float xe = x[2 * t], xo = x[2 * t + 1];
                            const float a0 = xe * c, a1 = xo * sn, b0 = xe * sn, b1 = xo * c;
                            y[2 * t] = a0 - a1;
                            y[2 * t + 1] = b0 + b1;
                        }
                        pk.x = pack_bf16x2(y[0], y[1]);
                        pk.y = pack_bf16x2(y[2], y[3]);
                    }
                    *reinterpret_cast<u32x2*>(buf + ((mi & 1) * 16 + lrow) * ROWB + (ni * 16 + lgrp * 4) * 2) = pk;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(buf + (i * 4 + r4) * ROWB + c16 * 16);
                __builtin_amdgcn_raw_buffer_store_b128(v, rout, dst_off[p & 1][i], 0, 0);
            }
        }
    } else if constexpr (Epi == EPI_SWIGLU) {
        // The wave's 128 columns are 64 gate columns (sub-tiles 0 to 3) and the 64 up columns
        // (sub-tiles 4 to 7) of the same 64 columns of h, so a lane holds every pair in its own
        // registers. gate and up are rounded to bf16 as the plain epilogue would have stored
        // them, then h = bf16(up * bf16(silu(gate))) -- the arithmetic of the SwiGLU producer
        // kernel on the same rounded inputs. A pass is 32 rows x 64 columns of h (one 128-byte
        // line per row, 144-byte rows in LDS); the maximum of |h| over the wave's 64 columns goes to
        // row_max[m, piece] (bf16 magnitudes order like their bit patterns, so the maximum is taken on the packed bits).
        constexpr int ROWB = 144, PASS_BYTES = 32 * ROWB;
        uint8_t* const mine = lds + wave * (2 * PASS_BYTES);
        const int hw = g.n >> 1;                       // width of h
        const uint32_t row_bytes = (uint32_t)hw * 2u;
        const __amdgpu_buffer_rsrc_t rout =
            make_rsrc(static_cast<uint16_t*>(g.out) + (size_t)m0 * hw, (uint32_t)rows_here * row_bytes);
        const int piece = nwv >> 7;                    // the wave's 64-column piece of h
        const int pieces = g.n >> 7;
        const int r8 = lane >> 3, c8 = lane & 7;
        const uint32_t lane_off = (nwv < g.n)
            ? (uint32_t)(wave_m * 128 + r8) * row_bytes + (uint32_t)(piece * 64 + c8 * 8) * 2u
            : kOutOfRange;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint8_t* const buf = mine + (p & 1) * PASS_BYTES;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int mi = 2 * p + h;
                uint32_t mx = 0u;
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) {
                    float gt[4], up[4];
                    dequant(ni, mi, gt);
                    dequant(ni + 4, mi, up);
                    u32x2 pk;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const uint32_t gb = pack_bf16x2(gt[2 * t], gt[2 * t + 1]);
                        const uint32_t ub = pack_bf16x2(up[2 * t], up[2 * t + 1]);
                        const uint32_t sb2 = pack_bf16x2(silu_hw(__uint_as_float(gb << 16)),
                                                         silu_hw(__uint_as_float(gb & 0xffff0000u)));
                        const uint32_t hb = pack_bf16x2(
                            __uint_as_float(ub << 16) * __uint_as_float(sb2 << 16),
                            __uint_as_float(ub & 0xffff0000u) * __uint_as_float(sb2 & 0xffff0000u));
                        pk[t] = hb;
                        const uint32_t mag = hb & 0x7fff7fffu;
                        mx = max(mx, max(mag & 0xffffu, mag >> 16));
                    }
                    *reinterpret_cast<u32x2*>(buf + (h * 16 + lrow) * ROWB + (ni * 16 + lgrp * 4) * 2) = pk;
                }
                // the row's other columns sit in the lanes 16, 32 and 48 away
                mx = max(mx, (uint32_t)__shfl_xor((int)mx, 16, 64));
                mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32, 64));
                const int m = mw + mi * 16 + lrow;
                if (lgrp == 0 && m < g.m && nwv < g.n) g.row_max[(size_t)m * pieces + piece] = __uint_as_float(mx << 16);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(buf + (i * 8 + r8) * ROWB + c8 * 16);
                __builtin_amdgcn_raw_buffer_store_b128(v, rout, lane_off + (uint32_t)(p * 32 + i * 8) * row_bytes, 0, 2);
            }
        }
    } else {
        constexpr int ROWB = Cfg::EPI_ROW_BYTES, PASS_BYTES = Cfg::EPI_PASS_BYTES;
        uint8_t* const mine = lds + wave * (2 * PASS_BYTES);
        const uint16_t* bias = static_cast<const uint16_t*>(g.bias);
        const uint32_t row_bytes = (uint32_t)g.n * 2u;
        const __amdgpu_buffer_rsrc_t rout =
            make_rsrc(static_cast<uint16_t*>(g.out) + (size_t)m0 * g.n, (uint32_t)rows_here * row_bytes);
        [[maybe_unused]] u32x2 braw[8];
        if constexpr (Epi == EPI_PLAIN) {
#pragma unroll
            for (int ni = 0; ni < 8; ++ni) {
                const int n = nwv + ni * 16 + lgrp * 4;
                braw[ni] = (bias && n < g.n) ? *reinterpret_cast<const u32x2*>(bias + n) : u32x2{0u, 0u};
            }
        }
        const int r4 = lane >> 4, c16 = lane & 15;
        const int nst = nwv + c16 * 8;
        const uint32_t lane_off = (nst < g.n)
            ? (uint32_t)(wave_m * 128 + r4) * row_bytes + (uint32_t)nst * 2u
            : kOutOfRange;
        // EPI_RESID: the residual rows of this tile, addressed like the output
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t rres = make_rsrc(
            static_cast<const uint16_t*>(Epi == EPI_RESID ? g.resid : g.out) + (size_t)m0 * g.n,
            (uint32_t)rows_here * row_bytes);
        // the eight residual pieces of a pass live in a ring: each is requested again for the
        // next pass as soon as it has been used, a whole pass ahead of its use
        [[maybe_unused]] u32x4 rr[8];
        if constexpr (Epi == EPI_RESID) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                rr[i] = buf_load16(rres, lane_off + (uint32_t)(i * 4) * row_bytes, 0);
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint8_t* const buf = mine + (p & 1) * PASS_BYTES;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int ni = 0; ni < 8; ++ni) {
                    float v[4];
                    dequant(ni, 2 * p + h, v);
                    if constexpr (Epi == EPI_PLAIN) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
#pragma clang fp contract(off)
                            v[j] += __uint_as_float((j & 1) ? braw[ni][j >> 1] & 0xffff0000u : braw[ni][j >> 1] << 16);
                        }
                    }
                    u32x2 pk;
                    pk.x = pack_bf16x2(v[0], v[1]);
                    pk.y = pack_bf16x2(v[2], v[3]);
                    *reinterpret_cast<u32x2*>(buf + (h * 16 + lrow) * ROWB + (ni * 16 + lgrp * 4) * 2) = pk;
                }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                u32x4 v = *reinterpret_cast<const u32x4*>(buf + (i * 4 + r4) * ROWB + c16 * 16);
                if constexpr (Epi == EPI_RESID) {
                    // bf16(y + residual) on the rounded y, element by element
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t y2 = v[e], r2 = rr[i][e];
                        v[e] = pack_bf16x2(__uint_as_float(y2 << 16) + __uint_as_float(r2 << 16),
                                           __uint_as_float(y2 & 0xffff0000u) + __uint_as_float(r2 & 0xffff0000u));
                    }
                    if (p + 1 < 4)
                        rr[i] = buf_load16(rres, lane_off + (uint32_t)((p + 1) * 32 + i * 4) * row_bytes, 0);
                }
                __builtin_amdgcn_raw_buffer_store_b128(v, rout, lane_off + (uint32_t)(p * 32 + i * 4) * row_bytes, 0, 2);
            }
        }
    }
}

template <int Epi = EPI_PLAIN>
inline void launch_wave128_i8(const GemmArgs& g, hipStream_t stream, const RopeCacheArgs& rc = RopeCacheArgs{}) {
    using Cfg = Wave128Cfg;
    const int tiles = ((g.m + Cfg::BM - 1) / Cfg::BM) * ((g.n + Cfg::BN - 1) / Cfg::BN);
    auto kern = gemm_wave128_i8_kernel<Epi>;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::LDS_BYTES, lds_allowed);
    note_kernel(Epi == EPI_SWIGLU ? "wave128_swiglu" : Epi == EPI_ROPE ? "wave128_rope" : Epi == EPI_RESID ? "wave128_resid" : "wave128");
    kern<<<dim3((unsigned)tiles), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream>>>(g, rc);
}

}  // namespace w8a8
