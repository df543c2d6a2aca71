// The gated delta rule of mix_delta.hip over blocks of 64 tokens. What makes a prompt of few heads slow there is the chain
// of chunks: 16 tokens cost some 1400 cycles of exchanges and roundings whatever they compute, and a compute unit that walks a
// column block has nothing else to do. Here a block is one step of the chain. With G_t, L_tj, M and P as there over 64 tokens,
//   T = (I + M)^-1 diag(beta),   W = T (G K),   V' = T V          (prep, every block of every head at once)
//   U = V' - W S,   O = (G Q) S + P U,   S <- diag(G_63) S + (L_63 K)^T U       (walk)
// so that nothing but W S, the difference and L K^T U lies between two states. 16 heads of 128 x 128, 4096 tokens: 211 us there,
// 162 here (prep 80, walk 82). Pairs (t, j) meet at the middle of their common
// block of 2, 4 .. 64 tokens, where both factors of L_tj are at most 1. 32-bit factors enter the matrix cores as bf16 terms: two
// and, where 64 tokens' writes nearly cancel, three (T, G K in T's product, U in the state's) and the product of both low terms;
// the inverse is formed on fp32 matrix instructions. Against 64 bits the state is 2 to 45% closer than in chunks of 16 over head
// sizes 32 to 256, random, slow and strong decays, and up to 35 times with one key over and over; two terms throughout were 5 to
// 40% further off, 4 times with equal keys.
#include <algorithm>

#include "mix_common.cuh"
#include "mix_launchers.h"

namespace astrai_mix {

namespace {

constexpr int kBlock = 64;   // tokens
constexpr float kUnitEps = 1e-6f;
constexpr int kAhead = 3;
using w8a8::kOutOfRange;

// Operands of a block, fragments of 64 lanes x 16 bytes, the high terms' fragment and then the low terms':
//   W, G Q     [token tile i][step s of 32 channels]: lane (g, c16): row 16 i + c16, channels 32 s + 4 g .. and 32 s + 16 + 4 g ..
//   L_63 K     [channel tile][step p of 32 tokens]: row = channel, tokens 32 p + 4 g .. and 32 p + 16 + 4 g ..
//   P          [token tile i][p <= i / 2] likewise
//   G_63       DP floats, in whole KiB
//   V'         [value tile][token tile]: lane (g, c16): fp32, tokens 16 i + 4 g .., column c16
template <int DP>
struct Operands {
    static constexpr int NS = DP / 32;
    static constexpr int kW = 0, kQ = 8 * NS, kL = 16 * NS, kP = 24 * NS, kG = kP + 12, kV = kG + (DP * 4 + 1023) / 1024;   // fragments
    __host__ __device__ static constexpr int pieces(int vp) { return kV + vp / 16 * 4; }
};

__device__ __forceinline__ void split4(f32x4 v, u32x2& hi, u32x2& lo) {
    uint32_t h0, l0, h1, l1;
    split2(v[0], v[1], h0, l0);
    split2(v[2], v[3], h1, l1);
    hi = u32x2{h0, h1};
    lo = u32x2{l0, l1};
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// three terms
__device__ __forceinline__ void split4(f32x4 v, u32x2& hi, u32x2& mid, u32x2& lo) {
    split4(v, hi, mid);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t h = hi[e >> 1], m = mid[e >> 1];
        v[e] = v[e] - __uint_as_float(e & 1 ? h & 0xffff0000u : h << 16) - __uint_as_float(e & 1 ? m & 0xffff0000u : m << 16);
    }
    lo = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// An operand of 32 tokens, its second tile only where that one is behind the product's own: a NaN there times the zeros of a
// triangle would reach tokens ahead of it.
__device__ __forceinline__ u32x4 own_half(u32x4 v, bool both) { return u32x4{v.x, v.y, both ? v.z : 0, both ? v.w : 0}; }

constexpr int kPrepThreads = 512;

// A wave holds eight tokens, a lane two channels (of each 128) of them. LDS: the matrices of one level of pairs, then M, P
// and T in fp32 in their place, then values and operands on their way out. All loads come before the first store (those of
// the values, behind the stores at first, took a quarter of the time: 91 us in place of 80), and the operands that need no T
// leave before it, so that their factors' registers are free for its terms (162 us for the whole rule, 213 with 87 registers in
// scratch memory). A third of what is left is the wait for the first loads, which two workgroups a compute unit begin together:
// 225 MB at 2.9 TB/s in all. The heads of a token run side by side (8 heads of 256, 2048 tokens: 106 us in place of 112).
template <int DP>
__global__ __launch_bounds__(kPrepThreads, DP <= 128 ? 4 : 2) void delta_block_prep_kernel(DeltaArgs a, int blocks, int first) {
    using Op = Operands<DP>;
    constexpr int NS = Op::NS, NB = (DP + 127) / 128, CH = DP < 128 ? DP : 128;   // channels at a time
    constexpr int kRow = CH * 2 + 16, kMat = kBlock * kRow, kLd = kBlock + 4;      // bytes; floats
    constexpr int kTile = 6 * 1024 + 16;    // bytes from a channel tile's fragments to the next's
    constexpr int kFp32 = kBlock * kLd * 4, kArea = 4 * kMat > 3 * kFp32 + 4 * 1088 ? 4 * kMat : 3 * kFp32 + 4 * 1088;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    float* const ms = reinterpret_cast<float*>(lds);                       // [64][kLd]
    float* const ps = reinterpret_cast<float*>(lds + kFp32);
    float* const ts = reinterpret_cast<float*>(lds + 2 * kFp32);
    float* const xs = reinterpret_cast<float*>(lds + 3 * kFp32);           // [4][16][17] inverses of the diagonal tiles
    float* const whole = reinterpret_cast<float*>(lds + kArea);            // [8][DP] decays of eight tokens
    float* const inv = whole + 8 * DP;                                     // [2][64]: factor of k, of q
    float* const diag = inv + 2 * kBlock;                                  // [64]
    float* const beta = diag + kBlock;                                     // [64]
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int block = (int)blockIdx.x / a.heads, h = (int)blockIdx.x % a.heads, b = blockIdx.y, grp = h / (a.heads / a.kv_heads);
    const int t0 = (first + block) * kBlock, n = min(kBlock, a.seq - t0);
    const int64_t row0 = (int64_t)b * a.seq + t0;
    const uint16_t* q = static_cast<const uint16_t*>(a.qkv) + row0 * a.ldq + grp * a.dp;
    const uint16_t* k = q + a.kv_heads * a.dp;
    uint8_t* const image = static_cast<uint8_t*>(a.image) + (((int64_t)b * a.heads + h) * blocks + block) * ((int64_t)Op::pieces(a.vp) * 1024);

    // this wave's tokens: decays, keys and queries of the lane's two channels
    const int r0 = wave * 8;
    const bool lane_live = lane * 2 < CH;
    f32x2 dec[NB][8], xk[NB][8], xq[NB][8], bias[NB];
    uint32_t kk[NB][8], qq[NB][8];
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        const int d = p * 128 + lane * 2;
        const bool in = lane_live && d < a.dp;
        bias[p] = in ? *reinterpret_cast<const f32x2*>(a.dt_bias + h * a.dp + d) : f32x2{0, 0};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int t = r0 + i;
            const bool live = in && t < n;
            dec[p][i] = live ? *reinterpret_cast<const f32x2*>(a.z + (row0 + t) * a.heads * a.dp + h * a.dp + d) : f32x2{0, 0};
            kk[p][i] = live ? *reinterpret_cast<const uint32_t*>(k + (int64_t)t * a.ldq + d) : 0;
            qq[p][i] = live ? *reinterpret_cast<const uint32_t*>(q + (int64_t)t * a.ldq + d) : 0;
        }
    }
    __builtin_amdgcn_sched_barrier(0);   // (under way while the norms' are awaited)
    // norms, eight lanes to a token, which also give q . k of the same token
    {
        const int t = tid >> 3, l = tid & 7;
        float sq = 0.0f, sk = 0.0f, qk = 0.0f;
        if (t < n)
            for (int c = l * 8; c < a.dp; c += 64) {
                float x[8], y[8];
                w8a8::unpack8(*reinterpret_cast<const u32x4*>(q + (int64_t)t * a.ldq + c), x);
                w8a8::unpack8(*reinterpret_cast<const u32x4*>(k + (int64_t)t * a.ldq + c), y);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sq = fmaf(x[e], x[e], sq);
                    sk = fmaf(y[e], y[e], sk);
                    qk = fmaf(x[e], y[e], qk);
                }
            }
#pragma unroll
        for (int off = 4; off; off >>= 1) {
            sq += __shfl_xor(sq, off, kWave);
            sk += __shfl_xor(sk, off, kWave);
            qk += __shfl_xor(qk, off, kWave);
        }
        if (l == 0) {
            const float fq = a.q_scale / sqrtf(sq + kUnitEps), fk = 1.0f / sqrtf(sk + kUnitEps);
            inv[t] = fk;
            inv[kBlock + t] = fq;
            diag[t] = qk * fq * fk;
            beta[t] = t < n ? sigmoid(Elem<uint16_t>::get(static_cast<const uint16_t*>(a.proj) + (row0 + t) * a.ld + a.b_off + h)) : 0.0f;
        }
    }
    {
        const float decay = -kLog2e * a.decay[h];
#pragma unroll
        for (int p = 0; p < NB; ++p) {
            const int d = p * 128 + lane * 2;
            const bool in = lane_live && d < a.dp;
            f32x2 all = {1.0f, 1.0f};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool live = in && r0 + i < n;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    dec[p][i][e] = live ? __builtin_amdgcn_exp2f(decay * softplus_fast(dec[p][i][e] + bias[p][e])) : 1.0f;
                    all[e] *= dec[p][i][e];
                }
                xk[p][i] = f32x2{__uint_as_float(kk[p][i] << 16), __uint_as_float(kk[p][i] & 0xffff0000u)};
                xq[p][i] = f32x2{__uint_as_float(qq[p][i] << 16), __uint_as_float(qq[p][i] & 0xffff0000u)};
            }
            if (lane_live) *reinterpret_cast<f32x2*>(whole + wave * DP + d) = all;
        }
    }
    __syncthreads();
    auto scale = [](f32x2 u, f32x2 v) { return f32x2{u[0] * v[0], u[1] * v[1]}; };
#pragma unroll
    for (int p = 0; p < NB; ++p)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float fk = inv[r0 + i], fq = inv[kBlock + r0 + i];
            xk[p][i] = scale(xk[p][i], f32x2{fk, fk});
            xq[p][i] = scale(xq[p][i], f32x2{fq, fq});
        }
    // decays of the waves (eights of tokens) from .. to - 1
    auto eights = [&](int p, int from, int to) {
        f32x2 w = {1.0f, 1.0f};
        for (int i = from; i < to; ++i) w = scale(w, *reinterpret_cast<const f32x2*>(whole + i * DP + p * 128 + lane * 2));
        return w;
    };
    // both terms of a pair, the low ones a matrix further
    auto put = [&](uint8_t* hi, int t, f32x2 v) {
        uint32_t h2, l2;
        split2(v[0], v[1], h2, l2);
        *reinterpret_cast<uint32_t*>(hi + t * kRow + lane * 4) = h2;
        *reinterpret_cast<uint32_t*>(hi + kMat + t * kRow + lane * 4) = l2;
    };
    uint8_t* const mk = lds;              // keys of a level: high, low terms; then its queries (upper tokens only)
    uint8_t* const mq = lds + 2 * kMat;
    const bool is_q = wave >= 4;          // waves 0 .. 3 form M, 4 .. 7 P
    const int w4 = wave & 3;
    f32x4 near = {0, 0, 0, 0}, mid = {0, 0, 0, 0}, far = {0, 0, 0, 0};   // pairs in a tile of 16, a block of 32, across
    // the product of token tiles i (upper) and j of the matrices in LDS
    auto pairs = [&](int i, int j, f32x4 acc) {
        const uint8_t* left = (is_q ? mq : mk) + (i * 16 + c16) * kRow + 16 * g;
        const uint8_t* right = mk + (j * 16 + c16) * kRow + 16 * g;
        f32x4 acc2 = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < CH / 32; ++s) {
            const u32x4 lh = *reinterpret_cast<const u32x4*>(left + s * 64), ll = *reinterpret_cast<const u32x4*>(left + kMat + s * 64);
            const u32x4 kh = *reinterpret_cast<const u32x4*>(right + s * 64), kl = *reinterpret_cast<const u32x4*>(right + kMat + s * 64);
            acc = mfma16(lh, kh, acc);
            acc2 = mfma16(lh, kl, acc2);
            acc2 = mfma16(ll, kh, acc2);
        }
        return acc + acc2;
    };
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        // blocks of 2 HB tokens: upper tokens take the decays from the middle on, lower ones those up to it
        auto level = [&](auto hb_tag) {
            constexpr int HB = decltype(hb_tag)::value;
            if (p || HB != 32) __syncthreads();   // the level before is no longer read
            if (lane_live) {
                if constexpr (HB >= 8) {
                    constexpr int E = HB / 8;   // eights
                    if (wave & E) {
                        f32x2 w = eights(p, wave & ~(E - 1), wave);
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            w = scale(w, dec[p][i]);
                            put(mk, r0 + i, scale(xk[p][i], w));
                            put(mq, r0 + i, scale(xq[p][i], w));
                        }
                    } else {
                        f32x2 w = eights(p, wave + 1, (wave & ~(E - 1)) + E);
#pragma unroll
                        for (int i = 7; i >= 0; --i) {
                            put(mk, r0 + i, scale(xk[p][i], w));
                            w = scale(w, dec[p][i]);
                        }
                    }
                } else {
#pragma unroll
                    for (int m = HB; m < 8; m += 2 * HB) {
                        f32x2 w = {1.0f, 1.0f};
#pragma unroll
                        for (int i = m; i < m + HB; ++i) {
                            w = scale(w, dec[p][i]);
                            put(mk, r0 + i, scale(xk[p][i], w));
                            put(mq, r0 + i, scale(xq[p][i], w));
                        }
                        w = f32x2{1.0f, 1.0f};
#pragma unroll
                        for (int i = m - 1; i >= m - HB; --i) {
                            put(mk, r0 + i, scale(xk[p][i], w));
                            w = scale(w, dec[p][i]);
                        }
                    }
                }
            }
            __syncthreads();
            if constexpr (HB == 32) {
                far = pairs(2 + (w4 >> 1), w4 & 1, far);
            } else if constexpr (HB == 16) {
                if (w4 < 2) mid = pairs(2 * w4 + 1, 2 * w4, mid);
            } else {
                const f32x4 v = pairs(w4, w4, f32x4{0, 0, 0, 0});
#pragma unroll
                for (int e = 0; e < 4; ++e) {   // the level of (t, j) is the highest bit of t ^ j
                    const int t = 4 * g + e, x = t ^ c16;
                    near[e] += t > c16 && x >= HB && x < 2 * HB ? v[e] : 0.0f;
                }
            }
        };
        level(std::integral_constant<int, 32>{});
        level(std::integral_constant<int, 16>{});
        level(std::integral_constant<int, 8>{});
        level(std::integral_constant<int, 4>{});
        level(std::integral_constant<int, 2>{});
        level(std::integral_constant<int, 1>{});
    }
    // the values, 128 columns of them, loaded before the first store: loads behind stores would wait for those
    const uint16_t* const values = static_cast<const uint16_t*>(a.qkv) + row0 * a.ldq + 2 * a.kv_heads * a.dp + h * a.vp;
    u32x4 vv[2];
    auto load_v = [&](int from) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = (tid >> 4) + 32 * u, col = from + (tid & 15) * 8;
            vv[u] = t < n && col < a.vp ? *reinterpret_cast<const u32x4*>(values + (int64_t)t * a.ldq + col) : u32x4{0, 0, 0, 0};
        }
    };
    load_v(0);
    __builtin_amdgcn_sched_barrier(0);
    // a matrix [channel][token] as fragments, two or three terms of it: this thread's two channels, its eight tokens
    auto stage = [&](uint8_t* to, int tile, const f32x2 (&v)[8], auto terms) {
        constexpr int N = decltype(terms)::value;
        if (!lane_live) return;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int ch = 2 * lane + e;
#pragma unroll
            for (int gg = 0; gg < 2; ++gg) {
                u32x2 hi, mid, lo;
                split4(f32x4{v[4 * gg][e], v[4 * gg + 1][e], v[4 * gg + 2][e], v[4 * gg + 3][e]}, hi, mid, lo);
                uint8_t* dst = to + (ch >> 4) * tile + (wave >> 2) * N * 1024 + (((wave & 1) * 2 + gg) * 16 + (ch & 15)) * 16 + ((wave >> 1) & 1) * 8;
                *reinterpret_cast<u32x2*>(dst) = hi;
                *reinterpret_cast<u32x2*>(dst + 1024) = mid;
                if constexpr (N == 3) *reinterpret_cast<u32x2*>(dst + 2048) = lo;
            }
        }
    };
    auto leave_fragment = [&](int at, u32x4 v) { *reinterpret_cast<u32x4*>(image + (int64_t)at * 1024 + lane * 16) = v; };
    // the operands that need no T leave here, so that their factors' registers are free for it
    constexpr int kLTile = 4 * 1024 + 16;
    uint8_t* const ls = lds + 2 * kMat;
    f32x2 gk[NB][8];
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        __syncthreads();
        if (lane_live) {
            f32x2 v[8], w = eights(p, wave + 1, 8);
#pragma unroll
            for (int i = 7; i >= 0; --i) {   // L_63 K
                v[i] = scale(xk[p][i], w);
                w = scale(w, dec[p][i]);
            }
            stage(ls, kLTile, v, std::integral_constant<int, 2>{});
            w = eights(p, 0, wave);
#pragma unroll
            for (int i = 0; i < 8; ++i) {   // G K, G Q
                w = scale(w, dec[p][i]);
                gk[p][i] = scale(xk[p][i], w);
                put(lds, r0 + i, scale(xq[p][i], w));
            }
            if (wave == 7) *reinterpret_cast<f32x2*>(image + (int64_t)Op::kG * 1024 + (p * 128 + lane * 2) * 4) = w;
        }
        __syncthreads();
        for (int i = wave; i < CH / 16 * 4; i += 8)
            leave_fragment(Op::kL + p * 32 + i, *reinterpret_cast<const u32x4*>(ls + (i >> 2) * kLTile + (i & 3) * 1024 + lane * 16));
        for (int f = wave; f < 4 * (CH / 32) * 2; f += 8) {
            const int hl = f & 1, s = (f >> 1) % (CH / 32), i = (f >> 1) / (CH / 32);
            const uint8_t* from = lds + hl * kMat + (16 * i + c16) * kRow + s * 64 + 8 * g;
            leave_fragment(Op::kQ + (i * NS + p * 4 + s) * 2 + hl, join(*reinterpret_cast<const u32x2*>(from), *reinterpret_cast<const u32x2*>(from + 32)));
        }
    }
    __syncthreads();
    {
        float* const dst = is_q ? ps : ms;
        auto leave = [&](int i, int j, f32x4 v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * i + 4 * g + e;
                dst[t * kLd + 16 * j + c16] = is_q ? v[e] : beta[t] * v[e];
            }
        };
        f32x4 d = near;
        if (is_q) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * g + e == c16) d[e] = diag[16 * w4 + c16];
        }
        leave(w4, w4, d);
        if (w4 < 2) {
            leave(2 * w4 + 1, 2 * w4, mid);
            leave(2 * w4, 2 * w4 + 1, f32x4{0, 0, 0, 0});
        }
        leave(2 + (w4 >> 1), w4 & 1, far);
    }
    __syncthreads();
    // fragments whose lanes hold rows 16 i + c16, columns 32 p + 4 g .. and 32 p + 16 + 4 g .. of an fp32 matrix
    auto fragment = [&](const float* m, int i, int p, u32x4& hi, u32x4& mid, u32x4& lo) {
        const float* row = m + (16 * i + c16) * kLd + 32 * p + 4 * g;
        u32x2 h0, m0, l0, h1, m1, l1;
        split4(*reinterpret_cast<const f32x4*>(row), h0, m0, l0);
        split4(*reinterpret_cast<const f32x4*>(row + 16), h1, m1, l1);
        hi = join(h0, h1);
        mid = join(m0, m1);
        lo = join(l0, l1);
    };
    if (!is_q) {
        // row c16 of X = (I + M)^-1 of a diagonal tile from X (I + M) = I, last column first
        const float* m0 = ms + (16 * w4) * kLd + 16 * w4;
        float y[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) y[j] = j == c16 ? 1.0f : 0.0f;
#pragma unroll
        for (int s = 15; s >= 1; --s) {
            float m[16];
#pragma unroll
            for (int j = 0; j < s; j += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(m0 + s * kLd + j);
#pragma unroll
                for (int e = 0; e < 4; ++e) m[j + e] = v[e];
            }
#pragma unroll
            for (int j = 0; j < s; ++j) y[j] = fmaf(-y[s], m[j], y[j]);
        }
        if (g == 0) {
#pragma unroll
            for (int j = 0; j < 16; ++j) xs[(w4 * 16 + c16) * 17 + j] = y[j];
        }
    } else {   // P's fragments: tile w4, steps 0 .. w4 / 2 (two of tiles 0 and 1, four of 2 and 3)
        const int at = Op::kP + (w4 < 2 ? 2 * w4 : 4 * (w4 - 1));
#pragma unroll
        for (int p = 0; p < 2; ++p)
            if (p <= w4 / 2) {
                u32x4 hi, mid, lo;
                fragment(ps, w4, p, hi, mid, lo);
                leave_fragment(at + 2 * p, hi);
                leave_fragment(at + 2 * p + 1, mid);
            }
    }
    __syncthreads();
    if (!is_q) {
        // block column w4 of the inverse: X_i = -X_ii (sum over k of M_ik X_k), fp32 throughout; a product's rows 4 g + e are
        // the next one's contraction index 4 g + e as they are
        f32x4 x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = f32x4{0, 0, 0, 0};
            if (i == w4) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][e] = xs[(16 * i + 4 * g + e) * 17 + c16];
            } else if (i > w4) {
                f32x4 z = {0, 0, 0, 0};
#pragma unroll
                for (int kk = 0; kk < i; ++kk) {
                    if (kk < w4) continue;
                    const f32x4 m = *reinterpret_cast<const f32x4*>(ms + (16 * i + c16) * kLd + 16 * kk + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) z = mfma_f32(m[e], x[kk][e], z);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i] = mfma_f32(xs[(16 * i + c16) * 17 + 4 * g + e], -z[e], x[i]);
            }
            const float f = beta[16 * w4 + c16];
#pragma unroll
            for (int e = 0; e < 4; ++e) ts[(16 * i + 4 * g + e) * kLd + 16 * w4 + c16] = i < w4 ? 0.0f : x[i][e] * f;
        }
    }
    __syncthreads();   // M and P are no longer read: their place takes values, then operands on their way out
    constexpr int kVRow = 128 * 2 + 16;
    static_assert(kBlock * kVRow <= kFp32);
    for (int from = 0; from < a.vp; from += 128) {   // V' = T V
        if (from) {
            load_v(from);
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(lds + ((tid >> 4) + 32 * u) * kVRow + (tid & 15) * 16) = vv[u];
        __syncthreads();
        if (from + wave * 16 < a.vp) {
            const uint8_t* const src = lds + (4 * g + (c16 >> 2)) * kVRow + wave * 32 + (c16 & 3) * 8;
            const u32x4 vf[2] = {join(lds_read_tr(src), lds_read_tr(src + 16 * kVRow)), join(lds_read_tr(src + 32 * kVRow), lds_read_tr(src + 48 * kVRow))};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f32x4 acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
#pragma unroll
                for (int p = 0; p <= i / 2; ++p) {
                    u32x4 th, tm, tl;
                    fragment(ts, i, p, th, tm, tl);
                    const u32x4 v = own_half(vf[p], 2 * p < i);
                    acc = mfma16(th, v, acc);
                    acc2 = mfma16(tm, v, acc2);
                    acc2 = mfma16(tl, v, acc2);
                }
                __builtin_amdgcn_sched_barrier(0);   // (one tile's terms at a time in registers)
                leave_fragment(Op::kV + (from / 16 + wave) * 4 + i, __builtin_bit_cast(u32x4, acc + acc2));
            }
        }
    }
    u32x4 th[2][2], tm[2][2], tl[2][2];   // this wave's two token tiles of T, 2 (wave % 2) ..
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int pp = 0; pp < 2; ++pp) fragment(ts, 2 * (wave & 1) + x, pp, th[x][pp], tm[x][pp], tl[x][pp]);
    __syncthreads();
    uint8_t* const staged = lds + kFp32;   // (behind the values)
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        if (p) __syncthreads();
        stage(staged, kTile, gk[p], std::integral_constant<int, 3>{});
        __syncthreads();
        // W^T = (G K)^T T^T: channels as rows, so that a lane's four are W's operand order already
        for (int s = wave >> 1; s < CH / 32; s += 4) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int ii = 2 * (wave & 1) + x;
                u32x2 hi[2], lo[2];
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const uint8_t* src = staged + (2 * s + half) * kTile + lane * 16;
                    f32x4 acc = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
#pragma unroll
                    for (int pp = 0; pp < 2; ++pp) {
                        if (pp > (wave & 1)) break;
                        u32x4 gh = *reinterpret_cast<const u32x4*>(src + pp * 3072), gm = *reinterpret_cast<const u32x4*>(src + pp * 3072 + 1024),
                              gl = *reinterpret_cast<const u32x4*>(src + pp * 3072 + 2048);
                        gh = own_half(gh, 2 * pp < ii);
                        gm = own_half(gm, 2 * pp < ii);
                        gl = own_half(gl, 2 * pp < ii);
                        acc = mfma16(gh, th[x][pp], acc);
                        acc2 = mfma16(gh, tm[x][pp], acc2);
                        acc2 = mfma16(gm, th[x][pp], acc2);
                        acc2 = mfma16(gm, tm[x][pp], acc2);
                        acc2 = mfma16(gh, tl[x][pp], acc2);
                        acc2 = mfma16(gl, th[x][pp], acc2);
                    }
                    split4(acc + acc2, hi[half], lo[half]);
                }
                const int at = Op::kW + (ii * NS + p * 4 + s) * 2;
                leave_fragment(at, join(hi[0], hi[1]));
                leave_fragment(at + 1, join(lo[0], lo[1]));
            }
        }
    }
}

// One workgroup per 16 value columns. Waves 0 .. 3 are the chain: wave w forms U of the block's tokens 16 w .. and owns the
// state's channels 32 s .., s = w, w + 4 .. Waves 4 .. 7, one to each SIMD too, form the outputs of the tokens 16 w .. beside
// them. The state and U change hands through LDS in operand order: a product's accumulators are the next one's right operand
// once split. Two barriers a block. What bounds it is the compute unit's load path, 124 KiB a block or 2000 cycles of the 2900
// that a block takes; so every operand register is refilled for the next block as soon as it has been multiplied (97 us for 64
// blocks with the loads in rows, whose issue the chain waited for, 82 now), and no branch lies between a load and its use: where
// paths meet, every load would be waited for. The column blocks of a head run on one XCD and find its operands in that L2, into
// which each touches its share of a block three ahead (84 us without).
template <int DP>
__global__ __launch_bounds__(512, 1) void delta_block_walk_kernel(DeltaArgs a, int blocks, int first) {
    using Op = Operands<DP>;
    constexpr int NS = Op::NS, NO = (NS + 3) / 4;    // steps of channels; of them a wave's own
    __shared__ u32x4 s_hi[NS][64], s_lo[NS][64], u_hi[2][64], u_lo[2][64], u_end[2][64];
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = all & 3;
    const int tiles = a.vp / 16, turn = (int)blockIdx.x / 8;
    const int bh = turn / tiles * 8 + (int)blockIdx.x % 8, vt = turn % tiles;
    if (bh >= a.batch * a.heads) return;
    const int b = bh / a.heads, h = bh % a.heads, v = vt * 16 + c16;
    const int64_t bytes = (int64_t)Op::pieces(a.vp) * 1024;
    const uint8_t* next = static_cast<const uint8_t*>(a.image) + (int64_t)bh * blocks * bytes;
    __amdgpu_buffer_rsrc_t r = w8a8::make_rsrc(next, (uint32_t)bytes);
    auto advance = [&](int c) {
        next += c + 1 < blocks ? bytes : 0;   // (past the end: the last one once more, for nothing)
        r = w8a8::make_rsrc(next, (uint32_t)bytes);
    };
    auto frag = [&](int i) { return w8a8::buf_load16(r, lane * 16, i * 1024); };
    if (all >= 4) {
        u32x4 q[NS][2], p[2][2];
        auto load_q = [&](int s) {
#pragma unroll
            for (int hl = 0; hl < 2; ++hl) q[s][hl] = frag(Op::kQ + (wave * NS + s) * 2 + hl);
        };
        auto load_p = [&](int pp) {   // (what P does not have: zeros, from past the operands' end)
            const int at = Op::kP + (wave < 2 ? 2 * wave : 4 * (wave - 1));
#pragma unroll
            for (int hl = 0; hl < 2; ++hl) p[pp][hl] = w8a8::buf_load16(r, pp <= wave / 2 ? lane * 16 : kOutOfRange, (at + 2 * pp + hl) * 1024);
        };
        const int ldo = a.heads * a.vp;
        uint16_t* out = static_cast<uint16_t*>(a.out) + ((int64_t)b * a.seq + (int64_t)first * kBlock) * ldo;
        const uint32_t out_lane = (uint32_t)((16 * wave + 4 * g) * ldo + h * a.vp + v) * 2;
#pragma unroll
        for (int s = 0; s < NS; ++s) load_q(s);
        load_p(0);
        load_p(1);
        // This column block's share of the lines of a later block's operands, touched so that the loads find them in the L2.
        const int lines = (int)(bytes / 128), share = (lines + tiles - 1) / tiles, mine = (tid & 255) < share ? vt * share + (tid & 255) : lines;
        const uint8_t* const image = next;
        auto touch = [&](int c) {
            const __amdgpu_buffer_rsrc_t rt = w8a8::make_rsrc(image + (int64_t)min(c, blocks - 1) * bytes, (uint32_t)bytes);
            return __builtin_amdgcn_raw_buffer_load_b32(rt, (uint32_t)mine * 128, 0, 0);
        };
        uint32_t seen = touch(1);
        asm volatile("" ::"v"(seen));
        seen = touch(2);
        __syncthreads();
        for (int c = 0; c < blocks; ++c) {
            advance(c);
            asm volatile("" ::"v"(seen));
            seen = touch(c + kAhead);
            u32x4 sh[NS], sl[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                sh[s] = s_hi[s][lane];
                sl[s] = s_lo[s][lane];
            }
            f32x4 o0 = {0, 0, 0, 0}, o1 = {0, 0, 0, 0}, o2 = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                o0 = mfma16(q[s][0], sh[s], o0);
                o1 = mfma16(q[s][1], sh[s], o1);
                o2 = mfma16(q[s][0], sl[s], o2);
                asm volatile("" : "+v"(o0), "+v"(o1), "+v"(o2));   // (here, and not further down)
                __builtin_amdgcn_sched_barrier(0);
                load_q(s);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();   // U is there, the state's operands have been read
            u32x4 uh[2], ul[2];
#pragma unroll
            for (int pp = 0; pp < 2; ++pp) {
                uh[pp] = own_half(u_hi[pp][lane], 2 * pp < wave);
                ul[pp] = own_half(u_lo[pp][lane], 2 * pp < wave);
                if (pp > wave / 2) uh[pp] = ul[pp] = u32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (int pp = 0; pp < 2; ++pp) {
                o0 = mfma16(p[pp][0], uh[pp], o0);
                o1 = mfma16(p[pp][1], uh[pp], o1);
                o2 = mfma16(p[pp][0], ul[pp], o2);
                load_p(pp);
            }
            const f32x4 o = o0 + (o1 + o2);
            const __amdgpu_buffer_rsrc_t ro = w8a8::make_rsrc(out, (uint32_t)(min(kBlock, a.seq - (first + c) * kBlock) * ldo) * 2);   // (ends at the last token)
#pragma unroll
            for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b16(w8a8::f32_to_bf16(o[e]), ro, out_lane + (uint32_t)(e * ldo) * 2, 0, 0);
            out += kBlock * ldo;
            __syncthreads();   // the state is there, U has been read
        }
        return;
    }
    float* state = a.state + ((int64_t)b * a.heads + h) * a.dp * a.vp + v;
    auto owns = [&](int o) { return NS % 4 == 0 || wave + 4 * o < NS; };
    f32x4 st[NO][2];   // rows 32 s + 16 i + 4 g + e, column v
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = 32 * (wave + 4 * o) + 16 * i + 4 * g + e;
                st[o][i][e] = d < a.dp ? state[(int64_t)d * a.vp] : 0.0f;
            }
    u32x4 w[NS][2], l[NO][2][2][2];
    f32x4 vp, decay[NO][2];
    auto load_w = [&](int s) {
#pragma unroll
        for (int hl = 0; hl < 2; ++hl) w[s][hl] = frag(Op::kW + (wave * NS + s) * 2 + hl);
    };
    auto load_v = [&]() { vp = __builtin_bit_cast(f32x4, frag(Op::kV + vt * 4 + wave)); };
    auto load_decay = [&]() {
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (owns(o)) decay[o][i] = __builtin_bit_cast(f32x4, w8a8::buf_load16(r, g * 16, Op::kG * 1024 + (2 * (wave + 4 * o) + i) * 64));
    };
    auto load_l = [&](int pp, int o) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int hl = 0; hl < 2; ++hl)
                if (owns(o)) l[o][i][pp][hl] = frag(Op::kL + ((2 * (wave + 4 * o) + i) * 2 + pp) * 2 + hl);
    };
    auto give_state = [&]() {
#pragma unroll
        for (int o = 0; o < NO; ++o)
            if (owns(o)) {
                u32x2 h0, l0, h1, l1;
                split4(st[o][0], h0, l0);
                split4(st[o][1], h1, l1);
                s_hi[wave + 4 * o][lane] = join(h0, h1);
                s_lo[wave + 4 * o][lane] = join(l0, l1);
            }
    };
    // (in the order in which they are waited for)
#pragma unroll
    for (int s = 0; s < NS; ++s) load_w(s);
    load_v();
    load_decay();
#pragma unroll
    for (int pp = 0; pp < 2; ++pp)
#pragma unroll
        for (int o = 0; o < NO; ++o) load_l(pp, o);
    give_state();
    __syncthreads();
    for (int c = 0; c < blocks; ++c) {
        advance(c);
        u32x4 sh[NS], sl[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            sh[s] = s_hi[s][lane];
            sl[s] = s_lo[s][lane];
        }
        f32x4 y0 = {0, 0, 0, 0}, y1 = {0, 0, 0, 0}, y2 = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y0 = mfma16(w[s][0], sh[s], y0);
            y1 = mfma16(w[s][1], sh[s], y1);
            y2 = mfma16(w[s][0], sl[s], y2);
            y1 = mfma16(w[s][1], sl[s], y1);
            __builtin_amdgcn_sched_barrier(0);
            load_w(s);
            __builtin_amdgcn_sched_barrier(0);
        }
        {
            const f32x4 u = vp - (y0 + (y1 + y2));
            u32x2 hi, lo, end;
            split4(u, hi, lo, end);
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint8_t*>(&u_end[wave >> 1][lane]) + (wave & 1) * 8) = end;
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint8_t*>(&u_hi[wave >> 1][lane]) + (wave & 1) * 8) = hi;
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint8_t*>(&u_lo[wave >> 1][lane]) + (wave & 1) * 8) = lo;
        }
        load_v();
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) st[o][i] *= decay[o][i];
        load_decay();
        __syncthreads();   // U is there, the state's operands have been read
        u32x4 uh[2], ul[2], ue[2];
#pragma unroll
        for (int pp = 0; pp < 2; ++pp) {
            uh[pp] = u_hi[pp][lane];
            ul[pp] = u_lo[pp][lane];
            ue[pp] = u_end[pp][lane];
        }
#pragma unroll
        for (int pp = 0; pp < 2; ++pp)
#pragma unroll
            for (int o = 0; o < NO; ++o)
                if (owns(o)) {
#pragma unroll
                    for (int t = 0; t < 5; ++t)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            st[o][i] = mfma16(l[o][i][pp][t == 1 || t == 4], t == 3 ? ue[pp] : t == 2 || t == 4 ? ul[pp] : uh[pp], st[o][i]);
                    __builtin_amdgcn_sched_barrier(0);
                    load_l(pp, o);
                    __builtin_amdgcn_sched_barrier(0);
                }
        give_state();
        __syncthreads();   // the state is there, U has been read
    }
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = 32 * (wave + 4 * o) + 16 * i + 4 * g + e;
                if (d < a.dp) state[(int64_t)d * a.vp] = st[o][i][e];
            }
}

int64_t pieces_of(int dp, int vp) {
    return dp <= 32 ? Operands<32>::pieces(vp) : dp <= 64 ? Operands<64>::pieces(vp) : dp <= 128 ? Operands<128>::pieces(vp) : Operands<256>::pieces(vp);
}

// Blocks that are prepared and walked at a time. Operands take 141 KiB a block and head of 128 where chunks of 16 take 108 for as
// many tokens; prompts whose operands are more than this go in equal parts, from whose states each next one starts, so that they
// need less than they would in chunks (16 heads of 128, 1 x 32768 tokens: 376 MiB, 864 in chunks), others 120 MiB more at most.
constexpr int64_t kImageMost = (int64_t)512 << 20;
int64_t blocks_at_a_time(int64_t heads, int64_t seq, int dp, int vp) {
    const int64_t blocks = (seq + kBlock - 1) / kBlock, bytes = heads * blocks * pieces_of(dp, vp) * 1024;
    const int64_t parts = std::min((bytes + kImageMost - 1) / kImageMost, blocks);
    return parts > 1 ? (blocks + parts - 1) / parts : blocks;
}

template <int DP>
void blocks_t(const DeltaArgs& a, hipStream_t stream) {
    constexpr int CH = DP < 128 ? DP : 128, mat = 4 * kBlock * (CH * 2 + 16), fp32 = 3 * kBlock * (kBlock + 4) * 4 + 4 * 1088;
    constexpr int shared = (mat > fp32 ? mat : fp32) + (8 * DP + 4 * kBlock) * 4;
    static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_block_prep_kernel<DP>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, shared);
    (void)once;
    const int all = (a.seq + kBlock - 1) / kBlock, groups = (a.batch * a.heads + 7) / 8;
    const int most = (int)blocks_at_a_time((int64_t)a.batch * a.heads, a.seq, a.dp, a.vp);
    for (int first = 0; first < all; first += most) {
        const int blocks = std::min(most, all - first);
        delta_block_prep_kernel<DP><<<dim3((unsigned)blocks * (unsigned)a.heads, (unsigned)a.batch), kPrepThreads, shared, stream>>>(a, blocks, first);
        delta_block_walk_kernel<DP><<<(unsigned)(groups * 8 * (a.vp / 16)), 512, 0, stream>>>(a, blocks, first);
    }
}

}  // namespace

int64_t delta_blocks_bytes(int64_t batch, int64_t heads, int64_t seq, int dp, int vp) {
    return batch * heads * blocks_at_a_time(batch * heads, seq, dp, vp) * pieces_of(dp, vp) * 1024;
}

// (a dimension of a launch holds fewer than 2^32 threads, a descriptor 2^32 bytes: 64 rows of out, a block's operands)
bool delta_blocks_supported(int64_t batch, int64_t heads, int64_t seq, int dp, int vp) {
    constexpr int64_t most = ((int64_t)1 << 32) - 1;
    return delta_chunk_supported(dp, vp) && heads * vp * kBlock * 2 <= most && pieces_of(dp, vp) * 1024 <= most &&
           (batch * heads + 7) / 8 * 8 * (vp / 16) * 512 <= most && blocks_at_a_time(batch * heads, seq, dp, vp) * heads * kPrepThreads <= most;
}

void launch_delta_blocks(const DeltaArgs& a, hipStream_t stream) {
    if (a.dp <= 32) blocks_t<32>(a, stream);
    else if (a.dp <= 64) blocks_t<64>(a, stream);
    else if (a.dp <= 128) blocks_t<128>(a, stream);
    else blocks_t<256>(a, stream);
}

}  // namespace astrai_mix
