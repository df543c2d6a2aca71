// y = x W^T for the few tokens of a decode step (up to 64 rows), bf16 operands, fp32 sums: bound by the
// stream of the weights, which are read exactly once with the streaming cache hint. Three epilogues: bf16 with
// a bias, fp32 (what leaves the accumulators), and act(gate) * up of a weight that holds the rows of gate, then
// those of up, so that the pair of products never reaches memory.
//
// The weight rows are dealt out in equal contiguous ranges over about one workgroup per compute unit; the
// waves of a workgroup split K into contiguous slices of 256-byte items (128 values) and keep all tokens and
// row groups of their slice, so a workgroup reads x once. Every load moves 4 rows x 256 contiguous bytes; an
// item of 16 rows is turned into MFMA operand order (lane = row, 16 bytes of K) through a wave-private LDS
// patch whose XOR chunk swizzle keeps the row-major writes and the operand reads free of conflicts. Weights
// and x take the same route, so any order of K inside an item is the same for both. Each unit's registers are
// refilled for the next item as soon as it has been consumed: the bytes in flight stay the same from the first
// instruction to the last, when nothing is left to request. The waves' partial sums are added through LDS in wave order.
//
// Several ranges of K by workgroups of their own (splits) make the row ranges longer and the part of x that a workgroup reads
// shorter: x is most of the bytes that a workgroup pulls out of L2 where the weights have few rows. The fp32 sums of the
// ranges lie in planes that the row norm behind the product adds up. With that norm (us, one range / four): 64 rows of 5632 ->
// 2048 18.7 / 12.4, 2048 -> 2048 10.9 / 9.0; 32 rows 13.8 / 11.0, 8.7 / 7.9; 16 rows 11.7 / 9.9, 8.1 / 7.2; 1 row 9.9 / 9.6, 7.3 / 6.8.
//
// What bounds it (graph replays over weights that no cache holds): the stream from 20 MB on (2048 -> 32000, 131 MB, 22.5 us at 1
// token, 5.8 TB/s), below it launch and the load path's 16 cycles for every 1 KiB instruction, of x as much as of the
// weights: leaving out those for rows and tokens that are not there and those past the last item took 2048 -> 2048 from 4.3
// to 3.8 us (1 token) and 5.6 to 5.3 (32), 2048 -> 6656 from 7.6 to 6.8 and 8.4 to 8.2, gate|up of 5632 9.85 -> 9.6 and 11.3 -> 11.0.
#include <type_traits>

#include "mix_common.cuh"
#include "mix_launchers.h"

namespace astrai_mix {

namespace {

constexpr int kItem = 256;  // bytes of K per item
constexpr int kMaxGroups = 3;

template <int ACT>
__device__ __forceinline__ float act_of(float z) {
    return ACT == kActGelu ? gelu_as<uint16_t>(z) : silu_fast(z);
}

__device__ __forceinline__ void to_operand_order(uint8_t* patch, int lane, const u32x4 (&in)[4], u32x4 (&out)[4]) {
    const int c16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = i * 4 + g;
        *reinterpret_cast<u32x4*>(patch + row * 256 + ((c16 ^ row) << 4)) = in[i];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = *reinterpret_cast<const u32x4*>(patch + c16 * 256 + (((4 * j + g) ^ c16) << 4));
}

// RG: groups of 16 weight rows per workgroup (ACT >= 0: of gate and of up each); MB: groups of 16 tokens;
// NW: waves. ACT: -1 none. IB: items under way (two where a wave's eight rows leave too few bytes in flight). WH, XH: of the last group of weight rows / of tokens at most 8 are there.
template <int RG, int MB, int NW, int ACT, bool F32, bool WH, bool XH, int IB>
__global__ __launch_bounds__(NW * 64) void few_rows_linear_kernel(FewRowsArgs a, int rows_per_wg) {
    constexpr int HALVES = ACT >= 0 ? 2 : 1;
    constexpr int WG = RG * HALVES;              // weight units per item
    constexpr int P = MB + WG;
    constexpr int PATCH = 8192, RED = WG * MB * 1024;
    constexpr int WAVE_LDS = PATCH > RED ? PATCH : RED;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int items = a.k / (kItem / 2);
    const int part = blockIdx.y * NW + wave, parts = gridDim.y * NW;   // (blockIdx.y: a range of K whose sums stand by themselves)
    const int i0 = part * items / parts, i1 = (part + 1) * items / parts;
    const int r0 = blockIdx.x * rows_per_wg, r1 = min(r0 + rows_per_wg, a.n);
    const uint32_t w_row = (uint32_t)a.k * 2, x_row = (uint32_t)a.ldx * 2;
    const __amdgpu_buffer_rsrc_t rw = w8a8::make_rsrc(a.w, (uint32_t)(HALVES * a.n) * w_row);
    const __amdgpu_buffer_rsrc_t rx = w8a8::make_rsrc(a.x, (uint32_t)(a.m - 1) * x_row + w_row);

    f32x4 acc[WG][MB];
#pragma unroll
    for (int r = 0; r < WG; ++r)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[r][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    uint8_t* const wpatch = smem + wave * WAVE_LDS;
    uint8_t* const xpatch = wpatch + 4096;
    u32x4 ring[IB][P][4] = {};
    // (a load past every row costs the unit's one load path its 16 cycles as any other: left out)
    auto loads_of = [](int s) { return s < MB ? (XH && s == MB - 1 ? 2 : 4) : (WH && (s - MB) % RG == RG - 1 ? 2 : 4); };
    auto issue = [&](u32x4 (&dst)[4], int item, int s) {
        const uint32_t k0 = (uint32_t)item * kItem;
        if (s < MB) {
#pragma unroll
            for (int i = 0; i < loads_of(s); ++i)  // tokens past m lie past the descriptor: zeros
                dst[i] = w8a8::buf_load16(rx, (uint32_t)(s * 16 + i * 4 + g) * x_row + (uint32_t)c16 * 16, k0);
        } else {
            const int u = s - MB, half = u / RG;
#pragma unroll
            for (int i = 0; i < loads_of(s); ++i) {
                const int row = r0 + (u - half * RG) * 16 + i * 4 + g;
                dst[i] = __builtin_amdgcn_raw_buffer_load_b128(
                    rw, row < r1 ? (uint32_t)(half * a.n + row) * w_row + (uint32_t)c16 * 16 : w8a8::kOutOfRange,
                    k0, 2);  // 2: not kept once delivered
            }
        }
    };
    // an item; NEXT: the item that many further on is requested into its registers, a unit at a time
    auto consume = [&](u32x4 (&units)[P][4], auto next_tag, int item) {
        constexpr int NEXT = decltype(next_tag)::value;
        u32x4 xf[MB][4];
#pragma unroll
        for (int s = 0; s < P; ++s) {
            if (s < MB) {
                to_operand_order(xpatch, lane, units[s], xf[s < MB ? s : 0]);
            } else {
                u32x4 wf[4];
                to_operand_order(wpatch, lane, units[s], wf);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int b = 0; b < MB; ++b) acc[s < MB ? 0 : s - MB][b] = mfma16(wf[j], xf[b][j], acc[s < MB ? 0 : s - MB][b]);
            }
            if constexpr (NEXT > 0) issue(units[s], item + NEXT, s);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto request = [&](u32x4 (&units)[P][4], int item) {
#pragma unroll
        for (int s = 0; s < P; ++s) issue(units[s], item, s);
    };
    constexpr std::integral_constant<int, 0> none{};
    constexpr std::integral_constant<int, IB> next{};
    if (i0 < i1) {
        int item = i0;
        request(ring[0], item);
        if constexpr (IB == 1) {
            for (; item + 1 < i1; ++item) consume(ring[0], next, item);
            consume(ring[0], none, item);
        } else if (i1 - i0 == 1) {
            consume(ring[0], none, item);
        } else {
            request(ring[1], item + 1);
            for (; item + 3 < i1; item += 2) {
                consume(ring[0], next, item);
                consume(ring[1], next, item + 1);
            }
            if (item + 2 < i1) {
                consume(ring[0], next, item);
                consume(ring[1], none, item + 1);
                consume(ring[0], none, item + 2);
            } else {
                consume(ring[0], none, item);
                consume(ring[1], none, item + 1);
            }
        }
    }

    __syncthreads();  // the patches are free
    f32x4* const red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int r = 0; r < WG; ++r)
#pragma unroll
        for (int b = 0; b < MB; ++b) red[wave * (WAVE_LDS / 16) + (r * MB + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    auto total = [&](int unit) {
        f32x4 s = red[unit * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += red[w * (WAVE_LDS / 16) + unit * 64 + lane];
        return s;
    };
#pragma unroll
    for (int t = wave; t < RG * MB; t += NW) {
        const int m = (t % MB) * 16 + c16, row = r0 + (t / MB) * 16 + g * 4;
        if (m >= a.m || row >= r1) continue;
        f32x4 v = total(t);
        const int64_t at = ((int64_t)blockIdx.y * a.m + m) * a.n + row;
        if constexpr (ACT >= 0) {
            const f32x4 up = total(t + RG * MB);
#pragma unroll
            for (int e = 0; e < 4; ++e) {  // both factors as the products' own bf16 output would hold them
                const float gate = w8a8::bf16_to_f32(f32_to_bf16(v[e]));
                v[e] = act_of<ACT>(gate) * w8a8::bf16_to_f32(f32_to_bf16(up[e]));
            }
        } else if (a.bias) {
            v += Elem<uint16_t>::get4(static_cast<const uint16_t*>(a.bias) + row);
        }
        if constexpr (F32) Elem<float>::put4(static_cast<float*>(a.out) + at, v);
        else Elem<uint16_t>::put4(static_cast<uint16_t*>(a.out) + at, v);
    }
}

template <int RG, int MB, int NW, int ACT, bool F32, bool WH, bool XH, int IB = 1>
void launch_inst(const FewRowsArgs& a, int rows, hipStream_t stream) {
    constexpr int units = RG * (ACT >= 0 ? 2 : 1) * MB * 1024;
    constexpr int lds = NW * (units > 8192 ? units : 8192);
    static_assert(lds <= 64 * 1024, "within the limit that needs no attribute");
    few_rows_linear_kernel<RG, MB, NW, ACT, F32, WH, XH, IB>
        <<<dim3((unsigned)((a.n + rows - 1) / rows), (unsigned)a.splits), dim3(NW * 64), lds, stream>>>(a, rows);
}

template <int RG, int NW, int ACT, bool F32, bool WH>
void launch_mb(const FewRowsArgs& a, int rows, hipStream_t stream) {
    if constexpr (RG == 1 && NW == 8 && ACT < 0) {
        // Up to 8 tokens x costs little, and two items under way feed the stream (5632 -> 2048, 1 token 8.0 -> 6.6 us, 8 tokens
        // 8.0 -> 7.2), if a wave has more than two in all (2048 -> 2048 3.8 -> 3.9). 16 tokens and more are bound by x.
        if (a.m <= 8 && a.k >= 4096) return launch_inst<RG, 1, NW, ACT, F32, WH, true, 2>(a, rows, stream);
    }
    if (a.m <= 8) launch_inst<RG, 1, NW, ACT, F32, WH, true>(a, rows, stream);
    else if (a.m <= 16) launch_inst<RG, 1, NW, ACT, F32, WH, false>(a, rows, stream);
    else if (a.m <= 32) launch_inst<RG, 2, NW, ACT, F32, WH, false>(a, rows, stream);
    else launch_inst<RG, 4, NW, ACT, F32, WH, false>(a, rows, stream);
}

template <int RG, int NW, int ACT, bool F32>
void launch_wh(const FewRowsArgs& a, int rows, hipStream_t stream) {
    if (rows <= RG * 16 - 8) launch_mb<RG, NW, ACT, F32, true>(a, rows, stream);
    else launch_mb<RG, NW, ACT, F32, false>(a, rows, stream);
}

template <int ACT, bool F32>
void launch_rg(const FewRowsArgs& a, hipStream_t stream) {
    // rows dealt out over 256 workgroups (a multiple of them where a range would be over GROUPS * 16 rows),
    // in fours: one load instruction
    constexpr int GROUPS = ACT >= 0 ? 2 : kMaxGroups;
    const int round = 256 / a.splits, wgs = round * ((a.n + round * GROUPS * 16 - 1) / (round * GROUPS * 16));
    const int rows = ((a.n + wgs - 1) / wgs + 3) & ~3;
    if (rows > 32) {
        if constexpr (GROUPS == 3) launch_wh<3, 4, ACT, F32>(a, rows, stream);
    } else if (rows > 16) {
        launch_wh<2, 4, ACT, F32>(a, rows, stream);
    } else if (a.k >= 1024) {
        launch_wh<1, 8, ACT, F32>(a, rows, stream);
    } else {
        launch_wh<1, 4, ACT, F32>(a, rows, stream);
    }
}

}  // namespace

bool few_rows_linear_supported(int64_t m, int64_t n, int64_t k, bool act) {
    return m > 0 && m <= kFewRowsMax && n > 0 && n % 4 == 0 && k > 0 && k % (kItem / 2) == 0 &&
           n * k * (act ? 4 : 2) < ((int64_t)1 << 31);
}

bool launch_few_rows_linear(const FewRowsArgs& a, int act, bool out_float, hipStream_t stream) {
    if (!few_rows_linear_supported(a.m, a.n, a.k, act >= 0) || a.ldx < a.k || a.ldx % 8 ||
        (int64_t)kFewRowsMax * a.ldx * 2 >= ((int64_t)1 << 31))
        return false;
    if (a.splits != 1 && (a.splits < 1 || a.splits > kMaxParts || act >= 0 || !out_float || a.bias)) return false;
    if (act == kActGelu) launch_rg<kActGelu, false>(a, stream);
    else if (act == kActSilu) launch_rg<kActSilu, false>(a, stream);
    else if (out_float) launch_rg<-1, true>(a, stream);
    else launch_rg<-1, false>(a, stream);
    return true;
}

}  // namespace astrai_mix
