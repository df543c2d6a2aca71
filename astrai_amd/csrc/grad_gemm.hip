// The two products of a Linear's backward on bf16 tensors as they lie in memory: grad_x = g W (g [m, n], W [n, k]) and
// grad_w = g^T x (x [m, k]), fp32 sums, rounded once. W, x and, in grad_w, g hold the contraction in their rows, so
// their tiles arrive row by row and are turned on their way out of LDS (ds_read_b64_tr_b16), not by a pass over memory.
//
// 128 x 128 output tiles, four waves of 64 x 64 on 16x16x32 MFMAs, slabs of 64 values of the contraction through a ring of S
// LDS stages of 32 KiB filled by direct-to-LDS loads; a wave reads the fragments of slab k + 1 into a second register set
// between the MFMAs of slab k, and one barrier a slab publishes slab k + 1 and frees slab k's stage (the scheme of
// gemm_mid128.cuh). Rows past the contraction's end, and past the output's in g's own order, read as zeros; columns
// past the output's are never stored.
//
// What bounds it: with one workgroup to a compute unit the instructions that a wave issues beside its 32 MFMAs of 16 cycles a slab
// (24 LDS reads, 8 loads): addresses that are constants away and scalar load offsets took 66 vector instructions out of a slab,
// 1140 cycles -> 850; with two the power limit (4096^3: matrix pipe busy 69% at 1.6 GHz, LDS 37%). Tiles of 256 x 128 (one wave a
// SIMD, 64 MFMAs a barrier) were slower at every size (4096^3 142 us against 119).
// Measured against the vendor library's products and torch's column sums (us, both with the chip to themselves): grad_w and
// grad_bias 552 x 11264 x 2048 35 / 60 + 16, 1500 x 3072 x 2048 24 / 37 + 17, 2500 x 11008 x 4096 215 / 278 + 121, 700 x 2048 x 2048 11 / 18 + 11;
// grad_x 552 x 11264 x 2048 40 / 91, 1000 x 11008 x 4096 80 / 105, 700 x 2048 x 2048 15 / 22.
#include <type_traits>
#include <utility>

#include "gemm_tile.cuh"
#include "lds_dma.cuh"

namespace w8a8 {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 128, kSlab = 64;
constexpr int kOperand = kTile * kSlab * 2, kStage = 2 * kOperand;   // bytes
constexpr int kLoads = 8;                                            // of a wave and slab
constexpr int kRowB = 144;                                           // a row of the epilogue's 64 columns in LDS
constexpr uint32_t kPast = 0x80000000u;                              // an offset past any operand

template <int N>
__device__ __forceinline__ void wait_loads() {   // all but the N youngest
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_reads() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
}
__device__ __forceinline__ void meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// f(0), f(1), .. f(N - 1), each with its number as a type
template <class F, int... I>
__device__ __forceinline__ void repeat_(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void repeat(F&& f) {
    repeat_(f, std::make_integer_sequence<int, N>{});
}

// out [p, q] = sum over t of A(p, t) B(t, q). B is stored [t, q]; A [p, t] (ROWS) or [t, p].
// SUMS (not ROWS): tiles of the first columns also leave A's sums over t, on MFMAs against ones.
template <bool ROWS, bool SUMS, int S>
__global__ __launch_bounds__(256, 2) void grad_gemm_kernel(GradGemmArgs g) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_p = wave & 1, wave_q = wave >> 1;
    const int l16 = lane & 15, grp = lane >> 4;

    const TileCoord tc = map_tile<8>((g.p + kTile - 1) / kTile, (g.q + kTile - 1) / kTile);
    const int p0 = tc.tm * kTile, q0 = tc.tn * kTile;
    const int slabs = (g.t + kSlab - 1) / kSlab;
    const int first = (int)blockIdx.y * g.slabs_per_split, last = min(first + g.slabs_per_split, slabs);

    // The value of the contraction that a lane's fragment begins with, of a slab's half ks: 8 (4 ks + grp) where both operands
    // are turned, 8 (2 grp + ks) beside an A in its own order, whose 16-byte reads are free of bank conflicts that way.
    constexpr int GRP = ROWS ? 16 : 8, KS = ROWS ? 8 : 32;

    // ---- loads. An operand with the contraction in its rows: 64 rows of 256 bytes, sixteen 16-byte chunks, chunk c of row t at
    // position c ^ (4 (t & 3) + 2 (t / GRP & 1)): the eight rows that 32 lanes of a turning read touch lie in banks of their
    // own. Wave w fetches rows 16w .. 16w + 15, four an instruction. A in its own order: 128 rows of 128 bytes, as in
    // gemm_mid128.cuh; wave w fetches rows 32w .. 32w + 31, eight an instruction.
    const u32x4 da = make_desc(g.a, (uint32_t)g.p * (uint32_t)g.t * 2u), db = make_desc(g.b, (uint32_t)g.t * (uint32_t)g.q * 2u);
    uint32_t a_off[4], b_off[4];
    auto by_rows = [&](int r, int width, int col) -> uint32_t {
        const int row = wave * 16 + 4 * r + grp, chunk = l16 ^ (4 * grp + 2 * ((wave * 16 + 4 * r) / GRP & 1));
        return (uint32_t)row * (uint32_t)width * 2u + (uint32_t)col * 2u + (uint32_t)chunk * 16u;
    };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        b_off[r] = by_rows(r, g.q, q0);
        if constexpr (ROWS) {
            const int row = p0 + wave * 32 + 8 * r + (lane >> 3), chunk = (lane & 7) ^ (lane >> 3) ^ (r & 1);
            a_off[r] = (uint32_t)row * (uint32_t)g.t * 2u + (uint32_t)chunk * 16u;
        } else {
            a_off[r] = by_rows(r, g.p, p0);
        }
    }
    const uint32_t a_step = ROWS ? kSlab * 2 : (uint32_t)(kSlab * 2) * (uint32_t)g.p, b_step = (uint32_t)(kSlab * 2) * (uint32_t)g.q;
    const uint32_t lds_wave = lds0 + (uint32_t)wave * 4096u;
    uint32_t a_at = 0, b_at = 0;   // of the slab that is loaded
    auto load_slab = [&](int slab) __attribute__((always_inline)) {   // past the last one: no traffic
        a_at = slab < last ? (uint32_t)slab * a_step : kPast;
        b_at = slab < last ? (uint32_t)slab * b_step : kPast;
    };
    auto issue = [&](auto stage, auto load) __attribute__((always_inline)) {
        constexpr int L = decltype(load)::value, R = L >> 1, AT = decltype(stage)::value * kStage + R * 1024;
        if constexpr (L & 1) lds_dma16_at<AT + kOperand>(db, lds_wave, b_off[R], b_at);
        else lds_dma16_at<AT>(da, lds_wave, a_off[R], a_at);
    };

    // ---- fragments: lane (l16, grp) holds row or column l16 of a 16-wide sub-tile. Addresses that the compiler does not take
    // apart: stages, halves and rows of sub-tiles are constants away (a ds offset reaches two stages).
    uint32_t a_rd[4], b_rd[4];
    {
        const uint32_t turned = (uint32_t)(GRP * grp + (l16 >> 2)) * 256u +
                                (uint32_t)((((l16 & 3) >> 1) ^ (4 * (l16 >> 2) + 2 * (grp & 1))) << 4) + (uint32_t)((l16 & 1) << 3);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            b_rd[i] = lds0 + kOperand + (turned ^ (uint32_t)((wave_q * 4 + i) << 5));
            a_rd[i] = lds0 + (turned ^ (uint32_t)((wave_p * 4 + i) << 5));
            if constexpr (ROWS)   // [half of the slab]
                a_rd[i] = lds0 + (uint32_t)(wave_p * 8192 + l16 * 128 + (((2 * grp + (i & 1)) ^ (l16 & 7) ^ (l16 >> 3)) << 4));
            __asm__("" : "+v"(a_rd[i]), "+v"(b_rd[i]));
        }
    }
    uint32_t far_a[S > 2 ? 4 : 1], far_b[S > 2 ? 4 : 1];   // of stages 2 and 3
    if constexpr (S > 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            far_a[i] = a_rd[i] + 2 * kStage, far_b[i] = b_rd[i] + 2 * kStage;
            __asm__("" : "+v"(far_a[i]), "+v"(far_b[i]));
        }
    }
    struct Fragments {
        u32x4 a[2][4], b[2][4];   // [half of the slab][sub-tile]
    };
    auto read_turned = [&](uint32_t at) __attribute__((always_inline)) -> u32x4 {
        typedef __attribute__((address_space(3))) i16x4* Lds;
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)at));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(at + 4 * 256)));
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    auto read = [&](auto stage, auto fragment, Fragments& to) __attribute__((always_inline)) {   // in the order of their use
        constexpr int ST = decltype(stage)::value, F = decltype(fragment)::value, ks = F >> 3, i = (F >> 1) & 3;
        constexpr uint32_t at = (ST & 1) * kStage;
        const uint32_t(&ra)[4] = ST < 2 ? a_rd : reinterpret_cast<const uint32_t(&)[4]>(far_a);
        const uint32_t(&rb)[4] = ST < 2 ? b_rd : reinterpret_cast<const uint32_t(&)[4]>(far_b);
        if constexpr (F & 1) to.b[ks][i] = read_turned(rb[i] + at + ks * KS * 256);
        else if constexpr (ROWS) to.a[ks][i] = *(__attribute__((address_space(3))) u32x4*)(ra[ks] + at + i * 2048);
        else to.a[ks][i] = read_turned(ra[i] + at + ks * KS * 256);
    };

    f32x4 acc[4][4];   // [p sub-tile][q sub-tile]
    [[maybe_unused]] f32x4 sums[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        sums[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const bool sums_here = SUMS && tc.tn == 0 && wave_q == 0;
    Fragments even, odd;

    // slab k, of stage k % S, on `now`; the fragments of slab k + 1 into `next`
    auto slab = [&](auto stage, int k, const Fragments& now, Fragments& next) __attribute__((always_inline)) {
        constexpr int ST = decltype(stage)::value;
        constexpr std::integral_constant<int, (ST + 1) % S> after{};
        wait_reads();
        wait_loads<kLoads * (S - 2)>();   // slab k + 1 has landed
        meet();                           // for every wave, and every wave has read slab k: its stage is free
        load_slab(first + k + S);
        // 32 MFMAs; behind the first 16 the next fragments, behind every fourth a load of slab k + S
        repeat<32>([&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value, ks = n >> 4, i = (n >> 2) & 3, j = n & 3;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, now.b[ks][j]), __builtin_bit_cast(bf16x8, now.a[ks][i]),
                                                                acc[i][j], 0, 0, 0);
            if constexpr (n < 24 && n % 3 != 2) read(after, std::integral_constant<int, n / 3 * 2 + n % 3>{}, next);
            if constexpr (n % 4 == 2) issue(stage, std::integral_constant<int, n / 4>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        if (SUMS && sums_here) {
            const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
#pragma unroll
            for (int n = 0; n < 8; ++n)
                sums[n & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones),
                                                                      __builtin_bit_cast(bf16x8, now.a[n >> 2][n & 3]), sums[n & 3], 0, 0, 0);
        }
    };

    constexpr std::integral_constant<int, 0> s0{};
    constexpr std::integral_constant<int, 1> s1{};
    constexpr std::integral_constant<int, S - 2> s2{};
    constexpr std::integral_constant<int, S - 1> s3{};
    repeat<S>([&](auto t) __attribute__((always_inline)) {
        load_slab(first + decltype(t)::value);
        repeat<kLoads>([&](auto l) __attribute__((always_inline)) { issue(t, l); });
    });
    wait_loads<kLoads * (S - 1)>();
    meet();
    repeat<16>([&](auto f) __attribute__((always_inline)) { read(s0, f, even); });
    const int count = last - first;
    int k = 0;
    for (; k + S <= count; k += S) {
        slab(s0, k, even, odd);
        slab(s1, k + 1, odd, even);
        if constexpr (S == 4) {
            slab(s2, k + 2, even, odd);
            slab(s3, k + 3, odd, even);
        }
    }
    if (k < count) slab(s0, k, even, odd);
    if constexpr (S == 4) {
        if (k + 1 < count) slab(s1, k + 1, odd, even);
        if (k + 2 < count) slab(s2, k + 2, even, odd);
    }
    wait_reads();
    wait_loads<0>();

    // ---- out. A lane holds columns q 4 grp .. 4 grp + 3 of a sub-tile, of row p l16.
    const int pw = p0 + wave_p * 64, qw = q0 + wave_q * 64;
    if (SUMS && sums_here && grp == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = pw + i * 16 + l16;
            if (p >= g.p) continue;
            if (g.partial) g.partial[(size_t)blockIdx.y * g.plane + (size_t)g.p * g.q + p] = sums[i][0];
            else static_cast<uint16_t*>(g.sums)[p] = f32_to_bf16(sums[i][0]);
        }
    }
    if (g.partial) {   // one of several ranges of the contraction: grad_sum_kernel adds them
        float* const plane = g.partial + (size_t)blockIdx.y * g.plane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = pw + i * 16 + l16;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = qw + j * 16 + grp * 4;
                if (p < g.p && q < g.q) *reinterpret_cast<f32x4*>(plane + (size_t)p * g.q + q) = acc[i][j];
            }
        }
        return;
    }
    meet();   // the stages are free: every wave's reads of them, and loads into them, are behind it
    uint8_t* const mine = lds + wave * (64 * kRowB);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 v = acc[i][j];
            *reinterpret_cast<u32x2*>(mine + (i * 16 + l16) * kRowB + j * 32 + grp * 8) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    uint16_t* const out = static_cast<uint16_t*>(g.out);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = i * 8 + (lane >> 3), p = pw + row, q = qw + (lane & 7) * 8;
        const u32x4 v = *reinterpret_cast<const u32x4*>(mine + row * kRowB + (lane & 7) * 16);
        if (p < g.p && q < g.q) *reinterpret_cast<u32x4*>(out + (size_t)p * g.q + q) = v;
    }
}

// out = the planes' sum, in their order; the last p floats of a plane are the column sums'
__global__ __launch_bounds__(256) void grad_sum_kernel(GradGemmArgs g) {
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, body = (int64_t)g.p * g.q;
    if (at >= body + (g.sums ? g.p : 0)) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(g.partial + at);
    for (int s = 1; s < g.splits; ++s) v += *reinterpret_cast<const f32x4*>(g.partial + s * g.plane + at);
    uint16_t* const out = at < body ? static_cast<uint16_t*>(g.out) + at : static_cast<uint16_t*>(g.sums) + (at - body);
    *reinterpret_cast<u32x2*>(out) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

struct Plan {
    int tiles, splits, slabs_per_split;
    bool two;   // two stages and two workgroups to a compute unit, or four and one
};

// The quickest of a few ways by what their parts measured (ns). Alone on its compute unit a workgroup with four stages takes 400 a
// slab, one with two stages 620, two of these side by side 920 together; a round's start and end 5000 and, where two share a
// unit, 3500 (1408 tiles of five slabs 24 us with two stages, 30 with four; 640 of 172 slabs 248 and 210). Ranges of the
// contraction fill the chip where tiles do not, and cost a launch and their planes' way through memory (552 x 11264 x 2048, 80
// tiles of 176 slabs: 65 us whole, 44 / 40 / 47 in two, three and four).
Plan plan_of(int64_t p, int64_t q, int64_t t) {
    const int64_t tiles = ((p + kTile - 1) / kTile) * ((q + kTile - 1) / kTile);
    const int64_t slabs = (t + kSlab - 1) / kSlab;
    Plan plan{(int)tiles, 1, (int)slabs, true};
    const int64_t full = tiles / 512, rest = tiles % 512;
    int64_t least = full * (slabs * 920 + 3500);
    if (rest) least += slabs * (620 + (rest > 256 ? 300 * (rest - 256) / 256 : 0)) + 3500;
    for (int64_t s = 1; s <= 8 && (s == 1 || s <= slabs / 8); ++s) {
        const int64_t each = (slabs + s - 1) / s, ranges = (slabs + each - 1) / each;
        int64_t time = (tiles * ranges + 255) / 256 * (each * 400 + 5000);
        if (ranges > 1) time += 4500 + ranges * p * q / 560;   // (written and read: 8 bytes a value at 4.5 TB/s)
        if (time < least) least = time, plan = Plan{(int)tiles, (int)ranges, (int)each, false};
    }
    return plan;
}

template <bool ROWS, bool SUMS, int S>
void launch_inst(const GradGemmArgs& g, const Plan& plan, hipStream_t stream) {
    auto kern = grad_gemm_kernel<ROWS, SUMS, S>;
    constexpr int bytes = S * kStage;
    static std::atomic<uint64_t> lds_allowed{0};
    allow_dynamic_lds(reinterpret_cast<const void*>(kern), bytes, lds_allowed);
    kern<<<dim3((unsigned)plan.tiles, (unsigned)plan.splits), dim3(256), bytes, stream>>>(g);
}

template <bool ROWS, bool SUMS>
void launch_plan(GradGemmArgs g, float* scratch, hipStream_t stream) {
    const Plan plan = plan_of(g.p, g.q, g.t);
    g.splits = plan.splits;
    g.slabs_per_split = plan.slabs_per_split;
    g.plane = (int64_t)g.p * g.q + (ROWS ? 0 : g.p);
    g.partial = plan.splits > 1 ? scratch : nullptr;
    if (plan.two) launch_inst<ROWS, SUMS, 2>(g, plan, stream);
    else launch_inst<ROWS, SUMS, 4>(g, plan, stream);
    if (plan.splits > 1) {
        const int64_t values = (int64_t)g.p * g.q + (g.sums ? g.p : 0);
        grad_sum_kernel<<<dim3((unsigned)((values + 1023) / 1024)), dim3(256), 0, stream>>>(g);
    }
}

}  // namespace

bool linear_grad_bf16_supported(int64_t m, int64_t n, int64_t k) {
    constexpr int64_t kMost = (int64_t)1 << 30;   // values an operand's 32-bit byte offsets reach, with a tile's overhang
    if (m <= 0 || n <= 0 || k <= 0 || n % kSlab || k % 8) return false;
    return (m + 2 * 512) * (n + kTile) < kMost && (m + 2 * 512) * (k + kTile) < kMost && (n + 2 * 512) * (k + kTile) < kMost;
}

int64_t linear_grad_bf16_scratch_bytes(int64_t m, int64_t n, int64_t k) {
    const Plan x = plan_of(m, k, n), w = plan_of(n, k, m);
    const int64_t x_floats = x.splits > 1 ? x.splits * m * k : 0, w_floats = w.splits > 1 ? w.splits * (n * k + n) : 0;
    return 4 * (x_floats > w_floats ? x_floats : w_floats);
}

void launch_linear_grad_bf16(const void* g, const void* x, const void* w, void* scratch, void* gx, void* gw, void* gb, int64_t m,
                             int64_t n, int64_t k, hipStream_t stream) {
    GradGemmArgs a{};
    if (gx) {
        a.a = g, a.b = w, a.out = gx, a.p = (int)m, a.q = (int)k, a.t = (int)n;
        launch_plan<true, false>(a, static_cast<float*>(scratch), stream);
    }
    if (gw) {
        a.a = g, a.b = x, a.out = gw, a.sums = gb, a.p = (int)n, a.q = (int)k, a.t = (int)m;
        if (gb) launch_plan<false, true>(a, static_cast<float*>(scratch), stream);
        else launch_plan<false, false>(a, static_cast<float*>(scratch), stream);
    }
}

}  // namespace w8a8
