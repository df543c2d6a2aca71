// Merging the context splits of attention rows: each split left D unnormalised sums, their running maximum and the sum
// of their exponentials, fp32, rows of D + 2. Groups of D / 8 threads take a split each, as many groups to a head as
// there are splits, several heads to a workgroup of 256 where the splits are few: all of a row's splits are requested
// at once. A thread that walks them in turn pays a memory round trip for every few (64 splits of 8192 keys, 32 heads x
// 64: 38 us, here 5; with two to eight splits both take 4 to 5 us).
#pragma once
#include "common.cuh"

namespace w8a8 {

// thread groups to a head, heads to a workgroup (a power of two that divides the heads)
template <int D>
struct MergeShape {
    static constexpr int L = D / 8, G = 256 / L;
    int per_head = 1, heads = 1;
    __host__ __device__ MergeShape(int nsplit, int n_heads) {
        while (per_head < nsplit && per_head < G) per_head *= 2;
        while (heads * 2 * per_head <= G && n_heads % (heads * 2) == 0) heads *= 2;
    }
};

// `base_of(head)`: the head's row in split 0; `stride`: floats from a split to the next; `out`: the row of the first
// of the workgroup's heads; all 256 threads take part
template <int D, class F>
__device__ __forceinline__ void merge_splits(const MergeShape<D>& shape, F base_of, int64_t stride, int nsplit, uint16_t* out) {
    constexpr int L = MergeShape<D>::L, G = MergeShape<D>::G;
    constexpr float kNone = -1e30f;    // what a split without keys left as its maximum
    __shared__ __attribute__((aligned(16))) float sh_v[G][D + 8];
    __shared__ float sh_m[G], sh_l[G];
    const int ln = threadIdx.x % L, grp = threadIdx.x / L, head = grp / shape.per_head;
    float m = kNone, l = 0.0f, v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (head < shape.heads) {
        const float* base = base_of(head);
        for (int j = grp % shape.per_head; j < nsplit; j += shape.per_head) {
            const float* r = base + (int64_t)j * stride;
            const float rm = r[D], rl = r[D + 1];
            float x[8];    // (a caller's workspace is aligned to floats only)
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = r[ln * 8 + i];
            const float mn = fmaxf(m, rm), f0 = __expf(m - mn), f1 = __expf(rm - mn);
            m = mn;
            l = l * f0 + rl * f1;
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = v[i] * f0 + x[i] * f1;
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i += 4) *reinterpret_cast<f32x4*>(&sh_v[grp][ln * 8 + i]) = f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
    if (ln == 0) {
        sh_m[grp] = m;
        sh_l[grp] = l;
    }
    __syncthreads();
    const int n = min(shape.per_head, nsplit);
    for (int e = threadIdx.x * 2; e < shape.heads * D; e += 512) {
        const int g0 = e / D * shape.per_head, d = e % D;
        float mm = kNone;
        for (int i = 0; i < n; ++i) mm = fmaxf(mm, sh_m[g0 + i]);
        float ll = 0.0f, o0 = 0.0f, o1 = 0.0f;
        for (int i = 0; i < n; ++i) {
            const float f = __expf(sh_m[g0 + i] - mm);
            ll += sh_l[g0 + i] * f;
            o0 += sh_v[g0 + i][d] * f;
            o1 += sh_v[g0 + i][d + 1] * f;
        }
        const float inv = ll > 0.0f ? 1.0f / ll : 0.0f;  // a row with no visible key yields zeros
        *reinterpret_cast<uint32_t*>(out + e) = pack_bf16x2(o0 * inv, o1 * inv);
    }
}

}  // namespace w8a8
