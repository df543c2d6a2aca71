// Causal grouped-query attention of a block of new tokens (prefill, chunked or whole), head_dim
// 128 or 64, bf16 MFMAs, fp32 softmax: against the dense bf16 KV cache, against key / value tensors
// of any row, head and batch stride, or against a pool behind a slot table.
//
// The reference expands the KV heads and calls SDPA on [batch, heads, seq, head_dim]
// tensors with a mask tensor (astrai/extension/backend/attention.py:244-253,443-498,
// cached branch of astrai/model/components/attention.py:19-85). Here the mask is
// `key <= position` computed in the kernel, key blocks wholly above a query block
// are never visited, the n_rep query heads of a KV group share every key/value tile,
// and the output is written token-major [batch, seq, heads*head_dim], the layout the
// output projection reads.
//
// One workgroup per (batch, KV head, 32 * QSUB query tokens); wave r takes query head
// hk*n_rep + r % n_rep and the 32 tokens r / n_rep of the block. Keys are handled in 32-key tiles:
//   S^T = K.Q^T on v_mfma_f32_32x32x16_bf16 with keys as rows and queries as columns,
//     so a lane owns ONE query (column lane%32) and 16 of a tile's 32 scores: row maxima
//     and sums are per-lane reductions plus one exchange with lane^32;
//   O^T += V^T.P^T with the same instruction: P^T is the S^T accumulator itself,
//     rounded to bf16 in place (its register order fixes which 8 keys a lane half
//     contributes per 16-key step), and the V^T operand is read out of the row-major
//     value tile with ds_read_b64_tr_b16, the LDS read that hands each lane of a
//     16-lane group four values down a column (four keys of one dim). SPLIT instances (the
//     shapes that attn_rows.hip would take otherwise, whose probabilities have 16 bits of
//     mantissa) enter P as a bf16 head and a bf16 remainder, two MFMAs;
//   keys and values sit in LDS as rows of 16-byte chunks XOR-swizzled by row so that the 16 rows
//     a key operand read touches, and the 4 rows a transposing read touches, fall into
//     different banks.
// A wave's instruction stream is a software pipeline over tiles, written out and pinned with sched_barrier: a step issues
// the score MFMAs of tile T+1 and the P.V MFMAs of tile T-1 with the exponentials of tile T spread evenly behind all
// of them, an element behind each. A 32x32x16 MFMA leaves the vector ALU 24 of its 32 cycles (4 for most instructions, 8
// for an exponential); what exceeds that in one slot delays the next MFMA and what is left unused in another is lost: 16
// slots of 20 cycles take 536, eight of 44 and eight empty ones 640. Row maxima of tile T+1 go behind the last MFMAs,
// the question whether one has outgrown its reference into the next step. Keys and values arrive by direct-to-LDS
// loads into two rings of four tiles, values two tiles behind the keys, one 64-key block ahead (the first three tiles of
// both at once), one load to every second MFMA of a block's first step (all at once they stall the waves that issue
// them); one workgroup barrier per block; no staging registers. Dense loads keep their lane's offset, the descriptors move
// along instead; the loop over unmasked blocks goes once round the rings, so that its LDS offsets are constants. Tiles that
// every query of the wave sees whole skip the masking code; the accumulators are rescaled only when a row maximum has
// outgrown the reference maximum by 2^8.
//
// The direct-to-LDS loads are written in assembly (they have no output register): behind the
// builtin the compiler orders every transposing read after all loads in flight (s_waitcnt vmcnt(0)),
// which puts a whole memory round trip into each 64-key block. The blocks without and with masking
// are two loops, not two branches of one: at a join of the two the compiler moved all accumulators
// from one register set to another on every block.
// What bounds it: 53 vector instructions, 16 exponentials, 16 MFMAs and 24 LDS reads a tile and wave; a tile takes 890
// cycles alone on a SIMD, 790 with two waves (512 are the MFMAs'; operand reads 190, the branch and the barrier 100),
// under a clock that the power limit holds at 1.7 GHz for long sequences (2.1 for short ones).
// Counters of 4 x 2048 tokens: matrix pipe busy 57% of the SIMD cycles, vector ALU 56% (48 and 53 before the exponentials were spread).
// Measured (graph replays): 4 x 2048 causal tokens, 16/4 heads x 128 in [batch, seq, head] order 75 us (915 TFLOP/s), ragged
// 16 x 175..700 tokens of 32/8 heads x 64 in a pool 75.7 us (P in two terms); with the exponentials behind the score
// MFMAs alone, the loads in a burst and offsets formed for each (120 vector instructions a tile) 80.3 and 78.2. Prompts of up
// to 100 tokens were 0.2 to 0.3 us faster that way (8 x 100, 32/8 heads x 64: 6.8 and 7.15). Up to 238 /
// 168 registers: two / three workgroups per CU. 64 query tokens a workgroup halve the loads, but couple eight waves:
// 2 x 4096 126 us (133 here, same run), 4 x 2048 74 (74), 16 x 1024 89 (85), 1 x 4096 93 (76), 32 x 512 64.5 (58); not kept.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "lds_dma.cuh"
#include "launchers.h"

namespace w8a8 {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kKB = 64;            // keys per block
constexpr float kNegBig = -1e30f;  // finite stand-in for -inf: no inf - inf

// The offset of a row that is to read as zeros, and the most bytes a descriptor of this file spans: pools and heads
// go up to 4 GiB, past the 2 GiB of kOutOfRange.
constexpr uint32_t kMissing = 0xffffff00u;

typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxParts = 16;
typedef float f32x4_at4 __attribute__((ext_vector_type(4), aligned(4)));  // (a caller's workspace is aligned to floats only)
typedef float f32x2_at4 __attribute__((ext_vector_type(2), aligned(4)));

// What a wave leaves of a part: the accumulators as its lanes hold them, four dims of a row after four, then maximum
// (log2 units) and sum of its 32 rows. Waves in the order of the workgroups that a schedule without parts has.
__host__ __device__ constexpr int part_floats(int d) { return 32 * (d + 2); }

// Parts of the keys, for schedules with few (64-row tile, query head) pairs: n of them leave blocks / n of the 64-key
// blocks in the chain, 1 to 1.5 us each, and cost a write and a read of fp32 accumulators, 1 us for 48 to 64 pairs and part;
// the sum is least at about n = sqrt(96 blocks / pairs). A block of queries counts its own keys. The launch, which knows
// only how many there can be, has no parts where they would not save what they and the second launch cost.
// Measured (graph replays, us), attn_rows.hip with its split, which these schedules ran before, -> here; one part in brackets:
//   16/16 heads x 64:  1 x 33 tokens 8.9 -> 6.5, 1 x 256 15.8 -> 11.1, 3 x 64 behind 2000 24.0 -> 21.0 (41.5), 1 x 300
//   behind 1500 31.6 -> 23.6 (37.6);  32/8 x 64: 1 x 33 10.3 -> 5.8, 1 x 256 30.1 -> 9.5, 3 x 64 behind 2000 32.8 -> 19.4
//   (35.9), 1 x 300 behind 1500 53.6 -> 27.2 (32.8);  16/16 x 128: 10.6 -> 7.8, 21.0 -> 14.5, 35.5 -> 24.0 (58.3),
//   48.3 -> 29.8 (52.3).
// From 256 pairs on there are none: those schedules ran here before, in one launch, and with a wide table over short
// contexts the second would be paid for nothing (4 x 256 behind 1000, 16/16 x 64: 26 us with one part and two).
constexpr int kMaxPartPairs = 256, kPairsPerBlock = 96, kMergeBlocks = 1;

__host__ __device__ inline int part_count(int blocks, int64_t pairs, int nsplit) {
    int n = 1;
    while (n < nsplit && n < blocks && (int64_t)(n + 1) * (n + 1) * pairs <= (int64_t)blocks * kPairsPerBlock) ++n;
    return n;
}

// 64-key blocks of a part of `blocks` of them
__device__ __forceinline__ int part_blocks(const AttnPrefillArgs& a, int blocks) {
    const int n = part_count(blocks, (int64_t)a.num_q_tiles * a.n_heads, a.nsplit);
    return (blocks + n - 1) / n;
}

// PAGED: the queries are packed [total_q, heads, D] with per-request row ranges
// (qo_indptr), the caches are token-granular pools [slots, kv_heads, D] reached through
// req_to_token, and a 64-row query tile t of the caller's schedule belongs to request
// q_tile_to_batch[t], rows 64 * q_tile_to_index[t] .. of it (csrc/kernels/attention/
// paged_prefill.cu:4-34, layout_policies.cuh:67-93,174-232; the schedule is built in
// astrai/inference/cache/pool.py:219-234). Query row i of a
// request of q_len rows and kv_len keys sees keys 0 .. kv_len - q_len + i (all of them
// without the causal flag), so nothing has to be fetched to know the key range. Workgroups walk
// the schedule backwards: a sequence's last tiles see the most keys and start first.
// MASK (paged only): a bool tensor says, per sequence, (head,) (query row,) and position,
// what may be attended on top of the causal range (csrc/kernels/attention/mma_utils.cuh:190-199);
// every tile then takes the masking path.
// PARTS (paged, no mask, SPLIT): part `split` of a.nsplit takes the 64-key blocks part_blocks() gives it, of which nothing but
// the table and the limits know; a block of queries with more than one part leaves them to merge_parts_kernel.
template <int D, int NREP, int QSUB, bool PAGED, bool MASK, bool SPLIT, bool PARTS = false>
__global__ __launch_bounds__(64 * NREP * QSUB, NREP * QSUB < 4 ? 1 : D == 64 && NREP * QSUB == 4 ? 3 : 2) void attn_prefill_kernel(AttnPrefillArgs a) {
    constexpr int WAVES = NREP * QSUB;
    constexpr int QB = 32 * QSUB;                 // query tokens per workgroup
    constexpr int ROW = 2 * D;                    // bytes per key or value row in LDS
    constexpr int TILE = 32 * ROW;                // one 32-key tile
    constexpr int RING = 4 * TILE;                // keys; as much again for values
    constexpr int LPR = ROW / 16;                 // 16-byte chunks (lanes of a load) per row
    constexpr int RPI = 64 / LPR;                 // rows per 1 KiB load
    constexpr int DMA = kKB / RPI / WAVES;        // loads per wave, tensor and block
    constexpr int KS = D / 16;                    // score MFMAs per tile
    constexpr int DT = D / 32;                    // 32-dim output tiles
    static_assert(DMA >= 1 && (!PAGED || QB <= 64), "shape");
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * RING];
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = lane & 31, h = lane >> 5;
    const int rep = wave % NREP, qsub = wave / NREP;
    // XOR swizzles (in chunks) of key and value rows: see the file comment
    auto swz_k = [](int row) { return D == 128 ? (row & 15) : ((row >> 1) & 7); };
    auto swz_v = [](int row) { return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); };

    int hk, rows_total, row0;   // KV head; query rows of the sequence; first row of this block
    int64_t tok0;               // index of row 0 of the sequence in the token-major output
    const uint16_t* qbase;      // row 0 of the sequence, this wave's head
    int64_t q_row_stride;       // elements between consecutive query rows
    int pq, kmax;               // this lane's newest visible key; the block's newest
    [[maybe_unused]] int part = 0;
    [[maybe_unused]] bool whole = true;         // this part is all there is
    [[maybe_unused]] float* part_ws = nullptr;  // where it goes otherwise
    [[maybe_unused]] const int* table = nullptr;
    [[maybe_unused]] int b_dense = 0, seq_index = 0;
    [[maybe_unused]] int64_t block_pos = -1;  // dense, with positions: that of the block's row `lane`
    if constexpr (PAGED) {
        constexpr int SUBS = 64 / QB;  // workgroups that share a tile
        const int idx = (int)(gridDim.x - 1 - blockIdx.x);
        hk = idx % a.n_kv_heads;
        int sub = (idx / a.n_kv_heads) % SUBS, tile = idx / (SUBS * a.n_kv_heads);
        [[maybe_unused]] int item = 0;
        if constexpr (PARTS) {
            item = idx / a.n_kv_heads;
            part = item % a.nsplit;
            item /= a.nsplit;
            sub = item % SUBS, tile = item / SUBS;
        }
        const int req_i = a.q_tile_to_batch[tile];
        seq_index = req_i;
        const int q_start = a.qo_indptr[req_i];
        rows_total = a.qo_indptr[req_i + 1] - q_start;
        row0 = a.q_tile_to_index[tile] * 64 + sub * QB;
        if (row0 >= rows_total) return;  // this part of the tile lies past the request
        const int64_t req = a.req_pool_indices[req_i];
        const bool req_ok = req >= 0 && req < a.num_requests;  // a bad row reads as an empty sequence
        const int kv_len = req_ok ? (int)min((int64_t)(a.kv_indptr[req_i + 1] - a.kv_indptr[req_i]), a.rtt_stride) : 0;
        table = a.req_to_token + (req_ok ? req : 0) * a.rtt_stride;
        tok0 = q_start;
        q_row_stride = (int64_t)a.n_heads * D;
        qbase = static_cast<const uint16_t*>(a.q) + ((int64_t)q_start * a.n_heads + hk * NREP + rep) * D;
        const int last = min(row0 + QB, rows_total) - 1;
        const int shift = a.causal ? kv_len - rows_total : INT_MIN;
        pq = a.causal ? min(shift + row0 + qsub * 32 + qi, kv_len - 1) : kv_len - 1;
        kmax = a.causal ? min(shift + last, kv_len - 1) : kv_len - 1;
        if constexpr (PARTS) {
            const int blocks = max(kmax, 0) / kKB + 1, per = part_blocks(a, blocks);
            if (part * per >= blocks) return;
            const int key0 = part * per * kKB;
            whole = per >= blocks;
            table += key0;
            pq = min(pq - key0, per * kKB - 1);
            kmax = min(kmax - key0, per * kKB - 1);
            part_ws = a.ws + ((((int64_t)item * a.n_kv_heads + hk) * WAVES + wave) * a.nsplit + part) * part_floats(D);
        }
    } else {
        const int nqb = (a.seq + QB - 1) / QB;
        const int groups = a.batch * a.n_kv_heads;
        // Longest key ranges first; where all workgroups are resident at once, two to a compute unit (four waves
        // each), the second 256 run the other way, so that the longest share a unit with the shortest: 1 x 4096
        // tokens, 16/4 heads x 128, 97 -> 93 us. With eight waves a unit holds one, and the second 256 start as
        // units become free: longest first is the better order (32/4 heads: 140 us, reversed 161)
        const bool turned = WAVES <= 4 && gridDim.x <= 512 && blockIdx.x >= 256;
        const int order = turned ? (int)(gridDim.x + 255 - blockIdx.x) : (int)blockIdx.x;
        const int qb = nqb - 1 - order / groups;
        const int bk = order % groups;
        const int b = bk / a.n_kv_heads;
        b_dense = b;
        hk = bk % a.n_kv_heads;
        rows_total = a.seq;
        row0 = qb * QB;
        tok0 = (int64_t)b * a.seq;
        q_row_stride = a.q_stride.row;
        qbase = static_cast<const uint16_t*>(a.q) + b * a.q_stride.batch + (hk * NREP + rep) * a.q_stride.head;
        kmax = 0;
        if (a.positions) {
            // The positions are requested first and looked at last: the query rows and the first
            // key tiles do not depend on them. (Blocks of up to 64 rows: launch_attn_prefill.)
            block_pos = lane < QB && row0 + lane < a.seq ? a.positions[row0 + lane] : -1;
            pq = -1;
        } else {
            const int last = min(row0 + QB, rows_total) - 1;
            const int newest = (int)a.max_len - 1;
            pq = a.causal ? min(a.causal_offset + row0 + qsub * 32 + qi, newest) : newest;
            kmax = a.causal ? min(a.causal_offset + last, newest) : newest;
        }
    }
    const int head = hk * NREP + rep;
    const int s_row = row0 + qsub * 32 + qi;
    const bool row_live = s_row < rows_total;
    // this lane's row of the mask and how many of its positions the mask covers (none for a
    // query row the mask has no row for: nothing is read there and nothing attended)
    [[maybe_unused]] const uint8_t* mask_row = nullptr;
    [[maybe_unused]] int mask_keys = 0;
    if constexpr (MASK) {
        const bool covered = row_live && (a.mask_l_stride == 0 || s_row < a.mask_rows);
        mask_row = a.mask + (int64_t)seq_index * a.mask_b_stride + (int64_t)head * a.mask_h_stride +
                   (int64_t)(covered ? s_row : 0) * a.mask_l_stride;
        mask_keys = covered ? a.mask_width : 0;
    }

    const uint16_t* qrow = qbase + (int64_t)min(s_row, rows_total - 1) * q_row_stride;
    u32x4 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qrow + ks * 16 + h * 8);

    // keys: straight from memory into LDS, 1 KiB (RPI rows) per instruction; lane l
    // lands at row l / LPR, chunk position l % LPR and therefore asks for that chunk ^ swizzle(row).
    // Dense: the descriptor covers the whole row range of this (batch, KV head):
    // whatever a row past the newest position holds, its scores are replaced (not scaled)
    // by the mask. Paged: the descriptor covers the pool and each lane looks up the slot of
    // its row; rows past the sequence ask for an offset outside it and arrive as zeros.
    const uint32_t k_row = PAGED ? (uint32_t)a.n_kv_heads * ROW : (uint32_t)(a.k_stride.row * 2);  // bytes from row to row
    const uint32_t v_row = PAGED ? k_row : (uint32_t)(a.v_stride.row * 2);
    const uint16_t* kc = static_cast<const uint16_t*>(a.k_cache) +
                         (PAGED ? (int64_t)hk * D : b_dense * a.k_stride.batch + hk * a.k_stride.head);
    const uint16_t* vc = static_cast<const uint16_t*>(a.v_cache) +
                         (PAGED ? (int64_t)hk * D : b_dense * a.v_stride.batch + hk * a.v_stride.head);
    const uint32_t pool_bytes = PAGED ? (uint32_t)(a.num_slots * k_row - hk * ROW) : 0u;
    u32x4 rk = make_desc(kc, PAGED ? pool_bytes : (uint32_t)(a.max_len - 1) * k_row + ROW);
    // Paged: one load per wave fetches the slots of all rows its next loads cover (lane l <
    // RPW: this wave's l-th key row; the next RPW lanes: its value rows); the loads take each
    // row's slot from the lane that holds it. Looked up one block ahead, so that the table
    // access is not a second memory round trip in front of every load.
    constexpr int RPW = RPI * DMA;  // rows of a 64-row block that this wave loads
    auto lookup = [&](int t0, int v0) -> int {  // first key tile, first value tile (-1: before the first key)
        const int l = lane & (2 * RPW - 1);  // (lanes past 2 RPW repeat the pattern, unused)
        const int key = l < RPW ? t0 * 32 + wave * RPW + l : v0 * 32 + wave * RPW + (l - RPW);
        const int slot = (key >= 0 && key <= kmax) ? table[key] : -1;
        return slot;
    };
    // the rows' offsets in the lanes that looked them up (kMissing: chunk offsets added to it stay past the pool)
    auto rows_of = [&](int slot) -> uint32_t {
        return slot >= 0 && slot < a.num_slots ? (uint32_t)slot * k_row : kMissing;
    };
    auto paged_off = [&](uint32_t rows, int src_lane, int swz) -> uint32_t {
        return (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane << 2, (int)rows) + (uint32_t)(((lane & (LPR - 1)) ^ swz) << 4);
    };
    // Dense: the descriptors move along with the keys, so that a load's offset is a constant of its lane
    auto advance = [](u32x4& desc, uint64_t bytes) {
        const uint64_t addr = (((uint64_t)desc.y << 32) | desc.x) + bytes;
        desc.x = (uint32_t)addr;
        desc.y = (uint32_t)(addr >> 32);
        desc.z = desc.z > bytes ? desc.z - (uint32_t)bytes : 0u;
    };
    [[maybe_unused]] uint32_t k_voff[DMA];
    if constexpr (!PAGED) {
#pragma unroll
        for (int j = 0; j < DMA; ++j) {
            const int row = (wave * DMA + j) * RPI + lane / LPR;
            k_voff[j] = (uint32_t)row * k_row + (uint32_t)(((lane & (LPR - 1)) ^ swz_k(row)) << 4);
        }
    }
    // tiles t0 and t0+1 (64 keys) into their ring slots: where in memory, and one load of them
    constexpr int TI = 32 / RPI;  // loads per tile
    auto k_off = [&](int j, [[maybe_unused]] uint32_t rows) -> uint32_t {
        const int inst = wave * DMA + j;  // 64 / RPI loads; half of them per tile
        return PAGED ? paged_off(rows, j * RPI + lane / LPR, swz_k(inst * RPI + lane / LPR)) : k_voff[j];
    };
    auto dma_k = [&](int j, int t0, uint32_t off) {
        const int inst = wave * DMA + j;
        lds_dma16<false>(rk, lds0 + ((t0 + inst / TI) & 3) * TILE + (inst % TI) * 1024, off);
    };
    // The first three tiles, keys and values alike: load i of the workgroup's is rows i * RPI .. of them, and wave i % WAVES's
    constexpr int I3 = 3 * TI, T3 = (I3 + WAVES - 1) / WAVES;
    [[maybe_unused]] uint32_t start_rows = 0;
    auto start_load = [&](const u32x4& desc, int ring, int t, uint32_t stride, auto swz) __attribute__((always_inline)) {
        const int i = wave + t * WAVES, row = i * RPI + lane / LPR;
        if (I3 % WAVES && i >= I3) return;
        const uint32_t chunk = (uint32_t)(((lane & (LPR - 1)) ^ swz(row)) << 4);
        uint32_t off;
        if constexpr (PAGED) off = (uint32_t)__builtin_amdgcn_ds_bpermute((t * RPI + lane / LPR) << 2, (int)start_rows) + chunk;
        else off = (uint32_t)min((uint64_t)row * stride + chunk, (uint64_t)kMissing);
        lds_dma16<false>(desc, lds0 + ring + i * 1024, off);
    };
    [[maybe_unused]] int slots = 0;
    if constexpr (PAGED) {
        const int key = (wave + lane / RPI * WAVES) * RPI + lane % RPI;
        const int first = (key < 96 && key <= kmax) ? table[key] : -1;
        slots = lookup(3, 1);  // what the first block's loads will ask for
        start_rows = rows_of(first);
    }
#pragma unroll
    for (int t = 0; t < T3; ++t) start_load(rk, 0, t, k_row, swz_k);
    if constexpr (!PAGED) advance(rk, (uint64_t)k_row * 96);

    if constexpr (!PAGED) {
        if (a.positions) {
            // (a token past the cache sees what it holds; positions are whole 64-bit numbers)
            const int newest = (int)max(min(block_pos, a.max_len - 1), (int64_t)-1);
            pq = __shfl(newest, qsub * 32 + qi, kWave);
            // what the block's queries may see: every lane ends up with the same value
            kmax = newest;
#pragma unroll
            for (int off = 32; off; off >>= 1) kmax = max(kmax, __shfl_xor(kmax, off, kWave));
        }
        kmax = __builtin_amdgcn_readfirstlane(kmax);
    }
    // (rows that lie before the first key count from below it: -1 for all of them, so that every wave of the
    // workgroup walks the same blocks, one of masked keys)
    kmax = max(kmax, -1);
    // what this wave's queries see: all of them up to pmin, none past kmax_w (equal to kmax with one
    // group of 32 tokens per workgroup)
    int pmin = row_live ? pq : 1 << 30, kmax_w = row_live ? pq : -1;
#pragma unroll
    for (int off = 16; off; off >>= 1) {
        pmin = min(pmin, __shfl_xor(pmin, off, kWave));
        kmax_w = max(kmax_w, __shfl_xor(kmax_w, off, kWave));
    }
    pmin = __builtin_amdgcn_readfirstlane(pmin);
    kmax_w = max(__builtin_amdgcn_readfirstlane(min(kmax_w, kmax)), -1);
    if (!row_live) pq = kmax_w;  // rows past the end see everything and are never stored
    const int nkb = kmax / kKB + 1;     // (kmax = -1, an empty sequence: one block of masked keys)
    const int tiles_w = kmax_w / 32 + 1;  // tiles this wave computes

    // values: the same way into a ring of their own, two tiles behind the keys. Rows past kmax arrive as zeros, so a
    // stale cache row can never meet a zero probability as 0 * NaN. (With far strides those rows' offsets pass 32
    // bits: they must not come round to a place inside. Keys may: their scores are replaced.)
    u32x4 rv = make_desc(vc, PAGED ? pool_bytes : kmax >= 0 ? (uint32_t)kmax * v_row + ROW : 0u);
    [[maybe_unused]] uint32_t v_voff[DMA];
    if constexpr (!PAGED) {
#pragma unroll
        for (int j = 0; j < DMA; ++j) {
            const int row = (wave * DMA + j) * RPI + lane / LPR;
            v_voff[j] = (uint32_t)min((uint64_t)row * v_row + (((lane & (LPR - 1)) ^ swz_v(row)) << 4), (uint64_t)kMissing);
        }
    }
    auto v_off = [&](int j, [[maybe_unused]] uint32_t rows) -> uint32_t {
        const int inst = wave * DMA + j;
        return PAGED ? paged_off(rows, RPW + j * RPI + lane / LPR, swz_v(inst * RPI + lane / LPR)) : v_voff[j];
    };
    auto dma_v = [&](int j, int t0, uint32_t off) {
        const int inst = wave * DMA + j;
        lds_dma16<false>(rv, lds0 + RING + ((t0 + inst / TI) & 3) * TILE + (inst % TI) * 1024, off);
    };

    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = 0.0f;
    // m_run is the reference maximum the probabilities are taken against, in log2 units.
    // It follows the true running maximum lazily: only when some query of the wave has
    // outgrown it by more than kSlack does the wave pay for rescaling its accumulators;
    // until then probabilities may reach 2^kSlack, which fp32 sums and bf16 operands hold.
    constexpr float kSlack = 8.0f;
    // It starts half way between any score and a hidden key's, whose probability is then an exact zero: started at
    // the stand-in itself, a row whose first tiles are hidden took it for a maximum, and the rounding of c times it
    // for a probability, infinite at every other scale.
    const float c = a.scale * 1.44269504088896340736f;  // scores to log2 units
    float m_run = 0.5f * kNegBig * fminf(c, 1.0f), l_run = 0.0f, m_lim = m_run + kSlack;
    const f32x16 zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f,
                           0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // V^T operand of 32 dims x 16 keys: two transposing reads. In each 16-lane group, lane
    // 4j+q points at row j, dims 4q..4q+3 of a 4-row x 16-dim patch and receives dim (its
    // index in the group) of rows 0..3. Lane half h takes rows 4h..4h+3 and 8+4h..8+4h+3 of
    // the 16-key step: the keys its P^T registers hold (register 4g+j = key 8g + 4h + j).
    // (the swizzle leaves the chunk bits of the dim tile free: it is XORed into the offset as well)
    const int v_lane0 = [&] {
        const int sl = lane & 15, j = sl >> 2, q = sl & 3, g1 = (lane >> 4) & 1;
        return (4 * h + j) * ROW + ((((2 * g1 + (q >> 1)) ^ swz_v(j)) << 4) | ((q & 1) << 3));
    }();
    // key operand of k-step ks: chunk (2ks + h) ^ swizzle(row) of this lane's row. The tile
    // offset and the row offset are multiples of the row size, so the k-step can be XORed into the
    // whole byte offset: one address register per tile instead of one per k-step.
    const int k_lane0 = qi * ROW + ((h ^ swz_k(qi)) << 4);
    auto k_frag = [&](int tile_off, int ks) -> u32x4 {
        return *reinterpret_cast<const u32x4*>(lds + tile_off + (k_lane0 ^ (ks << 5)));
    };
    // T0: first key of the tile; PARTIAL with several token groups per workgroup: rows past this
    // wave's newest key are other queries' keys and are replaced by zeros (their probabilities here
    // are zero, and 0 * NaN would not be)
    auto v_frag = [&](auto mask_tag, int T0, int vt_off, int t, int dt) -> u32x4 {
        typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
        const uint8_t* src = lds + vt_off + (v_lane0 ^ (dt << 6)) + t * 16 * ROW;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + 8 * ROW));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        u32x4 v = {l2.x, l2.y, h2.x, h2.y};
        if constexpr (QSUB > 1 && decltype(mask_tag)::value) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int key = T0 + t * 16 + (w >> 1) * 8 + 4 * h + 2 * (w & 1);
                v[w] &= (key <= kmax_w ? 0xffffu : 0u) | (key < kmax_w ? 0xffff0000u : 0u);
            }
        }
        return v;
    };
    // the larger of this lane's and lane^32's value, without a round trip through LDS
    auto max_halves = [](float m) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        float both;
        __asm__("v_max_f32 %0, %1, %2" : "=v"(both) : "v"(r[0]), "v"(r[1]));  // (fmaxf would make each quiet first)
        return both;
    };
    // masking and this lane's share of the row maximum of tile T (raw scores; c > 0 keeps order)
    auto mask_max4 = [&](auto mask_tag, int T, f32x16& s, int g, float m) __attribute__((always_inline)) -> float {
        constexpr bool PARTIAL = decltype(mask_tag)::value;  // some score of the tile may be hidden
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = 4 * g + j;
            if (PARTIAL) {
                const int key = T * 32 + g * 8 + h * 4 + j;
                bool visible = key <= pq;
                if constexpr (MASK) {
                    // (the byte is fetched whether or not it is needed, from a clamped index:
                    // four independent loads per group instead of four dependent branches)
                    const uint8_t keep = mask_row[max(min(key, mask_keys - 1), 0)];
                    visible = visible && key < mask_keys && keep != 0;
                }
                s[e] = visible ? s[e] : kNegBig;
            }
            m = fmaxf(m, s[e]);
        }
        return m;
    };

    // the same of a whole tile, chosen at run time (65 vector instructions more if some score may be hidden)
    const int tfull = (pmin + 1) / 32;  // tiles every query of the wave sees whole
    auto tile_max = [&](int T, f32x16& s) __attribute__((always_inline)) -> float {
        float m = kNegBig;
        if (!MASK && T < tfull) {
#pragma unroll
            for (int g = 0; g < 4; ++g) m = mask_max4(std::false_type{}, T, s, g, m);
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) m = mask_max4(std::true_type{}, T, s, g, m);
        }
        return max_halves(m);
    };

    constexpr int NV = 2 * DT;                 // value operands of a tile
    constexpr int NM = NV * (SPLIT ? 2 : 1);   // P.V MFMAs
    constexpr int NS = KS + NM;                // slots (MFMAs) of a step
    constexpr int KD = KS / 2, V0 = SPLIT ? 2 : 4;  // key / value operands are requested that many ahead
    static_assert(V0 <= KS && V0 <= NV && KD <= NM, "lead");
    // P of a tile: bf16 pairs, and their remainders
    struct Probs {
        uint32_t hi[8];
        uint32_t lo[SPLIT ? 8 : 1];
    };
    // element e of P; the even one of a pair waits in `even` for the odd one
    auto prob = [&](int e, const f32x16& s, Probs& out, float& even, float& l_add) __attribute__((always_inline)) {
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], c, -m_run));
        __asm__ volatile("" : "+v"(p));  // here: its uses are a step away, and the compiler would move it there
        if ((e & 1) == 0) {
            even = p;
            return;
        }
        l_add += even + p;
        uint32_t hi = pack_bf16x2(even, p);
        __asm__ volatile("" : "+v"(hi), "+v"(l_add));
        out.hi[e >> 1] = hi;
        if constexpr (SPLIT) {
            uint32_t lo = pack_bf16x2(even - __uint_as_float(hi << 16), p - __uint_as_float(hi & 0xffff0000u));
            __asm__ volatile("" : "+v"(lo));
            out.lo[e >> 1] = lo;
        }
    };
    auto pv = [&](const Probs& p, int n, u32x4 (&vf)[NV]) __attribute__((always_inline)) {
        const int i = SPLIT ? n >> 1 : n, t = i / DT, dt = i % DT;
        u32x4 pf = {p.hi[4 * t], p.hi[4 * t + 1], p.hi[4 * t + 2], p.hi[4 * t + 3]};
        if constexpr (SPLIT)
            if (n & 1) pf = u32x4{p.lo[4 * t], p.lo[4 * t + 1], p.lo[4 * t + 2], p.lo[4 * t + 3]};
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8, vf[i]), __builtin_bit_cast(bf16x8, pf), o[dt], 0, 0, 0);
    };
    auto k_first = [&](int T, u32x4 (&kf)[KS]) __attribute__((always_inline)) {  // a step's first key operands
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) kf[ks] = k_frag((T & 3) * TILE, ks);
    };
    [[maybe_unused]] uint32_t k_at[DMA], v_at[DMA];  // where the block's loads go to (paged: looked up at its start)

    // One step: the scores of tile T+1, P of tile T, and P.V of tile T-1, the exponentials spread evenly over all of
    // its MFMAs. In: s_in = raw (masked) scores of tile T; grow_in: some row's maximum m_in (both lane halves) has
    // outgrown the reference. Out: p_out = P of tile T; s_out, m_out, grow_out the same for tile T+1.
    // first_tag: 1: a block's first step, which issues its loads (K tiles T+3, T+4, V tiles T+1, T+2), and reads the
    // second step's first key operands; 2: a second one that chooses at run time whether the scores are masked.
    auto step = [&](auto mask_tag, auto ring_tag, auto first_tag, int T, f32x16& s_in, float m_in, bool grow_in, f32x16& s_out,
                    float& m_out, bool& grow_out, const Probs& p_in, Probs& p_out, u32x4 (&kf)[KS])
                    __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_tag)::value == 1, CHOOSE = decltype(first_tag)::value == 2;
        constexpr int RING0 = decltype(ring_tag)::value;  // ring slot of the block's first tile; -1: from T
        constexpr int AT = RING0 + (FIRST ? 0 : 1);
        auto slot_of = [&](int d) { return RING0 >= 0 ? (AT + d + 4) & 3 : (T + d) & 3; };
        float alpha = 1.0f;
        if (__builtin_expect(grow_in, 0)) {
            __asm__ volatile("" ::: "memory");  // (a branch, not four selects)
            const float m_new = fmaxf(m_run, m_in * c);
            alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            m_lim = m_new + kSlack;
            l_run *= alpha;
        }
        const int kt = slot_of(1) * TILE, vt = RING + slot_of(-1) * TILE;
        float l_add = 0.0f, e0 = 0.0f, m = kNegBig;
        u32x4 vf[NV];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            // operands of later MFMAs
            if (n + KD < KS) kf[n + KD] = k_frag(kt, n + KD);
            if (n >= KS - V0 && n < KS)
                vf[n - (KS - V0)] = v_frag(mask_tag, (T - 1) * 32, vt, (n - (KS - V0)) / DT, (n - (KS - V0)) % DT);
            if (n >= KS && (!SPLIT || ((n - KS) & 1) == 0)) {
                const int i = (SPLIT ? (n - KS) >> 1 : n - KS) + V0;
                if (i < NV) vf[i] = v_frag(mask_tag, (T - 1) * 32, vt, i / DT, i % DT);
            }
            if constexpr (FIRST)
                if (n >= NS - KD) kf[n - (NS - KD)] = k_frag(slot_of(2) * TILE, n - (NS - KD));
            if (n < KS) {
                s_out = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, kf[n]), __builtin_bit_cast(bf16x8, qf[n]), n == 0 ? zero16 : s_out, 0, 0, 0);
            } else {
                pv(p_in, n - KS, vf);
            }
            if constexpr (FIRST) {
                // the block's loads, one at a time: together they stall the waves that issue them
#pragma unroll
                for (int l = 0; l < 2 * DMA; ++l)
                    if (n == 1 + l * (NS - 2) / (2 * DMA)) {
                        if (l < DMA) dma_k(l, slot_of(3), PAGED ? k_at[l] : k_off(l, 0));
                        else dma_v(l - DMA, slot_of(1), PAGED ? v_at[l - DMA] : v_off(l - DMA, 0));
                    }
            }
            // exponentials: element e behind MFMA e * NS / 16
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (n == e * NS / 16) prob(e, s_in, p_out, e0, l_add);
            if constexpr (!CHOOSE) {
                if (n >= NS - 6 && n < NS - 2) m = mask_max4(mask_tag, T + 1, s_out, n - (NS - 6), m);
                if (n == NS - 2) m_out = max_halves(m);
                if (n == NS - 1) grow_out = __any(m_out * c > m_lim);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (CHOOSE) {
            m_out = tile_max(T + 1, s_out);
            grow_out = __any(m_out * c > m_lim);
        }
        l_run += l_add;
        if (__builtin_expect(grow_in, 0)) {  // P.V of tile T-1 was still against the old reference
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
        }
    };

    // ---- prologue: key tiles 0..2, value tiles 0..2; scores of tile 0
    const int nfast = MASK ? 0 : min(max(tfull - 1, 0), tiles_w) / 2;  // blocks whose steps only produce unmasked tiles
#pragma unroll
    for (int t = 0; t < T3; ++t) start_load(rv, RING, t, v_row, swz_v);
    if constexpr (!PAGED) advance(rv, (uint64_t)v_row * 32);  // (the first block moves it on to tile 3)
    // the scores need the queries and the key tiles, not the values, the newest of this wave's loads
    __builtin_amdgcn_s_waitcnt(0x0f70 | (I3 / WAVES));  // vmcnt(I3 / WAVES)
    static_assert(I3 / WAVES < 16, "vmcnt's low bits");
    __syncthreads();
    f32x16 sa, sb;
    float ma, mb;
    bool ga, gb;
    Probs pa, pb;
    {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8, k_frag(0, ks)), __builtin_bit_cast(bf16x8, qf[ks]),
                ks == 0 ? zero16 : sa, 0, 0, 0);
        ma = tile_max(0, sa);
        ga = __any(ma * c > m_lim);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __syncthreads();  // tile 0's ring slot is overwritten by the first block's loads
    u32x4 kf[KS];
    k_first(1, kf);
    auto begin_block = [&](int kb) {
        if (kb + 1 >= nkb) rk.z = 0;  // nobody is left to read them (paged: no such slots)
        if constexpr (PAGED) {
#pragma unroll
            for (int j = 0; j < DMA; ++j) k_at[j] = k_off(j, rows_of(slots)), v_at[j] = v_off(j, rows_of(slots));
            slots = lookup(2 * kb + 5, 2 * kb + 3);  // for the next block's loads
        }
    };
    auto end_block = [&](int next_tile) {  // (or its ring slot)
        if constexpr (!PAGED) {
            advance(rk, (uint64_t)k_row * 64);
            advance(rv, (uint64_t)v_row * 64);
        }
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        k_first(next_tile, kf);
    };
    auto block = [&](auto mask_tag, auto ring_tag, int kb) __attribute__((always_inline)) {
        constexpr int R = decltype(ring_tag)::value;
        begin_block(kb);
        step(mask_tag, ring_tag, std::true_type{}, 2 * kb, sa, ma, ga, sb, mb, gb, pb, pa, kf);
        step(mask_tag, ring_tag, std::false_type{}, 2 * kb + 1, sb, mb, gb, sa, ma, ga, pa, pb, kf);
        end_block(R >= 0 ? R + 3 : 2 * kb + 3);
    };
    auto last_pv = [&](const Probs& p) __attribute__((always_inline)) {
        const int vt = RING + ((tiles_w - 1) & 3) * TILE;
        u32x4 vf[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) vf[i] = v_frag(std::true_type{}, (tiles_w - 1) * 32, vt, i / DT, i % DT);
#pragma unroll
        for (int n = 0; n < NM; ++n) pv(p, n, vf);
    };
    // The first block by itself, which for a short prompt is most of the way: no P.V in its first step, beside which the
    // first values land; scores of a second tile only if there is one; masked only where some query needs it (as any other
    // block, behind zeros as value tile -1 and with tile 1's values waited for at the end: 1 x 33 tokens, 16/4 heads x 128,
    // 6.5 us, here 6.2; 8 x 100, 32/8 x 64, 7.35 and 7.15; 16 x 700 + 500 in a pool, 16/16 x 64, 64 and 61)
    begin_block(0);
    if (__builtin_expect(ga, 0)) {
        m_run = fmaxf(m_run, ma * c);
        m_lim = m_run + kSlack;
    }
    float even = 0.0f;
    if (tiles_w > 1) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < KS; ++n) {
            if (n + KD < KS) kf[n + KD] = k_frag(TILE, n + KD);
            sb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8, kf[n]), __builtin_bit_cast(bf16x8, qf[n]), n == 0 ? zero16 : sb, 0, 0, 0);
#pragma unroll
            for (int l = 0; l < DMA; ++l)
                if (n == l * KS / DMA) dma_k(l, 3, PAGED ? k_at[l] : k_off(l, 0));
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (n == e * KS / 16) prob(e, sa, pa, even, l_run);
            __builtin_amdgcn_sched_barrier(0);
        }
        k_first(2, kf);
        mb = tile_max(1, sb);
        gb = __any(mb * c > m_lim);
    } else {
#pragma unroll
        for (int l = 0; l < DMA; ++l) dma_k(l, 3, PAGED ? k_at[l] : k_off(l, 0));
#pragma unroll
        for (int e = 0; e < 16; ++e) prob(e, sa, pa, even, l_run);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70 | DMA);  // vmcnt(DMA): the values (its key loads are newer)
    __syncthreads();
    if (tiles_w > 1)
        step(std::true_type{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 2>{}, 1, sb, mb, gb, sa, ma, ga, pa, pb, kf);
    else
        last_pv(pa);
    end_block(3);
    int kb = 1;
    for (; kb + 1 < nfast; kb += 2) {  // two blocks: once round the rings, so that every LDS offset is a constant
        block(std::false_type{}, std::integral_constant<int, 2>{}, kb);
        block(std::false_type{}, std::integral_constant<int, 0>{}, kb + 1);
    }
    if (kb < nfast) {
        block(std::false_type{}, std::integral_constant<int, -1>{}, kb);
        ++kb;
    }
    for (; kb < tiles_w / 2; ++kb) block(std::true_type{}, std::integral_constant<int, -1>{}, kb);
    if (tiles_w > 1) {
        if (tiles_w & 1) {  // a last block of one tile, whose values are there already (the next block's loads replace them)
            begin_block(kb);
            step(std::true_type{}, std::integral_constant<int, -1>{}, std::true_type{}, 2 * kb, sa, ma, ga, sb, mb, gb, pb, pa, kf);
            last_pv(pa);
            end_block(2 * kb + 3);
            ++kb;
        } else {
            last_pv(pb);
        }
    }
    for (; kb < nkb; ++kb) {  // keys that only later tokens of the workgroup see
        begin_block(kb);
#pragma unroll
        for (int j = 0; j < DMA; ++j) {
            dma_k(j, 2 * kb + 3, PAGED ? k_at[j] : k_off(j, 0));
            dma_v(j, 2 * kb + 1, PAGED ? v_at[j] : v_off(j, 0));
        }
        end_block(2 * kb + 3);
    }
    if constexpr (WAVES * TILE > RING) __syncthreads();  // some staging areas lie over the values
    // ---- normalise and write [batch, seq, heads*D]: through this wave's part of the
    // (now idle) LDS, so that the 32 x D tile leaves as whole rows
    l_run += __shfl_xor(l_run, 32, kWave);
    // a row that meets no key (empty sequence, more queries than keys, all of them masked) has a sum of zero and
    // yields zeros. A NaN in l_run comes from a score the row sees, and goes out.
    const bool has_value = l_run != 0.0f;
    const float inv = has_value ? 1.0f / l_run : 0.0f;
    // (its accumulators hold zeros times what the value rows held)
    if (!has_value) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] = 0.0f;
    }
    if constexpr (PARTS)
        if (!whole) {
#pragma unroll
            for (int g = 0; g < D / 8; ++g) {
                const f32x16& v = o[g / 4];
                *reinterpret_cast<f32x4_at4*>(part_ws + g * 256 + lane * 4) = f32x4_at4{v[g % 4 * 4], v[g % 4 * 4 + 1], v[g % 4 * 4 + 2], v[g % 4 * 4 + 3]};
            }
            if (h == 0) *reinterpret_cast<f32x2_at4*>(part_ws + 32 * D + 2 * qi) = f32x2_at4{has_value ? m_run : kNegBig, l_run};
            return;
        }
    {
        uint8_t* const mine = lds + wave * TILE;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 w;
                w.x = pack_bf16x2(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv);
                w.y = pack_bf16x2(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
                // row qi, dims 32dt + 8g + 4h ..+3: chunk 4dt+g (XOR-swizzled by row), half h
                *reinterpret_cast<u32x2*>(mine + qi * ROW + (((4 * dt + g) ^ (qi & (LPR - 1))) << 4) + h * 8) = w;
            }
        const int first = row0 + qsub * 32;
        uint16_t* const obase = static_cast<uint16_t*>(a.out) + ((tok0 + first) * a.n_heads + head) * D;
        const int r = lane / LPR, ch = lane & (LPR - 1);
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
            const int row = i * RPI + r;
            const u32x4 v = *reinterpret_cast<const u32x4*>(mine + row * ROW + ((ch ^ (row & (LPR - 1))) << 4));
            if (first + row < rows_total)
                *reinterpret_cast<u32x4*>(obase + (size_t)row * a.n_heads * D + ch * 8) = v;
        }
    }
}

// A wave merges eight dims of the 32 rows that a wave above had. Everything the workspace could hold is requested
// before the schedule is, which says how much of it there is: two memory round trips, not four.
template <int D, int NREP, int QSUB>
__global__ __launch_bounds__(256) void merge_parts_kernel(AttnPrefillArgs a, int64_t waves) {
    constexpr int WAVES = NREP * QSUB, QB = 32 * QSUB, SUBS = 64 / QB;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int64_t idx = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t src = idx / (D / 8);
    const int g = (int)(idx % (D / 8));
    if (src >= waves) return;
    const float* const ws = a.ws + src * a.nsplit * part_floats(D);
    f32x4 x[kMaxParts];
    float pm[kMaxParts], pl[kMaxParts];
#pragma unroll
    for (int j = 0; j < kMaxParts; ++j) {
        pm[j] = kNegBig;
        if (j < a.nsplit) {
            const float* const p = ws + j * part_floats(D);
            x[j] = *reinterpret_cast<const f32x4_at4*>(p + g * 256 + lane * 4);
            const f32x2_at4 ml = *reinterpret_cast<const f32x2_at4*>(p + 32 * D + 2 * (lane & 31));
            pm[j] = ml.x;
            pl[j] = ml.y;
        }
    }
    const int wave = (int)(src % WAVES), hk = (int)(src / WAVES % a.n_kv_heads);
    const int64_t item = src / WAVES / a.n_kv_heads, tile = item / SUBS;
    const int req_i = a.q_tile_to_batch[tile], q_start = a.qo_indptr[req_i];
    const int rows_total = a.qo_indptr[req_i + 1] - q_start;
    const int row0 = a.q_tile_to_index[tile] * 64 + (int)(item % SUBS) * QB, row = row0 + wave / NREP * 32 + (lane & 31);
    const int64_t req = a.req_pool_indices[req_i];
    const int kv_len = req >= 0 && req < a.num_requests ? (int)min((int64_t)(a.kv_indptr[req_i + 1] - a.kv_indptr[req_i]), a.rtt_stride) : 0;
    const int last = min(row0 + QB, rows_total) - 1;
    const int kmax = a.causal ? min(kv_len - rows_total + last, kv_len - 1) : kv_len - 1;
    const int blocks = max(kmax, 0) / kKB + 1, per = part_blocks(a, blocks), parts = (blocks + per - 1) / per;
    if (row >= rows_total || parts == 1) return;  // (the one part wrote the output)
    float m = kNegBig;
#pragma unroll
    for (int j = 0; j < kMaxParts; ++j)
        if (j < parts) m = fmaxf(m, pm[j]);
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    float l = 0.0f;
#pragma unroll
    for (int j = 0; j < kMaxParts; ++j)
        if (j < parts) {
            const float f = __builtin_amdgcn_exp2f(pm[j] - m);
            l += pl[j] * f;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += x[j][i] * f;
        }
    const float inv = l != 0.0f ? 1.0f / l : 0.0f;  // a row with no visible key yields zeros
    const int dim = 8 * g + 4 * h;
    uint16_t* const out = static_cast<uint16_t*>(a.out) + ((int64_t)(q_start + row) * a.n_heads + hk * NREP + wave % NREP) * D + dim;
    *reinterpret_cast<u32x2*>(out) = u32x2{pack_bf16x2(v[0] * inv, v[1] * inv), pack_bf16x2(v[2] * inv, v[3] * inv)};
}

template <int D, int NREP, int QSUB, bool SPLIT>
bool launch_shape(const AttnPrefillArgs& a, hipStream_t stream) {
    // tokens per workgroup: a schedule tile has 64 rows, and the kernel reads the positions of 64
    constexpr int QP = 32 * QSUB <= 64 ? QSUB : 2;
    const bool paged = a.req_to_token != nullptr, narrow = paged || a.positions;
    const int rows = 32 * (narrow ? QP : QSUB);
    const int64_t wgs = paged ? (int64_t)a.num_q_tiles * (64 / rows) * a.n_kv_heads
                              : (int64_t)((a.seq + rows - 1) / rows) * a.batch * a.n_kv_heads;
    if (wgs * std::max(a.nsplit, 1) > INT_MAX) return false;
    const dim3 grid((unsigned)wgs), block(64 * NREP * (narrow ? QP : QSUB));
    if (paged && a.mask) {
        if constexpr (!SPLIT)
            attn_prefill_kernel<D, NREP, QP, true, true, SPLIT><<<grid, block, 0, stream>>>(a);
        else
            return false;
    } else if (paged && a.nsplit > 1) {
        if constexpr (SPLIT) {
            const int64_t waves = wgs * NREP * QP, merges = (waves * (D / 8) + 3) / 4;
            if (merges > INT_MAX) return false;
            attn_prefill_kernel<D, NREP, QP, true, false, SPLIT, true><<<dim3((unsigned)(wgs * a.nsplit)), block, 0, stream>>>(a);
            merge_parts_kernel<D, NREP, QP><<<dim3((unsigned)merges), dim3(256), 0, stream>>>(a, waves);
        } else {
            return false;
        }
    } else if (paged) {
        attn_prefill_kernel<D, NREP, QP, true, false, SPLIT><<<grid, block, 0, stream>>>(a);
    } else if (narrow) {
        attn_prefill_kernel<D, NREP, QP, false, false, SPLIT><<<grid, block, 0, stream>>>(a);
    } else {
        attn_prefill_kernel<D, NREP, QSUB, false, false, SPLIT><<<grid, block, 0, stream>>>(a);
    }
    return true;
}

}  // namespace

bool attn_prefill_supported(int n_heads, int n_kv_heads, int head_dim) {
    if (head_dim != 128 || n_kv_heads <= 0 || n_heads % n_kv_heads) return false;
    const int n_rep = n_heads / n_kv_heads;
    return n_rep == 2 || n_rep == 4 || n_rep == 8;
}

bool attn_prefill_split_supported(int n_heads, int n_kv_heads, int head_dim) {
    if (n_kv_heads <= 0 || n_heads % n_kv_heads) return false;
    const int n_rep = n_heads / n_kv_heads;
    return head_dim == 64 ? n_rep == 1 || n_rep == 2 || n_rep == 4 || n_rep == 8 : head_dim == 128 && n_rep == 1;
}

bool attn_prefill_pool_ok(int64_t num_slots, int n_kv_heads, int head_dim) {
    return num_slots <= (int64_t)kMissing / (2 * (int64_t)n_kv_heads * head_dim);
}

int attn_prefill_parts(int64_t tiles, int n_heads, int64_t max_keys, int nsplit) {
    const int64_t pairs = tiles * n_heads;
    if (nsplit <= 1 || pairs >= kMaxPartPairs) return 1;
    const int blocks = (int)((max_keys + kKB - 1) / kKB), n = part_count(blocks, pairs, std::min(nsplit, kMaxParts));
    const int64_t cost = 2 * n * pairs / kPairsPerBlock + kMergeBlocks;
    return blocks - (blocks + n - 1) / n >= cost ? n : 1;
}

bool launch_attn_prefill(const AttnPrefillArgs& a, hipStream_t stream) {
    if (a.nsplit > 1 && (a.nsplit > kMaxParts || !a.ws || a.mask || !a.req_to_token)) return false;
    const bool split = attn_prefill_split_supported(a.n_heads, a.n_kv_heads, a.head_dim);
    if (!split && !attn_prefill_supported(a.n_heads, a.n_kv_heads, a.head_dim)) return false;
    const bool paged = a.req_to_token != nullptr;
    if (a.mask && (!paged || a.mask_width <= 0 || a.mask_rows <= 0)) return false;
    const int n_rep = a.n_heads / a.n_kv_heads;
    if (paged) {
        if (!a.req_pool_indices || !a.kv_indptr || !a.qo_indptr || !a.q_tile_to_batch || !a.q_tile_to_index ||
            a.num_q_tiles <= 0 || a.rtt_stride <= 0 || a.num_slots <= 0 || a.num_requests <= 0)
            return false;
        if (!attn_prefill_pool_ok(a.num_slots, a.n_kv_heads, a.head_dim)) return false;
    } else {
        if (a.batch <= 0 || a.seq <= 0 || a.max_len <= 0) return false;
        if (a.max_len * std::max(a.k_stride.row, a.v_stride.row) * 2 > (int64_t)kMissing) return false;  // 32-bit offsets
    }
    if (a.head_dim == 64) {
        if (n_rep == 1) return launch_shape<64, 1, 4, true>(a, stream);
        if (n_rep == 2) return launch_shape<64, 2, 2, true>(a, stream);
        if (n_rep == 4) return launch_shape<64, 4, 1, true>(a, stream);
        return launch_shape<64, 8, 1, true>(a, stream);
    }
    if (n_rep == 1) return launch_shape<128, 1, 4, true>(a, stream);
    if (n_rep == 2) return launch_shape<128, 2, 2, false>(a, stream);
    if (n_rep == 4) return launch_shape<128, 4, 1, false>(a, stream);
    return launch_shape<128, 8, 1, false>(a, stream);
}

}  // namespace w8a8
