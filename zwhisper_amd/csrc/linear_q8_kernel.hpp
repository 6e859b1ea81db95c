// Linear layers over int8 block weights on gfx950 MFMA: ops.linear with a gemm.Q8
// (src/ops.zig:283-306, src/gemm.zig:188-351).  q int8 [n][k], scales f32 [n][k / 32]:
//
//     out[i][o] = sum_b scales[o][b] * (sum_{p in block b} x[i][p] * q[o][p])  (+ bias[o])
//
// with blocks of 32 along k, each block's partial dot product scaled once (gemm.dotQ,
// src/gemm.zig:274-286, and micro4x4Q, :289-327, do the same per vector lane).
//
// Precision.  An int8 weight is exact in f16.  Each f32 activation is split into two f16 terms,
// x = hi + lo (hi = f16(x), lo = f16(x - hi)), which keep 22 of x's 24 significand bits; a
// block's two MFMAs per term accumulate hi*q and lo*q in f32, and the block sum is scaled in f32
// on the VALU.  |x| must stay within f16's range (65504).
//
// Three families of kernels (linear.hip chooses):
//
// * linear_q8p_short_kernel, linear_q8p_long_kernel: resident weights in the packed layout (Q8Packed),
//   token steps, logits, prompt batches of up to 256 rows and the longer calls that they win.  32- or
//   64-row blocks; each stage of x sits in LDS split into hi/lo halves in the MFMA A-operand order, and
//   every wave streams its own slabs of 32 weight rows into registers.
//
// * linear_q8_stream_kernel<MT, S>: weights as the caller has them (int8 [n][k]), m <= 64.  The
//   weights are the stream: every int8 byte is read from HBM once, 16 bytes per lane per load (one Q8
//   block of 32 weight rows per wave-load).  A workgroup of 4 waves owns 4*S slabs of 32 weight
//   rows and walks k in chunks of 256 (8 blocks).  x is split into hi/lo halves once per call by
//   linear_q8_xprep_kernel, in the exact order the MFMA A operand wants it; each workgroup copies
//   a chunk of it into LDS with direct global-to-LDS loads (no VGPRs, no VALU), issued before the
//   chunk's weight loads so the wait for x never waits on the weights.  An operand read is then
//   1 KB contiguous per wave (conflict-free ds_read_b128).
//
// * linear_mfma_kernel<BM, BN, kWQ8 or kWQ8P> (linear_kernel.hpp): the remaining calls of more rows, the
//   tiled GEMM with the weight tile widened to f16 on its way into LDS and the same per-block scaling.
//
// The first two use v_mfma_f32_32x32x16_f16 with A = x rows, B = weight rows: lane l's 16 weight bytes
// q[row l%32][kb + 16 (l/32) .. +16] feed the block's two k-steps (bytes 0-7, then 8-15), and
// the result column l%32 is the weight row, so the block's scale is one f32 per lane.  When the
// weight rows alone give too few workgroups to fill the chip, k is split over gridDim.y and a
// split-sum kernel adds the partial sums in a fixed order.
//
// MFMA operand layout (v_mfma_f32_32x32x16_f16, measured on the device): lane l, half s of A is
// A[l % 32][8 (l / 32) + s], of B is B[8 (l / 32) + s][l % 32]; result register r of lane l is
// C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "linear_kernel.hpp"

namespace zwg_lin {

constexpr int kQ8Block = 32;                // src/gemm.zig:194
constexpr int kQ8Chunk = 256;               // k per chunk: of the packed layout, the split x and the stream kernel's LDS
constexpr int kQ8ChunkBlocks = kQ8Chunk / kQ8Block;
constexpr int kQ8Threads = 256;
// Cache policy nt: packed weights that one row block reads once stream past the caches, which keep the
// x stages that every workgroup reuses (Q8pTile::POLICY).
constexpr int kQ8CachePolicyNT = 2;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding: vmcnt in bits 3:0 and 15:14,
// expcnt 6:4 and lgkmcnt 11:8 left at their maxima).
__host__ __device__ constexpr int q8_vmcnt(int n) {
    return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8);
}

struct Q8Args {
    const float *x;      // [m][k]
    const int8_t *q;     // [n][k]
    const float *scales; // [n][nb]
    const float *bias;   // [n] or nullptr
    float *out;          // [m][n]
    float *part;         // [n_split][m][n] when n_split > 1
    int32_t m, n, k, nb;
    int32_t chunks_per_split, n_split;
    uint32_t epi; // zwg_ew::kEpi*, applied where `out` is written (here, or by the split sum)
};

// Layout of x's hi/lo halves, per chunk of 256 k: [block][m-tile][hi/lo][k-step][lane][8 halves],
// 32 KB per m-tile.  Lane l, k-step s of (block b, m-tile i) holds x[32 i + l % 32][kb + 16 (l / 32)
// + 8 s + 0..7], kb = 32 b.  One [hi/lo][k-step] piece of a (block, m-tile) is 1 KB: 64 lanes x 16 B,
// lane l at place l ^ 4 s: a write of four consecutive k of each row touches both k-steps, which
// then sit on different banks.
template <int MT>
__host__ __device__ constexpr int q8_chunk_halves() {
    return kQ8ChunkBlocks * MT * 2 * 2 * 64 * 8;
}
template <int MT>
__device__ __forceinline__ int q8_xs_at(int b, int i, int hl, int s, int lane) {
    return ((((b * MT + i) * 2 + hl) * 2 + s) * 64 + (lane ^ (4 * s))) * 8;
}

// x[row][gk .. gk + 3] (gk % 4 == 0) split into f16 hi/lo halves at its place in xcvt's chunk
// layout above: hi = f16(v), lo = f16(v - hi)
template <int MT>
__device__ __forceinline__ void q8_xs_store(_Float16 *xcvt, int row, int gk, f32x4 v) {
    const int c = gk / kQ8Chunk, kk = gk % kQ8Chunk;
    const int b = kk >> 5, kb = kk & 31;
    const int gg = kb >> 4, s = (kb >> 3) & 1, j = kb & 7;
    const int i = row >> 5, l = (row & 31) + 32 * gg;
    half4 hi, lo;
    zwg_split::split4(v, hi, lo);
    _Float16 *base = xcvt + (int64_t)c * q8_chunk_halves<MT>();
    *reinterpret_cast<half4 *>(base + q8_xs_at<MT>(b, i, 0, s, l) + j) = hi;
    *reinterpret_cast<half4 *>(base + q8_xs_at<MT>(b, i, 1, s, l) + j) = lo;
}

// One element of such a row: v at x[row][gk]
template <int MT>
__device__ __forceinline__ void q8_xs_store1(_Float16 *xcvt, int row, int gk, float v) {
    const int c = gk / kQ8Chunk, b = gk % kQ8Chunk >> 5, kb = gk & 31;
    const int s = (kb >> 3) & 1, j = kb & 7, i = row >> 5, l = (row & 31) + 32 * (kb >> 4);
    _Float16 *base = xcvt + (int64_t)c * q8_chunk_halves<MT>();
    const _Float16 hi = (_Float16)v;
    base[q8_xs_at<MT>(b, i, 0, s, l) + j] = hi;
    base[q8_xs_at<MT>(b, i, 1, s, l) + j] = (_Float16)(v - (float)hi);
}

// x f32 [m][k] -> xcvt f16 [blocks of 32 MT rows][n_chunks][chunk layout above]; rows >= m and columns
// >= k are 0.  One thread per 4 consecutive k of one row.
template <int MT>
__global__ __launch_bounds__(256) void linear_q8_xprep_kernel(const float *x, _Float16 *xcvt, int32_t m, int32_t k,
                                                             int32_t n_chunks) {
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int per_chunk = MT * 32 * (kQ8Chunk / 4);
    const int64_t zc = f / per_chunk; // row block z, chunk c
    const int rem = (int)(f % per_chunk);
    const int z = (int)(zc / n_chunks), c = (int)(zc % n_chunks);
    const int row = rem / (kQ8Chunk / 4), gk = c * kQ8Chunk + 4 * (rem % (kQ8Chunk / 4));
    const int64_t r = (int64_t)z * MT * 32 + row;
    if (z * MT * 32 >= m) return;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (r < m && gk < k) v = *reinterpret_cast<const f32x4 *>(x + r * k + gk);
    q8_xs_store<MT>(xcvt + (int64_t)z * n_chunks * q8_chunk_halves<MT>(), row, gk, v);
}

template <int MT, int S>
__global__ __launch_bounds__(kQ8Threads) void linear_q8_stream_kernel(Q8Args a, const _Float16 *xcvt) {
    constexpr int NB = kQ8ChunkBlocks;
    constexpr int ROWS = 4 * S * 32;                   // weight rows per workgroup
    constexpr int PIECES = q8_chunk_halves<MT>() / 512; // 1 KB pieces of an x chunk
    constexpr int XL = PIECES / 4;                      // pieces each wave copies
    __shared__ __align__(16) _Float16 xs[q8_chunk_halves<MT>()];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r32 = lane & 31, g = lane >> 5;
    const int n0 = blockIdx.x * ROWS;
    const int wrow0 = wave * S * 32; // this wave's first row within the workgroup's slab group
    const int split = blockIdx.y;
    const int n_chunks = (a.k + kQ8Chunk - 1) / kQ8Chunk;
    const int c_begin = split * a.chunks_per_split;
    const int c_end = min(c_begin + a.chunks_per_split, n_chunks);

    // q / scales: rows past n read as 0.  x_src: the call's prepared x chunks.
    const __amdgpu_buffer_rsrc_t x_src = rsrc(xcvt, (uint32_t)n_chunks * (uint32_t)PIECES * 1024u);
    const int rows_w = min(ROWS, a.n - n0);
    const __amdgpu_buffer_rsrc_t q_src = rsrc(a.q + (int64_t)n0 * a.k, (uint32_t)((int64_t)rows_w * a.k));
    const __amdgpu_buffer_rsrc_t s_src = rsrc(a.scales + (int64_t)n0 * a.nb, (uint32_t)((int64_t)rows_w * a.nb * 4));
    uint32_t qbase[S], sbase[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int row = wrow0 + s * 32 + r32;
        qbase[s] = (uint32_t)(row * a.k + 16 * g);
        sbase[s] = (uint32_t)(row * a.nb) * 4u;
    }

    f32x16 acc[MT][S];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[i][s] = (f32x16){0};

    for (int c = c_begin; c < c_end; ++c) {
        const int k0 = c * kQ8Chunk;
        __syncthreads(); // the previous chunk's operand reads are done
        // x chunk into LDS: wave w copies pieces w, w + 4, ...; lane l's 16 bytes land at l * 16
#pragma unroll
        for (int u = 0; u < XL; ++u) {
            const int piece = wave + 4 * u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(x_src, (__attribute__((address_space(3))) void *)(xs + piece * 512), 16,
                                                 (uint32_t)((c * PIECES + piece) * 1024 + lane * 16), 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // This wave's weights for the chunk (slab s, block b: 16 bytes per lane) and the blocks'
        // scales.  A block past k gets scale 0 (its offset is out of range), so whatever the
        // weight load returned there adds exactly nothing.
        u32x4 wq[S][NB];
        float sc[S][NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int kb = k0 + b * kQ8Block;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                wq[s][b] = __builtin_bit_cast(
                    u32x4, __builtin_amdgcn_raw_buffer_load_b128(q_src, (int)(qbase[s] + (uint32_t)kb), 0, 0));
                const uint32_t soff = kb < a.k ? sbase[s] + (uint32_t)(kb / kQ8Block) * 4u : kOutOfRange;
                sc[s][b] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s_src, (int)soff, 0, 0));
            }
        }
        // wait for this wave's x pieces only (loads complete in order; the 2 S NB weight and
        // scale loads were issued after them), then for every wave's
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(q8_vmcnt(2 * S * NB));
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);

#pragma unroll
        for (int b = 0; b < NB; ++b) {
            half8 ah[MT][2], al[MT][2];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    ah[i][s] = *reinterpret_cast<const half8 *>(&xs[q8_xs_at<MT>(b, i, 0, s, lane)]);
                    al[i][s] = *reinterpret_cast<const half8 *>(&xs[q8_xs_at<MT>(b, i, 1, s, lane)]);
                }
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const half8 w0 = int8x8_to_half8(wq[s][b][0], wq[s][b][1]);
                const half8 w1 = int8x8_to_half8(wq[s][b][2], wq[s][b][3]);
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    f32x16 t = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i][0], w0, (f32x16){0}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i][0], w0, t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i][1], w1, t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i][1], w1, t, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][s][r] = __builtin_fmaf(t[r], sc[s][b], acc[i][s][r]);
                }
            }
        }
    }

    // register r of lane l: row 32 i + 8 (r / 4) + 4 (l / 32) + r % 4, column (weight row) l % 32
    float *dst = a.n_split > 1 ? a.part + (int64_t)split * a.m * a.n : a.out;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int col = n0 + wrow0 + s * 32 + r32;
        if (col >= a.n) continue;
        const float bj = (a.n_split == 1 && a.bias) ? a.bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row < a.m) {
                    if (a.n_split > 1) dst[(int64_t)row * a.n + col] = acc[i][s][r];
                    else zwg_ew::epilogue_store(&dst[(int64_t)row * a.n + col], acc[i][s][r] + bj, a.epi);
                }
            }
    }
}

// Packed device weights (zwg_q8w): the same int8 and scales, laid out for the packed kernels so
// that every wave-load is contiguous.  n is padded to whole slabs of 32 rows, k to whole chunks
// of 256 (8 blocks); padding is zero (scale 0).
//   q:      [slab][block][lane][16 bytes], lane l of (slab s, block b) holding
//           q[32 s + l % 32][32 b + 16 (l / 32) .. +16]: one 1 KB tile per (slab, block).
//   scales: [slab][chunk][32 rows][8 blocks] f32: a lane's 8 block scales of a chunk are 32
//           contiguous bytes, and the 32 rows of a slab 1 KB.
struct Q8Packed {
    const uint8_t *q;
    const float *scales;
    int32_t n_slabs, n_chunks;
};

// Weight sets of one token-step launch over the same x (a decode step's q/k/v, or gate/up): set j
// takes workgroups block_start[j] .. block_start[j + 1] - 1 of the packed kernel and elements
// elem_start[j] .. elem_start[j + 1] - 1 of the split sum; all sets share x, k and the k split.
constexpr int kQ8MaxGroup = 4;
struct Q8Group {
    int32_t count;
    int32_t n_chunks; // k / 256, rounded up: the same for every set
    int32_t block_start[kQ8MaxGroup + 1];
    int64_t elem_start[kQ8MaxGroup + 1];
    const uint8_t *q[kQ8MaxGroup]; // packed weights of set j (Q8Packed)
    const float *scales[kQ8MaxGroup];
    int32_t n_slabs[kQ8MaxGroup];
    int32_t n[kQ8MaxGroup];
    const float *bias[kQ8MaxGroup];
    float *out[kQ8MaxGroup];
    float *part[kQ8MaxGroup]; // [n_split][m][n[j]] when the call is split
    // 1: a SwiGLU pair (count 2, n[0] == n[1]: the MLP's gate and up, src/llm.zig:207-210): each
    // workgroup takes the same columns of both sets and the call stores silu(gate) * up into
    // out[0] (Q8pTile::store; split calls through linear_split_sum_swiglu_kernel)
    int32_t swiglu;
    // a SwiGLU pair of more than 32 rows: nullptr, or silu(gate) * up goes here split into f16 hi/lo
    // halves for the next 64-row-block call (linear_q8_xprep_kernel's layout; n % 128 == 0, so every
    // column its stages read is written) instead of into out[0]
    _Float16 *xcvt_out;
};

// entry j of a group field, by selects on the uniform j (no dynamic indexing of the kernel-
// argument struct, which would go through scratch)
template <typename T, int N>
__device__ __forceinline__ T q8_pick(const T (&v)[N], int j) {
    T r = v[0];
#pragma unroll
    for (int i = 1; i < N; ++i) r = j == i ? v[i] : r;
    return r;
}
__device__ __forceinline__ int q8_group_of_block(const Q8Group &g, int bx) {
    int j = 0;
#pragma unroll
    for (int i = 1; i < kQ8MaxGroup; ++i) j += (i < g.count && bx >= g.block_start[i]) ? 1 : 0;
    return j;
}
__device__ __forceinline__ int q8_group_of_elem(const Q8Group &g, int64_t e) {
    int j = 0;
#pragma unroll
    for (int i = 1; i < kQ8MaxGroup; ++i) j += (i < g.count && e >= g.elem_start[i]) ? 1 : 0;
    return j;
}

__host__ __device__ inline int64_t q8p_q_bytes(int64_t n_slabs, int64_t n_chunks) {
    return n_slabs * n_chunks * kQ8ChunkBlocks * 1024;
}
__host__ __device__ inline int64_t q8p_scale_bytes(int64_t n_slabs, int64_t n_chunks) {
    return n_slabs * n_chunks * 32 * kQ8ChunkBlocks * 4;
}

// Pack q [n][k] (int8) and scales [n][k / 32] into the layout above: one thread per 16-byte
// piece of a q tile (and, for the first 8 lanes of a slab's chunk, nothing else); scales by a
// second grid-stride pass in the same kernel.
__global__ __launch_bounds__(256) void linear_q8_pack_kernel(const int8_t *q, const float *scales, int32_t n,
                                                            int32_t k, uint8_t *pq, float *ps, int32_t n_slabs,
                                                            int32_t n_chunks) {
    const int32_t nb = k / kQ8Block, nbp = n_chunks * kQ8ChunkBlocks;
    const int64_t pieces = (int64_t)n_slabs * nbp * 64;
    const int64_t sc_elems = (int64_t)n_slabs * n_chunks * 32 * kQ8ChunkBlocks;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t f = (int64_t)blockIdx.x * 256 + threadIdx.x; f < pieces; f += stride) {
        const int lane = (int)(f & 63);
        const int64_t tile = f >> 6;
        const int b = (int)(tile % nbp);
        const int64_t slab = tile / nbp;
        const int64_t row = slab * 32 + (lane & 31);
        const int kk = b * kQ8Block + 16 * (lane >> 5);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (row < n && kk < k) v = *reinterpret_cast<const u32x4 *>(q + row * k + kk);
        *reinterpret_cast<u32x4 *>(pq + f * 16) = v;
    }
    for (int64_t f = (int64_t)blockIdx.x * 256 + threadIdx.x; f < sc_elems; f += stride) {
        const int b8 = (int)(f & 7);
        const int r = (int)((f >> 3) & 31);
        const int64_t sc_chunk = f >> 8; // slab * n_chunks + chunk
        const int c = (int)(sc_chunk % n_chunks);
        const int64_t slab = sc_chunk / n_chunks;
        const int64_t row = slab * 32 + r;
        const int b = c * kQ8ChunkBlocks + b8;
        ps[f] = (row < n && b < nb) ? scales[row * nb + b] : 0.f;
    }
}

// The packed-weight kernels: a workgroup of NS x MS x KB waves computes 32 MT rows x 32 NS columns
// (weight rows); wave (ws, ms, kg) takes slab ws, m-tiles ms MT / MS .. of it and blocks
// kg SB / KB .. of every stage.  k is walked in stages of SB blocks.  x stages sit in LDS in the MFMA
// A-operand order (q8_xs_at) and are shared by the waves; a wave's weights and scales go to its own
// registers.  Each block's sum starts from zero (four MFMAs) and is scaled into the accumulator in
// block order, so every tile shape with KB = 1 gives the same bits; with KB = 2 the two waves' sums
// are added at the end.
//
// Loads run ahead of their use.  Past the last stage the same loads go out with out-of-range
// offsets: they return zeros without touching memory, and every path through a loop then has the
// same loads in flight, so the compiler's in-order wait counts stay exact.  Two x paths:
//   XS = false: x was split into f16 hi/lo halves in the MFMA A-operand order by
//     linear_q8_xprep_kernel (or the previous call's row kernel); each stage's pieces are copied into
//     LDS by direct global-to-LDS loads (no VGPRs, no VALU).
//   XS = true: no separate pass.  A stage's f32 x rows arrive in registers and the workgroup splits
//     them into the LDS stage itself.  A wave's load takes 16 rows x 64 bytes (four lanes per row:
//     full 64-byte requests), which its LDS writes then scatter without bank conflicts; with one
//     load per 512 contiguous bytes of two rows, 16 lanes of every write met on the same banks
//     (0.9 us of a 2.2 us stage).
// Padding blocks (k is padded to 256) have scale 0 and x 0; a stage wholly past k is not run.
//
// Stores.  The accumulators go through LDS (rows of 36 floats per wave, the x buffers' space) so
// that a lane stores 16 bytes: 4-byte stores cost the same address cycles each, four times as many
// (1.9 -> 0.5 us at the end of a 64 x 128 tile).
//
// PAIR: a SwiGLU pair (Q8Group swiglu), a form of its own so the other calls carry none of it: the
// first NS / 2 slabs are the gate's, the others the up's over the same columns.
// GRP = false: one weight set (set 0), without the choice of a set.
constexpr int kQ8OutLd = 36; // floats per row of a wave's 32-column output tile in LDS (16-byte rows, spread banks)

template <int MT, int NS, int MS, int KB, int SB, bool XS, bool PAIR, bool GRP>
struct Q8pTile {
    static constexpr int NW = NS * MS * KB;           // waves
    static constexpr int NB = SB / KB;                // blocks of a stage per wave
    static constexpr int WT = MT / MS;                // m-tiles per wave
    static constexpr int K = SB * kQ8Block;           // k per stage
    static constexpr int SPC = kQ8Chunk / K;          // stages per chunk
    static constexpr int PIECES = SB * MT * 4;        // 1 KB pieces of an x stage
    static constexpr int XL = PIECES / NW;            // pieces each wave copies (XS = false)
    static constexpr int STAGE_HALVES = PIECES * 512; // one x stage in LDS
    // XS: the x stage's quads go to the waves by groups of 16 rows (RG of them) x 16 k; CW waves
    // share a row group's 2 SB column groups
    static constexpr int RG = 2 * MT, CW = NW / RG;
    static constexpr int XQ = XS ? 2 * SB / CW : 1;
    static_assert(PIECES % NW == 0 && NW % RG == 0 && (2 * SB) % CW == 0 && MT % MS == 0, "x stage divides among the waves");
    static constexpr int OT = WT * 32 * kQ8OutLd; // floats of one wave's output tile
    static constexpr int OUT_BYTES = NW * OT * 4;
    static constexpr int HS = NS / 2;
    static constexpr int OS = PAIR ? HS : NS;   // output slabs
    static constexpr int PW = OS * MT * 4 / NW; // pieces of 8 rows x 32 columns each wave stores
    static constexpr int WPS = NW / OS;         // waves per output slab
    static_assert(PW >= 1 && WPS * OS == NW && PW * WPS == MT * 4, "whole pieces per wave, one slab each");
    static constexpr int NP = PAIR ? 2 : 1;
    // the packed weights are streamed past the caches when nothing reads them again (32-row calls);
    // a 64-row call's row blocks do, and its loads run at twice the rate per CU without the policy
    // (a 1001 x 1536 x 8960 call 85 -> 71 us, the 64-row logits of 151936 rows 82 -> 79 us; the
    // one-row logits 31 us with it, 33 without)
    static constexpr int POLICY = MT == 1 ? kQ8CachePolicyNT : 0;

    struct Scales {
        float s[NB];
    };

    int lane, wave, ws, ms, kg, set, bx, slab, r0, m, m_all, n, k, split, n_split, t_begin, t_end;
    uint32_t epi;
    __amdgpu_buffer_rsrc_t x_src, q_src, s_src;
    int x_r, x_p, x_g0;
    uint32_t x_lane, w_lane, s_lane;
    int o_s, o_r, o_c, col;
    f32x4 bv[NP];

    __device__ __forceinline__ Q8pTile(const Q8Args &a, const Q8Group &grp, const _Float16 *xcvt) {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); // uniform: the LDS DMA base is per wave
        ws = wave % NS;
        ms = wave / NS % MS;
        kg = wave / (NS * MS);
        constexpr bool pick = PAIR || GRP;
        set = PAIR ? (ws >= HS ? 1 : 0) : GRP ? q8_group_of_block(grp, (int)blockIdx.x) : 0;
        bx = (int)blockIdx.x - (PAIR || !GRP ? 0 : q8_pick(grp.block_start, set));
        const uint8_t *q = pick ? q8_pick(grp.q, set) : grp.q[0];
        const float *scales = pick ? q8_pick(grp.scales, set) : grp.scales[0];
        const int n_slabs = pick ? q8_pick(grp.n_slabs, set) : grp.n_slabs[0];
        n = pick ? q8_pick(grp.n, set) : grp.n[0];
        k = a.k;
        epi = a.epi;
        // a call of more rows than one x stage holds runs gridDim.z blocks of 32 MT rows: block z
        // takes rows r0 = 32 MT z .. of x and of the outputs; the partial sums keep the whole
        // call's [split][m][n] layout
        m_all = a.m;
        r0 = (int)blockIdx.z * MT * 32;
        m = min(MT * 32, m_all - r0);
        slab = bx * (PAIR ? HS : NS) + (PAIR ? ws - set * HS : ws); // this wave's slab
        split = blockIdx.y;
        n_split = a.n_split;
        const int n_stages = (a.k + K - 1) / K;
        t_begin = split * a.chunks_per_split * SPC;
        t_end = min(t_begin + a.chunks_per_split * SPC, n_stages); // at least one stage
        // XS: x [m][k] f32, rows past m read as 0 (range), columns past k get an out-of-range offset;
        // otherwise this row block's split x chunks
        const uint32_t xc_bytes = (uint32_t)grp.n_chunks * (uint32_t)(SPC * PIECES) * 1024u;
        x_src = XS ? rsrc(a.x + (int64_t)r0 * a.k, (uint32_t)m * (uint32_t)a.k * 4u)
                   : rsrc(reinterpret_cast<const char *>(xcvt) + (int64_t)blockIdx.z * xc_bytes, xc_bytes);
        // a slab past the matrix (in the last workgroup) reads as 0
        const bool live = slab < n_slabs;
        const uint32_t slab_q = (uint32_t)grp.n_chunks * kQ8ChunkBlocks * 1024u;
        const uint32_t slab_s = (uint32_t)grp.n_chunks * 32u * kQ8ChunkBlocks * 4u;
        q_src = rsrc(q + (live ? (int64_t)slab * slab_q : 0), live ? slab_q : 0u);
        s_src = rsrc(reinterpret_cast<const char *>(scales) + (live ? (int64_t)slab * slab_s : 0), live ? slab_s : 0u);
        // XS: quad e of this thread in a stage is row x_r, k 16 (x_g0 + e) + 4 x_p of the stage.  The
        // per-lane part of the offset is one VGPR, the stage's k goes in the scalar offset
        x_r = 16 * (wave % RG) + (lane >> 2);
        x_p = lane & 3;
        x_g0 = wave / RG * XQ;
        x_lane = ((uint32_t)x_r * (uint32_t)a.k + 4u * (uint32_t)x_p) * 4u;
        w_lane = (uint32_t)lane * 16u;
        s_lane = (uint32_t)(lane & 31) * (kQ8ChunkBlocks * 4u);
        // the output pieces of this wave: slab o_s, rows o_r + 8 p, this lane's four columns and their bias
        o_s = wave / WPS;
        o_r = (wave % WPS) * PW * 8 + (lane >> 3);
        o_c = 4 * (lane & 7);
        col = (bx * OS + o_s) * 32 + o_c;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const float *bias = a.n_split > 1 ? nullptr : PAIR ? grp.bias[j] : GRP ? q8_pick(grp.bias, set) : grp.bias[0];
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[j][e] = bias && col + e < n ? bias[col + e] : 0.f;
        }
    }

    // the loads of stage t: x quad e (XS) or this wave's pieces into an LDS buffer, this wave's block
    // b of its slab, and the stage's scales of this lane's row.  A load past the last stage has its
    // lane offset out of range (and scalar offset 0: the range check is against the size less that)
    static __device__ __forceinline__ int lane_at(bool in, uint32_t at) { return (int)(in ? at : kOutOfRange); }
    static __device__ __forceinline__ int scalar_at(bool in, uint32_t at) { return (int)(in ? at : 0u); }
    __device__ __forceinline__ f32x4 load_x(int t, int e) const {
        const int at = t * K + 16 * (x_g0 + e); // whole column groups: k % 32 == 0
        const bool in = t < t_end && at < k;
        return __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(x_src, lane_at(in, x_lane), scalar_at(in, (uint32_t)at * 4u), 0));
    }
    // (the copies are waited for by the count of the loads after them, so none of those may move up)
    __device__ __forceinline__ void dma_x(int t, _Float16 *buf) const {
        const bool in = t < t_end;
#pragma unroll
        for (int u = 0; u < XL; ++u) {
            const int piece = wave + NW * u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(x_src, (__attribute__((address_space(3))) void *)(buf + piece * 512), 16,
                                                     lane_at(in, w_lane), scalar_at(in, (uint32_t)((t * PIECES + piece) * 1024)),
                                                     0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ u32x4 load_w(int t, int b) const {
        const bool in = t < t_end;
        const uint32_t at = (uint32_t)(t * SB + kg * NB + b) * 1024u;
        return __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(q_src, lane_at(in, w_lane), scalar_at(in, at), POLICY));
    }
    __device__ __forceinline__ Scales load_s(int t) const {
        const bool in = t < t_end;
        const uint32_t at = (uint32_t)(t / SPC) * (32u * kQ8ChunkBlocks * 4u) + 4u * (uint32_t)(t % SPC * SB + kg * NB);
        const int lo = lane_at(in, s_lane), so = scalar_at(in, at);
        if constexpr (NB == 4)
            return __builtin_bit_cast(Scales, __builtin_amdgcn_raw_buffer_load_b128(s_src, lo, so, POLICY));
        else if constexpr (NB == 2)
            return __builtin_bit_cast(Scales, __builtin_amdgcn_raw_buffer_load_b64(s_src, lo, so, POLICY));
        else
            return __builtin_bit_cast(Scales, __builtin_amdgcn_raw_buffer_load_b32(s_src, lo, so, POLICY));
    }
    // XS: quad e split into an LDS buffer (a quad is half of one lane's 8-element piece)
    __device__ __forceinline__ void put_x(_Float16 *buf, int e, const f32x4 &v) const {
        half4 hi, lo;
        zwg_split::split4(v, hi, lo);
        const int cg = x_g0 + e, l = (x_r & 31) + 32 * (cg & 1), i = x_r >> 5, s = x_p >> 1, j = 4 * (x_p & 1);
        *reinterpret_cast<half4 *>(buf + q8_xs_at<MT>(cg >> 1, i, 0, s, l) + j) = hi;
        *reinterpret_cast<half4 *>(buf + q8_xs_at<MT>(cg >> 1, i, 1, s, l) + j) = lo;
    }
    // x operands of (this wave's block b, its m-tile i): hi and lo of k-step 0, hi and lo of k-step 1
    __device__ __forceinline__ void read_a(half8 (&A)[4], const _Float16 *buf, int b, int i) const {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int hl = 0; hl < 2; ++hl)
                A[2 * s + hl] = *reinterpret_cast<const half8 *>(buf + q8_xs_at<MT>(kg * NB + b, ms * WT + i, hl, s, lane));
    }

    // The stores, through the output tiles in `lds` (which every wave is done with): the bias, then
    // the partial sums, or the epilogue and the output
    __device__ __forceinline__ void store(const f32x16 (&acc)[WT], float *lds, const Q8Group &grp) const {
        const int r32 = lane & 31, g = lane >> 5;
        float *tile = lds + wave * OT;
        // register r of lane l: row 32 i + 8 (r / 4) + 4 (l / 32) + r % 4, column (weight row) l % 32
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) tile[(32 * i + 8 * (r >> 2) + 4 * g + (r & 3)) * kQ8OutLd + r32] = acc[i][r];
        __syncthreads();
        if (col >= n) return;
        f32x4 v[NP][PW];
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int p = 0; p < PW; ++p) {
                const int row = o_r + 8 * p;
                const float *at = lds + (o_s + j * HS + row / (32 * WT) * NS) * OT + row % (32 * WT) * kQ8OutLd + o_c;
                f32x4 q = *reinterpret_cast<const f32x4 *>(at);
#pragma unroll
                for (int g2 = 1; g2 < KB; ++g2) q += *reinterpret_cast<const f32x4 *>(at + g2 * NS * MS * OT);
                v[j][p] = q + bv[j];
            }
        bool vec = n % 4 == 0; // rows 16-byte aligned (outputs start so; a group's partial sums may not)
        auto put = [&](float *o, f32x4 q) {
            if (vec) *reinterpret_cast<f32x4 *>(o) = q;
            else
                for (int e = 0; e < 4 && col + e < n; ++e) o[e] = q[e];
        };
        const int64_t o_at = (int64_t)(r0 + o_r) * n + col;
        if (n_split > 1) {
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                float *part = (PAIR ? grp.part[j] : GRP ? q8_pick(grp.part, set) : grp.part[0]) + (int64_t)split * m_all * n + o_at;
                vec = n % 4 == 0 && (reinterpret_cast<uintptr_t>(part) & 15) == 0;
#pragma unroll
                for (int p = 0; p < PW; ++p)
                    if (o_r + 8 * p < m) put(part + (int64_t)8 * p * n, v[j][p]);
            }
            return;
        }
        float *o = (GRP && !PAIR ? q8_pick(grp.out, set) : grp.out[0]) + o_at;
        if constexpr (PAIR) {
#pragma unroll
            for (int p = 0; p < PW; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[0][p][e] = zwg_ew::silu_mul(v[0][p][e], v[1][p][e]);
            if (MT == 2 && grp.xcvt_out) { // (split from the rounded product: the asm keeps the two apart)
                _Float16 *xc = grp.xcvt_out + (int64_t)blockIdx.z * ((n + kQ8Chunk - 1) / kQ8Chunk) * q8_chunk_halves<2>();
#pragma unroll
                for (int p = 0; p < PW; ++p) {
                    asm volatile("" : "+v"(v[0][p]));
                    if (o_r + 8 * p < m) q8_xs_store<2>(xc, o_r + 8 * p, col, v[0][p]);
                }
                return;
            }
        } else if (epi == zwg_ew::kEpiAdd) { // every residual load before the first store
            f32x4 res[PW];
#pragma unroll
            for (int p = 0; p < PW; ++p) {
                const float *op = o + (int64_t)8 * p * n;
                if (o_r + 8 * p >= m) continue;
                if (vec) res[p] = *reinterpret_cast<const f32x4 *>(op);
                else
                    for (int e = 0; e < 4; ++e) res[p][e] = col + e < n ? op[e] : 0.f;
            }
#pragma unroll
            for (int p = 0; p < PW; ++p) v[0][p] = res[p] + v[0][p];
        } else if (epi == zwg_ew::kEpiGelu) {
#pragma unroll
            for (int p = 0; p < PW; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[0][p][e] = zwg_ew::gelu(v[0][p][e]);
        }
#pragma unroll
        for (int p = 0; p < PW; ++p)
            if (o_r + 8 * p < m) put(o + (int64_t)8 * p * n, v[0][p]);
    }
};

// Short calls (a chunk or so of k per workgroup, about one workgroup per CU): nothing but the order
// of a wave's own instructions hides latency.  Stages of 128 k.  32-row calls take any number of them
// through three LDS buffers: at stage t the buffers of t and t + 1 are complete and t + 2's is being
// filled, so a call of one or two stages has one barrier before its products and none after.  64-row
// calls take one chunk, at most two stages (launch_q8p_tile refuses more), both loaded up front into
// two buffers.  A stage is walked in units of one (block, m-tile): while a unit's four MFMAs run, the
// wave reads the next unit's x operands, widens the next block's weights, scales the previous unit's
// sums and splits its share of stage t + 2's x.
// Left to the compiler, each operand was read directly before its MFMA.  Measured back to back with
// weights from HBM, against one workgroup shape with a barrier per stage and 4-byte stores:
// 32 x 768 x 768 in 3 splits 5.8 -> 4.6 us, 64 x 1536 x 1536 in 6 splits 9.1 -> 6.0 us, 256 x 896 x
// 896 in 4 splits 9.4 -> 6.1 us (64-column tiles; 128-column ones 7.0 and 7.5 us).
template <int MT, int NS, int MS, bool XS, bool PAIR, bool GRP>
__global__ __launch_bounds__(64 * NS * MS) __attribute__((amdgpu_waves_per_eu(2)))
void linear_q8p_short_kernel(Q8Args a, Q8Group grp, const _Float16 *xcvt) {
    using Tile = Q8pTile<MT, NS, MS, 1, 4, XS, PAIR, GRP>;
    constexpr bool LOOP = MT == 1; // more than two stages
    static_assert(XS || !LOOP, "the loop splits its own x");
    constexpr int NB = 4, WT = Tile::WT, XQ = Tile::XQ, U = NB * WT, BUFS = LOOP ? 3 : 2;
    constexpr int XS_BYTES = BUFS * Tile::STAGE_HALVES * 2;
    __shared__ __align__(16) char lds_all[XS_BYTES > Tile::OUT_BYTES ? XS_BYTES : Tile::OUT_BYTES];
    auto &xs = *reinterpret_cast<_Float16(*)[BUFS][Tile::STAGE_HALVES]>(lds_all);
    const Tile w(a, grp, xcvt);

    f32x16 acc[WT];
#pragma unroll
    for (int i = 0; i < WT; ++i) acc[i] = (f32x16){0};
    f32x4 xr[XQ];
    u32x4 wq[BUFS][NB];
    typename Tile::Scales sc[BUFS];

    // stage t in buffer and register set `c`.  more: stages past t + 1 may follow (the last ones
    // load and put nothing)
    auto stage = [&](int t, auto c_c, auto more_c) {
        constexpr int c = decltype(c_c)::value, c2 = (c + 2) % 3;
        constexpr bool more = decltype(more_c)::value;
        static_assert(LOOP || !more);
        half8 A[2][4]; // a unit's x operands
        half8 W[2][2]; // a block's widened weights
        f32x16 T[2];   // a unit's sums
        auto widen = [&](int b) { // and reload the block's registers for stage t + 3
            W[b & 1][0] = int8x8_to_half8(wq[c][b][0], wq[c][b][1]);
            W[b & 1][1] = int8x8_to_half8(wq[c][b][2], wq[c][b][3]);
            if (more) wq[c][b] = w.load_w(t + 3, b);
        };
        auto scale = [&](int u) {
            const float s = sc[c].s[u / WT];
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u % WT][r] = __builtin_fmaf(T[u & 1][r], s, acc[u % WT][r]);
        };
        w.read_a(A[0], xs[c], 0, 0);
        widen(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const half8(&au)[4] = A[u & 1];
            const half8(&wu)[2] = W[(u / WT) & 1];
            f32x16 tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(au[0], wu[0], (f32x16){0}, 0, 0, 0);
            if (u + 1 < U) w.read_a(A[(u + 1) & 1], xs[c], (u + 1) / WT, (u + 1) % WT);
            if (u % WT == WT - 1 && u / WT + 1 < NB) widen(u / WT + 1);
            __builtin_amdgcn_sched_barrier(0);
            tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(au[1], wu[0], tt, 0, 0, 0);
            if constexpr (more) { // a share of stage t + 2's x into LDS, its registers reloaded for t + 3
#pragma unroll
                for (int e = u * XQ / U; e < (u + 1) * XQ / U; ++e) {
                    w.put_x(xs[c2], e, xr[e]);
                    xr[e] = w.load_x(t + 3, e);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(au[2], wu[1], tt, 0, 0, 0);
            if (u > 0) scale(u - 1);
            __builtin_amdgcn_sched_barrier(0);
            T[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(au[3], wu[1], tt, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        scale(U - 1);
        if (more) sc[c] = w.load_s(t + 3);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (more) __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    // first loads: x of stages 0 and 1, their weights and scales, then (LOOP) stage 2's
    f32x4 x0[XQ], x1[XQ];
    if constexpr (XS) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) x0[e] = w.load_x(w.t_begin, e);
#pragma unroll
        for (int e = 0; e < XQ; ++e) x1[e] = w.load_x(w.t_begin + 1, e);
    } else {
        w.dma_x(w.t_begin, xs[0]);
        w.dma_x(w.t_begin + 1, xs[1]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int b = 0; b < NB; ++b) wq[c][b] = w.load_w(w.t_begin + c, b);
        sc[c] = w.load_s(w.t_begin + c);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (LOOP) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) xr[e] = w.load_x(w.t_begin + 2, e);
#pragma unroll
        for (int b = 0; b < NB; ++b) wq[2][b] = w.load_w(w.t_begin + 2, b);
        sc[2] = w.load_s(w.t_begin + 2);
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (XS) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) w.put_x(xs[0], e, x0[e]);
#pragma unroll
        for (int e = 0; e < XQ; ++e) w.put_x(xs[1], e, x1[e]);
    } else {
        __builtin_amdgcn_s_waitcnt(q8_vmcnt(2 * (NB + 1)));
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    const int n_t = w.t_end - w.t_begin;
    int t = w.t_begin;
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    if constexpr (LOOP) {
        // turns of three stages, then the remaining one or two: the loop has no other way out, so the
        // wait counts at its top are those of its own loads
        constexpr std::integral_constant<int, 2> c2{};
        for (int p = n_t / 3; p > 0; --p, t += 3) {
            stage(t, c0, std::true_type{});
            stage(t + 1, c1, std::true_type{});
            stage(t + 2, c2, std::true_type{});
        }
        if (n_t % 3 > 0) stage(t, c0, std::false_type{});
        if (n_t % 3 > 1) stage(t + 1, c1, std::false_type{});
    } else {
        stage(t, c0, std::false_type{});
        if (n_t > 1) stage(t + 1, c1, std::false_type{});
    }
    __syncthreads();
    w.store(acc, reinterpret_cast<float *>(lds_all), grp);
}

// Long calls (many stages per workgroup, or more workgroups than CUs): small stages of 64 k in two
// LDS buffers, so that three or four 4-wave workgroups share a CU and hide each other's loads,
// operand reads, first loads and stores.  Weights run two stages ahead in two register sets (block
// b's registers are reloaded as soon as they are widened), x one stage.  Such a call is bound by the
// bytes a CU can load (about 90-100 GB/s from L2 or the Infinity Cache, 32 KB of x and 16 KB of
// weights per 64 x 128 x 128 products) with the MFMAs close behind; stages of 128 k, three or four
// buffers, and eight-wave workgroups measured the same or slower.  Measured back to back, against
// 128 k stages with a barrier, an LDS round trip per operand and 4-byte stores: the 64-row
// logits of 151936 x 1536 91 -> 79 us, a 256-row SwiGLU pair of 4864 x 896 37 -> 20 us, the one-row
// logits of 151936 x 896 58 -> 31 us, 1001 x 1536 x 8960 (the tiled kernel before) 120 -> 71 us.
// The 64 x 128 tile is held to three workgroups per CU; its registers would allow four, which measured
// slower (1001 x 1536 x 8960 75.3 us for 73.6, the 64-row logits 88.6 for 86.9).
template <int MT, int NS, int KB, int SB, bool XS, bool PAIR, bool GRP>
__global__ __launch_bounds__(64 * NS * KB) __attribute__((amdgpu_waves_per_eu(
    SB == 2 ? 3 : MT == 1 && KB == 1 ? 4 : 2, SB == 2 && NS == 4 ? 3 : 8)))
void linear_q8p_long_kernel(Q8Args a, Q8Group grp, const _Float16 *xcvt) {
    using Tile = Q8pTile<MT, NS, 1, KB, SB, XS, PAIR, GRP>;
    constexpr int WT = Tile::WT, XQ = Tile::XQ, NB = Tile::NB;
    constexpr int XS_BYTES = 2 * Tile::STAGE_HALVES * 2;
    __shared__ __align__(16) char lds_all[XS_BYTES > Tile::OUT_BYTES ? XS_BYTES : Tile::OUT_BYTES];
    auto &xs = *reinterpret_cast<_Float16(*)[2][Tile::STAGE_HALVES]>(lds_all);
    const Tile w(a, grp, xcvt);

    f32x16 acc[WT];
#pragma unroll
    for (int i = 0; i < WT; ++i) acc[i] = (f32x16){0};
    f32x4 xr[XQ]; // XS: the next stage's x
    u32x4 wq[2][NB];
    typename Tile::Scales sc[2];

    // stage t in buffer and register set `c`; more: stages may follow
    auto stage = [&](int t, auto c_c, auto more_c) {
        constexpr int c = decltype(c_c)::value;
        constexpr bool more = decltype(more_c)::value;
        if constexpr (!XS && more) w.dma_x(t + 1, xs[c ^ 1]);
        if constexpr (XS && more) {
#pragma unroll
            for (int e = 0; e < XQ; ++e) {
                w.put_x(xs[c ^ 1], e, xr[e]);
                xr[e] = w.load_x(t + 2, e);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const half8 w0 = int8x8_to_half8(wq[c][b][0], wq[c][b][1]);
            const half8 w1 = int8x8_to_half8(wq[c][b][2], wq[c][b][3]);
            if (more) wq[c][b] = w.load_w(t + 2, b);
#pragma unroll
            for (int i = 0; i < WT; ++i) {
                half8 A[4];
                w.read_a(A, xs[c], b, i);
                f32x16 tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0], w0, (f32x16){0}, 0, 0, 0);
                tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[1], w0, tt, 0, 0, 0);
                tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[2], w1, tt, 0, 0, 0);
                tt = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[3], w1, tt, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(tt[r], sc[c].s[b], acc[i][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) sc[c] = w.load_s(t + 2);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (more) {
            // XS = false: the copies of stage t + 1; the weights and scales issued after them may still
            // be in flight
            if constexpr (!XS) __builtin_amdgcn_s_waitcnt(q8_vmcnt(NB + 1));
            __syncthreads();
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // first loads: stage 0's x, weights and scales, then stage 1's
    f32x4 x0[XQ];
    if constexpr (XS) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) x0[e] = w.load_x(w.t_begin, e);
    } else {
        w.dma_x(w.t_begin, xs[0]);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) wq[0][b] = w.load_w(w.t_begin, b);
    sc[0] = w.load_s(w.t_begin);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (XS) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) xr[e] = w.load_x(w.t_begin + 1, e);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) wq[1][b] = w.load_w(w.t_begin + 1, b);
    sc[1] = w.load_s(w.t_begin + 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (XS) {
#pragma unroll
        for (int e = 0; e < XQ; ++e) w.put_x(xs[0], e, x0[e]);
    } else {
        __builtin_amdgcn_s_waitcnt(q8_vmcnt(2 * (NB + 1)));
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    // pairs of stages, then an odd one (the loop has no other way out, as above)
    const int n_t = w.t_end - w.t_begin;
    int t = w.t_begin;
    for (int p = n_t / 2; p > 0; --p, t += 2) {
        stage(t, std::integral_constant<int, 0>{}, std::true_type{});
        stage(t + 1, std::integral_constant<int, 1>{}, std::true_type{});
    }
    if (n_t & 1) stage(t, std::integral_constant<int, 0>{}, std::false_type{});
    if constexpr (!XS) __builtin_amdgcn_s_waitcnt(q8_vmcnt(0)); // the last, out-of-range copies into LDS
    __syncthreads();
    w.store(acc, reinterpret_cast<float *>(lds_all), grp);
}

// out[i][o] (row stride ldo) = epilogue(sum over splits (in split order) of part[split][i][o],
// + bias[o]).  V consecutive elements of one row per thread (V = 4 needs n % 4 == 0 and 16-byte
// aligned partials).  The loads of up to kSumBatch splits are all issued before the first add, so
// a sum waits for one memory latency per batch rather than one per split; the adds stay in split
// order.
constexpr int kSumBatch = 16;
template <int V>
__global__ __launch_bounds__(256) void linear_split_sum_kernel(const float *part, const float *bias, float *out,
                                                              int64_t mn, int32_t n, int32_t n_split, uint32_t epi,
                                                              int64_t ldo) {
    using vec = typename std::conditional<V == 1, float, float __attribute__((ext_vector_type(4)))>::type;
    static_assert(V == 1 || V == 4, "one or four elements per thread");
    const int64_t e = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (e >= mn) return;
    const vec *p = reinterpret_cast<const vec *>(part + e);
    const int64_t step = mn / V;
    vec s{};
    for (int q0 = 0; q0 < n_split; q0 += kSumBatch) {
        vec v[kSumBatch];
#pragma unroll
        for (int j = 0; j < kSumBatch; ++j)
            if (q0 + j < n_split) v[j] = p[(q0 + j) * step];
#pragma unroll
        for (int j = 0; j < kSumBatch; ++j)
            if (q0 + j < n_split) s = q0 + j == 0 ? v[j] : s + v[j];
    }
    const int64_t row = e / n, col = e - row * n;
    if constexpr (V == 1) {
        zwg_ew::epilogue_store(&out[row * ldo + col], bias ? s + bias[col] : s, epi);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
            zwg_ew::epilogue_store(&out[row * ldo + col + v], bias ? s[v] + bias[col + v] : s[v], epi);
    }
}

// The split sum over a group: element e of the concatenated outputs is element e - elem_start[j]
// of set j, summed over the splits in split order, + bias, through the epilogue.
__global__ __launch_bounds__(256) void linear_split_sum_group_kernel(Q8Group grp, int32_t m, int32_t n_split,
                                                                    uint32_t epi) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= grp.elem_start[kQ8MaxGroup]) return;
    const int set = q8_group_of_elem(grp, e);
    const int64_t le = e - q8_pick(grp.elem_start, set);
    const int32_t n = q8_pick(grp.n, set);
    const int64_t mn = (int64_t)m * n;
    const float *part = q8_pick(grp.part, set);
    const float *bias = q8_pick(grp.bias, set);
    const float *p = part + le;
    float s = 0.f;
    for (int q0 = 0; q0 < n_split; q0 += kSumBatch) { // loads of a batch issued together, adds in split order
        float v[kSumBatch];
#pragma unroll
        for (int j = 0; j < kSumBatch; ++j)
            if (q0 + j < n_split) v[j] = p[(q0 + j) * mn];
#pragma unroll
        for (int j = 0; j < kSumBatch; ++j)
            if (q0 + j < n_split) s = q0 + j == 0 ? v[j] : s + v[j];
    }
    if (bias) s += bias[le % n];
    zwg_ew::epilogue_store(&q8_pick(grp.out, set)[le], s, epi);
}

// A split SwiGLU pair's sum (Q8Group swiglu): out[0][e] = silu(gate) * up, gate and up each their
// splits added in split order then their bias, as linear_split_sum_group_kernel forms them, then
// zwg_ew::silu_mul (the separate SiLU-mul kernel's function).  e over m n[0].
__global__ __launch_bounds__(256) void linear_split_sum_swiglu_kernel(Q8Group grp, int32_t m, int32_t n_split) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int32_t n = grp.n[0];
    const int64_t mn = (int64_t)m * n;
    if (e >= mn) return;
    float gu[2];
#pragma unroll
    for (int set = 0; set < 2; ++set) {
        const float *p = (set ? grp.part[1] : grp.part[0]) + e;
        float s = 0.f;
        for (int q0 = 0; q0 < n_split; q0 += kSumBatch) {
            float v[kSumBatch];
#pragma unroll
            for (int j = 0; j < kSumBatch; ++j)
                if (q0 + j < n_split) v[j] = p[(q0 + j) * mn];
#pragma unroll
            for (int j = 0; j < kSumBatch; ++j)
                if (q0 + j < n_split) s = q0 + j == 0 ? v[j] : s + v[j];
        }
        const float *bias = set ? grp.bias[1] : grp.bias[0];
        if (bias) s += bias[e % n];
        gu[set] = s;
    }
    float v = zwg_ew::silu_mul(gu[0], gu[1]);
    if (!grp.xcvt_out) {
        grp.out[0][e] = v;
        return;
    }
    asm volatile("" : "+v"(v)); // split from the rounded product
    const int row = (int)(e / n);
    q8_xs_store1<2>(grp.xcvt_out + (int64_t)(row >> 6) * ((n + kQ8Chunk - 1) / kQ8Chunk) * q8_chunk_halves<2>(), row & 63,
                    (int)(e % n), v);
}

// The q/k/v group's split sum with the cache append fused into its stores (set 0 q, 1 k, 2 v of a
// Q8Group; n = heads * D).  Where the split sum writes rows and kv_append_kernel then reads them
// back, this kernel takes the same sums -- the splits added in split order, then the bias -- and
// does what the append does with them:
//   - q and k at their token's position get NeoX rotary positions (pairs (j, j + D/2), rounded
//     product by product as the reference does, src/llm.zig:221-238) when the cache has tables;
//   - q is written to q_out; k into the key cache, transposed ([head][dim][n_ctx]) or as a row; v
//     as a row; a token whose position is outside [0, n_ctx) writes no cache rows and an unrotated q.
// So the caches and q equal, bit for bit, the group call into rows followed by zwg_kv_append_batch.
// A thread takes one (token, set, head, 4 dims j .. j+3) and the 4 dims j + D/2 .. of the pair.
struct Q8KvStore {
    float *q_out;           // [m][n_head * D]
    float *k_cache;         // the layer's caches: token i's sequence seq0 + i at + (seq0 + i) * per_seq
    float *v_cache;
    const float *cos;       // [n_ctx][D/2], or nullptr: no rotary positions
    const float *sin;
    const int32_t *pos_dev; // [m] positions, or nullptr: token i at pos0 + i
    int32_t *n_kv_out;      // or nullptr: [m] keys each sequence's cache then holds, pos + 1 (0 off the cache)
    int64_t per_seq;
    int32_t seq0, n_ctx, n_head, n_head_kv, kt;
    int32_t pos0;     // the first position when pos_dev is nullptr
    int32_t seq_step; // token i's sequence is seq0 + i seq_step: 1 (a decode step), 0 (one sequence's rows)
    int32_t d; // the kernel's D (host side: which instantiation)
};

template <int D>
__global__ __launch_bounds__(256) void linear_split_sum_qkv_kernel(Q8Group grp, Q8KvStore kv, int32_t m,
                                                                  int32_t n_split) {
#pragma clang fp contract(off) // the rotation rounds each product and sum, as the reference does
    constexpr int HALF = D / 2, QH = D / 8; // pair quads per head
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int per_tok = (kv.n_head + 2 * kv.n_head_kv) * QH;
    if (e >= (int64_t)m * per_tok) return;
    const int i = (int)(e / per_tok);
    int u = (int)(e - (int64_t)i * per_tok);
    const int set = u < kv.n_head * QH ? 0 : u < (kv.n_head + kv.n_head_kv) * QH ? 1 : 2;
    u -= set == 0 ? 0 : set == 1 ? kv.n_head * QH : (kv.n_head + kv.n_head_kv) * QH;
    const int h = u / QH, j = 4 * (u - h * QH);
    const int32_t n = q8_pick(grp.n, set);
    const int64_t mn = (int64_t)m * n;
    const float *part = q8_pick(grp.part, set) + (int64_t)i * n + h * D + j;
    const float *bias = q8_pick(grp.bias, set);
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
    for (int q0 = 0; q0 < n_split; q0 += kSumBatch) { // as linear_split_sum_group_kernel: loads first
        f4 vl[kSumBatch], vh[kSumBatch];
#pragma unroll
        for (int t = 0; t < kSumBatch; ++t)
            if (q0 + t < n_split) {
                vl[t] = *reinterpret_cast<const f4 *>(part + (q0 + t) * mn);
                vh[t] = *reinterpret_cast<const f4 *>(part + (q0 + t) * mn + HALF);
            }
#pragma unroll
        for (int t = 0; t < kSumBatch; ++t)
            if (q0 + t < n_split) {
                lo = q0 + t == 0 ? vl[t] : lo + vl[t];
                hi = q0 + t == 0 ? vh[t] : hi + vh[t];
            }
    }
    if (bias) {
        const f4 bl = *reinterpret_cast<const f4 *>(bias + h * D + j);
        const f4 bh = *reinterpret_cast<const f4 *>(bias + h * D + j + HALF);
        lo += bl;
        hi += bh;
    }
    const int p = kv.pos_dev ? kv.pos_dev[i] : kv.pos0 + i;
    const bool live = p >= 0 && p < kv.n_ctx;
    if (kv.n_kv_out && set == 0 && h == 0 && j == 0) kv.n_kv_out[i] = live ? p + 1 : 0;
    if (set < 2 && kv.cos && live) {
        const f4 c = *reinterpret_cast<const f4 *>(kv.cos + (int64_t)p * HALF + j);
        const f4 s = *reinterpret_cast<const f4 *>(kv.sin + (int64_t)p * HALF + j);
        const f4 x0 = lo, x1 = hi;
        lo = x0 * c - x1 * s;
        hi = x0 * s + x1 * c;
    }
    if (set == 0) {
        float *qr = kv.q_out + (int64_t)i * kv.n_head * D + h * D + j;
        *reinterpret_cast<f4 *>(qr) = lo;
        *reinterpret_cast<f4 *>(qr + HALF) = hi;
        return;
    }
    if (!live) return;
    const int kvw = kv.n_head_kv * D;
    const int64_t seq = (int64_t)(kv.seq0 + i * kv.seq_step) * kv.per_seq;
    if (set == 1 && kv.kt) {
        float *kc = kv.k_cache + seq + (int64_t)(h * D + j) * kv.n_ctx + p;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            kc[(int64_t)t * kv.n_ctx] = lo[t];
            kc[(int64_t)(t + HALF) * kv.n_ctx] = hi[t];
        }
        return;
    }
    float *row = (set == 1 ? kv.k_cache : kv.v_cache) + seq + (int64_t)p * kvw + h * D + j;
    *reinterpret_cast<f4 *>(row) = lo;
    *reinterpret_cast<f4 *>(row + HALF) = hi;
}

// A one-set call's split sum added to the residual stream and normalised, for the decoder blocks'
// ops.linear + ops.add + next ops.layerNorm (src/decoder.zig:185-188, :192-195, :200 with the
// next block's :178) and Qwen2's + ops.rmsNorm (src/llm.zig:203-204, :206-207 with :178): row i
// of x += sum over splits (in split order) of part[s][i] + bias -- as
// linear_split_sum_group_kernel with the add epilogue forms it -- then ln_out[i] = the norm of
// x[i] (NORM: zwg_ew::kNormLayer or kNormRms, through the functions layer_norm_kernel and
// rms_norm_kernel use).  So x and ln_out equal the split sum and the norm launch bit for bit.  One thread
// per float4 column (R waves per row, n <= 256 R floats), with up to 24 of its column's splits in flight
// at once: with a wave per row instead, each lane walked R columns in batches of 48 / R splits (the
// Qwen2.5-1.5B down projection's 35 splits of 1536-float rows: 18 batches of loads one after another;
// per step, paired: Whisper small.en decoder over 32 windows 1563 us so, 1537 with a thread per column,
// Qwen2.5-1.5B decode over 64 sequences 4394 and 4198).  The new row goes through LDS to the first wave,
// which normalises it.
struct Q8ResLn {
    float *x; // [m][n] residual stream, updated in place
    const float *ln_w, *ln_b; // ln_b unused by the RMS norm
    float *ln_out; // [m][n]
    float eps;
    int32_t norm; // zwg_ew::kNormLayer or kNormRms (host side: which instantiation)
    // nullptr, or the normalised rows also split into f16 hi/lo halves for the next call of 64-row blocks
    // (linear_q8_xprep_kernel's layout and values, the last block's rows past m zero)
    _Float16 *xcvt;
};

template <int R, int NORM>
__global__ __launch_bounds__(64 * R) void linear_split_sum_add_ln_wide_kernel(const float *part, const float *bias,
                                                                              Q8ResLn r, int32_t m, int32_t n,
                                                                              int32_t n_split) {
#pragma clang fp contract(off)
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int B = 24;
    constexpr bool kLayerNorm = NORM != zwg_ew::kNormRms;
    constexpr bool kPass = R * (kLayerNorm ? 2 : 1) > 8; // the norm's weights through LDS, below
    __shared__ f4 rowbuf[64 * R], wbuf[kPass ? 64 * R : 1], bbuf[kPass && kLayerNorm ? 64 * R : 1];
    const int c = threadIdx.x; // this thread's float4 column
    const int row = (int)blockIdx.x;
    if (row >= m) return;
    const int n4 = n >> 2;
    const bool live = c < n4;
    const int64_t step = (int64_t)m * n4;
    const f4 *p = reinterpret_cast<const f4 *>(part) + (int64_t)row * n4 + c;
    f4 *xr = reinterpret_cast<f4 *>(r.x + (int64_t)row * n);
    f4 xo = {0.f, 0.f, 0.f, 0.f}, bo = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        xo = xr[c];
        if (bias) bo = reinterpret_cast<const f4 *>(bias)[c];
    }
    // the norm's weights for the first wave, in flight with the partials rather than a round trip behind
    // them (the small.en decoder step 1460 -> 1436 us over its 36 launches).  Up to eight float4s go
    // straight to its registers (which every wave then has, at no loss: these rows are few workgroups);
    // of wider rows each thread loads its column's and passes them on through LDS, as in registers they
    // took a wave per SIMD and spilled (layer norm from R = 10, RMS from 14: a step of eight layers of 4096
    // floats, 64 rows, 961 us so, 771 through LDS; the Qwen2.5-0.5B prompt's batch, R = 4, 2140 through
    // LDS, 2134 so)
    f4 nw[kPass ? 1 : R], nb[kPass || !kLayerNorm ? 1 : R];
#pragma unroll
    for (int i = 0; i < (kPass ? 1 : R); ++i) {
        const int at = kPass ? c : c + 64 * i;
        if (at >= n4 || (!kPass && c >= 64)) continue;
        nw[i] = reinterpret_cast<const f4 *>(r.ln_w)[at];
        if constexpr (kLayerNorm) nb[i] = reinterpret_cast<const f4 *>(r.ln_b)[at];
    }
    f4 s = {0.f, 0.f, 0.f, 0.f};
    for (int q0 = 0; q0 < n_split; q0 += B) {
        f4 t[B];
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (live && q0 + j < n_split) t[j] = p[(q0 + j) * step];
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (live && q0 + j < n_split) s = q0 + j == 0 ? t[j] : s + t[j];
    }
    f4 nx = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        f4 val = s;
        if (bias) val = val + bo;
        nx = xo + val;
        xr[c] = nx;
    }
    rowbuf[c] = nx;
    if constexpr (kPass) {
        wbuf[c] = nw[0];
        if constexpr (kLayerNorm) bbuf[c] = nb[0];
    }
    __syncthreads();
    if (c < 64) {
        zwg_ew::ew_f32x4 v[R];
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = rowbuf[c + 64 * i];
        // with xcvt the normalised row also goes back into rowbuf (past n4 it stays zero)
        float *const orow = r.ln_out + (int64_t)row * n;
        f4 *const copy = r.xcvt ? rowbuf : nullptr;
        const auto w = [&](int i) { return kPass ? wbuf[c + 64 * i] : nw[kPass ? 0 : i]; };
        if constexpr (kLayerNorm)
            zwg_ew::layer_norm_with<R>(
                v, c, n4, w, [&](int i) { return kPass ? bbuf[c + 64 * i] : nb[kPass ? 0 : i]; }, r.eps, orow, copy);
        else
            zwg_ew::rms_norm_with<R>(v, c, n4, w, r.eps, orow, copy);
    }
    if (r.xcvt) {
        __syncthreads();
        const int n_cols = (n + kQ8Chunk - 1) / kQ8Chunk * (kQ8Chunk / 4); // float4 columns of whole chunks
        if (c < n_cols) {
            const int64_t per_z = (int64_t)(n_cols / (kQ8Chunk / 4)) * q8_chunk_halves<2>();
            q8_xs_store<2>(r.xcvt + (row >> 6) * per_z, row & 63, 4 * c, rowbuf[c]);
            for (int z = row + m; z < (m + 63) / 64 * 64; z += m)
                q8_xs_store<2>(r.xcvt + (z >> 6) * per_z, z & 63, 4 * c, (f32x4){0.f, 0.f, 0.f, 0.f});
        }
    }
}

// A decode step's token embeddings from the packed int8 token embedding (the tied output
// projection): x[i] = te.row(tok[i]) + pe[pos[i]] -- gemm.Q8.row (src/gemm.zig:257-265, q * scale
// in f32) then ops.add (src/decoder.zig:171-174) -- and ln_out[i] = the norm of x[i] (the first
// block's attn_ln, src/decoder.zig:178; for Qwen2, no position rows and the first block's RMS
// norm, src/llm.zig:175-178).  A token outside
// [0, n_vocab) gives a zero embedding row; a position outside [0, pe_rows) adds no position row
// (pos may be null when there are none).
// One wave per row of n <= 256 R floats; a lane's float4 is 4 bytes of one 16-byte lane piece of
// its block's tile (Q8Packed).
template <int R, int NORM>
__global__ __launch_bounds__(64) void q8p_embed_ln_kernel(Q8Packed te, int32_t n_vocab, const int32_t *tok,
                                                          const float *pe, const int32_t *pos, int32_t pe_rows,
                                                          int32_t m, int32_t n, float *x, Q8ResLn r) {
#pragma clang fp contract(off)
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x;
    const int row = (int)blockIdx.x; // one wave per workgroup, one row per wave
    if (row >= m) return;
    const int n4 = n >> 2;
    const int t = tok[row], ps = pos ? pos[row] : -1;
    const bool t_ok = t >= 0 && t < n_vocab, p_ok = ps >= 0 && ps < pe_rows;
    const int slab = t_ok ? t >> 5 : 0, r32 = t & 31;
    const int nbp = te.n_chunks * kQ8ChunkBlocks;
    zwg_ew::ew_f32x4 v[R];
    f4 *xr = reinterpret_cast<f4 *>(x + (int64_t)row * n);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int c = lane + 64 * i;
        f4 val = {0.f, 0.f, 0.f, 0.f};
        if (c < n4) {
            if (t_ok) {
                const int k0 = 4 * c, b = k0 >> 5;
                const uint32_t w4 = *reinterpret_cast<const uint32_t *>(
                    te.q + (((int64_t)slab * nbp + b) * 64 + r32 + 32 * ((k0 & 31) >> 4)) * 16 + (k0 & 15));
                const float sc =
                    te.scales[(((int64_t)slab * te.n_chunks + (b >> 3)) * 32 + r32) * kQ8ChunkBlocks + (b & 7)];
#pragma unroll
                for (int e = 0; e < 4; ++e) val[e] = (float)(int8_t)(uint8_t)(w4 >> (8 * e)) * sc;
            }
            if (p_ok) val = val + reinterpret_cast<const f4 *>(pe + (int64_t)ps * n)[c];
            xr[c] = val;
        }
        v[i] = val;
    }
    zwg_ew::norm_regs<NORM, R>(v, lane, n4, r.ln_w, r.ln_b, r.eps, r.ln_out + (int64_t)row * n);
}

} // namespace zwg_lin
