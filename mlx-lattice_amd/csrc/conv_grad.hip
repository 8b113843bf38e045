// Gradients of the sparse convolution (the reference's vjp:
// native/features/convolution/primitive.cpp:137-176, 597-680; CPU routines
// cpu/algorithms.cpp:355-481).
//
//  * Input gradient, CSR route: one lane per (input row, input channel)
//    walks the row's edges in the input-grouped CSR (in_row_offsets /
//    in_edge_ids) with an fp32 accumulator over the edges and every output
//    channel, one rounding at the end (eval_input_grad_typed).  Small
//    weights are staged once per block in LDS as fp32, (k, co, ci) with ci
//    fastest, so the lanes of a row read consecutive banks.
//  * Input gradient, matrix-core route: for a forward or submanifold
//    relation every (input row, k) pair has at most one output row, so the
//    relation transposes into a dense map in_out_map[in][k] with the same
//    row masks as the forward's out_in_map.  `transposed_map` scatters it
//    from the edges; the forward's sorted view and implicit-GEMM kernel then
//    compute grad[in][ci] = sum_k sum_co cot[map[in][k]][co] * W[k][ci][co]
//    with the weight transposed to (C_in, K, C_out).
//  * Weight gradient: dW[k] = sum over the edges of k of
//    feats[in]^T cot[out] (eval_weight_grad_typed), a contraction over
//    edges.  The matrix-core kernel splits each offset's kernel-grouped
//    edges (kernel_row_offsets / kernel_edge_ids, in output-row order) into
//    eight parts, one per XCD, and deals an XCD's blocks to the offsets in
//    proportion to their edge counts; an offset's blocks take its part's
//    64-edge chunks in turn, so the XCD's blocks sweep the same output rows
//    together and a cotangent row stays in L2 between the offsets that read
//    it.  Channel tiles are 128 x 128 when the channels fill them (an
//    edge's rows are gathered once for every channel pair).  A block stages
//    64 edges of both operands in LDS as edge rows, reads the MFMA
//    fragments (8 consecutive edges per lane) with transposing LDS reads
//    and accumulates in fp32.  Each block writes its partial tile; a second
//    kernel sums an offset's partials in a fixed order and rounds once, so
//    results are deterministic.  float32 contracts on 16x16x4 MFMAs over the
//    same steps; rows that are not whole 16-byte pieces are loaded value by
//    value.  Callers without a workspace take a one-lane-per-weight kernel,
//    whose lanes walk all of an offset's edges through three dependent
//    loads each: 64 -> 64 float32 over 60,001 rows (280k edges) 31,000 us
//    there, 42 us (plus 18 us of reduction) here.

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "lattice_common.h"
#include "scan.h"

namespace lattice {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

template <typename T> __device__ inline float to_f(T v) { return static_cast<float>(v); }

struct GradWeightIndex {
    int layout;  // LATTICE_WEIGHT_*
    int K, c_in, c_out;
    __device__ inline long long operator()(int k, int ci, int co) const {
        if (layout == LATTICE_WEIGHT_KERNEL_MAJOR) return (static_cast<long long>(k) * c_in + ci) * c_out + co;
        return (static_cast<long long>(co) * K + k) * c_in + ci;
    }
};

constexpr int kGradLdsFloats = 16384;
constexpr unsigned kGradStagedBlocks = 2048;

// ------------------------------------------------- input gradient (CSR) --

template <typename T>
__global__ void __launch_bounds__(256)
input_grad_csr(const T* __restrict__ cot, int out_capacity, const T* __restrict__ weights, GradWeightIndex widx,
               const int32_t* __restrict__ out_rows, const int32_t* __restrict__ kernel_ids,
               const int32_t* __restrict__ counts, int edge_capacity, const int32_t* __restrict__ in_row_offsets,
               const int32_t* __restrict__ in_edge_ids, int in_capacity, T* __restrict__ grad, bool staged) {
    extern __shared__ float wlds[];
    const int c_in = widx.c_in;
    const int c_out = widx.c_out;
    if (staged) {
        const int nw = widx.K * c_in * c_out;
        for (int i = threadIdx.x; i < nw; i += blockDim.x) {
            const int ci = i % c_in;
            const int kc = i / c_in;  // k * c_out + co
            wlds[i] = to_f(weights[widx(kc / c_out, ci, kc % c_out)]);
        }
        __syncthreads();
    }
    const int E = min(counts[0], edge_capacity);
    const long long total = static_cast<long long>(in_capacity) * c_in;
    for (long long t = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
         t += static_cast<long long>(gridDim.x) * blockDim.x) {
        const int row = static_cast<int>(t / c_in);
        const int ci = static_cast<int>(t - static_cast<long long>(row) * c_in);
        float acc = 0.0f;
        const int end = in_row_offsets[row + 1];
        for (int cur = in_row_offsets[row]; cur < end; ++cur) {
            const int e = in_edge_ids[cur];
            if (e < 0 || e >= E) continue;
            const int o = out_rows[e];
            const int k = kernel_ids[e];
            if (o < 0 || o >= out_capacity || k < 0 || k >= widx.K) continue;
            const T* g = cot + static_cast<long long>(o) * c_out;
            if (staged) {
                const float* wk = wlds + static_cast<long long>(k) * c_out * c_in + ci;
                for (int co = 0; co < c_out; ++co) acc += to_f(g[co]) * wk[co * c_in];
            } else {
                for (int co = 0; co < c_out; ++co) acc += to_f(g[co]) * to_f(weights[widx(k, ci, co)]);
            }
        }
        grad[t] = static_cast<T>(acc);
    }
}

// ---------------------------------------- transposed map (matrix cores) --

__global__ void __launch_bounds__(256)
transposed_map(const int32_t* __restrict__ in_rows, const int32_t* __restrict__ out_rows,
               const int32_t* __restrict__ kernel_ids, const int32_t* __restrict__ counts, int edge_capacity,
               int in_capacity, int K, int32_t* __restrict__ in_out_map, int32_t* __restrict__ status) {
    const int E = min(counts[0], edge_capacity);
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < E; e += gridDim.x * blockDim.x) {
        const int in = in_rows[e];
        const int o = out_rows[e];
        const int k = kernel_ids[e];
        if (in < 0 || in >= in_capacity || o < 0 || k < 0 || k >= K) continue;
        const int prev = atomicCAS(&in_out_map[static_cast<long long>(in) * K + k], -1, o);
        if (prev != -1 && status != nullptr) atomicOr(status, LATTICE_STATUS_REPEATED_PAIR);
    }
}

// The same from the dense map: entry (row, k) -> in.
__global__ void __launch_bounds__(256)
transposed_dense_map(const int32_t* __restrict__ out_in_map, long long entries, int K, int in_capacity,
                     int32_t* __restrict__ in_out_map, int32_t* __restrict__ status) {
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < entries;
         i += static_cast<long long>(gridDim.x) * blockDim.x) {
        const int in = out_in_map[i];
        if (in < 0 || in >= in_capacity) continue;
        const long long row = i / K;
        const int k = static_cast<int>(i - row * K);
        const int prev = atomicCAS(&in_out_map[static_cast<long long>(in) * K + k], -1, static_cast<int>(row));
        if (prev != -1 && status != nullptr) atomicOr(status, LATTICE_STATUS_REPEATED_PAIR);
    }
}

// Offset bits of each input row, from its row of the transposed map.  A
// block takes `rows_per_block` consecutive rows, copies their contiguous
// map rows into LDS with coalesced loads, and one lane per row then reads
// its row from LDS (a lane-per-row read of global memory would touch a
// different line per lane for each offset).
__global__ void __launch_bounds__(256)
transposed_masks(const int32_t* __restrict__ in_out_map, int in_capacity, int K, int words, int rows_per_block,
                 int32_t* __restrict__ row_masks) {
    extern __shared__ int32_t map_rows[];
    const int blocks = (in_capacity + rows_per_block - 1) / rows_per_block;
    for (int blk = blockIdx.x; blk < blocks; blk += gridDim.x) {
        const int r0 = blk * rows_per_block;
        const int n = min(rows_per_block, in_capacity - r0);
        const int32_t* src = in_out_map + static_cast<long long>(r0) * K;
        for (int i = threadIdx.x; i < n * K; i += blockDim.x) map_rows[i] = src[i];
        __syncthreads();
        for (int r = threadIdx.x; r < n; r += blockDim.x) {
            const int32_t* m = map_rows + r * K;
            for (int w = 0; w < words; ++w) {
                uint32_t bits = 0;
                for (int k = 32 * w; k < min(K, 32 * w + 32); ++k) bits |= (m[k] >= 0 ? 1u : 0u) << (k & 31);
                row_masks[static_cast<long long>(r0 + r) * words + w] = static_cast<int32_t>(bits);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------ edges grouped by the offset --
//
// A relation whose edges run in (out_row, offset) order and whose row masks
// hold one bit per edge groups by offset without a sort: the edges of offset
// k are the rows with bit k, in row order, and row r's is number
// popcount(mask & below k) of its run.  group_count counts the bits of every
// 1024-row block, group_scan places the blocks (offset by offset), and
// group_emit writes each edge's (input row, output row) pair and, when asked
// for, its id.  The masks, the run starts and the input rows are read once
// and the groups written once, against radix passes over the relation's
// whole capacity (K slots per row, used or not): 200k rows, 2.1M edges, both
// sorted groupings 440 us, the pairs 27 us (count 5, scan 5, emit 17).
constexpr int kGroupRows = 1024;   // rows per block, 64 per wave
constexpr int kGroupWaves = kGroupRows / kWave;
constexpr int kGroupBins = 32;     // offsets per block counter row

// counts of the wave's 64 masks: lane k (< 32) gets the rows with bit k
__device__ inline int wave_bit_counts(uint32_t mask, int K, int lane) {
    int mine = 0;
    for (int k = 0; k < K; ++k) {
        const int c = __popcll(ballot((mask >> k) & 1u));
        mine = lane == k ? c : mine;
    }
    return mine;
}

__global__ void __launch_bounds__(kGroupRows)
group_count(const int32_t* __restrict__ row_masks, int rows, int K, int32_t* __restrict__ block_counts) {
    __shared__ int32_t wave_counts[kGroupWaves][kGroupBins];
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const long long row = static_cast<long long>(blockIdx.x) * kGroupRows + threadIdx.x;
    const uint32_t mask = row < rows ? static_cast<uint32_t>(row_masks[row]) : 0u;
    const int c = wave_bit_counts(mask, K, lane);
    if (lane < kGroupBins) wave_counts[wave][lane] = c;
    __syncthreads();
    if (threadIdx.x < kGroupBins) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kGroupWaves; ++w) sum += wave_counts[w][threadIdx.x];
        block_counts[static_cast<long long>(blockIdx.x) * kGroupBins + threadIdx.x] = sum;
    }
}

// One workgroup: thread (segment, k) sums its run of blocks, the segments
// and offsets are scanned in LDS, and the counts become places in turn.
__global__ void __launch_bounds__(1024)
group_scan(int32_t* __restrict__ block_counts, int blocks, int K, int32_t* __restrict__ offsets) {
    constexpr int kSegments = 1024 / kGroupBins;
    __shared__ int32_t sums[kSegments][kGroupBins];
    __shared__ int32_t base[kGroupBins];
    const int k = threadIdx.x % kGroupBins;
    const int seg = threadIdx.x / kGroupBins;
    const int per = (blocks + kSegments - 1) / kSegments;
    const int lo = min(seg * per, blocks), hi = min(lo + per, blocks);
    int sum = 0;
    for (int b = lo; b < hi; ++b) sum += block_counts[static_cast<long long>(b) * kGroupBins + k];
    sums[seg][k] = sum;
    __syncthreads();
    if (threadIdx.x < kGroupBins) {
        int run = 0;
        for (int i = 0; i < kSegments; ++i) {
            const int v = sums[i][threadIdx.x];
            sums[i][threadIdx.x] = run;
            run += v;
        }
        base[threadIdx.x] = run;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int i = 0; i < kGroupBins; ++i) {
            const int v = base[i];
            base[i] = run;
            if (i <= K) offsets[i] = run;
            run += v;
        }
        if (K == kGroupBins) offsets[K] = run;
    }
    __syncthreads();
    int run = base[k] + sums[seg][k];
    for (int b = lo; b < hi; ++b) {
        int32_t* c = block_counts + static_cast<long long>(b) * kGroupBins + k;
        const int v = *c;
        *c = run;
        run += v;
    }
}

// A wave emits its 64 rows; their map rows pass through its own LDS, 16
// offsets at a time (coalesced reads, which the lanes then take offset by
// offset).  Reading the map by lane instead touches 64 lines per load.
// Bound by the scattered 8-byte stores and the latency of its few blocks:
// 200,000 rows of 27 offsets took 54 us in blocks of four waves with four
// such groups each and take 20 in blocks of sixteen waves.
constexpr int kEmitOffsets = 16;

__global__ void __launch_bounds__(kGroupRows)
group_emit(const int32_t* __restrict__ row_masks, const int32_t* __restrict__ out_in_map,
           const int32_t* __restrict__ row_offsets, int rows, int K, int edge_capacity,
           const int32_t* __restrict__ block_places, int2* __restrict__ pairs, int32_t* __restrict__ edge_ids) {
    constexpr int kStride = kEmitOffsets + 1;
    __shared__ int32_t place[kGroupWaves][kGroupBins];
    __shared__ int32_t stage[kGroupWaves][kWave * kStride];
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const long long row = static_cast<long long>(blockIdx.x) * kGroupRows + threadIdx.x;
    const long long row0 = row - lane;
    const int wave_rows = static_cast<int>(max(0ll, min(static_cast<long long>(kWave), rows - row0)));
    const uint32_t mask = row < rows ? static_cast<uint32_t>(row_masks[row]) : 0u;
    const int c = wave_bit_counts(mask, K, lane);
    if (lane < kGroupBins) place[wave][lane] = c;
    __syncthreads();
    if (threadIdx.x < kGroupBins) {
        int run = block_places[static_cast<long long>(blockIdx.x) * kGroupBins + threadIdx.x];
#pragma unroll
        for (int w = 0; w < kGroupWaves; ++w) {
            const int v = place[w][threadIdx.x];
            place[w][threadIdx.x] = run;
            run += v;
        }
    }
    __syncthreads();
    const int first = edge_ids != nullptr && row < rows ? row_offsets[row] : 0;
    for (int k0 = 0; k0 < K; k0 += kEmitOffsets) {
        const int n = min(kEmitOffsets, K - k0);
        if (pairs != nullptr) {
            const int step_rows = kWave / n;
            const int step_k = kWave % n;
            int r = lane / n;
            int k = lane % n;
            while (r < wave_rows) {
                stage[wave][r * kStride + k] = out_in_map[(row0 + r) * K + k0 + k];
                r += step_rows;
                k += step_k;
                if (k >= n) {
                    k -= n;
                    ++r;
                }
            }
        }
        __syncthreads();
        for (int j = 0; j < n; ++j) {
            const int k = k0 + j;
            const bool has = (mask >> k) & 1u;
            const uint64_t b = ballot(has);
            if (has) {
                const int pos = place[wave][k] + lanes_below(b);
                if (pos >= 0 && pos < edge_capacity) {
                    if (pairs != nullptr)
                        pairs[pos] = make_int2(stage[wave][lane * kStride + j], static_cast<int>(row));
                    if (edge_ids != nullptr) edge_ids[pos] = first + __popc(mask & ((1u << k) - 1u));
                }
            }
        }
        __syncthreads();
    }
}

size_t group_blocks(int rows) { return (static_cast<size_t>(std::max(rows, 0)) + kGroupRows - 1) / kGroupRows; }

// --------------------------------------- weight gradient (matrix cores) --

template <typename T> struct GradMfma;
template <> struct GradMfma<_Float16> {
    typedef half8_t vec;
    __device__ static float4_t mfma(vec a, vec b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct GradMfma<__bf16> {
    typedef bf16x8_t vec;
    __device__ static float4_t mfma(vec a, vec b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

// float32 contracts four edges per MFMA (16x16x4); the pieces are four
// channels.
template <> struct GradMfma<float> {
    typedef float4_t vec;
};

constexpr int kWgEdges = 64;   // edges per staged step (two 32-edge MFMA steps)

// LDS rows of a weight-gradient step: one row per edge, the operand's
// channels in 16-byte pieces (TC / 8 of them).  Piece q of row r sits at
// slot q ^ wg_swizzle(r): the waves' 16-byte stores (two rows of 8 pieces
// per 16 lanes) and the transposing fragment reads (16 rows x 2 pieces per
// instruction) then spread over all the banks.
__device__ inline int wg_swizzle(int r, int pieces) {
    return (2 * (r & 1) + 4 * ((r >> 1) & 1) + 8 * (((r >> 3) ^ r) & 1)) & (pieces - 1);
}

// float32 rows are read one 4-byte value per lane, 16 channels of four rows
// at a time: rows 16 floats apart in the banks spread them over all 64.
template <typename T, int TC>
constexpr int wg_row = sizeof(T) == 4 ? TC + 16 : TC;  // elements per staged row

template <typename T, int TC>
__device__ inline int wg_piece_slot(int r, int q) {
    if constexpr (sizeof(T) == 4) return r * wg_row<T, TC> + q * 4;
    return r * TC + ((q ^ wg_swizzle(r, TC / 8)) << 3);
}

typedef short short4_t __attribute__((ext_vector_type(4)));

// One MFMA operand fragment (16 channels x 32 edges) from edge-major LDS
// rows with two transposing reads.  In each 16-lane group, ds_read_b64_tr_b16
// gives lane i element i % 4 of the 8-byte chunks addressed by lanes
// i / 4 + 4j (j = 0..3).  Lane s of group g addresses row
// 32 ks + 8 g + 4 t + s / 4 at channel c0 + 4 (s % 4), so lane i receives
// channel c0 + i of four consecutive edges; the two reads (t = 0, 1) make
// the 8 edges 8 g .. 8 g + 7 the MFMA expects of lane i.
template <typename V, int TC, typename T>
__device__ inline V wg_fragment(const T* lds, int ks, int c0, int lane) {
    const int s = lane & 15;
    const int g = lane >> 4;
    const int q = (c0 >> 3) + ((s & 3) >> 1);
    short4_t h[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int r = 32 * ks + 8 * g + 4 * t + (s >> 2);
        const T* src = lds + wg_piece_slot<T, TC>(r, q) + 4 * (s & 1);
        h[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) short4_t*)(src));
    }
    typedef short short8_t __attribute__((ext_vector_type(8)));
    const short8_t both = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(V, both);
}

// Lock-step plan of the weight gradient.  The kernel-grouped edges of each
// offset are in output-row order, so part x (of kXcds equal parts) of every
// offset's edges covers about the same output rows.  The blocks of XCD x
// (launch index = x mod kXcds) all work on part x: S slots per XCD dealt
// to the offsets in proportion to their edge counts (at least one each),
// and the m_k blocks of offset k take its part's 64-edge chunks in turn
// (block j: chunks j, j + m_k, ...).  Every block then sums about the same
// number of edges, and all blocks of an XCD move through their part's
// output rows together, so the cotangent row of an output row, read once
// per offset, stays in that XCD's L2 between the offsets that read it.
constexpr int kXcds = 8;

// Blocks offset k gets on each XCD; first = blocks of the offsets before k.
__device__ inline void wg_share(const int32_t* koff, int K, int slots, int k, int* first, int* count) {
    const long long total = koff[K] - koff[0];
    int nz = 0;
    for (int i = 0; i < K; ++i) nz += koff[i + 1] > koff[i] ? 1 : 0;
    const long long spare = slots - nz;
    int acc = 0;
    *first = 0;
    *count = 0;
    for (int i = 0; i <= k; ++i) {
        const long long n = koff[i + 1] - koff[i];
        const int m = n > 0 ? 1 + static_cast<int>(spare * n / total) : 0;
        if (i == k) {
            *first = acc;
            *count = m;
        }
        acc += m;
    }
}

// Block (launch index): XCD x = index mod 8, then (tile, slot) from
// index / 8; channel tile TCI x TCO, four waves of (TCI/2) x (TCO/2).  Per
// step of 64 edges the block stages both operands into edge-major LDS rows.
// VEC: rows are whole 16-byte pieces (16-byte loads); otherwise every value
// is loaded by itself.  PAIRS: the grouped edges come as (input row, output
// row) pairs, one 8-byte load each, instead of as ids into the edge arrays
// (two dependent loads, the second of neighbours a row's degree apart).
template <typename T, int TCI, int TCO, bool VEC, bool PAIRS>
__global__ void __launch_bounds__(256, 3)
weight_grad_mfma(const T* __restrict__ feats, int n_in, int c_in, const T* __restrict__ cot, int n_out, int c_out,
                 const int32_t* __restrict__ in_rows, const int32_t* __restrict__ out_rows,
                 const int32_t* __restrict__ counts, int edge_capacity, const int32_t* __restrict__ koff,
                 const int32_t* __restrict__ kedges, const int2* __restrict__ kpairs, int K, int tiles, int tiles_co,
                 int slots, float* __restrict__ partial) {
    using V = typename GradMfma<T>::vec;
    constexpr int MB = TCI / 32;  // 16-row blocks per wave
    constexpr int NB = TCO / 32;  // 16-column blocks per wave
    constexpr int PE = 16 / static_cast<int>(sizeof(T));  // channels per 16-byte piece
    __shared__ __align__(16) T a_t[kWgEdges * wg_row<T, TCI>];
    __shared__ __align__(16) T b_t[kWgEdges * wg_row<T, TCO>];
    const int x = static_cast<int>(blockIdx.x) % kXcds;
    const int q = static_cast<int>(blockIdx.x) / kXcds;
    const int tile = q % tiles;
    const int slot = q / tiles;
    // The offset and the turn of this slot.
    int k = -1, turn = 0, turns = 0;
    {
        const long long total = koff[K] - koff[0];
        if (total <= 0) return;
        int nz = 0;
        for (int i = 0; i < K; ++i) nz += koff[i + 1] > koff[i] ? 1 : 0;
        const long long spare = slots - nz;
        int acc = 0;
        for (int i = 0; i < K; ++i) {
            const long long n = koff[i + 1] - koff[i];
            const int m = n > 0 ? 1 + static_cast<int>(spare * n / total) : 0;
            if (slot < acc + m) {
                k = i;
                turn = slot - acc;
                turns = m;
                break;
            }
            acc += m;
        }
    }
    if (k < 0) return;  // a spare slot: no partial tile is read for it
    const int ci0 = (tile / tiles_co) * TCI;
    const int co0 = (tile % tiles_co) * TCO;
    const int E = PAIRS ? edge_capacity : min(counts[0], edge_capacity);
    const int lo_k = koff[k];
    const long long n_k = koff[k + 1] - lo_k;
    const int lo = lo_k + static_cast<int>(n_k * x / kXcds);
    const int hi = lo_k + static_cast<int>(n_k * (x + 1) / kXcds);
    const int stride = turns * kWgEdges;  // the block's chunks: lo + 64 (turn + t turns)
    const int start = lo + turn * kWgEdges;

    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const int wm = wave & 1;
    const int wn = wave >> 1;
    const int lr = lane & 15;
    const int g = lane >> 4;
    float4_t acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[a][n] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Thread t stages edges t/8 and t/8 + 32 of the step: pieces t%8 + 8i of
    // their feature rows (i < PA) and cotangent rows (i < PB), so a wave's
    // loads cover eight whole 128-byte row lines.
    constexpr int PA = TCI / (8 * PE);
    constexpr int PB = TCO / (8 * PE);
    const int j = threadIdx.x >> 3;
    const int p = threadIdx.x & 7;
    V av[2][PA], bv[2][PB];
    bool aok[2][PA], bok[2][PB];
    // Three-stage pipeline over the steps: the edge ids of step s+3 and the
    // row indices of step s+2 are loaded while the rows of step s+1 are
    // gathered, so no step waits on a dependent index load.  Edges past the
    // share's end or outside the relation count as zeros.  Every load is
    // issued unconditionally (clamped address, validity kept aside) and the
    // index loads go out before the gathers: gfx950's vector-memory counter
    // retires in issue order, so a wait for an index issued after the
    // gathers would also wait for the gathers.
    const int last_edge = max(hi - 1, 0);
    auto issue_edges = [&](int base, int (&evr)[2], bool (&evv)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int cur = base + j + 32 * h;
            evv[h] = cur < hi;
            evr[h] = PAIRS ? cur : kedges[min(cur, last_edge)];
        }
    };
    auto edges_of = [&](const int (&evr)[2], const bool (&evv)[2], int (&ev)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) ev[h] = evv[h] ? evr[h] : -1;
    };
    auto issue_rows = [&](const int (&ev)[2], int (&rin)[2], int (&rout)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = ev[h] >= 0 && ev[h] < E ? ev[h] : 0;
            if constexpr (PAIRS) {
                const int2 io = kpairs[e];
                rin[h] = io.x;
                rout[h] = io.y;
            } else {
                rin[h] = in_rows[e];
                rout[h] = out_rows[e];
            }
        }
    };
    auto rows_of = [&](const int (&ev)[2], const int (&rin)[2], const int (&rout)[2], int (&ri)[2], int (&ro)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool ok = ev[h] >= 0 && ev[h] < E && rin[h] >= 0 && rin[h] < n_in && rout[h] >= 0 &&
                            rout[h] < n_out;
            ri[h] = ok ? rin[h] : -1;
            ro[h] = ok ? rout[h] : -1;
        }
    };
    // Channels c .. of a row (VEC: one load; c past the row re-reads its
    // start, masked when the piece is staged).
    auto load_piece = [&](const T* row, int c, int channels) {
        if constexpr (VEC) {
            return *reinterpret_cast<const V*>(row + (c < channels ? c : 0));
        } else {
            V v;
#pragma unroll
            for (int e = 0; e < PE; ++e) v[e] = row[min(c + e, channels - 1)];
            return v;
        }
    };
    auto staged_piece = [&](V v, bool ok, int c, int channels) {
        if constexpr (!VEC) {
#pragma unroll
            for (int e = 0; e < PE; ++e)
                if (c + e >= channels) v[e] = T(0);
        }
        return ok ? v : V{};
    };
    auto gather = [&](const int (&ri)[2], const int (&ro)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long long rin = ri[h] >= 0 ? ri[h] : 0, rout = ro[h] >= 0 ? ro[h] : 0;
#pragma unroll
            for (int i = 0; i < PA; ++i) {
                const int c = ci0 + PE * (p + 8 * i);
                aok[h][i] = ri[h] >= 0 && c < c_in;
                av[h][i] = load_piece(feats + rin * c_in, c, c_in);
            }
#pragma unroll
            for (int i = 0; i < PB; ++i) {
                const int c = co0 + PE * (p + 8 * i);
                bok[h][i] = ro[h] >= 0 && c < c_out;
                bv[h][i] = load_piece(cot + rout * c_out, c, c_out);
            }
        }
    };
    int ev[2], evr[2], ri[2], ro[2], rin[2], rout[2];
    bool evv[2];
    issue_edges(start, evr, evv);
    edges_of(evr, evv, ev);
    issue_rows(ev, rin, rout);
    rows_of(ev, rin, rout, ri, ro);
    gather(ri, ro);
    issue_edges(start + stride, evr, evv);
    edges_of(evr, evv, ev);
    issue_rows(ev, rin, rout);
    rows_of(ev, rin, rout, ri, ro);
    issue_edges(start + 2 * stride, evr, evv);
    edges_of(evr, evv, ev);
    for (int base = start; base < hi; base += stride) {
        // The thread's two edges take rows j and j + 32 (the order of edges
        // inside a step is free: the sum over them is in fp32).
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < PA; ++i)
                *reinterpret_cast<V*>(a_t + wg_piece_slot<T, TCI>(j + 32 * h, p + 8 * i)) =
                    staged_piece(av[h][i], aok[h][i], ci0 + PE * (p + 8 * i), c_in);
#pragma unroll
            for (int i = 0; i < PB; ++i)
                *reinterpret_cast<V*>(b_t + wg_piece_slot<T, TCO>(j + 32 * h, p + 8 * i)) =
                    staged_piece(bv[h][i], bok[h][i], co0 + PE * (p + 8 * i), c_out);
        }
        __syncthreads();
        issue_rows(ev, rin, rout);                   // row indices of step s+2
        int ev_next[2];
        {
            int evr_n[2];
            bool evv_n[2];
            issue_edges(base + 3 * stride, evr_n, evv_n);  // edge ids of step s+3
            // Keep the index loads ahead of the gathers in issue order.
            __builtin_amdgcn_sched_barrier(0);
            gather(ri, ro);  // rows of step s+1
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (sizeof(T) == 4) {
                // lane (lr, g): channel lr of edge 4 ks + g
#pragma unroll
                for (int ks = 0; ks < kWgEdges / 4; ++ks) {
                    float af[MB], bf[NB];
#pragma unroll
                    for (int m = 0; m < MB; ++m)
                        af[m] = a_t[(4 * ks + g) * wg_row<T, TCI> + (TCI / 2) * wm + 16 * m + lr];
#pragma unroll
                    for (int n = 0; n < NB; ++n)
                        bf[n] = b_t[(4 * ks + g) * wg_row<T, TCO> + (TCO / 2) * wn + 16 * n + lr];
#pragma unroll
                    for (int m = 0; m < MB; ++m)
#pragma unroll
                        for (int n = 0; n < NB; ++n)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[m], bf[n], acc[m][n], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    V af[MB], bf[NB];
#pragma unroll
                    for (int m = 0; m < MB; ++m)
                        af[m] = wg_fragment<V, TCI>(a_t, ks, (TCI / 2) * wm + 16 * m, lane);
#pragma unroll
                    for (int n = 0; n < NB; ++n)
                        bf[n] = wg_fragment<V, TCO>(b_t, ks, (TCO / 2) * wn + 16 * n, lane);
#pragma unroll
                    for (int m = 0; m < MB; ++m)
#pragma unroll
                        for (int n = 0; n < NB; ++n) acc[m][n] = GradMfma<T>::mfma(af[m], bf[n], acc[m][n]);
                }
            }
            edges_of(evr_n, evv_n, ev_next);
        }
        rows_of(ev, rin, rout, ri, ro);
        ev[0] = ev_next[0];
        ev[1] = ev_next[1];
        __syncthreads();
    }
    // D[m][n]: lane holds rows 4*(lane/16) + q, column lane%16 of each block.
    // The partial tile is stored as the lanes hold it (fragment order, one
    // 16-byte store per lane and block: whole 1 KB runs per wave); the
    // reduction maps each 4-float piece back to its (ci, co).
    float4_t* out = reinterpret_cast<float4_t*>(partial) +
                    (static_cast<long long>(x * slots + slot) * tiles + tile) * (TCI * TCO / 4);
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n) out[((wave * MB + m) * NB + n) * 64 + lane] = acc[m][n];
}

constexpr int kReduceBatch = 8;  // partial loads in flight per thread
constexpr int kReduceWaves = 4;

// dW[k] = sum of the partial tiles of offset k's blocks (XCD by XCD, then
// turn by turn), one rounding, written in the weight's layout.  Blocks
// (x, k): offset k's share is worked out once per thread, then the block
// strides over the partial matrix's 4-float pieces, 64 at a time; its four
// waves sum a quarter of the partials each, and the quarters are added in
// their order, so each entry keeps one summation order.  One thread per
// piece left a 64 x 64 weight 108 blocks of up to a hundred dependent
// additions: 18 us for fp32 over 60,001 rows, in quarters 10.  The pieces
// are in the fragment order of weight_grad_mfma: piece (tile, wave, m, n,
// lane) holds ci = ci0 + (TCI/2)*(wave&1) + 16m + 4(lane/16) + q, q < 4, and
// co = co0 + (TCO/2)*(wave>>1) + 16n + lane%16.
template <typename T>
__global__ void __launch_bounds__(kReduceWaves * kWave)
weight_grad_reduce(const float* __restrict__ partial, const int32_t* __restrict__ koff, int slots,
                   GradWeightIndex widx, int tci, int tco, int tiles, int tiles_co, T* __restrict__ grad) {
    const long long pieces = static_cast<long long>(tiles) * tci * tco / 4;  // per partial matrix
    const int mb = tci / 32, nb = tco / 32;
    const int k = blockIdx.y;
    int first = 0, count = 0;
    if (koff[widx.K] > koff[0]) wg_share(koff, widx.K, slots, k, &first, &count);
    const float4* p4 = reinterpret_cast<const float4*>(partial);
    __shared__ float4 quarter[kReduceWaves - 1][kWave];
    const int lane_of = lane_id();
    const int part = threadIdx.x / kWave;
    const int n = kXcds * count;
    const int begin = static_cast<int>(static_cast<long long>(n) * part / kReduceWaves);
    const int end = static_cast<int>(static_cast<long long>(n) * (part + 1) / kReduceWaves);
    // (tci * tco / 4 pieces per tile: whole 64s)
    for (long long w0 = static_cast<long long>(blockIdx.x) * kWave; w0 < pieces;
         w0 += static_cast<long long>(gridDim.x) * kWave) {
        const long long w4 = w0 + lane_of;
        // partial i of the (x, j) order: x = i / count, j = i % count;
        // kReduceBatch loads are issued before their adds, which run in that
        // order
        float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int i0 = begin; i0 < end; i0 += kReduceBatch) {
            float4 v[kReduceBatch];
#pragma unroll
            for (int u = 0; u < kReduceBatch; ++u) {
                const int i = i0 + u;
                const int x = count > 0 ? i / count : 0;
                const int j = i - x * count;
                v[u] = i < end ? p4[(x * slots + first + j) * pieces + w4] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
#pragma unroll
            for (int u = 0; u < kReduceBatch; ++u) {
                if (i0 + u < end) {
                    acc.x += v[u].x;
                    acc.y += v[u].y;
                    acc.z += v[u].z;
                    acc.w += v[u].w;
                }
            }
        }
        if (part > 0) quarter[part - 1][lane_of] = acc;
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int u = 0; u < kReduceWaves - 1; ++u) {
                const float4 v = quarter[u][lane_of];
                acc.x += v.x;
                acc.y += v.y;
                acc.z += v.z;
                acc.w += v.w;
            }
        }
        __syncthreads();
        if (part > 0) continue;
        const long long per_tile = static_cast<long long>(tci) * tco / 4;
        const int tile = static_cast<int>(w4 / per_tile);
        long long r = w4 - tile * per_tile;
        const int lane = static_cast<int>(r % 64);
        r /= 64;
        const int nn = static_cast<int>(r % nb);
        r /= nb;
        const int mm = static_cast<int>(r % mb);
        const int wave = static_cast<int>(r / mb);
        const int ci = (tile / tiles_co) * tci + (tci / 2) * (wave & 1) + 16 * mm + 4 * (lane >> 4);
        const int co = (tile % tiles_co) * tco + (tco / 2) * (wave >> 1) + 16 * nn + (lane & 15);
        const float a[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (ci + q < widx.c_in && co < widx.c_out) grad[widx(k, ci + q, co)] = static_cast<T>(a[q]);
        }
    }
}

// One lane per weight entry (k, ci, co), co fastest: the kernel-grouped
// edges of k in order with an fp32 accumulator (eval_weight_grad_typed's
// loop).  Used by callers that bring no workspace.
template <typename T>
__global__ void __launch_bounds__(256)
weight_grad_simple(const T* __restrict__ feats, int n_in, const T* __restrict__ cot, int n_out,
                   const int32_t* __restrict__ in_rows, const int32_t* __restrict__ out_rows,
                   const int32_t* __restrict__ counts, int edge_capacity, const int32_t* __restrict__ koff,
                   const int32_t* __restrict__ kedges, GradWeightIndex widx, T* __restrict__ grad) {
    const int c_in = widx.c_in;
    const int c_out = widx.c_out;
    const int E = min(counts[0], edge_capacity);
    const long long total = static_cast<long long>(widx.K) * c_in * c_out;
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<long long>(gridDim.x) * blockDim.x) {
        const int co = static_cast<int>(i % c_out);
        const int ci = static_cast<int>((i / c_out) % c_in);
        const int k = static_cast<int>(i / (static_cast<long long>(c_in) * c_out));
        float acc = 0.0f;
        for (int cur = koff[k]; cur < koff[k + 1]; ++cur) {
            const int e = kedges[cur];
            if (e < 0 || e >= E) continue;
            const int in = in_rows[e];
            const int o = out_rows[e];
            if (in < 0 || in >= n_in || o < 0 || o >= n_out) continue;
            acc += to_f(feats[static_cast<long long>(in) * c_in + ci]) * to_f(cot[static_cast<long long>(o) * c_out + co]);
        }
        grad[widx(k, ci, co)] = static_cast<T>(acc);
    }
}

int check_grad_dtype(int dtype) {
    LATTICE_REQUIRE(dtype == LATTICE_F32 || dtype == LATTICE_F16 || dtype == LATTICE_BF16,
                    "convolution gradients support float32, float16 and bfloat16.");
    return LATTICE_OK;
}

// Slots per XCD (blocks per channel tile = 8 x slots) of the matrix-core
// weight gradient: about 2,048 edge slots of the relation's capacity per
// block, at least one per offset, at most 96 (three blocks on each of an
// XCD's 32 CUs: one round, so the blocks of an XCD move together).
constexpr int kWgEdgesPerBlock = 2048;
constexpr int kWgMaxSlots = 96;
int weight_grad_slots(int edge_capacity, int kernel_count, int tiles) {
    const long long want =
        (static_cast<long long>(edge_capacity) + kXcds * kWgEdgesPerBlock - 1) / (kXcds * kWgEdgesPerBlock);
    return static_cast<int>(std::max<long long>(kernel_count, std::min<long long>(kWgMaxSlots / tiles, want)));
}

// Channel tiles of the matrix-core weight gradient: 128-channel tiles where
// the channels fill them, so one gather of an edge's rows serves every
// channel pair of the tile.
struct WgTiles {
    int tci, tco, tiles_ci, tiles_co;
    int tiles() const { return tiles_ci * tiles_co; }
};
// float32 takes tiles of 64 or 32: its MFMAs, a sixteenth of the 16-bit
// rate, cost more than a second gather of the rows, so padding to 128 or 64
// costs more than more tiles do (wider tiles' staged rows would also leave
// room for fewer blocks per CU).
// Rows that are not whole 16-byte pieces (vec false) take the narrow tile of
// their type: value by value, the wide tiles' loads spill.
WgTiles wg_tiles(int dtype, int c_in, int c_out, bool vec) {
    WgTiles t;
    const int wide = dtype == LATTICE_F32 ? 64 : 128;
    t.tci = vec && c_in > wide / 2 ? wide : wide / 2;
    t.tco = vec && c_out > wide / 2 ? wide : wide / 2;
    t.tiles_ci = (c_in + t.tci - 1) / t.tci;
    t.tiles_co = (c_out + t.tco - 1) / t.tco;
    return t;
}

// Block slots of the launch: one round of blocks per XCD whatever the number
// of channel tiles in float32 (its partial matrices would otherwise grow with
// their square); 16-bit tiles each take a round of their own.
int wg_slots(int dtype, int edge_capacity, int kernel_count, const WgTiles& t) {
    return weight_grad_slots(edge_capacity, kernel_count, dtype == LATTICE_F32 ? std::min(t.tiles(), 4) : 1);
}

// One fp32 partial matrix (every channel tile, in fragment order) per block
// slot; wide tiles (vec) need the most.
size_t weight_grad_partial_bytes(int dtype, int edge_capacity, int kernel_count, int c_in, int c_out) {
    const WgTiles t = wg_tiles(dtype, c_in, c_out, true);
    return static_cast<size_t>(kXcds) * wg_slots(dtype, edge_capacity, kernel_count, t) * t.tiles() * t.tci * t.tco *
           sizeof(float);
}

template <typename T>
void launch_input_grad(const void* cot, int out_capacity, const void* weights, GradWeightIndex widx,
                       const int32_t* out_rows, const int32_t* kernel_ids, const int32_t* counts, int edge_capacity,
                       const int32_t* in_row_offsets, const int32_t* in_edge_ids, int in_capacity, void* grad,
                       hipStream_t stream) {
    const long long nw = static_cast<long long>(widx.K) * widx.c_in * widx.c_out;
    const bool staged = nw <= kGradLdsFloats;
    const unsigned grid = grid_for(static_cast<long long>(in_capacity) * widx.c_in, 256,
                                   staged ? kGradStagedBlocks : 1u << 16);
    input_grad_csr<T><<<grid, 256, staged ? nw * sizeof(float) : 0, stream>>>(
        static_cast<const T*>(cot), out_capacity, static_cast<const T*>(weights), widx, out_rows, kernel_ids, counts,
        edge_capacity, in_row_offsets, in_edge_ids, in_capacity, static_cast<T*>(grad), staged);
}

template <typename T>
int launch_weight_grad(int dtype, const void* feats, int n_in, const void* cot, int n_out, GradWeightIndex widx,
                       const int32_t* in_rows, const int32_t* out_rows, const int32_t* counts, int edge_capacity,
                       const int32_t* koff, const int32_t* kedges, const int2* kpairs, void* grad, void* workspace,
                       size_t workspace_bytes, hipStream_t stream) {
    const size_t need = weight_grad_partial_bytes(dtype, edge_capacity, widx.K, widx.c_in, widx.c_out);
    // Without its workspace (or, for float32 and odd channel counts, with a
    // smaller one) the call runs one lane per weight value.
    const bool sixteens = dtype != LATTICE_F32 && widx.c_in % 8 == 0 && widx.c_out % 8 == 0;
    if (workspace != nullptr && (sixteens || workspace_bytes >= need)) {
        LATTICE_REQUIRE(workspace_bytes >= need, "weight gradient workspace too small.");
        float* partial = static_cast<float*>(workspace);
        const bool vec = (reinterpret_cast<uintptr_t>(feats) | reinterpret_cast<uintptr_t>(cot) |
                          (static_cast<uintptr_t>(widx.c_in) * sizeof(T)) |
                          (static_cast<uintptr_t>(widx.c_out) * sizeof(T))) %
                             16 ==
                         0;
        const WgTiles wt = wg_tiles(dtype, widx.c_in, widx.c_out, vec);
        const int slots = wg_slots(dtype, edge_capacity, widx.K, wt);
        const int tci = wt.tci, tco = wt.tco, tiles_co = wt.tiles_co, tiles = wt.tiles();
        const unsigned grid = static_cast<unsigned>(kXcds) * slots * tiles;
#define LATTICE_WG_KERNEL(A, B, VEC, PAIRS)                                                                     \
    weight_grad_mfma<T, A, B, VEC, PAIRS><<<grid, 256, 0, stream>>>(                                            \
        static_cast<const T*>(feats), n_in, widx.c_in, static_cast<const T*>(cot), n_out, widx.c_out, in_rows,   \
        out_rows, counts, edge_capacity, koff, kedges, kpairs, widx.K, tiles, tiles_co, slots, partial)
#define LATTICE_WG_LAUNCH(A, B, VEC)                                     \
    do {                                                                 \
        if (kpairs != nullptr) LATTICE_WG_KERNEL(A, B, VEC, true);       \
        else LATTICE_WG_KERNEL(A, B, VEC, false);                        \
    } while (0)
        constexpr int W = sizeof(T) == 4 ? 64 : 128;
        if (!vec) LATTICE_WG_LAUNCH(W / 2, W / 2, false);
        else if (tci == W && tco == W) LATTICE_WG_LAUNCH(W, W, true);
        else if (tci == W) LATTICE_WG_LAUNCH(W, W / 2, true);
        else if (tco == W) LATTICE_WG_LAUNCH(W / 2, W, true);
        else LATTICE_WG_LAUNCH(W / 2, W / 2, true);
#undef LATTICE_WG_LAUNCH
#undef LATTICE_WG_KERNEL
        LATTICE_LAUNCH_CHECK();
        const long long pieces = static_cast<long long>(tiles) * tci * tco / 4;
        const dim3 rgrid(grid_for(pieces, kWave, 1024), static_cast<unsigned>(widx.K));
        weight_grad_reduce<T><<<rgrid, kReduceWaves * kWave, 0, stream>>>(partial, koff, slots, widx, tci, tco, tiles, tiles_co,
                                                         static_cast<T*>(grad));
        LATTICE_LAUNCH_CHECK();
        return LATTICE_OK;
    }
    LATTICE_REQUIRE(kpairs == nullptr, "weight gradient workspace too small.");
    const long long total = static_cast<long long>(widx.K) * widx.c_in * widx.c_out;
    weight_grad_simple<T><<<grid_for(total, 256, 1u << 16), 256, 0, stream>>>(
        static_cast<const T*>(feats), n_in, static_cast<const T*>(cot), n_out, in_rows, out_rows, counts,
        edge_capacity, koff, kedges, widx, static_cast<T*>(grad));
    LATTICE_LAUNCH_CHECK();
    return LATTICE_OK;
}

}  // namespace
}  // namespace lattice

using namespace lattice;

extern "C" int lattice_hip_sparse_conv_input_grad(int dtype, const void* cot, int out_capacity, int c_out,
                                                  const void* weights, int weight_layout, int kernel_count, int c_in,
                                                  const int32_t* out_rows, const int32_t* kernel_ids,
                                                  const int32_t* counts, int edge_capacity,
                                                  const int32_t* in_row_offsets, const int32_t* in_edge_ids,
                                                  int in_capacity, void* grad, void* stream_ptr) {
    int rc = check_grad_dtype(dtype);
    if (rc != LATTICE_OK) return rc;
    LATTICE_REQUIRE(out_capacity >= 0 && in_capacity >= 0 && c_in > 0 && c_out > 0 && kernel_count > 0,
                    "gradient shapes must be positive.");
    LATTICE_REQUIRE(weight_layout == LATTICE_WEIGHT_KERNEL_MAJOR || weight_layout == LATTICE_WEIGHT_DENSE_5D,
                    "weights must have shape (K, C_in, C_out) or (C_out, Kx, Ky, Kz, C_in).");
    if (in_capacity == 0) return LATTICE_OK;
    LATTICE_REQUIRE(weights && out_rows && kernel_ids && counts && in_row_offsets && in_edge_ids && grad &&
                        (cot || out_capacity == 0),
                    "gradient pointers must be non-null.");
    hipStream_t stream = as_stream(stream_ptr);
    GradWeightIndex widx{weight_layout, kernel_count, c_in, c_out};
    if (dtype == LATTICE_F32) {
        launch_input_grad<float>(cot, out_capacity, weights, widx, out_rows, kernel_ids, counts, edge_capacity,
                                 in_row_offsets, in_edge_ids, in_capacity, grad, stream);
    } else if (dtype == LATTICE_F16) {
        launch_input_grad<_Float16>(cot, out_capacity, weights, widx, out_rows, kernel_ids, counts, edge_capacity,
                                    in_row_offsets, in_edge_ids, in_capacity, grad, stream);
    } else {
        launch_input_grad<__bf16>(cot, out_capacity, weights, widx, out_rows, kernel_ids, counts, edge_capacity,
                                  in_row_offsets, in_edge_ids, in_capacity, grad, stream);
    }
    LATTICE_LAUNCH_CHECK();
    return LATTICE_OK;
}

namespace lattice {
namespace {

// Offset masks of a transposed map.
int launch_transposed_masks(const int32_t* in_out_map, int in_capacity, int kernel_count, int32_t* row_masks,
                            hipStream_t stream) {
    const int words = (kernel_count + 31) / 32;
    // At most 64 KB of map rows per block, and at most one row per lane.
    const int rows_per_block = std::max(1, std::min(256, 16384 / kernel_count));
    const size_t lds = static_cast<size_t>(rows_per_block) * kernel_count * sizeof(int32_t);
    LATTICE_REQUIRE(lds <= 65536, "kernel count too large for the transposed masks.");
    transposed_masks<<<grid_for(in_capacity, rows_per_block, 1u << 16), 256, lds, stream>>>(
        in_out_map, in_capacity, kernel_count, words, rows_per_block, row_masks);
    LATTICE_LAUNCH_CHECK();
    return LATTICE_OK;
}

}  // namespace
}  // namespace lattice

extern "C" int lattice_hip_build_transposed_implicit_gemm_map(const int32_t* in_rows, const int32_t* out_rows,
                                                             const int32_t* kernel_ids, const int32_t* counts,
                                                             int edge_capacity, int in_capacity, int kernel_count,
                                                             int32_t* in_out_map, int32_t* row_masks,
                                                             int32_t* status, void* stream_ptr) {
    LATTICE_REQUIRE(edge_capacity >= 0 && in_capacity >= 0 && kernel_count > 0,
                    "transposed map shapes must be nonnegative with a positive kernel count.");
    if (status != nullptr) {
        const int rc = fill_i32(status, 1, 0, as_stream(stream_ptr));
        if (rc != LATTICE_OK) return rc;
    }
    if (in_capacity == 0) return LATTICE_OK;
    LATTICE_REQUIRE(in_out_map && row_masks && counts && (edge_capacity == 0 || (in_rows && out_rows && kernel_ids)),
                    "transposed map pointers must be non-null.");
    hipStream_t stream = as_stream(stream_ptr);
    int rc = fill_i32(in_out_map, static_cast<long long>(in_capacity) * kernel_count, -1, stream);
    if (rc != LATTICE_OK) return rc;
    if (edge_capacity > 0) {
        transposed_map<<<grid_for(edge_capacity, 256, 1u << 16), 256, 0, stream>>>(
            in_rows, out_rows, kernel_ids, counts, edge_capacity, in_capacity, kernel_count, in_out_map, status);
        LATTICE_LAUNCH_CHECK();
    }
    return launch_transposed_masks(in_out_map, in_capacity, kernel_count, row_masks, stream);
}

extern "C" int lattice_hip_build_transposed_map_from_dense(const int32_t* out_in_map, int out_capacity,
                                                           int in_capacity, int kernel_count, int32_t* in_out_map,
                                                           int32_t* row_masks, int32_t* status, void* stream_ptr) {
    LATTICE_REQUIRE(out_capacity >= 0 && in_capacity >= 0 && kernel_count > 0,
                    "transposed map shapes must be nonnegative with a positive kernel count.");
    hipStream_t stream = as_stream(stream_ptr);
    if (status != nullptr) {
        const int rc = fill_i32(status, 1, 0, stream);
        if (rc != LATTICE_OK) return rc;
    }
    if (in_capacity == 0) return LATTICE_OK;
    LATTICE_REQUIRE(in_out_map && row_masks && (out_capacity == 0 || out_in_map),
                    "transposed map pointers must be non-null.");
    int rc = fill_i32(in_out_map, static_cast<long long>(in_capacity) * kernel_count, -1, stream);
    if (rc != LATTICE_OK) return rc;
    const long long entries = static_cast<long long>(out_capacity) * kernel_count;
    if (entries > 0) {
        transposed_dense_map<<<grid_for(entries, 256, 1u << 16), 256, 0, stream>>>(out_in_map, entries, kernel_count,
                                                                                  in_capacity, in_out_map, status);
        LATTICE_LAUNCH_CHECK();
    }
    return launch_transposed_masks(in_out_map, in_capacity, kernel_count, row_masks, stream);
}

extern "C" size_t lattice_hip_conv_weight_grad_workspace_bytes(int dtype, int kernel_count, int c_in, int c_out,
                                                                int edge_capacity) {
    if (dtype != LATTICE_F32 && dtype != LATTICE_F16 && dtype != LATTICE_BF16) return 0;
    if (kernel_count <= 0 || c_in <= 0 || c_out <= 0) return 0;
    return weight_grad_partial_bytes(dtype, edge_capacity, kernel_count, c_in, c_out);
}

extern "C" int lattice_hip_sparse_conv_weight_grad(int dtype, const void* feats, int n_in, int c_in, const void* cot,
                                                   int out_capacity, int c_out, int weight_layout, int kernel_count,
                                                   const int32_t* in_rows, const int32_t* out_rows,
                                                   const int32_t* counts, int edge_capacity,
                                                   const int32_t* kernel_row_offsets,
                                                   const int32_t* kernel_edge_ids, void* grad, void* workspace,
                                                   size_t workspace_bytes, void* stream_ptr) {
    int rc = check_grad_dtype(dtype);
    if (rc != LATTICE_OK) return rc;
    LATTICE_REQUIRE(n_in >= 0 && out_capacity >= 0 && c_in > 0 && c_out > 0 && kernel_count > 0,
                    "gradient shapes must be positive.");
    LATTICE_REQUIRE(weight_layout == LATTICE_WEIGHT_KERNEL_MAJOR || weight_layout == LATTICE_WEIGHT_DENSE_5D,
                    "weights must have shape (K, C_in, C_out) or (C_out, Kx, Ky, Kz, C_in).");
    LATTICE_REQUIRE(grad && counts && kernel_row_offsets && (edge_capacity == 0 || (in_rows && out_rows && kernel_edge_ids)),
                    "gradient pointers must be non-null.");
    hipStream_t stream = as_stream(stream_ptr);
    GradWeightIndex widx{weight_layout, kernel_count, c_in, c_out};
    if (dtype == LATTICE_F32) {
        return launch_weight_grad<float>(dtype, feats, n_in, cot, out_capacity, widx, in_rows, out_rows, counts,
                                         edge_capacity, kernel_row_offsets, kernel_edge_ids, nullptr, grad, workspace,
                                         workspace_bytes, stream);
    }
    if (dtype == LATTICE_F16) {
        return launch_weight_grad<_Float16>(dtype, feats, n_in, cot, out_capacity, widx, in_rows, out_rows, counts,
                                            edge_capacity, kernel_row_offsets, kernel_edge_ids, nullptr, grad, workspace,
                                            workspace_bytes, stream);
    }
    return launch_weight_grad<__bf16>(dtype, feats, n_in, cot, out_capacity, widx, in_rows, out_rows, counts,
                                      edge_capacity, kernel_row_offsets, kernel_edge_ids, nullptr, grad, workspace,
                                      workspace_bytes, stream);
}

extern "C" size_t lattice_hip_kernel_pairs_workspace_bytes(int rows) {
    return aligned_bytes(std::max<size_t>(group_blocks(rows), 1) * kGroupBins * sizeof(int32_t)) + 256;
}

extern "C" int lattice_hip_build_kernel_pairs(const int32_t* row_masks, const int32_t* out_in_map,
                                              const int32_t* row_offsets, int rows, int kernel_count,
                                              int edge_capacity, int32_t* kernel_row_offsets, int32_t* pairs,
                                              int32_t* kernel_edge_ids, void* workspace, size_t workspace_bytes,
                                              void* stream_ptr) {
    LATTICE_REQUIRE(rows >= 0 && edge_capacity >= 0 && kernel_count > 0 && kernel_count <= kGroupBins,
                    "kernel pairs need nonnegative capacities and K <= 32.");
    LATTICE_REQUIRE(kernel_row_offsets != nullptr, "kernel pair pointers must be non-null.");
    LATTICE_REQUIRE(rows == 0 || edge_capacity == 0 ||
                        (row_masks && (pairs || kernel_edge_ids) && (!pairs || out_in_map) &&
                         (!kernel_edge_ids || row_offsets)),
                    "kernel pair pointers must be non-null.");
    LATTICE_REQUIRE(reinterpret_cast<uintptr_t>(pairs) % 8 == 0, "kernel pairs must be 8-byte aligned.");
    LATTICE_REQUIRE(workspace != nullptr && workspace_bytes >= lattice_hip_kernel_pairs_workspace_bytes(rows),
                    "kernel pairs workspace too small.");
    hipStream_t stream = as_stream(stream_ptr);
    if (rows == 0 || edge_capacity == 0) return fill_i32(kernel_row_offsets, kernel_count + 1, 0, stream);
    Workspace ws{static_cast<char*>(workspace), workspace_bytes};
    const int blocks = static_cast<int>(group_blocks(rows));
    int32_t* places = ws.take<int32_t>(static_cast<size_t>(blocks) * kGroupBins);
    LATTICE_REQUIRE(places != nullptr, "kernel pairs workspace too small.");
    group_count<<<blocks, kGroupRows, 0, stream>>>(row_masks, rows, kernel_count, places);
    LATTICE_LAUNCH_CHECK();
    group_scan<<<1, 1024, 0, stream>>>(places, blocks, kernel_count, kernel_row_offsets);
    LATTICE_LAUNCH_CHECK();
    group_emit<<<blocks, kGroupRows, 0, stream>>>(row_masks, out_in_map, row_offsets, rows, kernel_count,
                                                  edge_capacity, places, reinterpret_cast<int2*>(pairs),
                                                  kernel_edge_ids);
    LATTICE_LAUNCH_CHECK();
    return LATTICE_OK;
}

extern "C" int lattice_hip_sparse_conv_weight_grad_pairs(int dtype, const void* feats, int n_in, int c_in,
                                                         const void* cot, int out_capacity, int c_out,
                                                         int weight_layout, int kernel_count, const int32_t* pairs,
                                                         int edge_capacity, const int32_t* kernel_row_offsets,
                                                         void* grad, void* workspace, size_t workspace_bytes,
                                                         void* stream_ptr) {
    int rc = check_grad_dtype(dtype);
    if (rc != LATTICE_OK) return rc;
    LATTICE_REQUIRE(n_in >= 0 && out_capacity >= 0 && c_in > 0 && c_out > 0 && kernel_count > 0 && edge_capacity >= 0,
                    "gradient shapes must be positive.");
    LATTICE_REQUIRE(weight_layout == LATTICE_WEIGHT_KERNEL_MAJOR || weight_layout == LATTICE_WEIGHT_DENSE_5D,
                    "weights must have shape (K, C_in, C_out) or (C_out, Kx, Ky, Kz, C_in).");
    LATTICE_REQUIRE(grad && kernel_row_offsets && pairs && workspace, "gradient pointers must be non-null.");
    LATTICE_REQUIRE(reinterpret_cast<uintptr_t>(pairs) % 8 == 0, "kernel pairs must be 8-byte aligned.");
    hipStream_t stream = as_stream(stream_ptr);
    GradWeightIndex widx{weight_layout, kernel_count, c_in, c_out};
    const int2* p = reinterpret_cast<const int2*>(pairs);
    if (dtype == LATTICE_F32) {
        return launch_weight_grad<float>(dtype, feats, n_in, cot, out_capacity, widx, nullptr, nullptr, nullptr,
                                         edge_capacity, kernel_row_offsets, nullptr, p, grad, workspace,
                                         workspace_bytes, stream);
    }
    if (dtype == LATTICE_F16) {
        return launch_weight_grad<_Float16>(dtype, feats, n_in, cot, out_capacity, widx, nullptr, nullptr, nullptr,
                                            edge_capacity, kernel_row_offsets, nullptr, p, grad, workspace,
                                            workspace_bytes, stream);
    }
    return launch_weight_grad<__bf16>(dtype, feats, n_in, cot, out_capacity, widx, nullptr, nullptr, nullptr,
                                      edge_capacity, kernel_row_offsets, nullptr, p, grad, workspace, workspace_bytes,
                                      stream);
}
