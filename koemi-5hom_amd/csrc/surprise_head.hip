// Causal surprise from the prior states: the content head's product with the row
// scoring in its epilogue, and the backward of both.
//
// Reference: src/koemi/cuda_kernels/think/surprise_kernel.cu:194-328 (an fp32
// library product, a row kernel over its logits, and in the backward the
// product again, a row kernel writing the logits' gradient and two more library
// products). Here the forward's logits stay on chip (few rows of a wide state aside):
// a workgroup holds 64 rows x 256 or 64 vocabulary columns in its accumulators, scores
// them there and keeps (max, sum of exponentials, negative log-likelihood) per row
// for the backward, whose first kernel forms the logits again and writes their
// gradient G (fp32). The weight gradients contract G with the states and the weights, with G split into
// three bf16 planes that sum to it exactly (split_gemm.hpp): bf16 and fp16
// states and weights are never widened in memory, and a product with fp32 drops
// at most 2^-24 of itself, without bias.
#include "column_sum.hpp"
#include "common.hpp"
#include "detmath.hpp"
#include "split_gemm.hpp"

#include <algorithm>

namespace koemi {
namespace {

using split_gemm::kElementLoads;
using split_gemm::kThreads;

constexpr int kRows = 64;  // rows of a head tile
// Vocabulary columns of a head tile: 256, so that a byte vocabulary is scored in
// one, or 64 where the 256-column tiles would leave most CUs idle, with four K steps
// of loads in flight since no second workgroup hides them (256 rows x
// 1024, fp32: 66 -> 26 us; a tile step costs its latency there).
constexpr int kWide = 256, kNarrow = 64;

template <typename T, int BN>
using HeadTile = split_gemm::Tile<T, T, kRows, BN, false, false, BN == kNarrow ? 4 : 1>;
// fp32 rows of 128 to 255 wide tiles gain from the narrow ones ([8192, 1024], vocabulary
// 256, with gradients: 208 and 163 us), 16-bit ones only lose a launch.
inline int head_columns(int64_t rows, int64_t V, bool fp32) {
    return (rows + kRows - 1) / kRows * ((V + kWide - 1) / kWide) < (fp32 ? 256 : 128) ? kNarrow : kWide;
}

// The logits of the workgroup's rows and vocabulary columns [v0, v0 + BN), in
// the accumulators: lane l of wave (wm, wn) holds row 32 wm + l % 32, columns
// BN / 2 wn + 32 j + acc_column(v). Columns past V repeat column V - 1.
template <int BYTES, int BN, typename T>
__device__ __forceinline__ void head_logits(HeadTile<T, BN>& tile, char* lds, const T* __restrict__ prior,
                                            const T* __restrict__ weight, int64_t row0, int64_t v0, int64_t rows,
                                            int64_t D, int64_t V) {
    const int wn = threadIdx.x / kWave & 1;
    const uint64_t chains = tile.template run<BYTES, BYTES>(
        lds, D, D, 0, (D + HeadTile<T, BN>::BK - 1) / HeadTile<T, BN>::BK * HeadTile<T, BN>::BK,
        [&](int r) { return prior + min(row0 + r, rows - 1) * D; },
        [&](int r) { return weight + min(v0 + r, V - 1) * D; }, [&](int t) { return wn * (BN / 2) + t * 32; });
    if constexpr (!HeadTile<T, BN>::kNative) {
        if (__builtin_expect(__ballot(chains != 0) == 0, 1)) return;
        const int wm = threadIdx.x / kWave >> 1;
        const int64_t row = min(row0 + wm * 32 + (lane_id() & 31), rows - 1);
#pragma unroll
        for (int j = 0; j < HeadTile<T, BN>::NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (chains >> (j * 16 + v) & 1)
                    tile.acc[0][j][v] = split_gemm::scalar_dot(
                        prior + row * D, weight + min(v0 + wn * (BN / 2) + j * 32 + split_gemm::acc_column(v), V - 1) * D, D,
                        0.0f);
    }
}

// The score of a row from its logits' maximum, sum of exponentials and target
// logit (surprise_kernel.cu:84-134).
template <typename T>
__device__ __forceinline__ void finish_row(float m, float sum, float target, bool in, bool live, float log_vocab,
                                           int64_t row, int64_t rows, T* __restrict__ out, float* __restrict__ stats) {
#pragma clang fp contract(off)
    const float nll = (detmath::det_logf(sum) + m) - target;
    float s = 0.0f;
    if (live) s = in ? 1.0f - detmath::det_expf(-nll / log_vocab) : __builtin_nanf("");
    out[row] = from_f32<T>(s);
    stats[row] = m;
    stats[rows + row] = sum;
    stats[2 * rows + row] = nll;
}

// Scores: one workgroup per 64 rows and 256 columns. A vocabulary of one tile is
// finished here; with more, the tiles' (maximum, sum, target logit) go to `part`
// [tiles, 3, rows] and surprise_head_finish_kernel joins them. Bound by its one round
// of tiles (the states from HBM, the weights from L2); [32768, 512] bf16,
// vocabulary 256: 22 us, against two casts (21), the library's fp32 product (70)
// and the row kernel (9).
template <typename T, int BN, int BYTES>
__global__ __launch_bounds__(kThreads, 2) void surprise_head_forward_kernel(
    const T* __restrict__ prior, const T* __restrict__ weight, const T* __restrict__ bias,
    const int64_t* __restrict__ targets, const uint8_t* __restrict__ valid, T* __restrict__ out,
    float* __restrict__ stats, float* __restrict__ part, int64_t rows, int64_t D, int64_t V, int64_t v_tiles,
    float log_vocab) {
#pragma clang fp contract(off)
    using Tile = HeadTile<T, BN>;
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes];
    __shared__ __attribute__((aligned(16))) float bias_sh[BN];
    __shared__ float red[2][kRows], sums[2][kRows], target_sh[kRows];
    const int tid = threadIdx.x, wave = tid / kWave, wm = wave >> 1, wn = wave & 1;
    const int r = wm * 32 + (lane_id() & 31);
    const int64_t row0 = blockIdx.x / v_tiles * kRows, tile_v = blockIdx.x % v_tiles, v0 = tile_v * BN;
    const int64_t row = min(row0 + r, rows - 1);
    const int64_t t = targets[row];
    const int c0 = wn * (BN / 2) + 4 * (lane_id() >> 5);
    if (tid < BN) bias_sh[tid] = to_f32(bias[min(v0 + tid, V - 1)]);
    if (tid < kRows) target_sh[tid] = 0.0f;
    Tile tile;
    head_logits<BYTES, BN>(tile, lds, prior, weight, row0, v0, rows, D, V);  // barriers inside: the biases are visible
    // columns from this lane's first one: the tile's valid ones and the target
    const int here = static_cast<int>(min(V - v0, static_cast<int64_t>(BN))) - c0;
    const int hit = t >= v0 && t < v0 + BN ? static_cast<int>(t - v0) - c0 : -1;
    float m = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < Tile::NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int c = j * 32 + 8 * (v / 4) + v % 4;
            const float z = tile.acc[0][j][v] + bias_sh[c0 + c];
            if (c == hit) target_sh[r] = z;
            tile.acc[0][j][v] = c < here ? z : -__builtin_inff();
            m = fmaxf(m, tile.acc[0][j][v]);
        }
    m = fmaxf(m, __shfl_xor(m, 32, kWave));
    red[wn][r] = m;  // both halves of the wave hold the row's value
    __syncthreads();
    m = fmaxf(red[0][r], red[1][r]);
    // one of several tiles with no logit above minus infinity: its sum is 0, and NaN
    // where one of them is NaN (which fmaxf passes over)
    const float ref = v_tiles > 1 && !(m > -__builtin_inff()) ? 0.0f : m;
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < Tile::NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float e = detmath::det_expf_nonpos(tile.acc[0][j][v] - ref);
            if (j * 32 + 8 * (v / 4) + v % 4 < here) sum = sum + e;
        }
    sum = sum + __shfl_xor(sum, 32, kWave);
    sums[wn][r] = sum;
    __syncthreads();
    if (wn != 0 || lane_id() >= 32 || row0 + r >= rows) return;
    sum = sums[0][r] + sums[1][r];
    if (v_tiles == 1) {
        finish_row(m, sum, target_sh[r], t >= 0 && t < V, valid[row] != 0, log_vocab, row, rows, out, stats);
    } else {
        float* p = part + tile_v * 3 * rows + row;
        p[0] = m;
        p[rows] = sum;
        p[2 * rows] = target_sh[r];  // 0 in every tile but the target's
    }
}

// Joins the vocabulary tiles of surprise_head_forward_kernel: a thread per row, or a
// wave per row (LANES 64) where the tiles are many and one thread would load them one
// after the other ([16, 4096], vocabulary 50257: 326 -> 11 us).
constexpr int64_t kThreadTiles = 16;
template <typename T, int LANES>
__global__ void surprise_head_finish_kernel(const float* __restrict__ part, const int64_t* __restrict__ targets,
                                            const uint8_t* __restrict__ valid, T* __restrict__ out,
                                            float* __restrict__ stats, int64_t rows, int64_t V, int64_t v_tiles,
                                            int columns, float log_vocab) {
#pragma clang fp contract(off)
    const int64_t row = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / LANES;
    if (row >= rows) return;
    const int lane = threadIdx.x % LANES;
    const float* p = part + row;
    const int64_t t = targets[row];
    float m = -__builtin_inff(), sum = 0.0f;
    for (int64_t i = lane; i < v_tiles; i += LANES) m = fmaxf(m, p[i * 3 * rows]);
    if constexpr (LANES == kWave) m = wave_max_xor(m);
    for (int64_t i = lane; i < v_tiles; i += LANES)  // a tile of minus infinities adds 0, a NaN stays
        sum = sum + p[(i * 3 + 1) * rows] * detmath::det_expf_nonpos(p[i * 3 * rows] - m);
    if constexpr (LANES == kWave) sum = wave_sum_xor(sum);
    const bool in = t >= 0 && t < V;
    if (lane == 0)
        finish_row(m, sum, in ? p[(t / columns * 3 + 2) * rows] : 0.0f, in, valid[row] != 0, log_vocab, row, rows, out,
                   stats);
}

// Few 64 x 64 tiles and a wide state: each tile's sum over the width in chunks, so
// that the chip is full ([64, 4096] fp32, vocabulary 256: forward 85 -> 17 us, a
// tile's walk over its 128 K steps before). The chunks' logits go to part
// [chunks, rows, V] and are added (column_sum.hpp) for the two kernels after it. From
// 64 K steps on: two more launches cost a short walk more than it saves ([168, 1024]
// fp16, vocabulary 256: 137 us a call without, 150 with).
constexpr int64_t kLongWalk = 64;      // K steps
constexpr int64_t kSplitWidth = 256;   // width of a chunk at least
constexpr int64_t kMostSplitTiles = 512, kMostChunks = 16;
inline int64_t head_tiles_of(int64_t rows, int64_t V) { return (rows + 63) / 64 * ((V + 63) / 64); }
inline int64_t head_chunk(int64_t rows, int64_t D, int64_t V, bool fp32) {  // a chunk's width; D: one chunk
    if (D < kLongWalk * (fp32 ? HeadTile<float, kNarrow>::BK : HeadTile<bf16, kNarrow>::BK)) return D;
    // a workgroup to each CU, two of fp32 planes ([2048, 4096], vocabulary 256, with
    // gradients: 213 and 188 us; 16-bit operands: no shape gained)
    const int64_t tiles = (fp32 ? kMostSplitTiles : 256) / head_tiles_of(rows, V);
    const int64_t chunks = std::min({tiles, D / kSplitWidth, kMostChunks});
    return chunks < 2 ? D : ((D + chunks - 1) / chunks + 63) / 64 * 64;
}
inline int64_t head_chunks(int64_t rows, int64_t D, int64_t V, bool fp32) {
    const int64_t width = head_chunk(rows, D, V, fp32);
    return (D + width - 1) / width;
}
inline int64_t logits_floats(int64_t rows, int64_t V, int64_t chunks) {  // the logits and their chunks
    return (rows * V + 63) / 64 * 64 + chunks * rows * V;
}

template <typename T, int BYTES>
__global__ __launch_bounds__(kThreads, 2) void surprise_head_product_kernel(
    const T* __restrict__ prior, const T* __restrict__ weight, float* __restrict__ part, int64_t rows, int64_t D,
    int64_t V, int64_t v_tiles, int64_t tiles, int64_t chunk_width, int vec_out) {
    using Tile = HeadTile<T, kNarrow>;
    constexpr int kRegion = split_gemm::store_bytes<float, 1>();
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes > 4 * kRegion ? Tile::kLdsBytes : 4 * kRegion];
    const int64_t chunk = blockIdx.x / tiles, tile_id = blockIdx.x % tiles;
    const int64_t row0 = tile_id / v_tiles * kRows, v0 = tile_id % v_tiles * kNarrow;
    const int64_t k0 = chunk * chunk_width, k1 = min(D, k0 + chunk_width);  // chunk_width is a multiple of BK
    const int wave = threadIdx.x / kWave, wm = wave >> 1, wn = wave & 1;
    Tile tile;
    const uint64_t chains = tile.template run<BYTES, BYTES>(
        lds, D, D, k0, k1, [&](int r) { return prior + min(row0 + r, rows - 1) * D; },
        [&](int r) { return weight + min(v0 + r, V - 1) * D; }, [&](int) { return wn * 32; });
    if constexpr (Tile::kNative) split_gemm::lds_barrier();  // the output rows pass through LDS
    const int64_t row = row0 + wm * 32, first = v0 + wn * 32;
    float o[1][16];
#pragma unroll
    for (int v = 0; v < 16; ++v) o[0][v] = tile.acc[0][0][v];
    split_gemm::store_rows<float, 1>(lds + wave * kRegion, o, part + (chunk * rows + row) * V + first, V, rows - row,
                                     V - first, vec_out);
    split_gemm::fix_chains(chains, [&](int, int v) {
        const int64_t r = row + (lane_id() & 31), c = first + split_gemm::acc_column(v);
        if (r < rows && c < V)
            part[(chunk * rows + r) * V + c] = split_gemm::scalar_dot(prior + r * D + k0, weight + c * D + k0, k1 - k0, 0.0f);
    });
}

// Scores of logits [rows, V], a wave per row.
template <typename T>
__global__ __launch_bounds__(kThreads) void surprise_head_score_kernel(
    const float* __restrict__ logits, const T* __restrict__ bias, const int64_t* __restrict__ targets,
    const uint8_t* __restrict__ valid, T* __restrict__ out, float* __restrict__ stats, int64_t rows, int64_t V,
    float log_vocab) {
#pragma clang fp contract(off)
    const int64_t row = static_cast<int64_t>(blockIdx.x) * (kThreads / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;
    const float* z = logits + row * V;
    const int64_t t = targets[row];
    const bool in = t >= 0 && t < V;
    const float target = in ? z[t] + to_f32(bias[t]) : 0.0f;
    float m = -__builtin_inff();
#pragma unroll 4
    for (int64_t c = lane_id(); c < V; c += kWave) m = fmaxf(m, z[c] + to_f32(bias[c]));
    m = wave_max_xor(m);
    float sum = 0.0f;
#pragma unroll 4
    for (int64_t c = lane_id(); c < V; c += kWave) sum = sum + detmath::det_expf_nonpos((z[c] + to_f32(bias[c])) - m);
    sum = wave_sum_xor(sum);
    if (lane_id() == 0) finish_row(m, sum, target, in, valid[row] != 0, log_vocab, row, rows, out, stats);
}

// The logit gradient below of logits [rows, V]: 64 rows x 64 columns a workgroup,
// four rows to each of its waves (sixteen rows to a wave, one after the other: 15 us
// for 128 rows x 1000).
constexpr int kSplitGradThreads = 1024;
template <typename T>
__global__ __launch_bounds__(kSplitGradThreads) void surprise_head_split_grad_kernel(
    const float* __restrict__ logits, const T* __restrict__ bias, const int64_t* __restrict__ targets,
    const uint8_t* __restrict__ valid, const T* __restrict__ grad, const float* __restrict__ stats, float* __restrict__ G,
    float* __restrict__ bias_partial, int64_t rows, int64_t V, int64_t v_tiles, float log_vocab) {
#pragma clang fp contract(off)
    constexpr int kWaves = kSplitGradThreads / kWave;
    __shared__ float sums[kWaves][kWave];
    const int wave = threadIdx.x / kWave;
    const int64_t block = blockIdx.x / v_tiles, c = blockIdx.x % v_tiles * kWave + lane_id();
    const int64_t cc = min(c, V - 1);
    const float b = to_f32(bias[cc]);
    float acc[kRows / kWaves];
#pragma unroll
    for (int i = 0; i < kRows / kWaves; ++i) {
        const int64_t row = block * kRows + wave * (kRows / kWaves) + i, rr = min(row, rows - 1);
        const int64_t t = targets[rr];
        const bool live = row < rows && valid[rr] && t >= 0 && t < V;
        const float inv_sum = 1.0f / stats[rows + rr];
        const float gnll = to_f32(grad[rr]) * detmath::det_expf(-stats[2 * rows + rr] / log_vocab) / log_vocab;
        const float p = detmath::det_expf_nonpos((logits[rr * V + cc] + b) - stats[rr]) * inv_sum;
        acc[i] = live ? gnll * (p - (c == t ? 1.0f : 0.0f)) : 0.0f;
        if (row < rows && c < V) G[row * V + c] = acc[i];
    }
    static_assert(kRows / kWaves == 4, "the sum below");
    sums[wave][lane_id()] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
#pragma unroll
    for (int half = kWaves / 2; half > 0; half >>= 1) {
        if (wave < half) sums[wave][lane_id()] += sums[wave + half][lane_id()];
        __syncthreads();
    }
    if (wave == 0 && c < V) bias_partial[block * V + c] = sums[0][lane_id()];
}

// d score / d logits (surprise_kernel.cu:136-192), G [rows, V] fp32:
//   G_j = g exp(-nll / ln V) / ln V (softmax_j - [j == target]),
// zero for invalid rows, and the workgroup's 64-row column sums of it (the
// bias gradient's partial rows). At the sizes above 28 us, against the product
// (70), the row kernel (37) and the column sum (27).
template <typename T, int BN, int BYTES>
__global__ __launch_bounds__(kThreads, 2) void surprise_head_grad_logits_kernel(
    const T* __restrict__ prior, const T* __restrict__ weight, const T* __restrict__ bias,
    const int64_t* __restrict__ targets, const uint8_t* __restrict__ valid, const T* __restrict__ grad,
    const float* __restrict__ stats, float* __restrict__ G, float* __restrict__ bias_partial, int64_t rows, int64_t D,
    int64_t V, int64_t v_tiles, float log_vocab) {
#pragma clang fp contract(off)
    using Tile = HeadTile<T, BN>;
    constexpr int J = Tile::NT < 2 ? 1 : 2;
    constexpr int kRegion = split_gemm::store_bytes<float, J>();
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes > 4 * kRegion ? Tile::kLdsBytes : 4 * kRegion];
    __shared__ __attribute__((aligned(16))) float bias_sh[BN];
    __shared__ float column_sh[2][BN];
    const int tid = threadIdx.x, wave = tid / kWave, wm = wave >> 1, wn = wave & 1;
    const int r = wm * 32 + (lane_id() & 31);
    const int64_t block = blockIdx.x / v_tiles, row0 = block * kRows, v0 = blockIdx.x % v_tiles * BN;
    const int64_t row = min(row0 + r, rows - 1);
    const int64_t t = targets[row];
    const bool live = row0 + r < rows && valid[row] && t >= 0 && t < V;
    const float m = stats[row], inv_sum = 1.0f / stats[rows + row];
    const float gnll = to_f32(grad[row]) * detmath::det_expf(-stats[2 * rows + row] / log_vocab) / log_vocab;
    const int c0 = wn * (BN / 2) + 4 * (lane_id() >> 5);
    Tile tile;
    if (tid < BN) bias_sh[tid] = to_f32(bias[min(v0 + tid, V - 1)]);
    head_logits<BYTES, BN>(tile, lds, prior, weight, row0, v0, rows, D, V);
    if constexpr (Tile::kNative) split_gemm::lds_barrier();  // G passes through LDS
    const int hit = t >= v0 && t < v0 + BN ? static_cast<int>(t - v0) - c0 : -1;
#pragma unroll
    for (int j = 0; j < Tile::NT; j += J) {
        float o[J][16];
#pragma unroll
        for (int h = 0; h < J; ++h)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int c = (j + h) * 32 + 8 * (v / 4) + v % 4;
                const float p = detmath::det_expf_nonpos((tile.acc[0][j + h][v] + bias_sh[c0 + c]) - m) * inv_sum;
                o[h][v] = live ? gnll * (p - (c == hit ? 1.0f : 0.0f)) : 0.0f;
            }
        const int64_t first = v0 + wn * (BN / 2) + j * 32;
        split_gemm::store_rows<float, J>(lds + wave * kRegion, o, G + (row0 + wm * 32) * V + first, V,
                                         rows - row0 - wm * 32, V - first, V % 8 == 0);
        // lane l sums column l of the 32 rows the region still holds
        if (lane_id() < 32 * J) {
            const float* column = reinterpret_cast<const float*>(lds + wave * kRegion) + lane_id();
            // eight sums and a tree: few roundings follow a column's one large entry, its
            // target's (bias gradient of 128 rows, vocabulary 1000: 9.4e-8 from float64, 1.21e-7 in one sum)
            float acc[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = column[i * (kRegion / 32 / 4)];
#pragma unroll
            for (int i = 8; i < 32; ++i) acc[i % 8] += column[i * (kRegion / 32 / 4)];
#pragma unroll
            for (int n = 4; n > 0; n >>= 1)
#pragma unroll
                for (int i = 0; i < n; ++i) acc[i] += acc[i + n];
            column_sh[wm][wn * (BN / 2) + j * 32 + lane_id()] = acc[0];
        }
        asm volatile("" ::: "memory");  // the region is rewritten by the next columns
    }
    __syncthreads();
    if (tid < BN && v0 + tid < V)
        bias_partial[block * V + v0 + tid] = column_sh[0][tid] + column_sh[1][tid];
}

// grad_prior [rows, D] = G [rows, V] W [V, D]. Bound by its few K steps (eight at a
// vocabulary of 256) and the splits beside them. At the sizes above 50 us, against
// 77 for the library's fp32 product and 11 for the cast of its result. Of few tiles
// and a long vocabulary each takes the vocabulary [chunk * chunk_v, + chunk_v)
// (head_workspace), Out fp32 partial sums then ([16, 4096], vocabulary 50257:
// 2127 -> 563 us).
template <typename T, typename Out, int B, int BYTES>
__global__ __launch_bounds__(kThreads, 2) void surprise_head_grad_prior_kernel(
    const float* __restrict__ G, const T* __restrict__ weight, Out* __restrict__ grad_prior, int64_t rows, int64_t D,
    int64_t V, int64_t d_tiles, int64_t tiles, int64_t chunk_v, int vec_out) {
    constexpr int BM = B, BN = B;
    using Tile = split_gemm::Tile<float, T, BM, BN, false, true, B == 64 ? 4 : 1>;
    constexpr int J = Tile::NT < 2 ? 1 : 2;
    constexpr int kRegion = split_gemm::store_bytes<Out, J>();
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes > 4 * kRegion ? Tile::kLdsBytes : 4 * kRegion];
    const int64_t chunk = blockIdx.x / tiles, tile_id = blockIdx.x % tiles;
    const int64_t row0 = tile_id / d_tiles * BM, d0 = tile_id % d_tiles * BN;
    const int64_t k0 = chunk * chunk_v, k1 = min(V, k0 + chunk_v);  // chunk_v is a multiple of BK
    const int wave = threadIdx.x / kWave, wm = wave >> 1, wn = wave & 1;
    Tile tile;
    const uint64_t chains = tile.template run<BYTES, kElementLoads>(
        lds, V, V, k0, k1, [&](int r) { return G + min(row0 + r, rows - 1) * V; },
        [&](int r) { return weight + min(d0 + r, D - 1); }, [&](int t) { return wn * (BN / 2) + t * 32; }, 1, D);
#pragma unroll
    for (int i = 0; i < Tile::MT; ++i) {
        const int64_t block_row = row0 + wm * (BM / 2) + i * 32;
#pragma unroll
        for (int j0 = 0; j0 < Tile::NT; j0 += J) {
            const int64_t first = d0 + wn * (BN / 2) + j0 * 32;
            float o[J][16];
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[j][v] = tile.acc[i][j0 + j][v];
            split_gemm::store_rows<Out, J>(lds + wave * kRegion, o, grad_prior + (chunk * rows + block_row) * D + first, D,
                                           rows - block_row, D - first, vec_out);
        }
    }
    split_gemm::fix_chains(chains, [&](int block, int v) {
        const int64_t r = row0 + wm * (BM / 2) + block / Tile::NT * 32 + (lane_id() & 31);
        const int64_t c = d0 + wn * (BN / 2) + block % Tile::NT * 32 + split_gemm::acc_column(v);
        if (r < rows && c < D)
            grad_prior[(chunk * rows + r) * D + c] =
                from_f32<Out>(split_gemm::scalar_dot(G + r * V + k0, weight + k0 * D + c, k1 - k0, 0.0f, 1, D));
    });
}

// Partial sums of grad_weight [V, D] = G^T [V, rows] prior [rows, D] over the
// rows [chunk * chunk_rows, + chunk_rows): a vocabulary this small has few
// tiles, so the rows are split until the chip is full. At the sizes above 53 us (+ 7 for
// the sum of the chunks), against 406 for the library's fp32 product on few tiles. One
// chunk writes the gradient itself (Out T).
template <typename T, typename Out>
__global__ __launch_bounds__(kThreads, 2) void surprise_head_grad_weight_kernel(
    const float* __restrict__ G, const T* __restrict__ prior, Out* __restrict__ partial, int64_t rows, int64_t D,
    int64_t V, int64_t d_tiles, int64_t v_tiles, int64_t chunk_rows, int vec_out) {
    constexpr int BM = 128, BN = 128;
    using Tile = split_gemm::Tile<float, T, BM, BN, true, true>;
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes];
    const int64_t chunk = blockIdx.x / (d_tiles * v_tiles), tile_id = blockIdx.x % (d_tiles * v_tiles);
    const int64_t v0 = tile_id / d_tiles * BM, d0 = tile_id % d_tiles * BN;
    const int64_t k0 = chunk * chunk_rows, k1 = min(rows, k0 + chunk_rows);  // chunk_rows is a multiple of BK
    const int wave = threadIdx.x / kWave, wm = wave >> 1, wn = wave & 1;
    Tile tile;
    const uint64_t chains = tile.template run<kElementLoads, kElementLoads>(
        lds, rows, rows, k0, k1, [&](int r) { return G + min(v0 + r, V - 1); },
        [&](int r) { return prior + min(d0 + r, D - 1); }, [&](int t) { return wn * 64 + t * 32; }, V, D);
    constexpr int kRegion = split_gemm::store_bytes<Out, 1>();
    static_assert(4 * kRegion <= Tile::kLdsBytes, "the output regions fit the operands' LDS");
#pragma unroll
    for (int i = 0; i < Tile::MT; ++i) {
        const int64_t block_v = v0 + wm * (BM / 2) + i * 32;
#pragma unroll
        for (int j = 0; j < Tile::NT; ++j) {
            const int64_t first = d0 + wn * 64 + j * 32;
            float o[1][16];
#pragma unroll
            for (int e = 0; e < 16; ++e) o[0][e] = tile.acc[i][j][e];
            split_gemm::store_rows<Out, 1>(lds + wave * kRegion, o, partial + (chunk * V + block_v) * D + first, D,
                                           V - block_v, D - first, vec_out);
        }
    }
    split_gemm::fix_chains(chains, [&](int block, int e) {
        const int64_t r = v0 + wm * (BM / 2) + block / Tile::NT * 32 + (lane_id() & 31);
        const int64_t c = d0 + wn * 64 + block % Tile::NT * 32 + split_gemm::acc_column(e);
        if (r < V && c < D)
            partial[(chunk * V + r) * D + c] =
                from_f32<Out>(split_gemm::scalar_dot(G + k0 * V + r, prior + k0 * D + c, k1 - k0, 0.0f, V, D));
    });
}

// Workspace of the backward: G, the weight gradient's chunks, the prior gradient's
// and the logits' (each where there are several), the bias gradient's partial rows.
struct HeadWorkspace {
    int64_t chunks, chunk_rows, blocks;
    int64_t prior_tile, prior_tiles, prior_chunks, prior_chunk;  // tile rows and columns, tiles, chunks of the vocabulary
    int64_t head_chunks;
    size_t partial_off, prior_off, logits_off, bias_off, total;
};
inline size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }
constexpr int64_t kWeightTiles = 512;              // two workgroups per CU (256: 73 us, 512: 53)
constexpr int64_t kPriorTiles = 256;               // the prior gradient's, where the vocabulary is long
constexpr int64_t kPriorLong = 2048, kPriorChunk = 256;  // such a vocabulary, and a chunk's columns at least
constexpr int64_t kPartialFloats = int64_t(1) << 24;  // 64 MiB of partial sums at most

inline HeadWorkspace head_workspace(int64_t rows, int64_t D, int64_t V) {
    HeadWorkspace w;
    const int64_t tiles = (V + 127) / 128 * ((D + 127) / 128);
    int64_t chunks = kWeightTiles / tiles;
    if (chunks > (rows + 127) / 128) chunks = (rows + 127) / 128;  // at least four K steps each
    if (chunks > kPartialFloats / (V * D)) chunks = kPartialFloats / (V * D);
    if (chunks < 1) chunks = 1;
    w.chunk_rows = ((rows + chunks - 1) / chunks + 31) / 32 * 32;
    w.chunks = (rows + w.chunk_rows - 1) / w.chunk_rows;
    // 128 x 128 tiles, or 64 x 64 ones with four K steps of loads in flight where the
    // larger would give fewer than one to each CU (4000 rows x 300, vocabulary 1000,
    // fp32: 67 -> 39 us); then chunks of a long vocabulary
    w.prior_tile = (rows + 127) / 128 * ((D + 127) / 128) < 256 ? 64 : 128;
    w.prior_tiles = (rows + w.prior_tile - 1) / w.prior_tile * ((D + w.prior_tile - 1) / w.prior_tile);
    chunks = V < kPriorLong ? 1 : std::min(kPriorTiles / w.prior_tiles, V / kPriorChunk);
    if (chunks > kPartialFloats / (rows * D)) chunks = kPartialFloats / (rows * D);
    if (chunks < 1) chunks = 1;
    w.prior_chunk = ((V + chunks - 1) / chunks + 31) / 32 * 32;
    w.prior_chunks = (V + w.prior_chunk - 1) / w.prior_chunk;
    w.blocks = (rows + kRows - 1) / kRows;
    w.partial_off = align256(static_cast<size_t>(rows) * V * sizeof(float));
    w.prior_off = w.partial_off + (w.chunks > 1 ? align256(static_cast<size_t>(w.chunks) * V * D * sizeof(float)) : 0);
    w.head_chunks = std::max(head_chunks(rows, D, V, true), head_chunks(rows, D, V, false));  // of any type
    w.logits_off =
        w.prior_off + (w.prior_chunks > 1 ? align256(static_cast<size_t>(w.prior_chunks) * rows * D * sizeof(float)) : 0);
    w.bias_off =
        w.logits_off + (w.head_chunks > 1 ? align256(static_cast<size_t>(logits_floats(rows, V, w.head_chunks)) * sizeof(float)) : 0);
    w.total = w.bias_off + static_cast<size_t>(w.blocks) * V * sizeof(float);
    return w;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// run(kernel) with the columns and loads of a head tile.
#define KOEMI_HEAD_KERNEL(run, kernel, T, columns, bytes)                                               \
    ((columns) == kWide ? ((bytes) == 16 ? run(kernel<T, kWide, 16>)                                    \
                           : (bytes) == 8 ? run(kernel<T, kWide, 8>) : run(kernel<T, kWide, 0>))        \
                        : ((bytes) == 16 ? run(kernel<T, kNarrow, 16>)                                  \
                           : (bytes) == 8 ? run(kernel<T, kNarrow, 8>) : run(kernel<T, kNarrow, 0>)))

// Logits [rows, V] at part, the chunks' behind them.
template <typename T>
int head_product(const T* prior, const T* weight, float* part, int64_t rows, int64_t D, int64_t V, hipStream_t s) {
    const int64_t tiles = head_tiles_of(rows, V), chunks = head_chunks(rows, D, V, sizeof(T) == 4);
    const int bytes = std::min(split_gemm::load_bytes<T>(prior, D), split_gemm::load_bytes<T>(weight, D));
    float* const chunk_part = part + (rows * V + 63) / 64 * 64;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles * chunks)), dim3(kThreads), 0, s, prior, weight,
                           chunk_part, rows, D, V, (V + 63) / 64, tiles, head_chunk(rows, D, V, sizeof(T) == 4),
                           static_cast<int>(V % 8 == 0 && aligned16(chunk_part)));
        return check_launch("surprise head (product)");
    };
    const int st = bytes == 16  ? run(surprise_head_product_kernel<T, 16>)
                   : bytes == 8 ? run(surprise_head_product_kernel<T, 8>) : run(surprise_head_product_kernel<T, 0>);
    if (st != KOEMI_OK) return st;
    launch_column_sum(chunk_part, part, chunks, rows * V, s);
    return check_launch("surprise head (product sum)");
}

template <typename T>
int head_forward(const void* prior, const void* weight, const void* bias, const int64_t* targets, const uint8_t* valid,
                 void* out, float* stats, float* part, int64_t rows, int64_t D, int64_t V, float log_vocab,
                 hipStream_t s) {
    if (head_chunks(rows, D, V, sizeof(T) == 4) > 1) {
        const int st = head_product(static_cast<const T*>(prior), static_cast<const T*>(weight), part, rows, D, V, s);
        if (st != KOEMI_OK) return st;
        hipLaunchKernelGGL(surprise_head_score_kernel<T>, dim3(grid_for(rows, kThreads / kWave)), dim3(kThreads), 0, s, part,
                           static_cast<const T*>(bias), targets, valid, static_cast<T*>(out), stats, rows, V, log_vocab);
        return check_launch("koemi_surprise_head_forward(scores)");
    }
    const int columns = head_columns(rows, V, sizeof(T) == 4);
    const int bytes = std::min(split_gemm::load_bytes<T>(prior, D), split_gemm::load_bytes<T>(weight, D));
    const int64_t v_tiles = (V + columns - 1) / columns;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((rows + kRows - 1) / kRows * v_tiles)), dim3(kThreads), 0, s,
                           static_cast<const T*>(prior), static_cast<const T*>(weight), static_cast<const T*>(bias),
                           targets, valid, static_cast<T*>(out), stats, part, rows, D, V, v_tiles, log_vocab);
        return check_launch("koemi_surprise_head_forward");
    };
    const int st = KOEMI_HEAD_KERNEL(run, surprise_head_forward_kernel, T, columns, bytes);
    if (st != KOEMI_OK || v_tiles == 1) return st;
    const auto finish = [&](auto kernel, int64_t lanes) {
        hipLaunchKernelGGL(kernel, dim3(grid_for(rows * lanes, 256)), dim3(256), 0, s, part, targets, valid,
                           static_cast<T*>(out), stats, rows, V, v_tiles, columns, log_vocab);
    };
    if (v_tiles <= kThreadTiles) finish(surprise_head_finish_kernel<T, 1>, 1);
    else finish(surprise_head_finish_kernel<T, kWave>, kWave);
    return check_launch("koemi_surprise_head_forward(finish)");
}

template <typename T>
int head_backward(const void* prior, const void* weight, const void* bias, const int64_t* targets, const uint8_t* valid,
                  const float* stats, const void* grad, void* grad_prior, void* grad_weight, void* grad_bias,
                  int64_t rows, int64_t D, int64_t V, float log_vocab, const HeadWorkspace& ws, char* base,
                  hipStream_t s) {
    float* G = reinterpret_cast<float*>(base);
    float* partial = reinterpret_cast<float*>(base + ws.partial_off);
    float* bias_partial = reinterpret_cast<float*>(base + ws.bias_off);
    const T* p = static_cast<const T*>(prior);
    const T* w = static_cast<const T*>(weight);
    const int64_t d_tiles = (D + 127) / 128, v_tiles = (V + 127) / 128;
    int st;
    if (head_chunks(rows, D, V, sizeof(T) == 4) > 1) {
        float* const logits = reinterpret_cast<float*>(base + ws.logits_off);
        st = head_product(p, w, logits, rows, D, V, s);
        if (st != KOEMI_OK) return st;
        const int64_t tiles = (V + kWave - 1) / kWave;
        hipLaunchKernelGGL(surprise_head_split_grad_kernel<T>, dim3(static_cast<unsigned>(ws.blocks * tiles)),
                           dim3(kSplitGradThreads), 0, s, logits, static_cast<const T*>(bias), targets, valid,
                           static_cast<const T*>(grad), stats, G, bias_partial, rows, V, tiles, log_vocab);
        st = check_launch("koemi_surprise_head_backward(logits)");
    } else {
        const int columns = head_columns(rows, V, sizeof(T) == 4);
        const int head_bytes = std::min(split_gemm::load_bytes<T>(prior, D), split_gemm::load_bytes<T>(weight, D));
        const int64_t head_tiles = (V + columns - 1) / columns;
        const auto run = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ws.blocks * head_tiles)), dim3(kThreads), 0, s, p, w,
                               static_cast<const T*>(bias), targets, valid, static_cast<const T*>(grad), stats, G,
                               bias_partial, rows, D, V, head_tiles, log_vocab);
            return check_launch("koemi_surprise_head_backward(logits)");
        };
        st = KOEMI_HEAD_KERNEL(run, surprise_head_grad_logits_kernel, T, columns, head_bytes);
    }
    if (st != KOEMI_OK) return st;
    const int bytes = split_gemm::load_bytes<float>(G, V);
    const int64_t b = ws.prior_tile;
    const auto prior_run = [&](auto kernel, auto* out) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ws.prior_tiles * ws.prior_chunks)), dim3(kThreads), 0, s, G,
                           w, out, rows, D, V, (D + b - 1) / b, ws.prior_tiles, ws.prior_chunk,
                           static_cast<int>(D % 8 == 0 && aligned16(out)));
        return check_launch("koemi_surprise_head_backward(prior)");
    };
    T* const gp = static_cast<T*>(grad_prior);
    if (ws.prior_chunks > 1) {  // few tiles: 64 x 64
        float* const part = reinterpret_cast<float*>(base + ws.prior_off);
        st = bytes == 16  ? prior_run(surprise_head_grad_prior_kernel<T, float, 64, 16>, part)
             : bytes == 8 ? prior_run(surprise_head_grad_prior_kernel<T, float, 64, 8>, part)
                          : prior_run(surprise_head_grad_prior_kernel<T, float, 64, 0>, part);
        if (st != KOEMI_OK) return st;
        launch_column_sum(part, gp, ws.prior_chunks, rows * D, s);
        st = check_launch("koemi_surprise_head_backward(prior sum)");
    } else {
        st = b == 128 ? (bytes == 16  ? prior_run(surprise_head_grad_prior_kernel<T, T, 128, 16>, gp)
                         : bytes == 8 ? prior_run(surprise_head_grad_prior_kernel<T, T, 128, 8>, gp)
                                      : prior_run(surprise_head_grad_prior_kernel<T, T, 128, 0>, gp))
                      : (bytes == 16  ? prior_run(surprise_head_grad_prior_kernel<T, T, 64, 16>, gp)
                         : bytes == 8 ? prior_run(surprise_head_grad_prior_kernel<T, T, 64, 8>, gp)
                                      : prior_run(surprise_head_grad_prior_kernel<T, T, 64, 0>, gp));
    }
    if (st != KOEMI_OK) return st;
    const auto weight_run = [&](auto kernel, auto* out) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ws.chunks * d_tiles * v_tiles)), dim3(kThreads), 0, s, G, p,
                           out, rows, D, V, d_tiles, v_tiles, ws.chunk_rows,
                           static_cast<int>(D % 8 == 0 && aligned16(out)));
        return check_launch("koemi_surprise_head_backward(weight)");
    };
    T* const gw = static_cast<T*>(grad_weight);
    if (ws.chunks > 1) {
        st = weight_run(surprise_head_grad_weight_kernel<T, float>, partial);
        if (st != KOEMI_OK) return st;
        launch_column_sum(partial, gw, ws.chunks, V * D, s);
        st = check_launch("koemi_surprise_head_backward(weight sum)");
    } else {
        st = weight_run(surprise_head_grad_weight_kernel<T, T>, gw);
    }
    if (st != KOEMI_OK) return st;
    launch_column_sum(bias_partial, static_cast<T*>(grad_bias), ws.blocks, V, s);
    return check_launch("koemi_surprise_head_backward(bias sum)");
}

int check_head(int64_t rows, int64_t D, int64_t V, int dtype) {
    if (rows < 1 || D < 1 || V < 2) return fail(KOEMI_ERR_INVALID, "the surprise head needs rows, width >= 1 and vocab >= 2");
    if (!float_dtype(dtype)) return fail(KOEMI_ERR_UNSUPPORTED, "the surprise head does not support dtype %s", dtype_name(dtype));
    if ((rows + 63) / 64 * ((V + 63) / 64) > 0x7fffffffLL || (rows + 127) / 128 * ((D + 127) / 128) > 0x7fffffffLL ||
        (V + 127) / 128 * ((D + 127) / 128) > 0x7fffffffLL)
        return fail(KOEMI_ERR_UNSUPPORTED, "the surprise head's sizes are too large");
    return KOEMI_OK;
}

}  // namespace
}  // namespace koemi

using namespace koemi;

extern "C" size_t koemi_surprise_head_forward_workspace_bytes(int64_t rows, int64_t vocab) {
    if (rows < 1 || vocab < 2) return 0;
    const size_t row_bytes = static_cast<size_t>(rows) * sizeof(float);
    // chunks of the widest state, 12 MiB at most
    const int64_t chunks = std::min(kMostSplitTiles / head_tiles_of(rows, vocab), kMostChunks);
    const size_t split = chunks > 1 ? static_cast<size_t>(logits_floats(rows, vocab, chunks)) * sizeof(float) : 0;
    const int64_t columns = head_columns(rows, vocab, true);  // no wider than a 16-bit type's
    const size_t tiles = vocab > columns ? static_cast<size_t>((vocab + columns - 1) / columns * 3) * row_bytes : 0;
    return std::max(split, tiles);
}

extern "C" int koemi_surprise_head_forward(const void* prior, const void* weight, const void* bias,
                                           const int64_t* target_ids, const uint8_t* valid_mask, void* surprise,
                                           float* stats, int64_t rows, int64_t width, int64_t vocab, float log_vocab,
                                           int dtype, void* workspace, size_t workspace_bytes, koemi_stream_t stream) {
    const int st = check_head(rows, width, vocab, dtype);
    if (st != KOEMI_OK) return st;
    if (!prior || !weight || !bias || !target_ids || !valid_mask || !surprise || !stats)
        return fail(KOEMI_ERR_INVALID, "the surprise head received a null pointer");
    const size_t need = koemi_surprise_head_forward_workspace_bytes(rows, vocab);
    if (workspace_bytes < need || (need > 0 && !workspace))
        return fail(KOEMI_ERR_INVALID, "surprise head workspace too small: need %zu bytes", need);
    const auto run = [&](auto tag) {
        return head_forward<decltype(tag)>(prior, weight, bias, target_ids, valid_mask, surprise, stats,
                                           static_cast<float*>(workspace), rows, width, vocab, log_vocab,
                                           as_stream(stream));
    };
    return dtype == KOEMI_F32 ? run(float{}) : dtype == KOEMI_F16 ? run(f16{}) : run(bf16{});
}

extern "C" size_t koemi_surprise_head_backward_workspace_bytes(int64_t rows, int64_t width, int64_t vocab) {
    if (rows < 1 || width < 1 || vocab < 2) return 0;
    return head_workspace(rows, width, vocab).total;
}

extern "C" int koemi_surprise_head_backward(const void* prior, const void* weight, const void* bias,
                                            const int64_t* target_ids, const uint8_t* valid_mask, const float* stats,
                                            const void* grad_surprise, void* grad_prior, void* grad_weight,
                                            void* grad_bias, int64_t rows, int64_t width, int64_t vocab, float log_vocab,
                                            int dtype, void* workspace, size_t workspace_bytes, koemi_stream_t stream) {
    const int st = check_head(rows, width, vocab, dtype);
    if (st != KOEMI_OK) return st;
    if (!prior || !weight || !bias || !target_ids || !valid_mask || !stats || !grad_surprise || !grad_prior ||
        !grad_weight || !grad_bias)
        return fail(KOEMI_ERR_INVALID, "the surprise head received a null pointer");
    const HeadWorkspace ws = head_workspace(rows, width, vocab);
    if (!workspace || workspace_bytes < ws.total)
        return fail(KOEMI_ERR_INVALID, "surprise head workspace too small: need %zu bytes", ws.total);
    const auto run = [&](auto tag) {
        return head_backward<decltype(tag)>(prior, weight, bias, target_ids, valid_mask, stats, grad_surprise, grad_prior,
                                            grad_weight, grad_bias, rows, width, vocab, log_vocab, ws,
                                            static_cast<char*>(workspace), as_stream(stream));
    };
    return dtype == KOEMI_F32 ? run(float{}) : dtype == KOEMI_F16 ? run(f16{}) : run(bf16{});
}
