// Bounded recurrent gates for gfx950.
//
// Reference: model/memory.py:14-30 (BoundedRecurrentState.gates) and the
// masking of network.py:306-309:
//
//   retention = sigmoid(u W_r^T + b_r)
//   a = 2^-8 + ((1 - 2^-8) - 2^-8) * retention        (in [2^-8, 1 - 2^-8])
//   b = (1 - a) * tanh(u W_c^T + b_c)
//   invalid positions (valid mask given and false): a = 1, b = 0
//
// The two width x width products leave fp32 results in the workspace: fp32 inputs
// on the matrix cores as split bf16 planes (split_gemm.hpp; fp32 accumulation), 16-bit
// ones and few rows of some widths as plain GEMMs on rocBLAS. One HIP kernel then
// applies the biases, the bounded sigmoid, tanh and the mask and writes a and b in the
// input dtype, reading each fp32 product once (16-byte loads, four columns per
// thread). koemi_recurrent_scan (fp32) hands the two products straight to the
// affine-scan kernel, which applies the same expressions in registers, so a
// and b never reach memory.
#include "common.hpp"
#include "split_gemm.hpp"

#include <rocblas/rocblas.h>

#include <mutex>

namespace koemi {

// The rocBLAS handle of a device (blas.hip); callers hold g_blas_mutex.
rocblas_handle blas_handle(int device);
extern std::mutex g_blas_mutex;
// The fused gates + scan kernel (affine_scan.hip).
int launch_gated_scan(const float* zr, const float* zc, int64_t stride, const float* retention_bias,
                      const float* candidate_bias, const uint8_t* valid, const float* h0, float* h, void* h16,
                      int64_t h16_stride, int64_t B, int64_t L, int64_t F, hipStream_t stream, void* workspace,
                      size_t workspace_bytes);

namespace {


template <typename T>
__global__ __launch_bounds__(256) void gates_epilogue_kernel(
    const float* __restrict__ zr, const float* __restrict__ zc, const T* __restrict__ br, const T* __restrict__ bc,
    const uint8_t* __restrict__ valid, T* __restrict__ a_out, T* __restrict__ b_out, int64_t rows, int64_t D) {
    const int64_t quads = D / 4;
    const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= rows * quads) return;
    const int64_t row = q / quads;
    const int64_t c0 = (q - row * quads) * 4;
    const float4 r4 = *reinterpret_cast<const float4*>(zr + row * D + c0);
    const float4 z4 = *reinterpret_cast<const float4*>(zc + row * D + c0);
    const float r[4] = {r4.x, r4.y, r4.z, r4.w}, z[4] = {z4.x, z4.y, z4.z, z4.w};
    const bool keep = valid == nullptr || valid[row] != 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float a = kGateMinRetention + kGateRetentionSpan * gate_sigmoid(r[c] + to_f32(br[c0 + c]));
        const float b = (1.0f - a) * gate_tanh(z[c] + to_f32(bc[c0 + c]));
        a_out[row * D + c0 + c] = from_f32<T>(keep ? a : 1.0f);
        b_out[row * D + c0 + c] = from_f32<T>(keep ? b : 0.0f);
    }
}

rocblas_datatype gates_blas_type(int dtype) {
    return dtype == KOEMI_F16 ? rocblas_datatype_f16_r : dtype == KOEMI_BF16 ? rocblas_datatype_bf16_r : rocblas_datatype_f32_r;
}

size_t gates_workspace(int64_t rows, int64_t D) {
    const size_t one = (static_cast<size_t>(rows) * static_cast<size_t>(D) * sizeof(float) + 255) & ~size_t(255);
    return 2 * one;
}

// zr = u W_r^T, zc = u W_c^T for fp32: B x B tiles, a tile's columns all of one
// product. Workgroup b runs on XCD b % 8; an XCD takes a contiguous range of tiles,
// four row blocks at a time over every column, so that its L2 serves the rows and
// weights that concurrently running tiles share. Bound by the matrix cores (six
// bf16 products an fp32 one) and the splits beside them: [16384, 1024] with its scan
// 387 us against 559 with rocBLAS's fp32 products (about 325 us of it, 210 TFLOP/s,
// 1.27 PFLOP/s counting six), its error against float64 4.5e-7 against 5.1e-7.
template <int B, int BYTES>
__global__ __launch_bounds__(split_gemm::kThreads, 2) void gate_products_kernel(
    const float* __restrict__ u, const float* __restrict__ wr, const float* __restrict__ wc, float* __restrict__ zr,
    float* __restrict__ zc, int64_t rows, int64_t D, uint32_t row_tiles, uint32_t half_tiles) {
    using Tile = split_gemm::Tile<float, float, B, B, false, false, B == 64 ? 4 : 1>;
    constexpr int kRegion = split_gemm::store_bytes<float, 1>();
    static_assert(4 * kRegion <= Tile::kLdsBytes, "the output regions fit the operands' LDS");
    __shared__ __attribute__((aligned(16))) char lds[Tile::kLdsBytes];
    constexpr uint32_t kGroup = 4;
    const uint32_t columns = 2 * half_tiles, tiles = row_tiles * columns, per_xcd = (tiles + 7) / 8;
    if ((blockIdx.x >> 3) >= per_xcd) return;
    const uint32_t logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (logical >= tiles) return;
    const uint32_t first = logical / (kGroup * columns) * kGroup;
    const uint32_t group = min(kGroup, row_tiles - first), within = logical % (kGroup * columns);
    const uint32_t column = within / group;
    const int64_t row0 = static_cast<int64_t>(first + within % group) * B;
    const int64_t n0 = static_cast<int64_t>(column % half_tiles) * B;
    const float* w = column < half_tiles ? wr : wc;
    float* z = column < half_tiles ? zr : zc;
    const int wave = threadIdx.x / kWave, wm = wave >> 1, wn = wave & 1;
    Tile tile;
    const uint64_t chains = tile.template run<BYTES, BYTES>(
        lds, D, D, 0, (D + Tile::BK - 1) / Tile::BK * Tile::BK, [&](int r) { return u + min(row0 + r, rows - 1) * D; },
        [&](int r) { return w + min(n0 + r, D - 1) * D; }, [&](int t) { return wn * (B / 2) + t * 32; });
#pragma unroll
    for (int i = 0; i < Tile::MT; ++i) {
        const int64_t block_row = row0 + wm * (B / 2) + i * 32;
#pragma unroll
        for (int j = 0; j < Tile::NT; ++j) {
            const int64_t c0 = n0 + wn * (B / 2) + j * 32;
            float o[1][16];
#pragma unroll
            for (int v = 0; v < 16; ++v) o[0][v] = tile.acc[i][j][v];
            split_gemm::store_rows<float, 1>(lds + wave * kRegion, o, z + block_row * D + c0, D, rows - block_row, D - c0,
                                             D % 8 == 0);
        }
    }
    split_gemm::fix_chains(chains, [&](int block, int v) {
        const int64_t r = row0 + wm * (B / 2) + block / Tile::NT * 32 + (lane_id() & 31);
        const int64_t c = n0 + wn * (B / 2) + block % Tile::NT * 32 + split_gemm::acc_column(v);
        if (r < rows && c < D) z[r * D + c] = split_gemm::scalar_dot(u + r * D, w + c * D, D, 0.0f);
    });
}

int gate_products_f32(const float* u, const float* wr, const float* wc, float* zr, float* zc, int64_t rows, int64_t D,
                      hipStream_t s) {
    // 64 x 64 tiles with four K steps of loads in flight where the 128 x 128 ones would
    // give fewer than one to each CU (168 rows x 512 with its scan: 28 -> 19 us)
    const int64_t b = (rows + 127) / 128 * 2 * ((D + 127) / 128) < 256 ? 64 : 128;
    const int64_t row_tiles = (rows + b - 1) / b, half_tiles = (D + b - 1) / b;
    const int64_t blocks = (row_tiles * half_tiles * 2 + 7) / 8 * 8;
    if (blocks > 0x7fffffffLL) return fail(KOEMI_ERR_UNSUPPORTED, "recurrent gates sizes exceed the grid");
    // D is a multiple of 4, so rows start 16-byte aligned where the bases do; a base
    // from a C caller may not
    const auto bytes = [&](const void* p) { return split_gemm::load_bytes<float>(p, D); };
    const bool wide = bytes(u) == 16 && bytes(wr) == 16 && bytes(wc) == 16;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(split_gemm::kThreads), 0, s, u, wr, wc, zr,
                           zc, rows, D, static_cast<uint32_t>(row_tiles), static_cast<uint32_t>(half_tiles));
        return check_launch("recurrent gates (products)");
    };
    if (b == 128) return wide ? run(gate_products_kernel<128, 16>) : run(gate_products_kernel<128, 0>);
    return wide ? run(gate_products_kernel<64, 16>) : run(gate_products_kernel<64, 0>);
}

// zr = u W_r^T, zc = u W_c^T (row-major [rows, D], fp32); 16-bit inputs and few rows of
// some widths on rocBLAS: in its column-major terms Z' (D x rows) = W'^T (D x D) . u' (D x rows).
int gate_products(const void* input, const void* retention_weight, const void* candidate_weight, float* zr,
                  float* zc, int64_t rows, int64_t width, int dtype, hipStream_t s) {
    // Few rows between 768 and 2048 wide leave most CUs idle for a long walk over K,
    // and rocBLAS splits K there. us with the scan, library / these tiles: [64, 768]
    // 26.4 / 25.4, [16, 1024] 25.3 / 30.0, [256, 1024] 26.5 / 30.8, [384, 1024] 31.9 /
    // 34.0, [168, 1280] 26.4 / 35.4, [256, 1280] 33.1 / 36.2, [384, 1280] 50.7 / 38.7,
    // [96, 1536] 29.4 / 40.6, [128, 1536] 55.4 / 40.8, [16, 2048] 72.4 / 50.5, [16, 4096]
    // 235.9 / 91.0. Its error is the larger (5.1e-7 from float64 at [64, 1024], 2.3e-7 on
    // the tiles), as it is where the tiles took its place.
    const bool few = width > 768 && width < 2048 && rows * width * width < (width <= 1280 ? 430000000 : 300000000);
    if (dtype == KOEMI_F32 && !few)
        return gate_products_f32(static_cast<const float*>(input), static_cast<const float*>(retention_weight),
                                 static_cast<const float*>(candidate_weight), zr, zc, rows, width, s);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail(KOEMI_ERR_LAUNCH, "recurrent gates: no device");
    std::lock_guard<std::mutex> lock(g_blas_mutex);
    rocblas_handle h = blas_handle(dev);
    if (!h) return fail(KOEMI_ERR_LAUNCH, "recurrent gates: no rocBLAS handle");
    if (rocblas_set_stream(h, s) != rocblas_status_success ||
        rocblas_set_pointer_mode(h, rocblas_pointer_mode_host) != rocblas_status_success)
        return fail(KOEMI_ERR_LAUNCH, "recurrent gates: rocblas stream setup failed");
    const rocblas_datatype t = gates_blas_type(dtype);
    const rocblas_int d = static_cast<rocblas_int>(width), n = static_cast<rocblas_int>(rows);
    const float one = 1.0f, zero = 0.0f;
    for (int g = 0; g < 2; ++g) {
        const void* w = g == 0 ? retention_weight : candidate_weight;
        float* z = g == 0 ? zr : zc;
        const rocblas_status st = rocblas_gemm_ex(h, rocblas_operation_transpose, rocblas_operation_none, d, n, d, &one,
                                                  w, t, d, input, t, d, &zero, z, rocblas_datatype_f32_r, d, z,
                                                  rocblas_datatype_f32_r, d, rocblas_datatype_f32_r,
                                                  rocblas_gemm_algo_standard, 0, 0);
        if (st != rocblas_status_success)
            return fail(KOEMI_ERR_LAUNCH, "recurrent gates: rocblas_gemm_ex failed (%s)", rocblas_status_to_string(st));
    }
    return KOEMI_OK;
}

}  // namespace
}  // namespace koemi

using namespace koemi;

extern "C" size_t koemi_recurrent_gates_workspace_bytes(int64_t rows, int64_t width) {
    if (rows < 0 || width < 1) return 0;
    return gates_workspace(rows, width);
}

extern "C" int koemi_recurrent_gates(const void* input, const void* retention_weight, const void* retention_bias,
                                     const void* candidate_weight, const void* candidate_bias, const uint8_t* valid,
                                     void* retention_out, void* increment_out, int64_t rows, int64_t width, int dtype,
                                     void* workspace, size_t workspace_bytes, koemi_stream_t stream) {
    if (rows < 0 || width < 1) return fail(KOEMI_ERR_INVALID, "recurrent gates need non-negative rows and positive width");
    if (!float_dtype(dtype)) return fail(KOEMI_ERR_UNSUPPORTED, "recurrent gates do not support dtype %s", dtype_name(dtype));
    if (width % 4 != 0) return fail(KOEMI_ERR_UNSUPPORTED, "recurrent gates need width % 4 == 0");
    if (rows == 0) return KOEMI_OK;
    if (rows > 0x7fffffffLL || width > 0x7fffffffLL / 4)
        return fail(KOEMI_ERR_UNSUPPORTED, "recurrent gates sizes exceed 32-bit GEMM dimensions");
    if (!input || !retention_weight || !retention_bias || !candidate_weight || !candidate_bias || !retention_out ||
        !increment_out)
        return fail(KOEMI_ERR_INVALID, "recurrent gates received a null pointer");
    const size_t need = gates_workspace(rows, width);
    if (!workspace || workspace_bytes < need)
        return fail(KOEMI_ERR_INVALID, "recurrent gates workspace too small: need %zu bytes", need);
    float* zr = static_cast<float*>(workspace);
    float* zc = reinterpret_cast<float*>(static_cast<char*>(workspace) + need / 2);
    const hipStream_t s = as_stream(stream);

    {
        const int st = gate_products(input, retention_weight, candidate_weight, zr, zc, rows, width, dtype, s);
        if (st != KOEMI_OK) return st;
    }
    const int64_t quads = rows * (width / 4);
    const dim3 grid(static_cast<unsigned>((quads + 255) / 256)), block(256);
    switch (dtype) {
        case KOEMI_F32:
            hipLaunchKernelGGL(gates_epilogue_kernel<float>, grid, block, 0, s, zr, zc,
                               static_cast<const float*>(retention_bias), static_cast<const float*>(candidate_bias),
                               valid, static_cast<float*>(retention_out), static_cast<float*>(increment_out), rows, width);
            break;
        case KOEMI_F16:
            hipLaunchKernelGGL(gates_epilogue_kernel<f16>, grid, block, 0, s, zr, zc,
                               static_cast<const f16*>(retention_bias), static_cast<const f16*>(candidate_bias), valid,
                               static_cast<f16*>(retention_out), static_cast<f16*>(increment_out), rows, width);
            break;
        default:
            hipLaunchKernelGGL(gates_epilogue_kernel<bf16>, grid, block, 0, s, zr, zc,
                               static_cast<const bf16*>(retention_bias), static_cast<const bf16*>(candidate_bias),
                               valid, static_cast<bf16*>(retention_out), static_cast<bf16*>(increment_out), rows, width);
    }
    return check_launch("koemi_recurrent_gates");
}

extern "C" int koemi_recurrent_scan(const float* input, const float* retention_weight, const float* retention_bias,
                                    const float* candidate_weight, const float* candidate_bias, const uint8_t* valid,
                                    const float* initial, float* states, int64_t batch, int64_t length, int64_t width,
                                    void* workspace, size_t workspace_bytes, koemi_stream_t stream) {
    if (batch < 0 || length < 0 || width < 1)
        return fail(KOEMI_ERR_INVALID, "recurrent scan needs non-negative batch and length and a positive width");
    if (width % 4 != 0) return fail(KOEMI_ERR_UNSUPPORTED, "recurrent scan needs width % 4 == 0");
    const int64_t rows = batch * length;
    if (rows == 0) return KOEMI_OK;
    if (rows > 0x7fffffffLL || width > 0x7fffffffLL / 4)
        return fail(KOEMI_ERR_UNSUPPORTED, "recurrent scan sizes exceed 32-bit GEMM dimensions");
    if (batch * ((width + kWave - 1) / kWave) > 0x7fffffffLL)
        return fail(KOEMI_ERR_UNSUPPORTED, "recurrent scan grid too large");
    if (!input || !retention_weight || !retention_bias || !candidate_weight || !candidate_bias || !initial || !states)
        return fail(KOEMI_ERR_INVALID, "recurrent scan received a null pointer");
    const size_t need = gates_workspace(rows, width);
    if (!workspace || workspace_bytes < need)
        return fail(KOEMI_ERR_INVALID, "recurrent scan workspace too small: need %zu bytes", need);
    float* zr = static_cast<float*>(workspace);
    float* zc = reinterpret_cast<float*>(static_cast<char*>(workspace) + need / 2);
    const hipStream_t s = as_stream(stream);
    int st = gate_products(input, retention_weight, candidate_weight, zr, zc, rows, width, KOEMI_F32, s);
    if (st != KOEMI_OK) return st;
    return launch_gated_scan(zr, zc, width, retention_bias, candidate_bias, valid, initial, states, nullptr, width,
                             batch, length, width, s, nullptr, 0);
}
