// Fused RMSNorm + SiLU for gfx950.
//
// Reference: src/koemi/cuda_kernels/core/rmsnorm_silu.cu:62-132 (one block per
// row, two global passes over x). Here a row is held in registers by 16, 32 or
// 64 lanes (narrow rows share a wave): each lane loads NV 16-byte vectors (8
// bf16/f16 or 4 fp32 values), the sum of squares is reduced with a xor
// butterfly over the row's lanes, and y = silu(x * inv * w) is produced from
// the same registers, so x is read from HBM exactly once and y written once.
// Rows whose width does not fit that layout use a generic block-per-row path.
#include "column_sum.hpp"
#include "common.hpp"

namespace koemi {
namespace {

constexpr int kNormWaves = 4;
// Cache policy of the grouped forward by the size of x: non-temporal loads of
// x above KOEMI_NORM_NT_LOAD_BYTES, else non-temporal stores of y above
// KOEMI_NT_STORE_BYTES (measured at C2, [32768, 512] bf16: 13.4 -> 11.5 us in
// isolation; non-temporal loads and stores together were slower at both C2
// and C3).
#ifndef KOEMI_NORM_NT_LOAD_BYTES
#define KOEMI_NORM_NT_LOAD_BYTES (int64_t(128) << 20)
#endif

__device__ __forceinline__ float silu(float v) {
    // v * sigmoid(v) with the hardware exp2 and reciprocal (1 ulp each).
    const float e = __builtin_amdgcn_exp2f(v * -1.4426950408889634f);
    return v * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float silu_grad(float v) {
    const float e = __builtin_amdgcn_exp2f(v * -1.4426950408889634f);
    const float sg = __builtin_amdgcn_rcpf(1.0f + e);
    return sg * (1.0f + v * (1.0f - sg));
}

template <typename T>
struct Vec16 {
    static constexpr int N = 16 / sizeof(T);
    union {
        uint4 raw;
        T e[N];
    };
};

// NV vectors per lane; row width H must satisfy H % N == 0 and H <= NV*64*N.
// Each wave handles ROWS consecutive rows and issues all of their loads before
// any arithmetic, so ROWS*NV 16-byte loads per lane are in flight at once.
template <typename T, int NV, int ROWS>
__global__ __launch_bounds__(kWave * kNormWaves) void rmsnorm_silu_fwd_wave(
    const T* __restrict__ x, const T* __restrict__ w, T* __restrict__ y, float* __restrict__ inv_out,
    int64_t rows, int H, float eps) {
    constexpr int N = Vec16<T>::N;
    const int lane = lane_id();
    const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kNormWaves + threadIdx.x / kWave) * ROWS;
    if (row0 >= rows) return;
    // Unconditional loads at clamped addresses (no branch around a load), zeroed
    // afterwards where out of range, so all of them are in flight together.
    Vec16<T> xv[ROWS][NV], wv[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (v * kWave + lane) * N;
        wv[v].raw = *reinterpret_cast<const uint4*>(w + min(c, H - N));
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = (v * kWave + lane) * N;
            const int64_t rr = min(row0 + r, rows - 1);
            xv[r][v].raw = *reinterpret_cast<const uint4*>(x + rr * H + min(c, H - N));
        }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (v * kWave + lane) * N;
        if (c >= H) wv[v].raw = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            if (c >= H || row0 + r >= rows) xv[r][v].raw = make_uint4(0, 0, 0, 0);
    }
    float ss[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        ss[r] = 0.0f;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float f = to_f32(xv[r][v].e[i]);
                ss[r] = __builtin_fmaf(f, f, ss[r]);
            }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) ss[r] += __shfl_xor(ss[r], off, kWave);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if (row0 + r >= rows) break;
        const float inv = rsqrtf(ss[r] / static_cast<float>(H) + eps);
        if (lane == r) inv_out[row0 + r] = inv;
        T* yr = y + (row0 + r) * H;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = (v * kWave + lane) * N;
            if (c < H) {
                Vec16<T> o;
#pragma unroll
                for (int i = 0; i < N; ++i)
                    o.e[i] = from_f32<T>(silu(to_f32(xv[r][v].e[i]) * inv * to_f32(wv[v].e[i])));
                *reinterpret_cast<uint4*>(yr + c) = o.raw;
            }
        }
    }
}

// LPR lanes per row, 64 / LPR rows side by side in a wave (lane l serves row
// l / LPR); each lane holds NV 16-byte vectors of its row at columns
// (v * LPR + l % LPR) * N. Narrow rows keep every lane busy this way and the
// sum of squares needs only log2(LPR) butterfly steps for all rows at once.
// STREAM: x is read with non-temporal loads (inputs much larger than the
// 256 MiB Infinity Cache gain nothing from being cached there, and leaving it
// to the output measured 12% faster at [131072, 1024] bf16).
typedef unsigned int u32x4n __attribute__((ext_vector_type(4)));
template <bool STREAM>
__device__ __forceinline__ uint4 load16(const void* p) {
    if constexpr (STREAM) {
        const u32x4n v = __builtin_nontemporal_load(reinterpret_cast<const u32x4n*>(p));
        return make_uint4(v.x, v.y, v.z, v.w);
    } else {
        return *reinterpret_cast<const uint4*>(p);
    }
}

// VEC false: NV single elements per lane at columns v * LPR + l % LPR, for
// widths and alignments that 16-byte vectors do not fit: the row is still read
// once, coalesced. [32768, 511] bf16: 36 -> 18 us against a workgroup per row in
// two passes.
template <typename T, int NV, int LPR, bool STREAM, bool NT_STORE, bool VEC = true>
__global__ __launch_bounds__(kWave * kNormWaves) void rmsnorm_silu_fwd_group(
    const T* __restrict__ x, const T* __restrict__ w, T* __restrict__ y, float* __restrict__ inv_out,
    int64_t rows, int H, float eps) {
    constexpr int N = VEC ? Vec16<T>::N : 1;
    constexpr int kRowsPerWave = kWave / LPR;
    const int lane = lane_id();
    const int sub = lane % LPR;
    const int64_t wave_row0 = (static_cast<int64_t>(blockIdx.x) * kNormWaves + threadIdx.x / kWave) * kRowsPerWave;
    if (wave_row0 >= rows) return;
    const int64_t row = wave_row0 + lane / LPR;
    const int64_t rr = row < rows ? row : rows - 1;
    // Unconditional loads at clamped addresses, zeroed afterwards where out of range.
    Vec16<T> xv[NV], wv[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (v * LPR + sub) * N;
        if constexpr (VEC) {
            wv[v].raw = *reinterpret_cast<const uint4*>(w + min(c, H - N));
            xv[v].raw = load16<STREAM>(x + rr * H + min(c, H - N));
        } else {
            wv[v].e[0] = w[min(c, H - 1)];
            xv[v].e[0] = x[rr * H + min(c, H - 1)];
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (v * LPR + sub) * N;
        if (c >= H) {
            wv[v].raw = make_uint4(0, 0, 0, 0);
            xv[v].raw = make_uint4(0, 0, 0, 0);
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float f = to_f32(xv[v].e[i]);
            ss = __builtin_fmaf(f, f, ss);
        }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, kWave);
    if (row >= rows) return;
    const float inv = rsqrtf(ss / static_cast<float>(H) + eps);
    if (sub == 0) inv_out[row] = inv;
    T* yr = y + row * H;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (v * LPR + sub) * N;
        if (c < H) {
            Vec16<T> o;
#pragma unroll
            for (int i = 0; i < N; ++i) o.e[i] = from_f32<T>(silu(to_f32(xv[v].e[i]) * inv * to_f32(wv[v].e[i])));
            if constexpr (!VEC) yr[c] = o.e[0];
            else if constexpr (NT_STORE) store16_nt(yr + c, o.raw);
            else *reinterpret_cast<uint4*>(yr + c) = o.raw;
        }
    }
}

// Generic path: one 256-thread block per row, two passes over the row.
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_silu_fwd_block(const T* __restrict__ x,
                                                              const T* __restrict__ w,
                                                              T* __restrict__ y,
                                                              float* __restrict__ inv_out,
                                                              int64_t rows, int H, float eps) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    if (row >= rows) return;
    const T* xr = x + row * H;
    float ss = 0.0f;
    for (int c = threadIdx.x; c < H; c += 256) {
        const float f = to_f32(xr[c]);
        ss = __builtin_fmaf(f, f, ss);
    }
    ss = wave_sum_xor(ss);
    if (lane_id() == 0) red[threadIdx.x / kWave] = ss;
    __syncthreads();
    ss = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = rsqrtf(ss / static_cast<float>(H) + eps);
    if (threadIdx.x == 0) inv_out[row] = inv;
    for (int c = threadIdx.x; c < H; c += 256)
        y[row * H + c] = from_f32<T>(silu(to_f32(xr[c]) * inv * to_f32(w[c])));
}

// ------------------------------------------------------------------ backward --
// dx = inv * d * w - x * inv^3 / H * sum_c(d_c w_c x_c),  d = g * silu'(x inv w),
// dw = sum_rows d * x * inv. Stage 1 walks the rows with a fixed number of
// workgroups, each keeping its share of dw in registers and writing it once as
// an fp32 partial row; stage 2 (column_sum.hpp) adds the partial rows in a fixed order. No
// atomics: the same bits on every run.
constexpr int kBwdMaxBlocks = 1024;  // 4 workgroups per CU in flight; the partial rows stay in L2

// Partial rows the workspace has room for (stage 1 launches at most as many workgroups).
inline int64_t bwd_max_blocks(int64_t rows) { return rows < 1 ? 1 : (rows < kBwdMaxBlocks ? rows : kBwdMaxBlocks); }

// Stage 1 with the row held in registers by LPR lanes. LPR <= 64: 64 / LPR rows
// side by side in a wave, their sums by a butterfly over the row's lanes. LPR =
// 256: a row per workgroup, the four waves' sums through LDS. VEC: NV 16-byte
// vectors per lane at columns (v * LPR + sub) * N (H a multiple of N, aligned
// operands); otherwise NV single elements at columns v * LPR + sub, so that any
// H and alignment reads a row once and coalesced. Bound: HBM, x and g read once
// and dx written once. [32768, 512] bf16: 61 -> 21 us (a two-pass row per
// workgroup before, dw accumulated in global memory); [32768, 511]: 63 -> 22 us.
template <typename T, int NV, int LPR, bool VEC>
__global__ __launch_bounds__(kWave * kNormWaves) void rmsnorm_silu_bwd_rows(
    const T* __restrict__ g, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ inv_rms, T* __restrict__ dx, float* __restrict__ partial,
    int64_t rows, int H) {
    constexpr int N = VEC ? Vec16<T>::N : 1;
    constexpr int kThreads = kWave * kNormWaves;
    constexpr int kRowsPerBlock = kThreads / LPR;
    __shared__ float red[2][kNormWaves];
    const int tid = threadIdx.x;
    const int sub = tid % LPR;
    const float inv_h = 1.0f / static_cast<float>(H);
    T wv[NV][N];
    float dw[NV][N];
    auto column = [&](int v) { return (v * LPR + sub) * N; };
    auto load = [&](const T* p, T (&out)[NV][N]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = column(v);
            if constexpr (VEC) {
                Vec16<T> q;
                q.raw = *reinterpret_cast<const uint4*>(p + min(c, H - N));
#pragma unroll
                for (int i = 0; i < N; ++i) out[v][i] = q.e[i];
            } else {
                out[v][0] = p[min(c, H - 1)];
            }
        }
    };
    load(w, wv);
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < N; ++i) dw[v][i] = 0.0f;
    int parity = 0;
    // LPR = 256: every thread of the workgroup walks the same rows (the barrier
    // in the loop); otherwise rows past the end are clamped and not stored.
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock; base < rows;
         base += static_cast<int64_t>(gridDim.x) * kRowsPerBlock) {
        const int64_t row = base + tid / LPR;
        const bool live = row < rows;
        const int64_t rr = live ? row : rows - 1;
        T xv[NV][N], gv[NV][N];
        load(x + rr * H, xv);
        load(g + rr * H, gv);
        const float inv = inv_rms[rr];
        float d[NV][N];
        float dot = 0.0f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const bool in = live && column(v) < H;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float xf = to_f32(xv[v][i]), wf = to_f32(wv[v][i]);
                const float nrm = xf * inv;
                const float dv = to_f32(gv[v][i]) * silu_grad(nrm * wf);
                d[v][i] = in ? dv * wf : 0.0f;
                dot = __builtin_fmaf(d[v][i], in ? xf : 0.0f, dot);
                dw[v][i] += in ? dv * nrm : 0.0f;
            }
        }
#pragma unroll
        for (int off = (LPR < kWave ? LPR : kWave) / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, kWave);
        if constexpr (LPR > kWave) {
            if (lane_id() == 0) red[parity][tid / kWave] = dot;
            __syncthreads();  // the other parity is rewritten only after the next row's barrier
            dot = (red[parity][0] + red[parity][1]) + (red[parity][2] + red[parity][3]);
            parity ^= 1;
        }
        const float corr = inv * inv * inv * inv_h * dot;
        if (!live) continue;
        T* dr = dx + row * H;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = column(v);
            if (c >= H) continue;
            if constexpr (VEC) {
                Vec16<T> o;
#pragma unroll
                for (int i = 0; i < N; ++i) o.e[i] = from_f32<T>(inv * d[v][i] - to_f32(xv[v][i]) * corr);
                *reinterpret_cast<uint4*>(dr + c) = o.raw;
            } else {
                dr[c] = from_f32<T>(inv * d[v][0] - to_f32(xv[v][0]) * corr);
            }
        }
    }
    // One partial row per workgroup: its row slots' shares are added in slot
    // order, the slots of a wave by a butterfly, the waves' through LDS.
    float* part = partial + static_cast<int64_t>(blockIdx.x) * H;
    if constexpr (LPR > kWave) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = column(v);
            if (c >= H) continue;
#pragma unroll
            for (int i = 0; i < N; ++i) part[c + i] = dw[v][i];
        }
    } else {
        __shared__ float sums[kNormWaves][LPR * NV * N];
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int i = 0; i < N; ++i) {
#pragma unroll
                for (int off = kWave / 2; off >= LPR; off >>= 1) dw[v][i] += __shfl_xor(dw[v][i], off, kWave);
                if (lane_id() < LPR) sums[tid / kWave][column(v) + i] = dw[v][i];
            }
        __syncthreads();
        for (int c = tid; c < H; c += kThreads)
            part[c] = (sums[0][c] + sums[1][c]) + (sums[2][c] + sums[3][c]);
    }
}

// Stage 1 for rows wider than the register layouts: a workgroup per row, two
// passes over it.
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_silu_bwd_wide(
    const T* __restrict__ g, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ inv_rms, T* __restrict__ dx, float* __restrict__ partial,
    int64_t rows, int H) {
    __shared__ float red[4];
    __shared__ float total;
    const int64_t blocks = gridDim.x;
    float* part = partial + static_cast<int64_t>(blockIdx.x) * H;
    for (int c = threadIdx.x; c < H; c += 256) part[c] = 0.0f;
    for (int64_t row = blockIdx.x; row < rows; row += blocks) {
        const T* xr = x + row * H;
        const T* gr = g + row * H;
        const float inv = inv_rms[row];
        float dot = 0.0f;
        for (int c = threadIdx.x; c < H; c += 256) {
            const float xf = to_f32(xr[c]), wf = to_f32(w[c]);
            const float d = to_f32(gr[c]) * silu_grad(xf * inv * wf);
            dot = __builtin_fmaf(d * wf, xf, dot);
        }
        dot = wave_sum_xor(dot);
        __syncthreads();
        if (lane_id() == 0) red[threadIdx.x / kWave] = dot;
        __syncthreads();
        if (threadIdx.x == 0) total = (red[0] + red[1]) + (red[2] + red[3]);
        __syncthreads();
        const float corr = inv * inv * inv / static_cast<float>(H) * total;
        for (int c = threadIdx.x; c < H; c += 256) {
            const float xf = to_f32(xr[c]), wf = to_f32(w[c]);
            const float nrm = xf * inv;
            const float d = to_f32(gr[c]) * silu_grad(nrm * wf);
            dx[row * H + c] = from_f32<T>(inv * d * wf - xf * corr);
            part[c] += d * nrm;  // this thread is the only writer of part[c]
        }
    }
}

template <typename T>
int launch_forward(const void* x, const void* w, void* y, float* inv, int64_t rows, int64_t H,
                   float eps, hipStream_t stream) {
    constexpr int N = Vec16<T>::N;
    const T* xp = static_cast<const T*>(x);
    const T* wp = static_cast<const T*>(w);
    T* yp = static_cast<T*>(y);
    const bool aligned = (reinterpret_cast<uintptr_t>(x) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(w) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(y) % 16 == 0);
    const int Hi = static_cast<int>(H);
    const dim3 wblock(kWave * kNormWaves);
    if (aligned && H % N == 0) {
        const int64_t vecs = H / N;  // vectors per row
#define KOEMI_NORM_LAUNCH(NV, ROWS)                                                                      \
    hipLaunchKernelGGL((rmsnorm_silu_fwd_wave<T, NV, ROWS>), dim3(grid_for(rows, kNormWaves * ROWS)), wblock, 0, \
                       stream, xp, wp, yp, inv, rows, Hi, eps);                                           \
    return check_launch("koemi_rmsnorm_silu_forward")
        const int64_t bytes = rows * H * static_cast<int64_t>(sizeof(T));
        const bool stream_x = bytes > KOEMI_NORM_NT_LOAD_BYTES;
        const bool nt_store = bytes > KOEMI_NT_STORE_BYTES && !stream_x;  // both together measured slower
#define KOEMI_NORM_GROUP(NV, LPR)                                                                        \
    {                                                                                                    \
        const dim3 g(grid_for(rows, kNormWaves * (kWave / LPR)));                                        \
        if (stream_x)                                                                                    \
            hipLaunchKernelGGL((rmsnorm_silu_fwd_group<T, NV, LPR, true, false>), g, wblock, 0, stream, xp, wp, yp, \
                               inv, rows, Hi, eps);                                                      \
        else if (nt_store)                                                                               \
            hipLaunchKernelGGL((rmsnorm_silu_fwd_group<T, NV, LPR, false, true>), g, wblock, 0, stream, xp, wp, yp, \
                               inv, rows, Hi, eps);                                                      \
        else                                                                                             \
            hipLaunchKernelGGL((rmsnorm_silu_fwd_group<T, NV, LPR, false, false>), g, wblock, 0, stream, xp, wp, yp, \
                               inv, rows, Hi, eps);                                                      \
        return check_launch("koemi_rmsnorm_silu_forward");                                              \
    }
        if (vecs <= 16) { KOEMI_NORM_GROUP(1, 16); }
        if (vecs <= 32) { KOEMI_NORM_GROUP(2, 16); }
        if (vecs <= kWave * 1) { KOEMI_NORM_GROUP(4, 16); }
        if (vecs <= kWave * 2) { KOEMI_NORM_GROUP(4, 32); }
        if (vecs <= kWave * 4) { KOEMI_NORM_LAUNCH(4, 1); }
        if (vecs <= kWave * 8) { KOEMI_NORM_LAUNCH(8, 1); }
#undef KOEMI_NORM_LAUNCH
#undef KOEMI_NORM_GROUP
    } else if (H <= 1024) {
        auto run = [&](auto kernel, int lanes_per_row) {
            hipLaunchKernelGGL(kernel, dim3(grid_for(rows, kNormWaves * (kWave / lanes_per_row))), wblock, 0, stream, xp,
                               wp, yp, inv, rows, Hi, eps);
            return check_launch("koemi_rmsnorm_silu_forward");
        };
        if (H <= 128) return run(rmsnorm_silu_fwd_group<T, 8, 16, false, false, false>, 16);
        if (H <= 256) return run(rmsnorm_silu_fwd_group<T, 8, 32, false, false, false>, 32);
        if (H <= 512) return run(rmsnorm_silu_fwd_group<T, 8, 64, false, false, false>, 64);
        return run(rmsnorm_silu_fwd_group<T, 16, 64, false, false, false>, 64);
    }
    if (rows > 0x7fffffffLL) return fail(KOEMI_ERR_UNSUPPORTED, "rmsnorm_silu: too many rows for the generic path");
    hipLaunchKernelGGL(rmsnorm_silu_fwd_block<T>, dim3(static_cast<unsigned>(rows)), dim3(256), 0, stream, xp, wp, yp, inv, rows, Hi, eps);
    return check_launch("koemi_rmsnorm_silu_forward");
}

template <typename T>
int launch_backward(const void* g, const void* x, const void* w, const float* inv, void* dx,
                    void* dw, int64_t rows, int64_t H, float* partial, hipStream_t stream) {
    constexpr int N = Vec16<T>::N;
    if (rows == 0) {  // the operands may be null: only grad_weight is written, with zeros
        launch_column_sum(partial, static_cast<T*>(dw), 0, H, stream);
        return check_launch("koemi_rmsnorm_silu_backward");
    }
    const T* gp = static_cast<const T*>(g);
    const T* xp = static_cast<const T*>(x);
    const T* wp = static_cast<const T*>(w);
    T* dxp = static_cast<T*>(dx);
    const int Hi = static_cast<int>(H);
    int64_t blocks = bwd_max_blocks(rows);
    bool launched = false;
    // The narrowest lane group whose registers hold the row; 16-byte vectors
    // where the width and every pointer allow them, else single elements.
    auto run = [&](auto kernel, int64_t lanes_per_row) {
        const int64_t per_block = kWave * kNormWaves / lanes_per_row;
        const int64_t need = (rows + per_block - 1) / per_block;
        if (need < blocks) blocks = need;
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kWave * kNormWaves), 0, stream, gp, xp, wp,
                           inv, dxp, partial, rows, Hi);
        launched = true;
    };
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (H % N == 0 && aligned(g) && aligned(x) && aligned(w) && aligned(dx)) {
        const int64_t vecs = H / N;
        if (vecs <= 16) run(rmsnorm_silu_bwd_rows<T, 1, 16, true>, 16);
        else if (vecs <= 32) run(rmsnorm_silu_bwd_rows<T, 2, 16, true>, 16);
        else if (vecs <= 64) run(rmsnorm_silu_bwd_rows<T, 2, 32, true>, 32);
        else if (vecs <= 128) run(rmsnorm_silu_bwd_rows<T, 2, 64, true>, 64);
        else if (vecs <= 512) run(rmsnorm_silu_bwd_rows<T, 2, 256, true>, 256);
        else if (vecs <= 1024) run(rmsnorm_silu_bwd_rows<T, 4, 256, true>, 256);
    } else {
        if (H <= 128) run(rmsnorm_silu_bwd_rows<T, 8, 16, false>, 16);
        else if (H <= 256) run(rmsnorm_silu_bwd_rows<T, 8, 32, false>, 32);
        else if (H <= 512) run(rmsnorm_silu_bwd_rows<T, 8, 64, false>, 64);
        else if (H <= 1024) run(rmsnorm_silu_bwd_rows<T, 16, 64, false>, 64);
        else if (H <= 4096) run(rmsnorm_silu_bwd_rows<T, 16, 256, false>, 256);
    }
    if (!launched)
        hipLaunchKernelGGL(rmsnorm_silu_bwd_wide<T>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, gp, xp, wp,
                           inv, dxp, partial, rows, Hi);
    int st = check_launch("koemi_rmsnorm_silu_backward");
    if (st != KOEMI_OK) return st;
    launch_column_sum(partial, static_cast<T*>(dw), blocks, H, stream);
    return check_launch("koemi_rmsnorm_silu_backward");
}

}  // namespace
}  // namespace koemi

using namespace koemi;

extern "C" int koemi_rmsnorm_silu_forward(const void* input, const void* weight, void* output,
                                          float* inverse_rms, int64_t rows, int64_t hidden,
                                          double eps, int dtype, koemi_stream_t stream) {
    if (rows < 0 || hidden < 1) return fail(KOEMI_ERR_INVALID, "rmsnorm_silu needs rows >= 0 and a positive hidden dimension");
    if (hidden > 0x7fffffffLL) return fail(KOEMI_ERR_UNSUPPORTED, "rmsnorm_silu hidden dimension too large");
    if (!(eps > 0.0)) return fail(KOEMI_ERR_INVALID, "eps must be finite and positive");
    if (!float_dtype(dtype)) return fail(KOEMI_ERR_UNSUPPORTED, "rmsnorm_silu does not support dtype %s", dtype_name(dtype));
    if (rows == 0) return KOEMI_OK;
    if (!input || !weight || !output || !inverse_rms) return fail(KOEMI_ERR_INVALID, "rmsnorm_silu received a null pointer");
    hipStream_t s = as_stream(stream);
    const float e = static_cast<float>(eps);
    switch (dtype) {
        case KOEMI_F32: return launch_forward<float>(input, weight, output, inverse_rms, rows, hidden, e, s);
        case KOEMI_F16: return launch_forward<f16>(input, weight, output, inverse_rms, rows, hidden, e, s);
        default: return launch_forward<bf16>(input, weight, output, inverse_rms, rows, hidden, e, s);
    }
}

extern "C" size_t koemi_rmsnorm_silu_backward_workspace_bytes(int64_t rows, int64_t hidden) {
    if (rows < 0 || hidden < 1) return 0;
    return static_cast<size_t>(bwd_max_blocks(rows)) * static_cast<size_t>(hidden) * sizeof(float);
}

extern "C" int koemi_rmsnorm_silu_backward(const void* grad_output, const void* input,
                                           const void* weight, const float* inverse_rms,
                                           void* grad_input, void* grad_weight, int64_t rows,
                                           int64_t hidden, int dtype, void* workspace,
                                           size_t workspace_bytes, koemi_stream_t stream) {
    if (rows < 0 || hidden < 1) return fail(KOEMI_ERR_INVALID, "rmsnorm_silu backward needs rows >= 0 and a positive hidden dimension");
    if (hidden > 0x7fffffffLL) return fail(KOEMI_ERR_UNSUPPORTED, "rmsnorm_silu hidden dimension too large");
    if (!float_dtype(dtype)) return fail(KOEMI_ERR_UNSUPPORTED, "rmsnorm_silu does not support dtype %s", dtype_name(dtype));
    if (!grad_weight) return fail(KOEMI_ERR_INVALID, "rmsnorm_silu backward received a null pointer");
    if (rows > 0 && (!grad_output || !input || !weight || !inverse_rms || !grad_input))
        return fail(KOEMI_ERR_INVALID, "rmsnorm_silu backward received a null pointer");
    const size_t need = koemi_rmsnorm_silu_backward_workspace_bytes(rows, hidden);
    if (workspace_bytes < need || (need > 0 && !workspace))
        return fail(KOEMI_ERR_INVALID, "rmsnorm_silu backward workspace too small: need %zu bytes", need);
    hipStream_t s = as_stream(stream);
    float* partial = static_cast<float*>(workspace);
    switch (dtype) {
        case KOEMI_F32: return launch_backward<float>(grad_output, input, weight, inverse_rms, grad_input, grad_weight, rows, hidden, partial, s);
        case KOEMI_F16: return launch_backward<f16>(grad_output, input, weight, inverse_rms, grad_input, grad_weight, rows, hidden, partial, s);
        default: return launch_backward<bf16>(grad_output, input, weight, inverse_rms, grad_input, grad_weight, rows, hidden, partial, s);
    }
}
