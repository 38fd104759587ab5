// Matrix-core tiles for operands of any floating type, width and alignment.
//
// C = A B^T (both operands K-contiguous) on v_mfma_f32_32x32x16, fp32
// accumulation. Two operands of the same 16-bit type go to the matrix cores as
// they are (every product exact). Any other pair is split into bf16 planes that
// sum to the operand exactly: fp32 into three, fp16 into two, bf16 is its own.
// A plane is the upper 16 bits of what the planes before it left (truncation:
// no plane overflows where the operand does not, and the last remainder is
// exact). The products of planes i and j with i + j <= 2 are accumulated: six
// for fp32 x fp32, five for fp32 x fp16, three for fp32 x bf16; what is dropped
// is below 2^-23 of the product, the order of the rounding that an fp32
// multiply-add chain makes at every step.
//
// Infinities and NaN do not survive a split (inf x 0 between planes): callers
// recompute an output that is not finite with scalar_dot, the plain
// multiply-add chain, so that such inputs give what the chain gives.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace koemi {
namespace split_gemm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

constexpr int kThreads = 256;  // four waves, 2 x 2 over the block tile

// Planes of a T operand beside an operand of type Other.
template <typename T, typename Other>
constexpr int planes() {
    if (std::is_same<T, Other>::value && sizeof(T) == 2) return 1;
    return std::is_same<T, float>::value ? 3 : std::is_same<T, f16>::value ? 2 : 1;
}

// Eight consecutive K values of one row, packed as in memory.
template <typename T>
struct Octet {
    static constexpr int kWords = static_cast<int>(sizeof(T)) * 2;
    uint32_t w[kWords];
    __device__ float value(int i) const {
        if constexpr (sizeof(T) == 4) return __uint_as_float(w[i]);
        else return to_f32(__builtin_bit_cast(T, static_cast<uint16_t>(w[i / 2] >> (i % 2 * 16))));
    }
};

// K values [k, k + 8) of a row. VEC: K is a multiple of 8 and rows are 16-byte
// aligned, so an octet is all in or all out and is read by 16-byte loads;
// otherwise element by element. What lies past K is read at a clamped address
// and cleared by clear_past, which the caller runs when it uses the octet: a
// select beside the load would wait for it. K >= 1.
template <bool VEC, typename T>
__device__ __forceinline__ void load_octet(Octet<T>& o, const T* __restrict__ row, int64_t k, int64_t K) {
    if constexpr (VEC) {
        const uint4* p = reinterpret_cast<const uint4*>(row + min(k, K - 8));
#pragma unroll
        for (int i = 0; i < Octet<T>::kWords / 4; ++i) {
            const uint4 v = p[i];
            o.w[4 * i] = v.x, o.w[4 * i + 1] = v.y, o.w[4 * i + 2] = v.z, o.w[4 * i + 3] = v.w;
        }
    } else if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < 8; ++i) o.w[i] = __float_as_uint(row[min(k + i, K - 1)]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o.w[i] = __builtin_bit_cast(uint16_t, row[min(k + 2 * i, K - 1)]) |
                     static_cast<uint32_t>(__builtin_bit_cast(uint16_t, row[min(k + 2 * i + 1, K - 1)])) << 16;
    }
}
template <bool VEC, typename T>
__device__ __forceinline__ void clear_past(Octet<T>& o, int64_t k, int64_t K) {
    constexpr int kPerWord = 4 / static_cast<int>(sizeof(T));
#pragma unroll
    for (int i = 0; i < Octet<T>::kWords; ++i) {
        if (VEC ? k >= K : k + i * kPerWord >= K) o.w[i] = 0;
        else if (!VEC && kPerWord == 2 && k + i * 2 + 1 >= K) o.w[i] &= 0xffffu;
    }
}

// Joins the workgroup's waves once their LDS operations are done. Unlike
// __syncthreads it leaves global loads in flight (they only fill registers).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The next plane of eight values: their upper 16 bits, which are taken off them.
__device__ __forceinline__ uint4 take_plane(float (&f)[8]) {
    uint32_t hi[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        hi[i] = __float_as_uint(f[i]) & 0xffff0000u;
        f[i] -= __uint_as_float(hi[i]);
    }
    uint4 r;
    r.x = (hi[0] >> 16) | hi[1];
    r.y = (hi[2] >> 16) | hi[3];
    r.z = (hi[4] >> 16) | hi[5];
    r.w = (hi[6] >> 16) | hi[7];
    return r;
}

// A block tile of BM rows of A by BN rows of B, K in steps of BK through one LDS
// buffer; the next step's operands are loaded into registers before this step's
// products and split on their way into LDS. BK = 64 where neither operand is
// split (eight MFMAs a wave and step otherwise), else 32. An LDS row is BK
// 16-bit values of one plane; 16-byte group g of row r sits at group
// g ^ swizzle(r), so that the sixteen rows read by sixteen consecutive lanes
// fill 256 distinct bytes of banks.
template <typename TA, typename TB, int BM, int BN>
struct Tile {
    static constexpr int NA = planes<TA, TB>(), NB = planes<TB, TA>();
    static constexpr bool kNative = NA == 1 && NB == 1;
    static constexpr bool kHalf = kNative && std::is_same<TA, f16>::value;
    static constexpr int BK = kNative ? 64 : 32;
    static constexpr int kGroups = BK / 8;
    static constexpr int MT = BM / 64, NT = BN / 64;  // 32 x 32 tiles of a wave
    static constexpr int kRowBytes = BK * 2;
    static constexpr int kLdsBytes = (NA * BM + NB * BN) * kRowBytes;
    static constexpr int OA = BM * kGroups / kThreads, OB = BN * kGroups / kThreads;  // octets per thread
    static_assert(OA >= 1 && OB >= 1, "a thread stages at least one octet of each operand");

    __device__ static int swizzle(int r) { return BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; }
    __device__ static int at(int r, int g) { return r * kRowBytes + ((g ^ swizzle(r)) << 4); }

    f32x16 acc[MT][NT];

    // a_row(r), b_row(r): pointers to row r of the block tile's operands, for
    // rows this thread stages (already clamped to rows that exist).
    // b_first(t): the block tile's B row where this wave's n-tile t starts.
    template <bool VEC, typename ARow, typename BRow, typename BFirst>
    __device__ __forceinline__ void run(char* lds, int64_t KA, int64_t KB, int64_t k_begin, int64_t k_end, ARow a_row,
                                        BRow b_row, BFirst b_first) {
        const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
        const int wm = wave >> 1;
        const TA* ap[OA];
        const TB* bp[OB];
#pragma unroll
        for (int i = 0; i < OA; ++i) ap[i] = a_row((tid + i * kThreads) / kGroups);
#pragma unroll
        for (int i = 0; i < OB; ++i) bp[i] = b_row((tid + i * kThreads) / kGroups);
        const int g = tid % kGroups;  // kThreads is a multiple of kGroups: the same group in every octet
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
        char* const lds_b = lds + NA * BM * kRowBytes;
        Octet<TA> ao[OA];
        Octet<TB> bo[OB];
        auto load = [&](int64_t k0) {
#pragma unroll
            for (int i = 0; i < OA; ++i) load_octet<VEC>(ao[i], ap[i], k0 + g * 8, KA);
#pragma unroll
            for (int i = 0; i < OB; ++i) load_octet<VEC>(bo[i], bp[i], k0 + g * 8, KB);
        };
        load(k_begin);
        for (int64_t k0 = k_begin; k0 < k_end; k0 += BK) {
            lds_barrier();  // every wave is done with the previous step's planes
            if (k0 + BK > KA || k0 + BK > KB) {  // only the last step reaches past K
#pragma unroll
                for (int i = 0; i < OA; ++i) clear_past<VEC>(ao[i], k0 + g * 8, KA);
#pragma unroll
                for (int i = 0; i < OB; ++i) clear_past<VEC>(bo[i], k0 + g * 8, KB);
            }
            stage<TA, NA, OA, BM>(lds, ao, g);
            stage<TB, NB, OB, BN>(lds_b, bo, g);
            if (k0 + BK < k_end) load(k0 + BK);
            lds_barrier();
#pragma unroll
            for (int kk = 0; kk < BK / 16; ++kk) {
                const int fg = kk * 2 + (lane >> 5);
                uint4 af[NA][MT], bf[NB][NT];
#pragma unroll
                for (int p = 0; p < NA; ++p)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        af[p][t] = *reinterpret_cast<const uint4*>(
                            lds + p * BM * kRowBytes + at(wm * (BM / 2) + t * 32 + (lane & 31), fg));
#pragma unroll
                for (int p = 0; p < NB; ++p)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        bf[p][t] = *reinterpret_cast<const uint4*>(lds_b + p * BN * kRowBytes +
                                                                  at(b_first(t) + (lane & 31), fg));
                // smallest products first
#pragma unroll
                for (int s = 2; s >= 0; --s)
#pragma unroll
                    for (int p = 0; p < NA; ++p) {
                        const int q = s - p;
                        if (q < 0 || q >= NB) continue;
#pragma unroll
                        for (int i = 0; i < MT; ++i)
#pragma unroll
                            for (int j = 0; j < NT; ++j) {
                                if constexpr (kHalf)
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                        __builtin_bit_cast(f16x8, bf[q][j]), __builtin_bit_cast(f16x8, af[p][i]),
                                        acc[i][j], 0, 0, 0);
                                else
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                        __builtin_bit_cast(bf16x8, bf[q][j]), __builtin_bit_cast(bf16x8, af[p][i]),
                                        acc[i][j], 0, 0, 0);
                            }
                    }
            }
        }
    }

  private:
    template <typename T, int P, int O, int R>
    __device__ static __forceinline__ void stage(char* lds, Octet<T> (&o)[O], int g) {
#pragma unroll
        for (int i = 0; i < O; ++i) {
            const int off = at((threadIdx.x + i * kThreads) / kGroups, g);
            if constexpr (P == 1) {
                *reinterpret_cast<uint4*>(lds + off) = make_uint4(o[i].w[0], o[i].w[1], o[i].w[2], o[i].w[3]);
            } else {
                float f[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = o[i].value(e);
#pragma unroll
                for (int p = 0; p < P; ++p) *reinterpret_cast<uint4*>(lds + p * R * kRowBytes + off) = take_plane(f);
            }
        }
    }
};

// Element v of a lane's accumulators of n-tile t: A row `lane % 32` of the
// m-tile, B row 8 (v / 4) + 4 (lane / 32) + v % 4 of the n-tile.
__device__ __forceinline__ int acc_column(int v) { return 8 * (v / 4) + 4 * (lane_id() / 32) + v % 4; }

__device__ __forceinline__ bool finite(float v) { return fabsf(v) < __builtin_inff(); }

// start + sum_k a[k] b[k] as one fp32 multiply-add chain.
template <typename TA, typename TB>
__device__ __noinline__ float scalar_dot(const TA* a, const TB* b, int64_t K, float start) {
    for (int64_t k = 0; k < K; ++k) start = __builtin_fmaf(to_f32(a[k]), to_f32(b[k]), start);
    return start;
}

}  // namespace split_gemm
}  // namespace koemi
