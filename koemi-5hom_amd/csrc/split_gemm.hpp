// Matrix-core tiles for operands of any floating type, width and alignment.
//
// C = A B^T (both operands K-contiguous) on v_mfma_f32_32x32x16, fp32
// accumulation. Two operands of the same 16-bit type go to the matrix cores as
// they are (every product exact). Any other pair is split into bf16 planes that
// sum to the operand exactly: fp32 into three, fp16 into two, bf16 is its own.
// A plane is what the planes before it left, rounded to the nearest bf16: with x
// in [2^e, 2^(e+1)) the second plane is at most 2^(e-8) and the third 2^(e-17), of
// either sign, and the last remainder is exact. The products of planes i and j
// with i + j <= 2 are accumulated: six for fp32 x fp32, five for fp32 x fp16, three
// for fp32 x bf16 (all of them). Dropped are at most 2^-24 of the product (fp32 x
// fp32) or 2^-25 (x fp16), of either sign, so they average out as the roundings of
// an fp32 multiply-add chain do. Planes cut off by truncation instead drop up to
// 2^-21, always toward zero: with 4096 terms of one sign that bias is 191 units of
// 2^-24 of the result where a chain's rms error is 14 and these planes' 8.8 (256 x
// 256 uniform positive operands; 8 terms: 0.96, 0.75 and 0.44; 1024 normal ones:
// 0.41, 0.47 and 0.40 of the terms' sizes). One or two terms come out within 2.3
// units, where a chain's are within 1 and 1.8.
//
// Infinities and NaN do not survive a split (inf x 0 between planes), nor do
// values that round past bf16's range. A tile with an output that is not finite
// walks K again on one plane of what each operand is (classes): infinities and NaN
// as they are, any other value as 0 or a power of two whose products vanish, so
// that a NaN output becomes the infinity or NaN that multiply-adds give and the
// finite ones keep their bits. A NaN that finite operands made is left to the caller
// (scalar_dot). [16384, 1024] gates with their scan, every input NaN: 0.60 ms (0.44
// finite; 60 with a chain for each output, 0.61 with the library's fp32 products).
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

// Bytes per load that the rows of an operand allow: 16 or 8 where every row starts
// aligned to them (the base and the row length), else kElementLoads.
constexpr int kElementLoads = 0;
template <typename T>
inline int load_bytes(const void* base, int64_t K) {
    const uintptr_t both = reinterpret_cast<uintptr_t>(base) | static_cast<uintptr_t>(K * static_cast<int64_t>(sizeof(T)));
    return both % 16 == 0 ? 16 : both % 8 == 0 ? 8 : kElementLoads;
}

// K values [k, k + 8) of a row, in pieces of BYTES (load_bytes): a piece lies
// within K or past it. What lies past K is read at a clamped address and cleared
// by clear_past, which the caller runs when it uses the octet: a select beside
// the load would wait for it. K >= 1.
template <int BYTES, typename T>
__device__ __forceinline__ void load_octet(Octet<T>& o, const T* __restrict__ row, int64_t k, int64_t K) {
    if constexpr (BYTES != kElementLoads) {
        constexpr int n = BYTES / static_cast<int>(sizeof(T)), words = BYTES / 4;
#pragma unroll
        for (int i = 0; i < 8 / n; ++i) {
            const T* p = row + min(k + i * n, K - n);
            if constexpr (BYTES == 16) {
                const uint4 v = *reinterpret_cast<const uint4*>(p);
                o.w[i * words] = v.x, o.w[i * words + 1] = v.y, o.w[i * words + 2] = v.z, o.w[i * words + 3] = v.w;
            } else {
                const uint2 v = *reinterpret_cast<const uint2*>(p);
                o.w[i * words] = v.x, o.w[i * words + 1] = v.y;
            }
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
// The same from a K-strided operand: value k of the column at p is p[k * ld].
// tail (wave-uniform): the step reaches past K.
template <typename T>
__device__ __forceinline__ void load_octet_strided(Octet<T>& o, const T* __restrict__ p, int64_t ld, int64_t k, int64_t K,
                                                   bool tail) {
    T e[8];
    if (tail) {
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = p[min(k + i, K - 1) * ld];
    } else {
        const T* q = p + k * ld;
#pragma unroll
        for (int i = 0; i < 8; ++i, q += ld) e[i] = *q;
    }
#pragma unroll
    for (int i = 0; i < Octet<T>::kWords; ++i) {
        if constexpr (sizeof(T) == 4) o.w[i] = __float_as_uint(e[i]);
        else
            o.w[i] = __builtin_bit_cast(uint16_t, e[2 * i]) |
                     static_cast<uint32_t>(__builtin_bit_cast(uint16_t, e[2 * i + 1])) << 16;
    }
}
template <typename T>
__device__ __forceinline__ void clear_past(Octet<T>& o, int64_t k, int64_t K) {
    constexpr int kPerWord = 4 / static_cast<int>(sizeof(T));
#pragma unroll
    for (int i = 0; i < Octet<T>::kWords; ++i) {
        const bool out = k + i * kPerWord >= K;
        if (kPerWord == 2) o.w[i] &= out ? 0u : k + i * 2 + 1 >= K ? 0xffffu : 0xffffffffu;
        else o.w[i] = out ? 0u : o.w[i];
    }
}

// Joins the workgroup's waves once their LDS operations are done. Unlike
// __syncthreads it leaves global loads in flight (they only fill registers).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The next plane of eight values: the nearest bf16 of each, which is taken off it
// (one packed conversion a pair).
__device__ __forceinline__ uint4 take_plane(float (&f)[8]) {
    bf16x8 plane;
#pragma unroll
    for (int i = 0; i < 8; ++i) plane[i] = static_cast<__bf16>(f[i]);
    const uint4 r = __builtin_bit_cast(uint4, plane);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] -= __uint_as_float(i % 2 ? w[i / 2] & 0xffff0000u : w[i / 2] << 16);
    return r;
}

// Eight values as bf16 classes: infinities and NaN as they are, others as 0 or a
// signed 2^-100 (a product of two lies below fp32's smallest step).
template <typename T>
__device__ __forceinline__ uint4 classes(const Octet<T>& o) {
    bf16x8 c;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float f = o.value(i);
        c[i] = static_cast<__bf16>(fabsf(f) < __builtin_inff() ? f == 0.0f ? 0.0f : copysignf(0x1p-100f, f) : f);
    }
    return __builtin_bit_cast(uint4, c);
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) < __builtin_inff(); }

// Element v of a lane's accumulators of n-tile t: A row `lane % 32` of the
// m-tile, B row 8 (v / 4) + 4 (lane / 32) + v % 4 of the n-tile.
__device__ __forceinline__ int acc_column(int v) { return 8 * (v / 4) + 4 * (lane_id() / 32) + v % 4; }

// start + sum_k a[k a_ld] b[k b_ld] as one fp32 multiply-add chain.
template <typename TA, typename TB>
__device__ __noinline__ float scalar_dot(const TA* a, const TB* b, int64_t K, float start, int64_t a_ld = 1,
                                         int64_t b_ld = 1) {
    for (int64_t k = 0; k < K; ++k) start = __builtin_fmaf(to_f32(a[k * a_ld]), to_f32(b[k * b_ld]), start);
    return start;
}

// A block tile of BM rows of A by BN rows of B, K in steps of BK through one LDS
// buffer; the next step's operands are loaded into registers before this step's
// products and split on their way into LDS. BK = 64 where neither operand is
// split (eight MFMAs a wave and step otherwise), else 32. An LDS row is BK
// 16-bit values of one plane; 16-byte group g of row r sits at group
// g ^ swizzle(r), so that the sixteen rows read by sixteen consecutive lanes
// fill 256 distinct bytes of banks. A_STRIDED / B_STRIDED: the operand is stored
// K-major ([K, rows]); its octets are gathered by eight loads, each coalesced
// over the rows of consecutive lanes.
// DEPTH: K steps whose operands are on their way in registers; more than one where
// a launch has too few tiles to hide the loads behind other workgroups. Split
// operands then also start a new sum every DEPTH steps (kFold): for so few tiles
// the library splits K over workgroups, and its shorter sums err less ([168, 512]
// gates: 2.45e-7 from float64 with its product, 3.25e-7 in one sum, 2.16e-7 so).
template <typename TA, typename TB, int BM, int BN, bool A_STRIDED = false, bool B_STRIDED = false, int DEPTH = 1>
struct Tile {
    static constexpr int NA = planes<TA, TB>(), NB = planes<TB, TA>();
    static constexpr bool kNative = NA == 1 && NB == 1;
    static constexpr bool kHalf = kNative && std::is_same<TA, f16>::value;
    static constexpr int BK = kNative ? 64 : 32;
    static constexpr int kGroups = BK / 8;
    static constexpr int MT = BM / 64, NT = BN / 64;  // 32 x 32 tiles of a wave
    static constexpr int kRowBytes = BK * 2;
    static constexpr int kSets = kNative ? 2 : 1;  // fragment sets held by a wave
    static constexpr bool kFold = !kNative && DEPTH > 1;
    static constexpr int kLdsBytes = (NA * BM + NB * BN) * kRowBytes;
    static constexpr int OA = BM * kGroups / kThreads, OB = BN * kGroups / kThreads;  // octets per thread
    static_assert(OA >= 1 && OB >= 1, "a thread stages at least one octet of each operand");

    __device__ static int swizzle(int r) { return BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; }
    __device__ static int at(int r, int g) { return r * kRowBytes + ((g ^ swizzle(r)) << 4); }

    f32x16 acc[MT][NT];

    // Octet i of the thread, of an operand of R rows: its row and K group. Eight
    // or four consecutive threads share a row of a K-contiguous operand (its
    // 16-byte pieces), consecutive threads take consecutive rows of a strided one.
    template <int R, bool STRIDED>
    __device__ static int octet_row(int i, int tid = threadIdx.x) {
        return STRIDED ? (tid + i * kThreads) % R : (tid + i * kThreads) / kGroups;
    }
    template <int R, bool STRIDED>
    __device__ static int octet_group(int i, int tid = threadIdx.x) {
        return STRIDED ? (tid + i * kThreads) / R : tid % kGroups;
    }

    // a_row(r), b_row(r): pointers to row r of the block tile's operands, for
    // rows this thread stages (already clamped to rows that exist), read in pieces of
    // A_BYTES and B_BYTES; a strided
    // operand's row is the column whose value k lies at k * a_ld (b_ld).
    // b_first(t): the block tile's B row where this wave's n-tile t starts.
    // Split operands: the workgroup's waves are joined at the end (LDS is free). Returns
    // a bit ((i NT + j) 16 + v) for each output of the lane that the caller has to form
    // with scalar_dot (fix_chains).
    template <int A_BYTES, int B_BYTES, typename ARow, typename BRow, typename BFirst>
    __device__ __forceinline__ uint64_t run(char* lds, int64_t KA, int64_t KB, int64_t k_begin, int64_t k_end,
                                            ARow a_row, BRow b_row, BFirst b_first, int64_t a_ld = 1, int64_t b_ld = 1) {
        const int lane = lane_id(), wave = threadIdx.x / kWave;
        const int wm = wave >> 1;
        const TA* ap[OA];
        const TB* bp[OB];
#pragma unroll
        for (int i = 0; i < OA; ++i) ap[i] = a_row(octet_row<BM, A_STRIDED>(i));
#pragma unroll
        for (int i = 0; i < OB; ++i) bp[i] = b_row(octet_row<BN, B_STRIDED>(i));
        clear(acc);
        char* const lds_b = lds + NA * BM * kRowBytes;
        Octet<TA> a_ring[DEPTH][OA];
        Octet<TB> b_ring[DEPTH][OB];
        auto load = [&](int64_t k0, Octet<TA> (&ao)[OA], Octet<TB> (&bo)[OB]) {
#pragma unroll
            for (int i = 0; i < OA; ++i) {
                const int64_t k = k0 + octet_group<BM, A_STRIDED>(i) * 8;
                if constexpr (A_STRIDED) load_octet_strided(ao[i], ap[i], a_ld, k, KA, k0 + BK > KA);
                else load_octet<A_BYTES>(ao[i], ap[i], k, KA);
            }
#pragma unroll
            for (int i = 0; i < OB; ++i) {
                const int64_t k = k0 + octet_group<BN, B_STRIDED>(i) * 8;
                if constexpr (B_STRIDED) load_octet_strided(bo[i], bp[i], b_ld, k, KB, k0 + BK > KB);
                else load_octet<B_BYTES>(bo[i], bp[i], k, KB);
            }
        };
        auto step = [&](int64_t k0, Octet<TA> (&ao)[OA], Octet<TB> (&bo)[OB]) {
            lds_barrier();  // every wave is done with the previous step's planes
            if (k0 + BK > KA || k0 + BK > KB) {  // only the last step reaches past K
#pragma unroll
                for (int i = 0; i < OA; ++i) clear_past(ao[i], k0 + octet_group<BM, A_STRIDED>(i) * 8, KA);
#pragma unroll
                for (int i = 0; i < OB; ++i) clear_past(bo[i], k0 + octet_group<BN, B_STRIDED>(i) * 8, KB);
            }
            stage<TA, NA, OA, BM, A_STRIDED>(lds, ao);
            stage<TB, NB, OB, BN, B_STRIDED>(lds_b, bo);
            if (k0 + DEPTH * BK < k_end) load(k0 + DEPTH * BK, ao, bo);
            lds_barrier();
            // the fragments of K group kk + 1 are read under the products of group kk
            // where two sets fit the registers (one product each)
            uint4 af[kSets][NA][MT], bf[kSets][NB][NT];
            auto read = [&](int kk, int set) {
                const int fg = kk * 2 + (lane >> 5);
#pragma unroll
                for (int p = 0; p < NA; ++p)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        af[set][p][t] = *reinterpret_cast<const uint4*>(
                            lds + p * BM * kRowBytes + at(wm * (BM / 2) + t * 32 + (lane & 31), fg));
#pragma unroll
                for (int p = 0; p < NB; ++p)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        bf[set][p][t] = *reinterpret_cast<const uint4*>(lds_b + p * BN * kRowBytes +
                                                                       at(b_first(t) + (lane & 31), fg));
            };
            read(0, 0);
#pragma unroll
            for (int kk = 0; kk < BK / 16; ++kk) {
                const int set = kk % kSets;
                if (kSets == 2 && kk + 1 < BK / 16) read(kk + 1, 1 - set);
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
                                        __builtin_bit_cast(f16x8, bf[set][q][j]),
                                        __builtin_bit_cast(f16x8, af[set][p][i]), acc[i][j], 0, 0, 0);
                                else
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                        __builtin_bit_cast(bf16x8, bf[set][q][j]),
                                        __builtin_bit_cast(bf16x8, af[set][p][i]), acc[i][j], 0, 0, 0);
                            }
                    }
                if (kSets == 1 && kk + 1 < BK / 16) read(kk + 1, 0);
            }
        };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (k_begin + d * BK < k_end) load(k_begin + d * BK, a_ring[d], b_ring[d]);
        f32x16 total[MT][NT];
        if constexpr (kFold) clear(total);
        for (int64_t k0 = k_begin; k0 < k_end; k0 += DEPTH * BK) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d)
                if (k0 + d * BK < k_end) step(k0 + d * BK, a_ring[d], b_ring[d]);
            if constexpr (kFold) {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) total[i][j] += acc[i][j];
                clear(acc);
            }
        }
        if constexpr (kFold) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j];
        }
        uint64_t chains = 0;
        if constexpr (!kNative) {
            float zero[4] = {};  // NaN once an output is not finite: one multiply-add an output
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) zero[v % 4] = __builtin_fmaf(acc[i][j][v], 0.0f, zero[v % 4]);
            const bool whole = (zero[0] + zero[1]) + (zero[2] + zero[3]) == 0.0f;
            __shared__ __attribute__((aligned(16))) uint32_t votes[kThreads / kWave];
            const uint32_t vote = __ballot(!whole) != 0;
            if (lane == 0) votes[wave] = vote;
            lds_barrier();
            const uint4 any = *reinterpret_cast<const uint4*>(votes);
            if (__builtin_expect((any.x | any.y | any.z | any.w) != 0, 0)) {
                // an infinity came of finite operands (an infinite one makes NaN planes)
                // and stays; a NaN becomes what the classes say
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const bool nan = acc[i][j][v] != acc[i][j][v];
                            chains |= nan ? 1ull << ((i * NT + j) * 16 + v) : 0ull;
                            acc[i][j][v] = nan ? 0.0f : acc[i][j][v];
                        }
                // rows and addresses formed anew: kept from the loop above they would
                // cost every tile their registers
                int tid = threadIdx.x;
                asm volatile("" : "+v"(tid));
                for (int64_t k0 = k_begin; k0 < k_end; k0 += BK) {
                    lds_barrier();  // every wave is done with the previous step's classes
                    class_step<A_BYTES, BM, OA, A_STRIDED>(lds, tid, k0, KA, a_ld, a_row);
                    class_step<B_BYTES, BN, OB, B_STRIDED>(lds_b, tid, k0, KB, b_ld, b_row);
                    lds_barrier();
#pragma unroll
                    for (int kk = 0; kk < BK / 16; ++kk) {
                        const int fg = kk * 2 + (lane >> 5);
#pragma unroll
                        for (int i = 0; i < MT; ++i)
#pragma unroll
                            for (int j = 0; j < NT; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                    *reinterpret_cast<const bf16x8*>(lds_b + at(b_first(j) + (lane & 31), fg)),
                                    *reinterpret_cast<const bf16x8*>(lds + at(wm * (BM / 2) + i * 32 + (lane & 31), fg)),
                                    acc[i][j], 0, 0, 0);
                    }
                }
                // a NaN of finite operands (infinities of both signs, planes past bf16's range):
                // the caller's
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            chains &= finite(acc[i][j][v]) ? ~0ull : ~(1ull << ((i * NT + j) * 16 + v));
                lds_barrier();
            }
        }
        return chains;
    }

  private:
    // One operand's classes of the K step at k0 into LDS.
    template <int BYTES, int R, int O, bool STRIDED, typename Row>
    __device__ static __forceinline__ void class_step(char* lds, int tid, int64_t k0, int64_t K, int64_t ld, Row row) {
        using T = std::remove_const_t<std::remove_pointer_t<decltype(row(0))>>;
        Octet<T> o[O];
#pragma unroll
        for (int i = 0; i < O; ++i) {
            const int64_t k = k0 + octet_group<R, STRIDED>(i, tid) * 8;
            if constexpr (STRIDED) load_octet_strided(o[i], row(octet_row<R, STRIDED>(i, tid)), ld, k, K, k0 + BK > K);
            else load_octet<BYTES>(o[i], row(octet_row<R, STRIDED>(i, tid)), k, K);
        }
#pragma unroll
        for (int i = 0; i < O; ++i) {
            clear_past(o[i], k0 + octet_group<R, STRIDED>(i, tid) * 8, K);
            *reinterpret_cast<uint4*>(lds + at(octet_row<R, STRIDED>(i, tid), octet_group<R, STRIDED>(i, tid))) =
                classes(o[i]);
        }
    }

    __device__ static __forceinline__ void clear(f32x16 (&a)[MT][NT]) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) a[i][j] = f32x16{};
    }

    template <typename T, int P, int O, int R, bool STRIDED>
    __device__ static __forceinline__ void stage(char* lds, Octet<T> (&o)[O]) {
#pragma unroll
        for (int i = 0; i < O; ++i) {
            const int off = at(octet_row<R, STRIDED>(i), octet_group<R, STRIDED>(i));
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

// Runs fix(block, v) for every bit that Tile::run returned, after this lane's stores
// have left: a rolled loop, so that the rare case costs the kernel no registers.
template <typename Fix>
__device__ __forceinline__ void fix_chains(uint64_t chains, Fix fix) {
    if (__builtin_expect(__ballot(chains != 0) == 0, 1)) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    while (chains) {
        const int b = __builtin_ctzll(chains);
        chains &= chains - 1;
        fix(b / 16, b % 16);
    }
}

// Stores a wave's 32 x (32 J) outputs as full rows: o[j][v] is row lane % 32,
// column 32 j + acc_column(v) of the wave's block, whose first element goes to
// out[0] (rows ld apart). They pass through the wave's own LDS region of
// store_bytes<T, J>() and leave in 16-byte pieces of whole rows (without it every
// store would touch 32 rows). rows, cols: how many of them exist. VEC: rows of
// out start 16-byte aligned and cols is a multiple of 8; otherwise the pieces are
// stored element by element. The caller has joined the workgroup's waves after
// the tile's last LDS reads.
template <typename T, int J>
constexpr int store_bytes() {
    return 32 * (32 * J * static_cast<int>(sizeof(T)) + 16);
}
template <typename T, int J>
__device__ __forceinline__ void store_rows(char* region, const float (&o)[J][16], T* __restrict__ out, int64_t ld,
                                           int64_t rows, int64_t cols, bool vec) {
    constexpr int kRow = 32 * J * static_cast<int>(sizeof(T)) + 16, kPieces = (kRow - 16) / 16;
    constexpr int kPer = 16 / static_cast<int>(sizeof(T));
    const int lane = lane_id();
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            union {
                T e[4];
                uint32_t w[sizeof(T)];
            } u;
#pragma unroll
            for (int q = 0; q < 4; ++q) u.e[q] = from_f32<T>(o[j][v + q]);
            char* at = region + (lane & 31) * kRow + (j * 32 + acc_column(v)) * static_cast<int>(sizeof(T));
            if constexpr (sizeof(T) == 4) *reinterpret_cast<uint4*>(at) = make_uint4(u.w[0], u.w[1], u.w[2], u.w[3]);
            else *reinterpret_cast<uint2*>(at) = make_uint2(u.w[0], u.w[1]);
        }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own region: in order, no barrier
#pragma unroll
    for (int i = 0; i < 32 * kPieces / kWave; ++i) {
        const int piece = i * kWave + lane, r = piece / kPieces, c = piece % kPieces * kPer;
        union {
            uint4 raw;
            T e[kPer];
        } u;
        u.raw = *reinterpret_cast<const uint4*>(region + r * kRow + c * static_cast<int>(sizeof(T)));
        if (r >= rows) continue;
        T* p = out + r * ld + c;
        if (vec) {
            if (c < cols) *reinterpret_cast<uint4*>(p) = u.raw;
        } else {
#pragma unroll
            for (int q = 0; q < kPer; ++q)
                if (c + q < cols) p[q] = u.e[q];
        }
    }
    asm volatile("" ::: "memory");
}

}  // namespace split_gemm
}  // namespace koemi
