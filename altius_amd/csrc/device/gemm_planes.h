// A product's sums on the bf16 matrix cores where the second operand is a weight matrix kept as planes: the main loop of
// gemm_f32_tiles (matmul.hip) for such products.
//
// Every value times 2^24 is the exact sum of three bf16 numbers, down to the smallest denormal, and of the nine products of two values'
// parts six are taken, as in gemm_split.hip (the other three are below 2^-26 of the product).  The five small products of a step meet in
// sums of their own, 2^-8 of the large ones, so that only one in six additions is rounded to a large sum.  Against float64 (rel 2-norm,
// [1024,768] x [768,768] and [130,3072] x [3072,770]): 0.9e-7 and 1.0e-7 in four chains, 1.6e-7 and 1.6e-7 in one; with one sum for all six
// 2.1e-7 and 2.2e-7, 4.2e-7 and 4.3e-7; the fp32 kernel 2.5e-7 to 3.5e-7 and 5.0e-7 to 7.0e-7.  Sums of one sign are no worse off: uniform
// operands in [0, 1), or positive parts times positive weights, 0.5e-7 to 1.8e-7 where the fp32 kernel has 0.8e-7 to 8.4e-7 (k from 64 to
// 4096, all tiles), with a mean error of 1e-9.  Whole numbers whose sums fit 24 bits are exact.  Only where one or two products of a sum are
// not zero is it off by up to 1.04 times the fp32 kernel's (2.6e-8 and 2.5e-8); from eight on at most 0.6.  What does not come out finite
// (infinities, NaN, values beyond 2^103, sums beyond 2^79) is computed again by the caller.
//
// What bounds it: with every CU busy the power limit (4096^3 at 200 to 210 Tflop/s; 213 is what a large bf16 product reaches here, by six);
// otherwise a wavefront's instructions, one every four to five cycles, of which the 32 cycles of an instruction of the matrix cores cover
// six.  So the weights are split once, when a session is built (6 bytes a value instead of 4), and go from memory into registers in the
// order in which the instruction takes them; a value of the first operand is split once per block, on its way into LDS, in parts of four
// instructions or fewer behind each product; and a SIMD has two wavefronts.  Splitting both operands in registers behind LDS, by each
// wavefront: 12 to 18 instructions a product, 1024 x 768 x 3072 in 48 us instead of 33.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace altius {
// f(0) .. f(N - 1) with the number known when f is compiled.
template <class F, int... I> __device__ __forceinline__ void each_of(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>()), ...); }
template <int N, class F> __device__ __forceinline__ void each(F f) { each_of(f, std::make_integer_sequence<int, N>()); }

namespace planes {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) char *global_ptr;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// SET bytes for 32 columns (rows) and 16 values of k: three planes of 64 lanes with eight values each, in the order in which the
// instruction takes them.  Of 64 values of k set j (0 .. 3) has 8 j + 0 .. 7 and 32 more: lane l has column l % 32 and
// k = 8 j + 4 (l / 32) + 0 .. 3 and 32 more, so that neighbouring lanes that fetch a row of the first operand read whole lines.
constexpr uint32_t SET = 3072;
__device__ __forceinline__ uint32_t k_of(uint32_t set, uint32_t half, uint32_t e) { return set / 4 * 64 + set % 4 * 8 + 4 * half + e % 4 + e / 4 * 32; }
constexpr float SCALE = 0x1p24f, UNSCALE = 0x1p-48f;

__device__ __forceinline__ uint32_t pack(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// Four values on their way to three bf16 numbers each, in eight parts that products stand between.
struct Split4 {
    float x[4], t[4];
    u32x2 q0, q1, q2;
    template <int P> __device__ __forceinline__ u32x2 &q() {
        if constexpr (P == 0) return q0;
        else if constexpr (P == 1) return q1;
        else return q2;
    }
    template <int PART> __device__ __forceinline__ void part(const f32x4 &v) {
        if constexpr (PART == 0) {
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = v[e] * SCALE;
        } else if constexpr (PART == 1 || PART == 4 || PART == 7) {
#pragma unroll
            for (int e = 0; e < 2; e++) q<PART / 3>()[e] = pack(x[2 * e], x[2 * e + 1]);
        } else if constexpr (PART == 2 || PART == 5) {
#pragma unroll
            for (int e = 0; e < 4; e++) t[e] = __uint_as_float(e % 2 ? q<PART / 3>()[e / 2] & 0xffff0000u : q<PART / 3>()[e / 2] << 16);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] -= t[e];
        }
    }
};

// The tile of a block: WM x WN x WK wavefronts, WK of them along k, with TA x TB tiles of 32 x 32 each.  A step is one set of k per
// wavefront along k.  While step s multiplies, step s + 1's fragments of the first operand come out of LDS, step s + 2's values are split into
// the buffer that step s has left, and memory is asked for the values of step s + 2 + NA and the weights of step s + 1.  One barrier a step.
// Steps go in turns of U, the last turn with zeros behind the end of k.
template <int WM, int WN, int WK, int TA, int TB, int VEC, int NA> struct Tile {
    static constexpr int WAVES = WM * WN * WK, THREADS = 64 * WAVES, BM = 32 * WM * TA, BKT = 16 * WK;
    static constexpr int SETS = BM / 32 * WK, CH = BM * BKT / 8 / THREADS;
    static_assert(CH * THREADS * 8 == BM * BKT, "whole pieces");
    static constexpr int LDS_BYTES = 2 * SETS * (int)SET;
    static constexpr int U = 2;  // steps until registers and buffers are the same again
    static_assert(U % NA == 0, "whole turns");

    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[CH], kp[CH], to[CH], from;
    global_ptr b[TB];
    uint32_t k, last_set, lane16;
    int wk;
    char *lds;

    // a: the tile's first row at its first value of k, rows of them and k values; weights: of the tile's first column (of n32s left) and value of k.
    __device__ __forceinline__ void start(const float *a, uint32_t lda, uint32_t rows, uint32_t k_, const char *weights, uint32_t n32s, uint32_t col_sets,
                                          uint32_t sets_left, void *lds_, int tid, int wm, int wn, int wk_) {
        lds = static_cast<char *>(lds_);
        wk = wk_;
        k = (uint32_t)__builtin_amdgcn_readfirstlane((int)k_);
        last_set = (uint32_t)__builtin_amdgcn_readfirstlane((int)(sets_left - 1));
        const uint32_t bytes = k ? ((rows - 1) * lda + k) * 4u : 0;
        const uint64_t at = (uint64_t)(uintptr_t)a;
        const uint64_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32)) << 32;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(first), 0, __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const uint32_t f = c * THREADS + tid, piece = f % (2 * WK), row = f / (2 * WK);
            kp[c] = piece / 8 * 64 + piece % 8 * 4;
            off[c] = (row * lda + kp[c]) * 4;
            // The pieces of a row go to different banks.
            to[c] = ((piece / 2) * (BM / 32) + row / 32) * SET + ((piece % 2) * 32 + ((row % 32) ^ (piece * 8 / WK))) * 16;
        }
        const uint32_t lane = tid & 63, lr = lane & 31, lk = lane >> 5;
        from = (wk * (BM / 32) + wm * TA) * SET + (lk * 32 + (lr ^ ((2 * wk + lk) * 8 / WK))) * 16;
#pragma unroll
        for (int j = 0; j < TB; j++) {
            const uint64_t p = (uint64_t)(uintptr_t)weights + (uint64_t)min((uint32_t)(wn * TB + j), n32s - 1) * col_sets * SET;
            b[j] = (global_ptr)((uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32)) << 32);
        }
        lane16 = lane * 16;
    }
    __device__ __forceinline__ void load_a(f32x4 (&r)[2], int c, uint32_t step) const {
        const uint32_t first = step * WK / 4 * 64 + step * WK % 4 * 8, at = off[c] + first * 4, kk = kp[c] + first;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if constexpr (VEC == 4) {
                r[h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, kk + 32 * h < k ? at + 128 * h : 0x80000000u, 0, 0));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    r[h][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, kk + 32 * h + e < k ? at + 128 * h + 4 * e : 0x80000000u, 0, 0));
            }
        }
    }
    __device__ __forceinline__ u32x4 load_b(int j, int p, uint32_t step) const {
        const uint32_t set = min(step * WK + wk, last_set);
        const uint32_t at = set * SET + lane16;
        return *reinterpret_cast<const __attribute__((address_space(1))) u32x4 *>(b[j] + at + p * 1024);
    }
    __device__ __forceinline__ static void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

    __device__ __forceinline__ void run(floatx16 (&acc)[TA][TB]) {
        constexpr int BUF = SETS * (int)SET;
        f32x4 ra[NA][CH][2];
        u32x4 xa[2][TA][3], xb[2][TB][3];
        floatx16 low[TA][TB];
#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int j = 0; j < TB; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = low[i][j][e] = 0.0f;
        const uint32_t nk = ((k + 63) / 64 * 4 + WK - 1) / WK;
        auto write = [&](int c, Split4 (&s)[2], int buf) __attribute__((always_inline)) {
            each<3>([&](auto p) __attribute__((always_inline)) {
                *reinterpret_cast<u32x4 *>(lds + buf * BUF + to[c] + p * 1024) = __builtin_shufflevector(s[0].template q<p>(), s[1].template q<p>(), 0, 1, 2, 3);
            });
        };
        auto read = [&](int i, int p, int buf) __attribute__((always_inline)) {
            return *reinterpret_cast<const u32x4 *>(lds + buf * BUF + from + i * SET + p * 1024);
        };
        {
            f32x4 first[2][CH][2];
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int c = 0; c < CH; c++) load_a(first[s][c], c, s);
            // In the order in which the steps load, so that a wait for one of them leaves as many of the others on their way as later ones do.
            each<NA>([&](auto t) __attribute__((always_inline)) {
                constexpr int at = t - NA, sb = at + 1, sa = at + 2 + NA;
                if constexpr (sb >= 0) {
#pragma unroll
                    for (int j = 0; j < TB; j++)
#pragma unroll
                        for (int p = 0; p < 3; p++) xb[sb][j][p] = load_b(j, p, sb);
                }
                if constexpr (sa >= 2) {
#pragma unroll
                    for (int c = 0; c < CH; c++) load_a(ra[sa % NA][c], c, sa);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int c = 0; c < CH; c++) {
                    Split4 sp[2];
                    each<8>([&](auto p) __attribute__((always_inline)) {
                        sp[0].template part<p>(first[s][c][0]);
                        sp[1].template part<p>(first[s][c][1]);
                    });
                    write(c, sp, s);
                }
        }
        barrier();
#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int p = 0; p < 3; p++) xa[0][i][p] = read(i, p, 0);
        barrier();

        constexpr int Q = 6 * TA * TB, READS = 3 * TA, LOADS = 3 * TB, PARTS = 16 * CH, QR = Q / 3 > 0 ? Q / 3 : 1, QP = Q * 3 / 4;
        auto step = [&](auto at, uint32_t s) __attribute__((always_inline)) {
            constexpr int now = at % 2, next = (at + 1) % 2, slot = (at + 2) % NA;
            Split4 sp[CH][2];
            each<Q>([&](auto q) __attribute__((always_inline)) {
                constexpr int T = q / (TA * TB), i = q / TB % TA, j = q % TB;
                constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};  // smallest terms first
                floatx16 &sum = T < 5 ? low[i][j] : acc[i][j];
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, xa[now][i][PA[T]]), __builtin_bit_cast(bf16x8, xb[now][j][PB[T]]), sum, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                each<READS>([&](auto r) __attribute__((always_inline)) {
                    if constexpr (r * QR / READS == q) xa[next][r / 3][r % 3] = read(r / 3, r % 3, next);
                });
                each<LOADS>([&](auto l) __attribute__((always_inline)) {
                    if constexpr (l * Q / LOADS == q) xb[next][l / 3][l % 3] = load_b(l / 3, l % 3, s + 1);
                });
                each<PARTS>([&](auto u) __attribute__((always_inline)) {
                    constexpr int c = u / 16, p = u / 2 % 8, h = u % 2;
                    if constexpr (u * QP / PARTS == q) sp[c][h].template part<p>(ra[slot][c][h]);
                });
                each<CH>([&](auto c) __attribute__((always_inline)) {
                    constexpr int done = (16 * c + 15) * QP / PARTS;
                    if constexpr (done == q) {
                        write(c, sp[c], now);
                        load_a(ra[slot][c], c, s + 2 + NA);
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
            });
            barrier();
        };
        for (uint32_t s = 0; s < nk; s += U) each<U>([&](auto at) __attribute__((always_inline)) { step(at, s + at); });
#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int j = 0; j < TB; j++) {
                asm volatile("" : "+v"(low[i][j]));  // added behind the loop, not in it
                acc[i][j] += low[i][j];
            }
    }
};

}  // namespace planes
}  // namespace altius
