// fp32 matrix multiplication on the matrix cores: C = alpha * op(A) * op(B) + beta * C0, batched
// with broadcast batch strides.  Counterparts in the reference: compute_mat_mul
// (crates/session_interpreter/src/session.rs:621-684) and compute_gemm (686-794), both of which
// call sgemm (crates/session_interpreter/src/gemm.rs: the `matrixmultiply` crate or CBLAS).
//
// One kernel, gemm_f32_tiles, with v_mfma_f32_32x32x2_f32 (fp32 in, fp32 accumulate: 256 flop per cycle per CU, 157 Tflop/s
// on the part).  A block's wavefronts form a WM x WN grid over its tile of C, each with TA x TB tiles of 32 x 32, and WK such
// grids take different values of k (their sums are added in LDS at the end): small tiles for products with few of them, whose
// time is a chain of loads that WK cuts, large tiles where the chip is full and traffic per operation counts.
//
// Operand tiles go from memory to LDS directly (buffer loads, which read zeros behind an operand's end and wherever k is past
// its end), up to S tiles ahead, with one barrier per tile.  Nothing is transposed on the way: an operand whose k is the
// contiguous axis lies in LDS as [row][16], its 16-byte pieces exchanged by piece ^= (row / 4) % 4 so that a column of pieces
// covers the banks, and a lane reads four values of k at once; one whose rows are contiguous lies as [k][row], and a lane reads
// TA (TB) neighbouring rows, one for each of its tiles.  The instruction takes two values of k, one per half of the wavefront;
// a half takes k = 8 i + 4 half + 0 .. 3 in turn, the same for both layouts, so that a product does not depend on them.
//
// Products with a weight matrix of which planes are kept run their sums on the bf16 matrix cores instead (gemm_planes.h), in the same tiles'
// epilogue.
//
// A step's two halves take turns in registers: while one half's products run, the other's fragments come from LDS, and what else a step
// does (the next loads and their addresses) stands between the products, where the matrix pipe covers it.  With a step's fragments
// all read in front of its products and the addresses worked out anew in every step, the pipes were busy 60 to 84 % of the cycles:
//   [6304,768] x [768,768 / 2304 / 3072]: 72 -> 63 us, 192 -> 184, 258 -> 228;  [6304,3072] x [3072,768]: 262 -> 227
//   [1024,768] x [768,768 / 3072]: 16.4 -> 14.7, 45 -> 40;  [1024,3072] x [3072,768]: 51 -> 46
//   [197,768] x [768,768]: 8.6 -> 7.1;  [77,768] x [768,3072]: 12.0 -> 10.2
//   4096^3: 1061 -> 938 us (147 Tflop/s; 145 on another day's card);  [50432,768] x [768,3072]: 1788 -> 1670 (143)
// Single-value loads are taken for both operands where one of them needs them.
// What is left on large shapes: the blocks' first loads and their results (1 us of 12 in a 64 x 64 tile with 768 values of k), and a last
// round of blocks that is partly empty where a cut costs as much as it gives ([6304,768] x [768,768]: 4.6 rounds take five, cut 64 us).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "ctx.h"
#include "gemm_planes.h"
#include "math.h"

namespace altius {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr;

constexpr int BK = 16;  // values of k a wavefront multiplies between two barriers

struct GemmArgs {
    const float *a, *b, *c0, *residual;
    float *c;
    uint32_t m, n, k;
    // Row pitches of the stored matrices.  C0 (Gemm's third input) is read as c0[i * c0_rs + j * c0_cs]; either stride may be 0.
    uint32_t lda, ldb, ldc, c0_rs, c0_cs;
    // Batch z is (z / batch_inner, z % batch_inner); operand X starts at x + (z / batch_inner) * x_bs + (z % batch_inner) * x_bs2
    // (strides in elements, 0 = shared).
    uint64_t a_bs, b_bs, c_bs, a_bs2, b_bs2, c_bs2;
    uint32_t batch_inner;
    // Consecutive block ids go to the eight XCDs in turn, and each XCD (one L2) is given a contiguous run of `chunk` tiles, so
    // that the blocks it runs together share panels.  Within that order tiles go by groups of group_n tile columns, each group
    // walked row of tiles by row of tiles, so that those blocks cover few columns of B (they stay in its L2) and many rows of A.
    uint32_t tiles_m, tiles_n, tiles, chunk, group_n;  // tiles: of all batches
    // Of each XCD's run the first `full` tiles are whole; of the others k is cut into `slices` of slice_k values (whole steps of the
    // block; the last one takes the rest): see the epilogue.
    uint32_t full, slices, slice_k;
    // Steps that 32-bit byte offsets reach behind the tile whose first element they count from, for both operands.
    uint32_t window;
    float *partials;
    int *counters;
    float alpha, beta;
    int act;
    float act_alpha, act_beta;
    // The blocks of a CU all start together, and go out of step by priorities: one's first loads and results beside another's products.
    // (Of 256 blocks dealt in turn each of the part's 256 CUs gets one, the next 256 are its second: with fewer CUs the priorities
    // would not differ where they should, and the results would be the same.)
    int apart;
    // The second operand's planes where it has some, [n32s][k16s] sets (gemm_planes.h); b is the same operand as it lies in memory, b_kc: along k.
    const char *planes;
    uint32_t n32s, k16s;
    int b_kc;
};

// Four floats that blocks on any XCD read and write.
struct Halves {
    unsigned long long h[2];
};
__device__ __forceinline__ void store_shared(f32x4 *p, const f32x4 &v) {
    const Halves b = __builtin_bit_cast(Halves, v);
    unsigned long long *q = reinterpret_cast<unsigned long long *>(p);
    __hip_atomic_store(q, b.h[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, b.h[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4 load_shared(const f32x4 *p) {
    const unsigned long long *q = reinterpret_cast<const unsigned long long *>(p);
    Halves b;
    b.h[0] = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    b.h[1] = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(f32x4, b);
}

// What a lane holds of T tiles of an operand for four values of k, half a step: at(tile, step).  KC: k is the operand's contiguous axis.
template <bool KC, int T> struct Frag;
template <int T> struct Frag<true, T> {
    f32x4 v[T];
    __device__ __forceinline__ float at(int t, int s) const { return v[t][s]; }
    template <int PITCH> __device__ __forceinline__ void read(const float *p) {
#pragma unroll
        for (int t = 0; t < T; t++) v[t] = *reinterpret_cast<const f32x4 *>(p + t * (32 * BK));
    }
};
template <> struct Frag<false, 1> {
    float v[4];
    __device__ __forceinline__ float at(int, int s) const { return v[s]; }
    template <int PITCH> __device__ __forceinline__ void read(const float *p) {
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = p[s * PITCH];
    }
};
template <> struct Frag<false, 2> {
    f32x2 v[4];
    __device__ __forceinline__ float at(int t, int s) const { return v[s][t]; }
    template <int PITCH> __device__ __forceinline__ void read(const float *p) {
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = *reinterpret_cast<const f32x2 *>(p + s * PITCH);
    }
};

template <int N> __device__ __forceinline__ void wait_loads_and_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

// A wavefront's VEC floats per lane from a buffer to LDS, in asm: of loads it knows the compiler waits for all before any LDS read that it
// cannot prove independent of them, which would undo the prefetch.  Waits are wait_loads_and_barrier's.  (m0 and an SGPR that a vector
// instruction wrote need one and five cycles before the load reads them.  The compiler warns of any clobber that names m0, which it
// reserves; named, it does not take a value of its own in m0 to last across the asm.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int VEC> __device__ __forceinline__ void load_to_lds(i32x4 rsrc, uint32_t off, uint32_t to) {
    if constexpr (VEC == 4) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(to) : "m0", "memory");
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(to) : "m0", "memory");
}
#pragma clang diagnostic pop

// Copies an operand's tiles to LDS: [WK][W][BK] (KC, pieces exchanged) or [WK][BK][W], VEC floats per lane and instruction.  The
// operand is addressed as a buffer that ends behind its last element.  A lane whose k lies past the end asks for an offset behind any
// buffer, and lanes of rows past the edge for zeros or for values that only reach sums nobody stores.
template <bool KC, int W, int WK, int WAVES, int VEC> struct Loader {
    static constexpr int PER = 64 * VEC, TILE = W * BK, COUNT = TILE * WK / PER / WAVES;
    static_assert(COUNT * PER * WAVES == TILE * WK, "whole instructions");
    uint32_t off[COUNT];  // byte offsets of this lane's pieces of the tile to load next
    uint32_t lo = 0, hi = 0, bytes = 0;  // the buffer: from the first tile that off counts from to the operand's end; empty where there is none (k = 0)
    // A tile that starts at p, floats before the operand's end, with k_left values of k.
    __device__ __forceinline__ void start(const float *p, uint64_t floats, uint32_t ld, uint32_t k_left, int wave, int lane) {
        const uint64_t at = (uint64_t)(uintptr_t)p;
        lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at);
        hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32) & 0xffff);
        bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)min(floats, (uint64_t)0x3fffffff) * 4u));
        asm volatile("s_nop 4" ::"s"(lo), "s"(hi), "s"(bytes));
#pragma unroll
        for (int u = 0; u < COUNT; u++) {
            const uint32_t f = ((u * WAVES + wave) * 64 + lane) * VEC, sub = f / TILE, q = f % TILE;
            uint32_t k, o;
            if (KC) {
                const uint32_t row = q / BK, piece = (q % BK) / 4;
                k = sub * BK + ((piece ^ ((row >> 2) & 3)) * 4) + (q & 3);
                o = row * ld + k;
            } else {
                k = sub * BK + q / W;
                o = k * ld + q % W;
            }
            off[u] = k < k_left ? o * 4 : 0xffffffffu;
        }
    }
    __device__ __forceinline__ void next(uint32_t step_bytes) {
#pragma unroll
        for (int u = 0; u < COUNT; u++) off[u] += step_bytes;
    }
    __device__ __forceinline__ void nothing() {
#pragma unroll
        for (int u = 0; u < COUNT; u++) off[u] = 0xffffffffu;
    }
    __device__ __forceinline__ void load(int u, uint32_t stage, int wave) {
        const i32x4 rsrc = {(int)lo, (int)hi, (int)bytes, 0x00020000};
        load_to_lds<VEC>(rsrc, off[u], stage + (u * WAVES + wave) * (PER * 4));
    }
};

template <class X> struct PlaneRoom { static constexpr int FLOATS = X::LDS_BYTES / 4; };
template <> struct PlaneRoom<void> { static constexpr int FLOATS = 0; };

template <bool AKC, bool BKC, int WM, int WN, int WK, int TA, int TB, int VEC, class X = void>
__global__ __launch_bounds__(64 * WM * WN * WK, std::is_void<X>::value ? 1 : 2) void gemm_f32_tiles(GemmArgs g) {
    constexpr bool PLANES = !std::is_void<X>::value;
    static_assert(!PLANES || (AKC && BKC), "weights in planes: the first operand's k is contiguous, and a lane's columns are 32 apart");
    // Stages, and with them how many blocks a CU holds (48 KB of LDS: three).  A fourth is 3 to 10 % slower for the small tiles, which lose
    // a block by it.  Of 128 x 128 tiles a CU holds two: three in step end together, and the blocks left then fill the slots of few CUs
    // (4096^3, four rounds: 1153 us with three, 938 with two; five rounds, [4096,1024] x [1024,5120]: 354 and 304).
    constexpr int S = TA == 2 ? 4 : 3;
    constexpr int WAVES = WM * WN * WK, THREADS = 64 * WAVES, BM = 32 * WM * TA, BN = 32 * WN * TB, BKT = BK * WK;
    constexpr int STAGE_A = BM * BKT, STAGE = (BM + BN) * BKT;
    constexpr int CP = BN + 4, PASS_ROWS = 32 * WM, SUMS = WK * PASS_ROWS * CP;  // the epilogue's [WK][PASS_ROWS][CP]
    constexpr int ROOM = PLANES ? PlaneRoom<X>::FLOATS : S * STAGE;
    __shared__ __align__(16) float lds[ROOM > SUMS ? ROOM : SUMS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (WK == 4 && g.apart) __builtin_amdgcn_s_setprio(3);
    const int wk = wave / (WM * WN), wmn = wave % (WM * WN), wm = wmn / WN, wn = wmn % WN;
    const int lr = lane & 31, lk = lane >> 5;

    // block id -> (slice, tile): an XCD gets a run of consecutive tiles, the cut ones behind the whole ones, a tile's slices next to each other
    const uint32_t xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const bool cut = local >= g.full;
    const uint32_t cut_tile = cut ? (local - g.full) / g.slices : 0, slice = cut ? local - g.full - cut_tile * g.slices : 0;
    const uint32_t in_run = cut ? g.full + cut_tile : local;
    const uint32_t tile = xcd * g.chunk + in_run;
    if (in_run >= g.chunk || tile >= g.tiles) return;
    const uint32_t per_batch = g.tiles_m * g.tiles_n, z = tile / per_batch, t = tile - z * per_batch;
    const uint32_t per_group = g.tiles_m * g.group_n, grp = t / per_group, r = t - grp * per_group;
    const uint32_t width = min(g.group_n, g.tiles_n - grp * g.group_n);
    const uint32_t m0 = (r / width) * BM, n0 = (grp * g.group_n + r % width) * BN;
    const uint32_t zo = z / g.batch_inner, zi = z - zo * g.batch_inner;
    const uint32_t k0 = slice * g.slice_k, k = cut ? min(g.slice_k, g.k - k0) : g.k;
    const float *a = g.a + (size_t)zo * g.a_bs + (size_t)zi * g.a_bs2 + (AKC ? (size_t)m0 * g.lda + k0 : (size_t)k0 * g.lda + m0);
    const float *b = g.b + (size_t)zo * g.b_bs + (size_t)zi * g.b_bs2 + ((PLANES ? g.b_kc != 0 : BKC) ? (size_t)n0 * g.ldb + k0 : (size_t)k0 * g.ldb + n0);

    floatx16 acc[TA][TB];
    if constexpr (PLANES) {
        X x;
        x.start(a, g.lda, min(g.m - m0, (uint32_t)BM), k, g.planes + ((uint64_t)(n0 / 32) * g.k16s + k0 / BK) * planes::SET, g.n32s - n0 / 32, g.k16s,
                g.k16s - k0 / BK, lds, tid, wm, wn, wk);
        x.run(acc);
        // Where a sum is not finite an operand may have been infinite (inf - inf in the planes), or beyond 2^103, or the sum beyond 2^79: the
        // wavefront's sums over its values of k once more on the fp32 matrix cores, which have fp32 arithmetic's result for every value.
        // [1024,768] x [768,768] takes 13 us, 22 with one row infinite and 24 with a NaN in every row, [1024,3072] x [3072,768] 40, 72 and 73,
        // [6304,768] x [768,3072] 165, 225 and 446 (one value of k at a time: 60 and 70, 224 and 264, 336 and 910; the fp32 kernel 15, 42, 222).
        bool lost = false;
#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int j = 0; j < TB; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) lost |= !(__builtin_fabsf(acc[i][j][e]) < __builtin_inff());
        if (__builtin_expect(__any(lost), 0)) {
#pragma unroll
            for (int i = 0; i < TA; i++)
#pragma unroll
                for (int j = 0; j < TB; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
            // A set's values all on their way at once, those of the next set beside its products.
            const float *pa[TA], *pb[TB];
            const size_t b_step = g.b_kc ? 1 : g.ldb;
#pragma unroll
            for (int i = 0; i < TA; i++) pa[i] = a + (size_t)min(wm * (32 * TA) + lr + 32 * i, g.m - m0 - 1) * g.lda;
#pragma unroll
            for (int j = 0; j < TB; j++) pb[j] = b + (size_t)min(wn * (32 * TB) + lr + 32 * j, g.n - n0 - 1) * (g.b_kc ? g.ldb : 1);
            float va[2][8][TA], vb[2][8][TB];
            auto fetch = [&](auto to, uint32_t set) __attribute__((always_inline)) {
#pragma unroll
                for (uint32_t s = 0; s < 8; s += VEC) {  // VEC values of k lie side by side, all in front of its end or none
                    const uint32_t kk = planes::k_of(set, lk, s), at = min(kk, k - VEC);
#pragma unroll
                    for (int i = 0; i < TA; i++) {
                        float row[VEC];
                        __builtin_memcpy(row, __builtin_assume_aligned(pa[i] + at, VEC * sizeof(float)), sizeof(row));
#pragma unroll
                        for (uint32_t e = 0; e < VEC; e++) va[to][s + e][i] = kk < k ? row[e] : 0.0f;
                    }
#pragma unroll
                    for (uint32_t e = 0; e < VEC; e++)
#pragma unroll
                        for (int j = 0; j < TB; j++) vb[to][s + e][j] = kk < k ? pb[j][(at + e) * b_step] : 0.0f;
                }
            };
            auto multiply = [&](auto of) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int i = 0; i < TA; i++)
#pragma unroll
                        for (int j = 0; j < TB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[of][s][i], vb[of][s][j], acc[i][j], 0, 0, 0);
            };
            constexpr std::integral_constant<int, 0> even = {};
            constexpr std::integral_constant<int, 1> odd = {};
            fetch(even, wk);
#pragma unroll 1
            for (uint32_t set = wk; set / 4 * 64 < k; set += 2 * WK) {
                fetch(odd, set + WK);
                multiply(even);
                fetch(even, set + 2 * WK);
                multiply(odd);  // behind the end of k: zeros
            }
        } else {
#pragma unroll
            for (int i = 0; i < TA; i++)
#pragma unroll
                for (int j = 0; j < TB; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][j][e] *= planes::UNSCALE;
        }
    } else {
        Loader<AKC, BM, WK, WAVES, VEC> la;
        Loader<BKC, BN, WK, WAVES, VEC> lb;
        const uint64_t a_floats = k == 0 ? 0 : AKC ? (uint64_t)(min(g.m - m0, (uint32_t)BM) - 1) * g.lda + k : (uint64_t)(k - 1) * g.lda + (g.m - m0);
        const uint64_t b_floats = k == 0 ? 0 : BKC ? (uint64_t)(min(g.n - n0, (uint32_t)BN) - 1) * g.ldb + k : (uint64_t)(k - 1) * g.ldb + (g.n - n0);
        const uint64_t a_step = AKC ? (uint64_t)BKT : (uint64_t)BKT * g.lda, b_step = BKC ? (uint64_t)BKT : (uint64_t)BKT * g.ldb;
        constexpr int LOADS = decltype(la)::COUNT + decltype(lb)::COUNT;

#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int j = 0; j < TB; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

        // Where a tile and the one behind it are whole, and 32 bits reach, its addresses are the last tile's and a step (near: up to which
        // tile).  Per step that is an addition per load; a base, an end and a mask worked out anew each time held the products up by
        // 300 cycles a step (64 x 64 tiles: 18.8 ns a value of k for a CU's only block, 13.6 now).
        const uint32_t nk = (k + BKT - 1) / BKT, whole = k / BKT;
        uint32_t tile_k = 0, near = 0;
        auto advance_near = [&]() __attribute__((always_inline)) {
            la.next((uint32_t)a_step * 4);
            lb.next((uint32_t)b_step * 4);
            tile_k++;
        };
        auto advance_far = [&] __attribute__((always_inline)) {
            la.start(a + tile_k * a_step, a_floats - tile_k * a_step, g.lda, k - tile_k * BKT, wave, lane);
            lb.start(b + tile_k * b_step, b_floats - tile_k * b_step, g.ldb, k - tile_k * BKT, wave, lane);
            near = min(whole, tile_k + 1 + min(g.window, 0x7fffffffu - tile_k));
            tile_k++;
        };
        auto nothing_left = [&] __attribute__((always_inline)) {
            la.nothing();
            lb.nothing();
        };
        const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
        auto load = [&](auto u, uint32_t stage) __attribute__((always_inline)) {
            if constexpr (u < la.COUNT) la.load(u, lds0 + stage * (STAGE * 4), wave);
            else lb.load(u - la.COUNT, lds0 + (stage * STAGE + STAGE_A) * 4, wave);
        };
        // Behind the last tile 16-byte loads go on, for nothing: the waits and the steps stay as they are ([1872,3024] x [3024,2256] 202 us,
        // 209 without those loads).  Single-value loads are four times as many, and end (96 of [148,32] x [32,2821], one step each: 98 us
        // with the others', 77 without).
        constexpr bool TO_THE_END = VEC == 4;
#pragma unroll
        for (int s = 0; s < S; s++) {
            if (!TO_THE_END && tile_k >= nk) break;
            if (tile_k < near) advance_near();
            else if (tile_k < nk) advance_far();
            else nothing_left();
            each<LOADS>([&](auto u) __attribute__((always_inline)) { load(u, s); });
        }

        // This lane's fragments in stage 0, of either half of a step.
        const float *pa[2], *pb[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (AKC) {
                const int row = wm * (32 * TA) + lr;
                pa[h] = lds + (wk * BM + row) * BK + (((2 * h + lk) ^ ((row >> 2) & 3)) << 2);
            } else {
                pa[h] = lds + (wk * BK + 8 * h + 4 * lk) * BM + wm * (32 * TA) + TA * lr;
            }
            if (BKC) {
                const int row = wn * (32 * TB) + lr;
                pb[h] = lds + STAGE_A + (wk * BN + row) * BK + (((2 * h + lk) ^ ((row >> 2) & 3)) << 2);
            } else {
                pb[h] = lds + STAGE_A + (wk * BK + 8 * h + 4 * lk) * BN + wn * (32 * TB) + TB * lr;
            }
        }

        // Half a step's products while the next half's fragments are on their way.
        Frag<AKC, TA> fa[2];
        Frag<BKC, TB> fb[2];
        auto read = [&](int h, uint32_t stage) __attribute__((always_inline)) {
            fa[h].template read<BM>(pa[h] + stage * STAGE);
            fb[h].template read<BN>(pb[h] + stage * STAGE);
        };
        constexpr int Q = 4 * TA * TB;
        auto multiply = [&](int h, int q) __attribute__((always_inline)) {
            const int s = q / (TA * TB), i = q / TB % TA, j = q % TB;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[h].at(i, s), fb[h].at(j, s), acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (WK == 4 && g.apart) {
            const uint32_t turn = (blockIdx.x >> 8) % 3;
            if (turn == 0) __builtin_amdgcn_s_setprio(0);
            else if (turn == 1) __builtin_amdgcn_s_setprio(1);
            else __builtin_amdgcn_s_setprio(2);
        }
        // Waits until at most `behind` stages, whose loads are the last ones, are on their way.
        auto wait_behind = [&](uint32_t behind) __attribute__((always_inline)) {
            if (behind >= S - 1) wait_loads_and_barrier<(S - 1) * LOADS>();
            else if (S > 3 && behind == 2) wait_loads_and_barrier<2 * LOADS>();
            else if (behind == 1) wait_loads_and_barrier<LOADS>();
            else wait_loads_and_barrier<0>();
        };
        if (TO_THE_END) wait_loads_and_barrier<(S - 1) * LOADS>();
        else wait_behind(max(nk, 1u) - 1);
        read(0, 0);
        uint32_t cur = 0;
        // left: 0, or where the loads have ended how many steps there are from this one on.
        auto step = [&](auto is_near, uint32_t left) __attribute__((always_inline)) {
            each<Q>([&](auto q) __attribute__((always_inline)) {
                multiply(0, q);
                if constexpr (q == 0) read(1, cur);
                if constexpr (q == 1 && is_near) advance_near();
                __builtin_amdgcn_sched_barrier(0);
            });
            const uint32_t next = cur + 1 == S ? 0 : cur + 1;
            each<Q>([&](auto q) __attribute__((always_inline)) {
                constexpr int R = Q > 4 ? 1 : 0;
                multiply(1, q);
                if constexpr (q == 0) {  // this stage is read, the next one there
                    if (left) wait_behind(max(left, 2u) - 2);
                    else wait_loads_and_barrier<(S - 2) * LOADS>();
                }
                if constexpr (q == R) read(0, next);
                if (!left)
                    each<LOADS>([&](auto u) __attribute__((always_inline)) {
                        if constexpr (R + 1 + u * (Q - 1 - R) / LOADS == q) load(u, cur);
                    });
                __builtin_amdgcn_sched_barrier(0);
            });
            cur = next;
        };
        while (tile_k < nk) {
            if (tile_k >= near) {
                advance_far();
                step(std::false_type(), 0);
            }
            while (tile_k < near) step(std::true_type(), 0);
        }
        if (TO_THE_END) nothing_left();
        for (uint32_t left = min(nk, (uint32_t)S); left > 0; left--) step(std::false_type(), TO_THE_END ? 0 : left);
        wait_loads_and_barrier<0>();

    }
    if (WK == 4 && g.apart) __builtin_amdgcn_s_setprio(3);
    // Epilogue, TA passes of PASS_ROWS rows: accumulator e of lane l is row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32 of its
    // tile; through LDS the WK sums of an element meet and rows of C are stored 16 bytes per lane.
    const size_t c_at = (size_t)zo * g.c_bs + (size_t)zi * g.c_bs2;
    float *c = g.c + c_at;
    const float *residual = g.residual ? g.residual + c_at : nullptr;
    constexpr int PIECES = PASS_ROWS * BN / 4 / THREADS;  // per thread and pass
    static_assert(PIECES * THREADS * 4 == PASS_ROWS * BN, "whole pieces");
    // A thread's pieces lie in the same columns: a bias row is read once.
    static_assert(THREADS % (BN / 4) == 0, "a thread keeps its columns");
    const uint32_t col = n0 + tid % (BN / 4) * 4, w = col < g.n ? min(g.n - col, 4u) : 0;
    const bool bias = g.c0 && g.c0_rs == 0;
    f32x4 bias4 = {0.0f, 0.0f, 0.0f, 0.0f};
    if (bias) {
#pragma unroll
        for (uint32_t e = 0; e < 4; e++)
            if (e < w) bias4[e] = g.beta * g.c0[(size_t)(col + e) * g.c0_cs];
    }
    auto finish = [&](f32x4 v, int pass, int u) {
        const int pr = (u * THREADS + tid) / (BN / 4);
        const uint32_t row = m0 + (pr >> 5) * (32 * TA) + (AKC ? 32 * pass + (pr & 31) : TA * (pr & 31) + pass);
        if (row >= g.m || w == 0) return;
        const size_t at = (size_t)row * g.ldc + col;
        v = g.alpha * v;
        if (bias) v += bias4;
        if (w == 4) {
            if (g.c0 && !bias) {
                const float *q = g.c0 + (size_t)row * g.c0_rs + (size_t)col * g.c0_cs;
                const f32x4 x = {q[0], q[g.c0_cs], q[2 * (size_t)g.c0_cs], q[3 * (size_t)g.c0_cs]};
                v += g.beta * x;
            }
            if (g.act) {  // one look at act for the four
                auto each4 = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = f(v[e]);
                };
                if (g.act == AHIP_GELU) each4([](float x) { return dev::gelu_elem(x); });
                else if (g.act == AHIP_RELU) each4([](float x) { return dev::relu_elem(x); });
                else each4([&](float x) {
                    const float s = dev::hard_sigmoid_elem(x, g.act_alpha, g.act_beta);
                    return g.act == ACT_HARD_SWISH ? s * x : s;
                });
            }
            if (residual) v += *reinterpret_cast<const dev::v4f_dword *>(residual + at);
            *reinterpret_cast<dev::v4f_dword *>(c + at) = v;
        } else {
            for (uint32_t e = 0; e < w; e++) {
                float x = e == 0 ? v.x : e == 1 ? v.y : v.z;
                if (g.c0 && !bias) x += g.beta * g.c0[(size_t)row * g.c0_rs + (size_t)(col + e) * g.c0_cs];
                x = dev::activation(x, g.act, g.act_alpha, g.act_beta);
                if (residual) x += residual[at + e];
                c[at + e] = x;
            }
        }
    };
    const uint32_t idx = xcd * (g.chunk - g.full) + cut_tile;
    f32x4 *parts = reinterpret_cast<f32x4 *>(g.partials) + (size_t)idx * g.slices * (BM * BN / 4) + tid;
#pragma unroll
    for (int i = 0; i < TA; i++) {
        float *ct = lds + (size_t)wk * (PASS_ROWS * CP);
        if (i) __syncthreads();
#pragma unroll
        for (int e = 0; e < 16; e++)
#pragma unroll
            for (int j = 0; j < TB; j++)
                ct[(wm * 32 + 8 * (e >> 2) + 4 * lk + (e & 3)) * CP + wn * (32 * TB) + (BKC ? 32 * j + lr : TB * lr + j)] = acc[i][j][e];
        __syncthreads();
        auto sum_at = [&](int u) {
            const int f = u * THREADS + tid;
            const float *s = lds + f / (BN / 4) * CP + f % (BN / 4) * 4;
            f32x4 v = *reinterpret_cast<const f32x4 *>(s);
#pragma unroll
            for (int w = 1; w < WK; w++) v += *reinterpret_cast<const f32x4 *>(s + w * (PASS_ROWS * CP));
            return v;
        };
        if (cut) {
#pragma unroll
            for (int u = 0; u < PIECES; u++) store_shared(parts + (size_t)slice * (BM * BN / 4) + (i * PIECES + u) * THREADS, sum_at(u));
        } else if (g.act) {  // one copy of the activation's code: unrolled, it slowed every launch down
#pragma unroll 1
            for (int u = 0; u < PIECES; u++) finish(sum_at(u), i, u);
        } else {
#pragma unroll
            for (int u = 0; u < PIECES; u++) finish(sum_at(u), i, u);
        }
    }
    if (!cut) return;

    // A tile cut along k: the block that arrives last adds the slices' sums up in slice order, so the result does not depend on who
    // was last.  The sums pass by the L2s (agent-scope accesses), so it does not matter on which XCD a slice ran; vmcnt(0) says
    // that this block's are where the others look.
    __shared__ int arrived;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid == 0) arrived = atomicAdd(&g.counters[idx], 1);
    __syncthreads();
    if (arrived != (int)g.slices - 1) return;
    if (tid == 0) atomicExch(&g.counters[idx], 0);  // ready for the next launch
#pragma unroll 1
    for (int p = 0; p < TA * PIECES; p++) {
        f32x4 v = load_shared(parts + p * THREADS);
        for (uint32_t q = 1; q < g.slices; q++) v += load_shared(parts + (size_t)q * (BM * BN / 4) + p * THREADS);
        finish(v, p / PIECES, p % PIECES);
    }
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The block tiles, and what a launch of them takes: launch_us + rounds * (block_us + k_us * k / 768), rounds being the blocks that
// the busiest CU runs (dealt to the XCDs in turn), times `lone` where that is one: a CU's only block has nothing to fill its gaps
// with.  The tiles of a last round that is partly empty may be cut along k, so that it takes a part of a round: 0.8 us more, slice_us for
// each slice and the partial sums at 2.5 TB/s ([3152,3072] x [3072,768] 137 -> 116 us, [1536,1536] x [1536,1536] 65 -> 56,
// [2500,1000] x [1000,2000] 100 -> 79, against every tile cut alike or none; [197 and 77,3072] x [3072,768] in three slices, which only
// powers of two did not allow, 16.9 -> 16.0 and 11.7 -> 10.1; on nine sizes the choice is 0 to 4 % behind the best tile and cut).  Fitted to 120 products of 1e8 to
// 2e11 multiplications with every tile and 70 of up to 1500 tiles of 32 x 32 with every tile and cut (6, 4, 4 and 4 % rms); the choice
// is 0.4 % behind the best one on average.  Per value of C a small tile costs more (each of its operands serves fewer products), but its
// rounds come in smaller units.  A k_us of 10.24 per 64 x 64 would be the matrix cores' peak.
struct Shape {
    uint32_t bm, bn, step, threads;  // step: values of k that a cut counts in
    double launch_us, block_us, k_us, lone, slice_us;
};
constexpr Shape SHAPES[] = {{32, 32, 64, 256, 2.97, 0.72, 3.18, 1.02, 0.27},
                            {64, 64, 32, 256, 2.82, 1.06, 11.11, 1.04, 0.83},
                            {128, 64, 16, 256, 2.81, 1.38, 21.95, 1.04, 1.61},
                            {128, 128, 16, 256, 2.07, 3.63, 42.81, 1.02, 3.21}};
constexpr int N_SHAPES = 4;
// The same with a weight matrix's planes for the second operand: 64 x 64, 64 x 128 and 128 x 128 with eight wavefronts, of which a CU holds
// one block, and 128 x 128 with four, of which it holds two.  Fitted to 96 products of 256 to 12608 rows and 192 to 3072 values of k with
// every tile, and 898 of them with the last round cut (7 and 6 % rms); the choice is 0.8 % behind the best one on average.
constexpr Shape PLANE_SHAPES[] = {{64, 64, 64, 512, 1.18, 4.18, 7.38, 0.92, 0.59},
                                  {64, 128, 64, 512, 1.0, 6.32, 12.38, 0.89, 0.85},
                                  {128, 128, 64, 512, 1.0, 7.07, 24.52, 0.86, 1.5},
                                  {128, 128, 64, 256, 1.0, 4.14, 26.38, 1.3, 2.9}};
constexpr int N_PLANE_SHAPES = 4;

struct Choice {
    int shape = 0;
    uint32_t full = 0, slices = 1, slice_k = 0;  // full: whole tiles of an XCD's run where others are cut
    double us = 0.0;
};

// What a product adds up in which order is decided by the sizes alone, and by where a value lies in C: the values of a last round's
// tiles add up in slices, the others in one piece, so that equal rows of A need not give equal bits.  A product and the same product with
// an operand stored the other way round add up alike.  cut: k may be cut into slices.
// planes: of the tiles for weights as planes.
Choice choose(size_t batch, size_t m, size_t n, size_t k, size_t cus_per_xcd, bool cut, bool planes = false) {
    Choice best;
    const Shape *shapes = planes ? PLANE_SHAPES : SHAPES;
    const int n_shapes = planes ? N_PLANE_SHAPES : N_SHAPES;
    if (planes) k = (k + 63) / 64 * 64;
    for (int s = 0; s < n_shapes; s++) {
        const Shape &sh = shapes[s];
        const size_t chunk = (((m + sh.bm - 1) / sh.bm) * ((n + sh.bn - 1) / sh.bn) * batch + 7) / 8;
        const size_t rem = chunk % cus_per_xcd, whole = chunk / cus_per_xcd;  // tiles of a last round that is partly empty; rounds before it
        auto round_us = [&](size_t values) { return sh.block_us + sh.k_us * (double)std::max<size_t>(values, sh.step) / 768.0; };
        for (uint32_t want = 1; want <= 8; want++) {
            if (want > 1 && (!cut || batch != 1 || k < 128 * (size_t)want || rem == 0 || rem * 8 > GEMM_COUNTERS)) break;
            const size_t slice_k = ((k + want - 1) / want + sh.step - 1) / sh.step * sh.step, slices = slice_k ? (k + slice_k - 1) / slice_k : 1;
            if (want > 1 && slices != want) continue;
            // A grid ends at 2^32 threads: a few rows with 2^29 columns are more blocks of 32 x 32 than that.
            if ((s < n_shapes - 1 || want > 1) && (chunk + rem * (want - 1)) * 8 * sh.threads > 0xffffffffu) break;
            const size_t last = want == 1 ? rem != 0 : (rem * want + cus_per_xcd - 1) / cus_per_xcd;
            double us = sh.launch_us + ((double)whole * round_us(k) + (double)last * round_us(want == 1 ? k : slice_k)) * (whole + last == 1 ? sh.lone : 1.0);
            if (want > 1) us += 0.8 + want * (sh.slice_us + (double)(rem * 8) * sh.bm * sh.bn * sizeof(float) / 2.5e6);
            if (best.us == 0.0 || us < best.us) best = {s, (uint32_t)(whole * cus_per_xcd), want, (uint32_t)slice_k, us};
        }
    }
    return best;
}

// A product's grid: of each XCD's run of tiles those that are whole, and the slices of the others.
struct Grid {
    size_t gx = 0, gy = 0, tiles = 0, chunk = 0, full = 0, blocks = 0, threads = 256;
    Grid(const Choice &ch, size_t batch, size_t m, size_t n, bool planes = false) {
        const Shape &sh = planes ? PLANE_SHAPES[ch.shape] : SHAPES[ch.shape];
        threads = sh.threads;
        gy = (m + sh.bm - 1) / sh.bm, gx = (n + sh.bn - 1) / sh.bn, tiles = gx * gy * batch, chunk = (tiles + 7) / 8;
        full = ch.slices > 1 ? ch.full : chunk;
        blocks = (full + (chunk - full) * ch.slices) * 8;
    }
    bool fits(size_t batch) const {
        const size_t lim = (size_t)1 << 31;
        return gx * gy < lim && batch < lim && tiles < ((size_t)1 << 32) && blocks * threads <= 0xffffffffu;
    }
};

template <bool AKC, bool BKC> void launch_tiles(const DeviceCtx &ctx, const GemmArgs &g, int shape, bool vec) {
    const dim3 grid((g.full + (g.chunk - g.full) * g.slices) * 8), block(256);
#define TILES(...)                                                                                                                      \
    do {                                                                                                                                \
        if (vec) hipLaunchKernelGGL((gemm_f32_tiles<AKC, BKC, __VA_ARGS__, 4>), grid, block, 0, ctx.stream, g);                         \
        else hipLaunchKernelGGL((gemm_f32_tiles<AKC, BKC, __VA_ARGS__, 1>), grid, block, 0, ctx.stream, g);                             \
    } while (0)
    switch (shape) {
    case 0: TILES(1, 1, 4, 1, 1); break;
    case 1: TILES(2, 1, 2, 1, 2); break;
    case 2: TILES(4, 1, 1, 1, 2); break;
    default: TILES(2, 2, 1, 2, 2); break;
    }
#undef TILES
}

void launch_plane_tiles(const DeviceCtx &ctx, const GemmArgs &g, int shape, bool vec) {
    const dim3 grid((g.full + (g.chunk - g.full) * g.slices) * 8), block(PLANE_SHAPES[shape].threads);
#define TILES(WM, WN, WK, TA, TB, NA)                                                                                               \
    do {                                                                                                                            \
        if (vec) hipLaunchKernelGGL((gemm_f32_tiles<true, true, WM, WN, WK, TA, TB, 4, planes::Tile<WM, WN, WK, TA, TB, 4, NA>>),   \
                                    grid, block, 0, ctx.stream, g);                                                                 \
        else hipLaunchKernelGGL((gemm_f32_tiles<true, true, WM, WN, WK, TA, TB, 1, planes::Tile<WM, WN, WK, TA, TB, 1, NA>>),       \
                                grid, block, 0, ctx.stream, g);                                                                     \
    } while (0)
    switch (shape) {
    case 0: TILES(1, 2, 4, 2, 1, 2); break;
    case 1: TILES(1, 2, 4, 2, 2, 1); break;
    case 2: TILES(2, 2, 2, 2, 2, 1); break;
    default: TILES(2, 2, 1, 2, 2, 1); break;
    }
#undef TILES
}

// A weight matrix as planes: a wavefront per set, eight values a lane.  Element (k, n) is b[k * s_k + n * s_n].
__global__ __launch_bounds__(256) void pack_planes(const float *__restrict__ b, u32x4 *__restrict__ out, uint32_t n, uint32_t k, size_t s_k, size_t s_n,
                                                   uint32_t n32s, uint32_t k16s) {
    const uint64_t set = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (set >= (uint64_t)n32s * k16s) return;
    const uint32_t lane = threadIdx.x & 63, col = (uint32_t)(set / k16s) * 32 + (lane & 31), j = (uint32_t)(set % k16s);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const uint32_t kk = planes::k_of(j, lane >> 5, e);
        v[e] = col < n && kk < k ? b[(size_t)kk * s_k + (size_t)col * s_n] : 0.0f;
    }
    planes::Split4 s[2];
    each<8>([&](auto p) {
        s[0].part<p>(f32x4{v[0], v[1], v[2], v[3]});
        s[1].part<p>(f32x4{v[4], v[5], v[6], v[7]});
    });
    each<3>([&](auto p) { out[set * (planes::SET / 16) + p * 64 + lane] = __builtin_shufflevector(s[0].q<p>(), s[1].q<p>(), 0, 1, 2, 3); });
}

constexpr size_t TILE_SPAN = (size_t)1 << 30;  // floats from a tile's first element to its last: byte offsets are 32 bits

}  // namespace

namespace {
size_t weight_k16s(size_t k) { return (k + 63) / 64 * 4; }
// A tile's rows of the first operand lie within 31-bit byte offsets, and a set's within 32 bits of its column's first.
bool planes_reach(size_t lda, size_t k) { return k > 0 && k <= ((size_t)1 << 20) && 127 * lda + k < ((size_t)1 << 29); }
}

// Planes where they are reckoned 5 % faster, about what the estimates are off by, and where weights that come from HBM leave a gain: from a
// few hundred rows on, with the same weights again and again ([1024,768] x [768,768 / 3072] 13.7 -> 12.0 us, 39.8 -> 32.5, [1024,3072] x
// [3072,768] 42.3 -> 36.4; [6304,768] x [768,768 / 2304 / 3072] 62 -> 51, 171 -> 128, 225 -> 166, [6304,3072] x [3072,768] 223 -> 158;
// [12608,768] x [768,3072] 450 -> 315).  With fewer, a block's start and end and the 6 bytes a weight takes instead of 4 outweigh the products
// ([256,768] x [768,768] 6.8 and 10.1, [512,384] x [384,384] 5.4 and 8.0).
// A graph's weights are other ones in each product, and a block's few wavefronts wait for them longer than the estimates, fitted to one
// product alone, say.  In chains of 24 to 40 products planes took that much longer against the fp32 kernel than reckoned: -1.8 to 1.9 us for
// 1 to 6 MB of them, -1.4 to 8.5 for 10.6 and -0.3 to 12.1 for 14, the most where k is long and the columns are few ([1576,3072] x [3072,768]:
// 18.4 us reckoned, 6.2 gained); for 38 to 232 MB either kernel takes up to 50 us longer.  The estimates do not have that, so the line keeps a
// distance instead, by the weights' size: without it [256,768] x [768,3072] lost 1.3 us of 15, [512,3072] x [3072,768] 1.7 of 25 and
// [788,1536] x [1536,384] 1.1 of 15.  Of those 66 sizes none that is taken loses, and those left out would gain 1.9 us at most; of 216 more that
// are taken, with weights from HBM (128 to 2048 rows, k of 1024 to 16384, 256 to 1536 columns; 1000 to 16448 rows, k of 64 to 1024), one loses:
// [300,4096] x [4096,1024], 0.4 us of 31.
// A view that is not one tall matrix is copied first, a Transpose behind that the fp32 kernel writes ahead of copies the result; against that the
// fp32 kernel's tiles end with each matrix.  Copies of results take 2 us and 6 TB/s (58 products of 512 to 6304 rows and 192 to 3072 values of k
// with Transpose(1,0,2) behind: none that is taken loses, those left out would gain 2 % at most), of operands that Transpose(0,2,1) turns 5 us
// and 1.4 TB/s ([64,196,512] turned x [196,256] 36 us in place, 65 by planes; [16,1024,768] x [1024,256 / 2048] 54 and 107, 386 and 332).
bool gemm_takes_planes(const DeviceCtx &ctx, size_t m, size_t n, size_t k, size_t matrices, bool operand, bool result) {
    if (gemm_takes_split(ctx, m, n, k) || m < 64 || n < 64 || k < 64 || !planes_reach(k, k) || m >= ((size_t)1 << 31) || n >= ((size_t)1 << 31)) return false;
    const size_t cus = ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd : 32, parts = operand || result ? std::max<size_t>(matrices, 1) : 1;
    const Choice ch = choose(1, m, n, k, cus, ctx.gemm_split_k, true);
    const double us = choose(parts, m / parts, n, k, cus, ctx.gemm_split_k).us, from_hbm = std::min(1.5e-6 * (double)n * (double)k, 3.6);
    const double copies = (operand ? 5.0 + 8.0 * (double)m * (double)k / 1.4e6 : 0.0) + (result ? 2.0 + 8.0 * (double)m * (double)n / 6e6 : 0.0);
    return ch.us + copies + std::max(0.05 * us, from_hbm) < us && Grid(ch, 1, m, n, true).fits(1);
}

size_t gemm_weight_planes_bytes(size_t n, size_t k) { return (n + 31) / 32 * weight_k16s(k) * planes::SET; }

int gemm_pack_weights(DeviceCtx &ctx, void *planes, const float *b, size_t n, size_t k, size_t ld, bool k_contig) {
    const size_t n32s = (n + 31) / 32, k16s = weight_k16s(k);
    hipLaunchKernelGGL(pack_planes, dim3((unsigned)((n32s * k16s + 3) / 4)), dim3(256), 0, ctx.stream, b, static_cast<u32x4 *>(planes), (uint32_t)n,
                       (uint32_t)k, k_contig ? (size_t)1 : ld, k_contig ? ld : (size_t)1, (uint32_t)n32s, (uint32_t)k16s);
    return ctx.check(hipGetLastError(), "pack_planes launch");
}

bool gemm_takes_split(const DeviceCtx &ctx, size_t m, size_t n, size_t k) {
    return k > 0 && (ctx.gemm_algorithm == AHIP_GEMM_BF16X3 || (ctx.gemm_algorithm == AHIP_GEMM_AUTO && gemm_split_worthwhile(m, n, k)));
}

int launch_gemm(DeviceCtx &ctx, float *c, const float *a, const float *b, const float *c0, size_t batch, size_t m, size_t n,
                size_t k, int trans_a, int trans_b, size_t lda, size_t ldb, size_t ldc, size_t a_batch_stride,
                size_t b_batch_stride, size_t c_batch_stride, size_t c0_row_stride, size_t c0_col_stride, float alpha,
                float beta, const void *planes) {
    const size_t a_bs[2] = {a_batch_stride, 0}, b_bs[2] = {b_batch_stride, 0}, c_bs[2] = {c_batch_stride, 0};
    return launch_gemm_batch2(ctx, c, a, b, c0, batch, 1, m, n, k, trans_a, trans_b, lda, ldb, ldc, a_bs, b_bs, c_bs, c0_row_stride,
                              c0_col_stride, alpha, beta, nullptr, planes);
}

// The product in parts of at most `part` values of m (axis 0), n (1) or k (2; the parts' sums meet in C).
static int launch_gemm_far_rows(DeviceCtx &ctx, int axis, size_t part, float *c, const float *a, const float *b, const float *c0, size_t batch_outer,
                                size_t batch_inner, size_t m, size_t n, size_t k, int trans_a, int trans_b, size_t lda, size_t ldb, size_t ldc,
                                const size_t a_bs[2], const size_t b_bs[2], const size_t c_bs[2], size_t c0_rs, size_t c0_cs, float alpha, float beta,
                                const GemmPost *post) {
    const size_t none[2] = {0, 0};
    if (axis == 2 && batch_outer * batch_inner > 1) {  // C0 of the second part on is C, which has batches of its own
        for (size_t z = 0; z < batch_outer * batch_inner; z++) {
            const size_t zo = z / batch_inner, zi = z % batch_inner;
            GemmPost p;
            if (post) p = *post;
            if (p.residual) p.residual += zo * c_bs[0] + zi * c_bs[1];
            const int rc = launch_gemm_far_rows(ctx, axis, part, c + zo * c_bs[0] + zi * c_bs[1], a + zo * a_bs[0] + zi * a_bs[1],
                                                b + zo * b_bs[0] + zi * b_bs[1], c0, 1, 1, m, n, k, trans_a, trans_b, lda, ldb, ldc, none, none, none,
                                                c0_rs, c0_cs, alpha, beta, post ? &p : nullptr);
            if (rc) return rc;
        }
        return AHIP_OK;
    }
    const size_t extent = axis == 0 ? m : axis == 1 ? n : k;
    for (size_t i = 0; i < extent; i += part) {
        const size_t w = std::min(part, extent - i);
        int rc;
        if (axis == 2) {
            const bool last = i + w == extent;
            rc = launch_gemm_f32(ctx, c, a + (trans_a ? i * lda : i), b + (trans_b ? i : i * ldb), i ? c : c0, 1, 1, m, n, w, trans_a, trans_b, lda, ldb,
                                 ldc, none, none, none, i ? ldc : c0_rs, i ? 1 : c0_cs, alpha, i ? 1.0f : beta, last ? post : nullptr);
        } else {
            const size_t r = axis == 0 ? i : 0, q = axis == 1 ? i : 0;
            GemmPost p;
            if (post) p = *post;
            if (p.residual) p.residual += r * ldc + q;
            rc = launch_gemm_f32(ctx, c + r * ldc + q, a + (trans_a ? r : r * lda), b + (trans_b ? q * ldb : q), c0 ? c0 + r * c0_rs + q * c0_cs : nullptr,
                                 batch_outer, batch_inner, axis == 0 ? w : m, axis == 1 ? w : n, k, trans_a, trans_b, lda, ldb, ldc, a_bs, b_bs, c_bs,
                                 c0_rs, c0_cs, alpha, beta, post ? &p : nullptr);
        }
        if (rc) return rc;
    }
    return AHIP_OK;
}

int launch_gemm_batch2(DeviceCtx &ctx, float *c, const float *a, const float *b, const float *c0, size_t batch_outer,
                       size_t batch_inner, size_t m, size_t n, size_t k, int trans_a, int trans_b, size_t lda, size_t ldb, size_t ldc,
                       const size_t a_batch_strides[2], const size_t b_batch_strides[2], const size_t c_batch_strides[2],
                       size_t c0_row_stride, size_t c0_col_stride, float alpha, float beta, const GemmPost *post, const void *planes) {
    const bool has_post = post && (post->act != 0 || post->residual);
    if (!has_post && batch_outer * batch_inner == 1 && m && n && c && a && b && gemm_takes_split(ctx, m, n, k))
        return launch_gemm_split(ctx, c, a, b, c0, m, n, k, trans_a, trans_b, lda, ldb, ldc, c0_row_stride, c0_col_stride, alpha, beta);
    if (batch_outer * batch_inner != 1 || trans_a || !planes_reach(lda, k)) planes = nullptr;
    return launch_gemm_f32(ctx, c, a, b, c0, batch_outer, batch_inner, m, n, k, trans_a, trans_b, lda, ldb, ldc, a_batch_strides, b_batch_strides,
                           c_batch_strides, c0_row_stride, c0_col_stride, alpha, beta, post, planes);
}

// What choose() reckons is fitted to larger products with 16-byte loads; a convolution's, which decide between this and a kernel that reads
// x in place, take longer: 0.4 to 1.2 us of 4 to 7 ([144,48] x [48,196], 30 images, 5.7 reckoned and 6.8 measured), with single-value loads
// and a bias per row 1.3 and 2.6 us and 15 % ([576,96] x [96,49], 44 images: 7.1 and 10.8).  Without that, products were taken for images
// that the in-place kernels do in 5.9 and 9.3 us.
double gemm_f32_us(const DeviceCtx &ctx, size_t batch, size_t m, size_t n, size_t k, bool vec) {
    const size_t cus = ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd : 32;
    const Choice ch = choose(batch, m, n, k, cus, ctx.gemm_split_k);
    return vec ? ch.us + (ch.shape ? 1.2 : 0.4) : 1.15 * ch.us + (ch.shape ? 2.6 : 1.3);
}

int gemm_f32_chains(const DeviceCtx &ctx, size_t batch, size_t m, size_t n, size_t k) {
    if (gemm_small_batched_fits(batch, m, n, k)) return 0;
    const Choice ch = choose(batch, m, n, k, ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd : 32, ctx.gemm_split_k);
    return ch.slices > 1 ? 0 : (int)(SHAPES[ch.shape].step / BK);
}

int gemm_f32_grid(const DeviceCtx &ctx, size_t batch, size_t m, size_t n, size_t k, size_t *blocks, int *slices) {
    const Choice ch = choose(batch, m, n, k, ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd : 32, ctx.gemm_split_k);
    const Grid grid(ch, batch, m, n);
    *blocks = grid.blocks, *slices = (int)ch.slices;
    return grid.fits(batch) ? AHIP_OK : AHIP_ERR_UNSUPPORTED;
}

int launch_gemm_f32(DeviceCtx &ctx, float *c, const float *a, const float *b, const float *c0, size_t batch_outer, size_t batch_inner, size_t m,
                    size_t n, size_t k, int trans_a, int trans_b, size_t lda, size_t ldb, size_t ldc, const size_t a_batch_strides[2],
                    const size_t b_batch_strides[2], const size_t c_batch_strides[2], size_t c0_row_stride, size_t c0_col_stride, float alpha,
                    float beta, const GemmPost *post, const void *planes) {
    const size_t batch = batch_outer * batch_inner;
    if (batch == 0 || m == 0 || n == 0) return AHIP_OK;
    if (!c || (k && (!a || !b))) return ctx.fail(AHIP_ERR_ARG, "gemm: null pointer");
    const bool has_post = post && (post->act != 0 || post->residual);
    if (has_post && post->act != 0 && post->act != AHIP_GELU && post->act != AHIP_RELU && post->act != AHIP_HARDSIGMOID && post->act != ACT_HARD_SWISH)
        return ctx.fail(AHIP_ERR_UNSUPPORTED, "gemm: not an activation that can follow the product in its kernel");
    const size_t lim = (size_t)1 << 31;
    if (m >= lim || n >= lim || k >= lim || lda >= lim || ldb >= lim || ldc >= lim || m * ldc >= ((size_t)1 << 40))
        return ctx.fail(AHIP_ERR_UNSUPPORTED, "gemm: extent above 2^31");
    // Hundreds of small matrices (attention's two products per head): one block per matrix.
    // (its fetchers address a head's operand with 32-bit byte offsets: 2^29 floats per head at most)
    const size_t a_extent = (m - 1) * lda + k, b_extent = trans_b ? (n - 1) * ldb + k : (k ? k - 1 : 0) * ldb + n;
    if (!planes && !has_post && !trans_a && alpha == 1.0f && (!c0 || beta == 0.0f) && gemm_small_batched_fits(batch, m, n, k) &&
        a_extent < ((size_t)1 << 29) && b_extent < ((size_t)1 << 29))
        return launch_gemm_small_batched(ctx, c, a, b, batch_outer, batch_inner, m, n, k, trans_b, lda, ldb, ldc, a_batch_strides, b_batch_strides,
                                         c_batch_strides);
    const bool a_kc = !trans_a, b_kc = trans_b != 0;
    // Rows so far apart that a tile's would not lie within 32-bit offsets: fewer of them at a time.
    const size_t a_rows = a_kc ? std::min<size_t>(m, 128) : std::min<size_t>(k, 64), b_rows = b_kc ? std::min<size_t>(n, 128) : std::min<size_t>(k, 64);
    if (a_rows > 1 && a_rows * lda > TILE_SPAN)
        return launch_gemm_far_rows(ctx, a_kc ? 0 : 2, std::max<size_t>(1, TILE_SPAN / lda), c, a, b, c0, batch_outer, batch_inner, m, n, k, trans_a, trans_b,
                                    lda, ldb, ldc, a_batch_strides, b_batch_strides, c_batch_strides, c0_row_stride, c0_col_stride, alpha, beta, post);
    if (b_rows > 1 && b_rows * ldb > TILE_SPAN)
        return launch_gemm_far_rows(ctx, b_kc ? 1 : 2, std::max<size_t>(1, TILE_SPAN / ldb), c, a, b, c0, batch_outer, batch_inner, m, n, k, trans_a, trans_b,
                                    lda, ldb, ldc, a_batch_strides, b_batch_strides, c_batch_strides, c0_row_stride, c0_col_stride, alpha, beta, post);
    const size_t cus = ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd : 32;
    GemmArgs g = {};
    g.a = a;
    g.b = b;
    g.c0 = (c0 && beta != 0.0f) ? c0 : nullptr;
    g.c = c;
    g.m = (uint32_t)m;
    g.n = (uint32_t)n;
    g.k = (uint32_t)k;
    g.lda = (uint32_t)lda;
    g.ldb = (uint32_t)ldb;
    g.ldc = (uint32_t)ldc;
    g.c0_rs = (uint32_t)c0_row_stride;
    g.c0_cs = (uint32_t)c0_col_stride;
    g.a_bs = a_batch_strides[0];
    g.b_bs = b_batch_strides[0];
    g.c_bs = c_batch_strides[0];
    g.a_bs2 = a_batch_strides[1];
    g.b_bs2 = b_batch_strides[1];
    g.c_bs2 = c_batch_strides[1];
    g.batch_inner = (uint32_t)batch_inner;
    g.alpha = alpha;
    g.beta = beta;
    g.act = has_post ? post->act : 0;
    g.residual = has_post ? post->residual : nullptr;
    g.act_alpha = has_post ? post->alpha : 0.0f, g.act_beta = has_post ? post->beta : 0.0f;
    // 16-byte loads: every piece aligned, and whole inside its row.
    auto vec = [&](const float *p, size_t contiguous, size_t ld, const size_t bs[2]) {
        return aligned16(p) && contiguous % 4 == 0 && ld % 4 == 0 && bs[0] % 4 == 0 && bs[1] % 4 == 0;
    };
    const bool both = vec(a, a_kc ? k : m, lda, a_batch_strides) && (planes || vec(b, b_kc ? k : n, ldb, b_batch_strides));
    const Shape *shapes = planes ? PLANE_SHAPES : SHAPES;
    Choice ch = choose(batch, m, n, k, cus, ctx.gemm_split_k, planes);
    if (ch.slices > 1) {
        const Shape &cut = shapes[ch.shape];
        const Grid grid(ch, batch, m, n, planes);
        const int rc = gemm_partials(ctx, (grid.chunk - grid.full) * 8 * ch.slices * cut.bm * cut.bn * sizeof(float));
        if (rc == AHIP_ERR_OOM) ch = choose(batch, m, n, k, cus, false, planes);  // no room: whole
        else if (rc) return rc;
    }
    const Shape &sh = shapes[ch.shape];
    const Grid grid(ch, batch, m, n, planes);
    if (!grid.fits(batch)) return ctx.fail(AHIP_ERR_UNSUPPORTED, "gemm: more tiles than a grid holds");
    g.tiles_n = (uint32_t)grid.gx;
    g.tiles_m = (uint32_t)grid.gy;
    g.tiles = (uint32_t)grid.tiles;
    g.chunk = (uint32_t)grid.chunk;
    {
        // Groups of about 768 columns (measured on [50432,768]x[768,2304..3072] and 4096^3 .. 8192^3: widths of
        // 6 to 16 tile columns are within 1 % of each other and up to 3 % ahead of whole rows of tiles; a single
        // column is 3-6 % behind), all groups equally wide.
        const size_t group = 768 / sh.bn, groups = (grid.gx + group - 1) / group;
        g.group_n = (uint32_t)((grid.gx + groups - 1) / groups);
    }
    g.slices = ch.slices;
    g.full = (uint32_t)grid.full;
    g.slice_k = ch.slices > 1 ? ch.slice_k : (uint32_t)k;
    // Up to the three blocks of 32 x 32 that a CU holds ([197,768] x [768,2304 / 3072] 10.4 -> 10.15 us, 13.6 -> 13.25, [1024,768] x [768,768]
    // 13.9 -> 13.5, [1024,3072] x [3072,768] 42.8 -> 41.8; of 4713 tiles the later ones starve, 82 -> 87, cut ones gain nothing, and
    // 64 x 64 tiles lose 7 % of three rounds and more).
    g.apart = !planes && ch.slices == 1 && g.chunk <= 3 * cus;
    if (g.slices > 1) {
        g.partials = static_cast<float *>(ctx.gemm_partials);
        g.counters = ctx.gemm_counters;
    }
    auto window = [&](bool kc, size_t rows, size_t ld) {
        const size_t end = ((size_t)1 << 32) - 64, step = (kc ? (size_t)sh.step : sh.step * ld) * 4;
        const size_t span = (kc ? (rows - 1) * ld + sh.step : (sh.step - 1) * ld + rows) * 4;
        return span < end ? std::min<size_t>((end - span) / std::max<size_t>(step, 1), 0x7fffffff) : 0;
    };
    if (!planes) g.window = (uint32_t)std::min(window(a_kc, std::min<size_t>(sh.bm, a_kc ? m : sh.bm), lda), window(b_kc, std::min<size_t>(sh.bn, b_kc ? n : sh.bn), ldb));
    if (planes) {
        g.planes = static_cast<const char *>(planes);
        g.n32s = (uint32_t)((n + 31) / 32), g.k16s = (uint32_t)weight_k16s(k);
        g.b_kc = b_kc;
        launch_plane_tiles(ctx, g, ch.shape, both);
    } else if (a_kc && b_kc) launch_tiles<true, true>(ctx, g, ch.shape, both);
    else if (a_kc) launch_tiles<true, false>(ctx, g, ch.shape, both);
    else if (b_kc) launch_tiles<false, true>(ctx, g, ch.shape, both);
    else launch_tiles<false, false>(ctx, g, ch.shape, both);
    return ctx.check(hipGetLastError(), "gemm launch");
}

}  // namespace altius
