// Y[M, N] = X[M, K] * W[N, K]^T in float: the product of the 32-bit path, on the bfloat16 matrix cores.
//
// A float of 24 bits is the sum of three bfloat16 numbers, exactly (Henry, Tang, Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", 2019): x0 = x rounded, x1 = (x - x0) rounded, x2 = x - x0 - x1.
// (A number under 2^-110 may have a rest below 2^-133, which no bfloat16 number holds: its results are made as those that are not finite,
// below.)  A product of two parts is exact in float, and all but x2 w2, under 2^-32 of the whole, are summed.  The matrix cores multiply
// bfloat16 sixteen times as fast as float, so eight products are twice as fast, and weights that are bfloat16 numbers kept in 32
// bits (a checkpoint's) have parts w1 = w2 = 0 and need three.
//
// The order of sums, the same for every shape, whatever M is, so that a row's result does not depend on the other rows of a
// batch or on which kernel below runs:  the products x0 w0 of a chunk of 32 k are summed from zero (v_mfma_f32_16x16x32_bf16), and the chunks'
// sums added in order as floats; the small products have a sum of their own, on the matrix cores, which is added at the end.
// Where N is small, K is cut into slices that N and K alone decide (slices_of), and the slices' sums are added in order.  Leaving
// out the products of w1 and w2 where all of them are zero changes no bit: they add zero.  A result of one product is rounded as a float's
// (5.97e-8 at most; the matrix cores alone, which cut: 1.3e-7), of many it is nearer to 64 bits than with v_mfma_f32_16x16x4_f32 in
// four chains, which this replaces (2-norm, normal operands of 24 bits, k of 1, 2, 8, 64, 512, 2,048, 8,192: 2.54e-8, 3.1e-8, 5.3e-8, 8.3e-8,
// 2.07e-7, 4.07e-7, 8.1e-7 -> 2.54e-8, 2.6e-8, 2.8e-8, 4.7e-8, 7.3e-8, 8.8e-8, 1.27e-7).
//
// Infinities and NaN, and finite numbers that round to an infinite part: some product of parts is then not finite, and neither is
// the result.  A result that is not finite is made again from the floats as they are, on the float matrix cores (float_sums), 16 x 16
// results a wave at a time.  us, by a thread a result, k after k -> now (and without any):  a row of NaN among 303, x 128,256 x 2,048 8,450 -> 1,131
// (726), x 2,048 x 2,048 1,208 -> 67 (32), all 303 of them 2,996 -> 124;  one row alone, x 128,256 x 2,048 4,400 -> 401 (194).
//
// * Few rows: a workgroup's waves stream W past the step's rows.  Bound by reading W, or by what the workgroups fetch from L2.
// * More rows: X is split into its parts ahead, once, in the order in which the matrix cores read it; tiles of Y, X's parts and W as it
//   is staged through LDS by loads that pass no registers, W split where it is read.  Two sums a result
//   are what its registers hold: 128 x 256 outputs, which one sum allowed (303 x 128,256 x 2,048 664 us), would spill.
// Workspace: the parts, 6 bytes an element of X; where slices are apart their sums, a float a result and slice, 512 MiB at most.
// us, v_mfma_f32_16x16x4_f32 -> now, weights of 8 bits and of 24:  303 rows x 128,256 x 2,048 1,461 -> 594 and 1,204, x 16,384 x 2,048 203 -> 99
// and 168, x 2,048 x 8,192 136 -> 55 and 90, x 3,072 x 2,048 42.5 -> 31.6 and 45;  one row x 2,048 x 2,048 8.7 -> 6.1 and 7.3, x 2,048 x 8,192 23.4 -> 15.3
// and 19.9, x 14,336 x 4,096 50 -> 42 and 42;  64 rows x 2,048 x 2,048 11.6 -> 8.9 and 10.9.  Slower: 200 to 1,024 rows of 1,000 x 1,000 (512: 16.5 -> 19.5
// and 20.5, 1,024: 25 -> 28 and 41), one row x 128,256 x 2,048 (192 -> 198), and with weights of 24 bits 1 to 96 rows of 14,336 to 16,384 columns (17 x 16,384 x
// 2,048 28.8 -> 30.8, 32 x 14,336 x 4,096 50.5 -> 57.9) and 130 to 1,024 rows of 2,048 to 3,072 (512 x 2,048 x 2,048 42.7 -> 52.9, 303 x 3,072 x 2,048 42.6 -> 45).
#include "lds_load.h"

#include <algorithm>

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int CHUNK = 32;      // k that are summed from zero
constexpr int PARTS = 3;
constexpr int PART_BLOCK = PARTS * SIA_WAVE;      // 16-byte pieces of the parts of 16 rows of X in a chunk

// ---------------------------------------------------------------------------------------------------------
// parts and products
// ---------------------------------------------------------------------------------------------------------

// The parts of eight consecutive floats, each eight bfloat16 in order.  Returned: bits of which the low 16 are zero if the parts are all there
// is of them.  (What is left for the third part has eight bits; below 2^-126, of a number under 2^-110, they may reach lower than
// bfloat16 does.  NaN, where some part is not finite, ends in zeros too.)
__device__ __forceinline__ uint32_t split8(u32x4 first, u32x4 second, u32x4 (&part)[PARTS]) {
    uint32_t rest = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const u32x4& v = e < 2 ? first : second;
        float a = __uint_as_float(v[2 * (e & 1)]), b = __uint_as_float(v[2 * (e & 1) + 1]);
#pragma unroll
        for (int p = 0; p < PARTS - 1; ++p) {
            const uint32_t r = bf16_pair(a, b);
            part[p][e] = r;
            a -= __uint_as_float(r << 16), b -= __uint_as_float(r & 0xffff0000u);
        }
        part[PARTS - 1][e] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
        rest |= __float_as_uint(a) | __float_as_uint(b);
    }
    return rest;
}

// Whether any lane's parts leave something out.
__device__ __forceinline__ bool any_rest(uint32_t rest) { return __any((rest & 0xffffu) != 0); }

// NaN for the third part of those of the eight floats that have a rest: what they are multiplied with is then made again.
__device__ __forceinline__ void mark_rests(u32x4 first, u32x4 second, u32x4& third) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float v = __uint_as_float((e < 4 ? first : second)[e % 4]);
#pragma unroll
        for (int p = 0; p < PARTS - 1; ++p) v -= __uint_as_float(bf16_pair(v, v) << 16);
        if (__float_as_uint(v) & 0xffffu) third[e / 2] |= e % 2 ? 0x7fff0000u : 0x7fffu;
    }
}

// The first part of eight floats that have no other.
__device__ __forceinline__ u32x4 upper_halves(u32x4 a, u32x4 b) {
    return u32x4{__builtin_amdgcn_perm(a[1], a[0], 0x07060302), __builtin_amdgcn_perm(a[3], a[2], 0x07060302),
                 __builtin_amdgcn_perm(b[1], b[0], 0x07060302), __builtin_amdgcn_perm(b[3], b[2], 0x07060302)};
}

__device__ __forceinline__ uint32_t or_of(u32x4 a, u32x4 b) { return (a[0] | a[1] | a[2] | a[3]) | (b[0] | b[1] | b[2] | b[3]); }

__device__ __forceinline__ f32x4 product(u32x4 w, u32x4 x, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}

// A chunk's products of a block of 16 rows of X with TN blocks of 16 rows of W, added to their sums.  The matrix cores cut off where floats
// round: the large products, exact where one is alone, are added as floats, and the small ones, 2^-8 of them, stay on the matrix cores, in a
// sum of their own.  The blocks alternate: a product is done when the next one that adds to it begins.
// more: W has more parts than the first.  One body for both (as two branches the sums of each had registers of their own).
template <int TN>
__device__ __forceinline__ void add_chunk(const u32x4 (&w)[TN][PARTS], const u32x4 (&x)[PARTS], bool more, f32x4 (&total)[TN], f32x4 (&small)[TN]) {
    constexpr int MORE = 5, ORDER[MORE][2] = {{2, 1}, {1, 2}, {2, 0}, {1, 1}, {1, 0}};      // parts of W and X
    f32x4 large[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) large[j] = product(w[j][0], x[0], f32x4{0.f, 0.f, 0.f, 0.f});
    if (more)
#pragma unroll
        for (int o = 0; o < MORE; ++o)
#pragma unroll
            for (int j = 0; j < TN; ++j) small[j] = product(w[j][ORDER[o][0]], x[ORDER[o][1]], small[j]);
#pragma unroll
    for (int p = PARTS - 1; p > 0; --p)
#pragma unroll
        for (int j = 0; j < TN; ++j) small[j] = product(w[j][0], x[p], small[j]);
#pragma unroll
    for (int j = 0; j < TN; ++j) total[j] += large[j];
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= 3.402823466e38f; }

// A block of 16 x 16 results by v_mfma_f32_16x16x4_f32, for those that the parts do not give:  x and w are the rows r = lane % 16 of either
// operand, the lane gets row r and columns 4 g .. 4 g + 3, g = lane / 16.  All lanes take part.  Pieces of 16 k go to four sums in
// turn, (s0 + s1) + (s2 + s3): a result depends on its row and column alone, whoever asks for it.
__device__ __forceinline__ f32x4 float_sums(const float* __restrict__ x, const float* __restrict__ w, int K) {
    const int g = (threadIdx.x % SIA_WAVE) / 16;
    const bool wide = __all(K % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0);
    f32x4 sum[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) sum[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
    for (int k0 = 0; k0 < K; k0 += 64) {      // pieces of 16 k, 4 g .. 4 g + 3 of each in this lane; zeros behind the last k
        f32x4 a[4], b[4];
        if (wide) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int at = min(k0 + 16 * s + 4 * g, K - 4);
                a[s] = *(const f32x4*)(w + at), b[s] = *(const f32x4*)(x + at);
            }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int at = min(k0 + 16 * s + 4 * g + i, K - 1);
                    a[s][i] = w[at], b[s][i] = x[at];
                }
        }
        if (k0 + 64 > K)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (k0 + 16 * s + 4 * g + i >= K) a[s][i] = 0.f, b[s][i] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) sum[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i], b[s][i], sum[s], 0, 0, 0);
    }
    return (sum[0] + sum[1]) + (sum[2] + sum[3]);
}

// A KiB of 8 rows of a chunk into LDS by loads of 16 bytes a lane (WIDE: rows at multiples of 16 bytes, K a multiple of 4), or by four loads of a float
// a lane, of two rows each, for rows that begin anywhere; the places are the same (`turn`).  (Loaded into registers float by float, or copied to
// rows of 16 bytes first, us:  32 rows x 2,048 x 2,049 32.6 -> 12.0, 17 x 16,384 x 2,049 78 -> 37, 303 x 40,000 x 2,049 2,873 -> 294, 303 x 1,000 x 333 18.4 -> 10.6;
// slower 600 x 2,048 x 2,049 with weights of 24 bits, 70 -> 90.)  Lane's row of load q, and its k of a chunk:
template <bool WIDE> __device__ __forceinline__ int row_of_load(int q, int lane) { return WIDE ? lane / 8 : 2 * q + lane / 32; }
template <bool WIDE> __device__ __forceinline__ int k_of_load(int row, int lane) {      // row: of 16
    return WIDE ? ((lane & 7) ^ turn(row)) * 4 : (((lane % 32 / 4) ^ turn(row)) * 4 + lane % 4);
}
template <bool WIDE> __device__ __forceinline__ void load_chunk(const float* row, int k, int K, char* to, int q) {      // behind the last k: the last
    if constexpr (WIDE)
        load_to_lds(row + min(k, K - 4), to);
    else
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row + min(k, K - 1)),
                                         (__attribute__((address_space(3))) void*)(to + q * (LL_TILE / 4)), 4, 0, 0);
}

// Slices of K, in chunks: from N and K alone.  Few rows of W beside a long K are too little for the chip without; an output head
// is enough, and its tiles then need no second sum.
__host__ __device__ static inline int slices_of(int N, int K) { return N > 32 * 1024 || K <= 4 * CHUNK ? 1 : N > 12 * 1024 ? 2 : 8; }
__device__ __forceinline__ int slice_begin(int chunks, int slice, int slices) { return (int)((long long)chunks * slice / slices); }

// ---------------------------------------------------------------------------------------------------------
// few rows
// ---------------------------------------------------------------------------------------------------------

// A workgroup has MB blocks of 16 rows of X and WAVES / SLICES groups of NB blocks of 16 rows of W; a wave has a slice of K of one group.
// A wave's step is U chunks, whose sums do not depend on one another.  W's and X's rows come to LDS directly as they are, 128 bytes of eight
// rows an instruction, into a ring of SLOTS steps that the wave has for itself, and are split where they are read.  (Loaded into registers,
// an instruction touches 16 lines in pieces of 16 bytes: see gemm_skinny.hip.)  XI: tiles of 8 rows of X, 2 MB or 1.
// WIDE: see load_chunk.
template <int SLICES, int WAVES, int MB, int NB, int XI, int U, int SLOTS, bool WIDE>
__global__ __launch_bounds__(WAVES* SIA_WAVE) void gemm_f32_few_rows_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                                            float* __restrict__ Y, int M, int N, int K) {
    static_assert(WAVES % SLICES == 0, "a wave a slice");
    constexpr int GROUPS = WAVES / SLICES;
    static_assert(XI == 2 * MB || (MB == 1 && XI == 1), "tiles of 8 rows");
    constexpr int TILES = 2 * NB + XI, EACH = WIDE ? 1 : 4, LOADS = U * TILES * EACH;      // KiB of a chunk, loads of each
    constexpr int RING = WAVES * SLOTS * U * TILES * LL_TILE, SUMS = SLICES > 1 ? WAVES * MB * NB * 256 * 4 : 0;
    constexpr int LDS = RING > SUMS ? RING : SUMS > 0 ? SUMS : 16;
    static_assert(LDS <= LL_LDS, "a workgroup's LDS");
    __shared__ __attribute__((aligned(1024))) char lds[LDS];
    const int lane = threadIdx.x % SIA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SIA_WAVE);
    const int r = lane % 16, g = lane / 16;
    const int m0 = blockIdx.y * MB * 16, slice = wave % SLICES, group = wave / SLICES;
    const int n0 = (blockIdx.x * GROUPS + group) * NB * 16;
    const int chunks = (K + CHUNK - 1) / CHUNK;
    const int begin = slice_begin(chunks, slice, SLICES);
    const int steps = n0 < N ? slice_begin(chunks, slice + 1, SLICES) - begin : 0;      // chunks of this wave

    f32x4 total[MB][NB], small[MB][NB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int j = 0; j < NB; ++j) total[b][j] = small[b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t rest_x[MB], rest_w[NB];      // of the rows r (a branch at every split: 17 rows x 2,048 x 8,192 22.8 us, 22.0 so)
#pragma unroll
    for (int b = 0; b < MB; ++b) rest_x[b] = 0;
#pragma unroll
    for (int j = 0; j < NB; ++j) rest_w[j] = 0;
    // U chunks from s on; chunks behind the last are zeros, which change nothing
    auto multiply = [&](int s, u32x4 (&wa)[U][NB], u32x4 (&wb)[U][NB], u32x4 (&xa)[U][MB], u32x4 (&xb)[U][MB]) {
        const u32x4 none = {0, 0, 0, 0};
        uint32_t bits = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (begin + s + u) * CHUNK + 8 * g;
            if (s + u >= steps)
#pragma unroll
                for (int j = 0; j < NB; ++j) wa[u][j] = none, wb[u][j] = none;
            if (s + u >= steps || (begin + s + u + 1) * CHUNK > K)
#pragma unroll
                for (int b = 0; b < MB; ++b) {      // behind the last k too (W has there what was read instead)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {      // (wide: K is a multiple of 4)
                        if (s + u >= steps || k + (WIDE ? 0 : e) >= K) xa[u][b][e] = 0;
                        if (s + u >= steps || k + 4 + (WIDE ? 0 : e) >= K) xb[u][b][e] = 0;
                    }
                }
#pragma unroll
            for (int j = 0; j < NB; ++j) bits |= or_of(wa[u][j], wb[u][j]);
        }
        const bool more = __any((bits & 0xffffu) != 0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            u32x4 w[NB][PARTS];
#pragma unroll
            for (int j = 0; j < NB; ++j) w[j][0] = upper_halves(wa[u][j], wb[u][j]);
            if (more)
#pragma unroll
                for (int j = 0; j < NB; ++j) rest_w[j] |= split8(wa[u][j], wb[u][j], w[j]);
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                u32x4 x[PARTS];
                rest_x[b] |= split8(xa[u][b], xb[u][b], x);
                add_chunk(w, x, more, total[b], small[b]);
            }
        }
    };
    u32x4 wa[U][NB], wb[U][NB], xa[U][MB], xb[U][MB];
    // rows that do not exist are read as the last one and not stored
    const float* from[TILES * EACH];
    int piece[TILES * EACH];
#pragma unroll
    for (int l = 0; l < TILES; ++l)
#pragma unroll
        for (int q = 0; q < EACH; ++q) {
            const int row = (l < 2 * NB ? l : l - 2 * NB) * 8 + row_of_load<WIDE>(q, lane);
            from[l * EACH + q] = l < 2 * NB ? W + (size_t)min(n0 + row, N - 1) * K : X + (size_t)min(m0 + row, M - 1) * K;
            piece[l * EACH + q] = begin * CHUNK + k_of_load<WIDE>(row & 15, lane);
        }
    char* const ring = lds + wave * (SLOTS * U * TILES * LL_TILE);
    // steps of U chunks; the last one's chunks behind the end are loaded again, so that the waits count the same
    auto request = [&](int s, int slot) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int l = 0; l < TILES; ++l)
#pragma unroll
                for (int q = 0; q < EACH; ++q)
                    load_chunk<WIDE>(from[l * EACH + q], min(s + u, steps - 1) * CHUNK + piece[l * EACH + q], K,
                                     ring + ((slot * U + u) * TILES + l) * LL_TILE, q);
    };
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
        if (s * U < steps) request(s * U, s);
    const int at[2] = {r * 128 + ((2 * g) ^ turn(r)) * 16, r * 128 + ((2 * g + 1) ^ turn(r)) * 16};
    const int xr = XI == 1 ? r & 7 : r;
    const int x_at[2] = {xr * 128 + ((2 * g) ^ turn(xr)) * 16, xr * 128 + ((2 * g + 1) ^ turn(xr)) * 16};
    int slot = 0;
    for (int s = 0; s < steps; s += U) {
        wait_step<LOADS, SLOTS - 1>((steps - 1) / U - s / U);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const char* in = ring + (slot * U + u) * TILES * LL_TILE;
#pragma unroll
            for (int j = 0; j < NB; ++j)
                wa[u][j] = *(const u32x4*)(in + 2 * j * LL_TILE + at[0]), wb[u][j] = *(const u32x4*)(in + 2 * j * LL_TILE + at[1]);
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                const char* in_x = in + (2 * NB + 2 * b) * LL_TILE;
                xa[u][b] = *(const u32x4*)(in_x + x_at[0]), xb[u][b] = *(const u32x4*)(in_x + x_at[1]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the slot has been read: it may be filled again
        if (s + SLOTS * U < steps) request(s + SLOTS * U, slot);
        slot = slot + 1 < SLOTS ? slot + 1 : 0;
        multiply(s, wa, wb, xa, xb);
    }
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int j = 0; j < NB; ++j) total[b][j] += small[b][j];
    uint32_t rest = 0;
#pragma unroll
    for (int b = 0; b < MB; ++b) rest |= rest_x[b];
#pragma unroll
    for (int j = 0; j < NB; ++j) rest |= rest_w[j];
    if (any_rest(rest)) {      // the results of these rows of X and W are made again
        auto row_has = [&](uint32_t v) {
            v |= __shfl_xor(v, 16, SIA_WAVE);
            return ((v | __shfl_xor(v, 32, SIA_WAVE)) & 0xffffu) != 0;
        };
        bool has_x[MB], has_w[NB];
#pragma unroll
        for (int b = 0; b < MB; ++b) has_x[b] = row_has(rest_x[b]);
#pragma unroll
        for (int j = 0; j < NB; ++j) has_w[j] = row_has(rest_w[j]);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool column = __shfl(has_w[j], 4 * g + e, SIA_WAVE);
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    if (has_x[b] || column) total[b][j][e] = __builtin_nanf("");
            }
    }
    // a block of results from row m and column n on
    auto finish = [&](int m, int n, f32x4 v) {
        bool odd = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) odd |= m + r < M && n + 4 * g + e < N && !finite(v[e]);
        if (__any(odd)) {
            const f32x4 again = float_sums(X + (size_t)min(m + r, M - 1) * K, W + (size_t)min(n + r, N - 1) * K, K);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = finite(v[e]) ? v[e] : again[e];
        }
        if (m + r >= M) return;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + 4 * g + e < N) Y[(size_t)(m + r) * N + n + 4 * g + e] = v[e];
    };
    if (SLICES == 1) {
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int j = 0; j < NB; ++j) finish(m0 + b * 16, n0 + j * 16, total[b][j]);
        return;
    }
    f32x4* const part = (f32x4*)lds;
    __syncthreads();      // every wave has read its ring
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int j = 0; j < NB; ++j) part[(((slice * GROUPS + group) * MB + b) * NB + j) * SIA_WAVE + lane] = total[b][j];
    __syncthreads();
    constexpr int BLOCKS = GROUPS * MB * NB;
#pragma unroll
    for (int i = 0; i < (BLOCKS + WAVES - 1) / WAVES; ++i) {
        const int block = wave + i * WAVES;
        if (block >= BLOCKS) return;
        f32x4 v = part[block * SIA_WAVE + lane];
#pragma unroll
        for (int s = 1; s < SLICES; ++s) v += part[(s * BLOCKS + block) * SIA_WAVE + lane];
        finish(m0 + block / NB % MB * 16, (blockIdx.x * GROUPS + block / (MB * NB)) * NB * 16 + block % NB * 16, v);
    }
}

// Small rings, and more workgroups on a unit, are faster than deep ones (us for one row and weights of 8 bits, 8 waves, the best two of
// each:  2,048 x 2,048 6.4 with one step of two chunks, 6.8 with three;  28,672 x 4,096 78 and 86).
template <int MB, int NB, int XI, bool WIDE>
static void launch_few_rows(const float* X, const float* W, float* Y, int M, int N, int K, hipStream_t stream) {
    const int slices = slices_of(N, K), y = (M + MB * 16 - 1) / (MB * 16);
    auto columns = [&](int groups) { return dim3((N + groups * NB * 16 - 1) / (groups * NB * 16), y); };
    constexpr int EACH = 2 * NB + XI, U = MB * NB == 1 ? 2 : 1;
    constexpr int SLOTS2 = EACH <= 3 ? 3 : EACH <= 8 ? 2 : 1, SLOTS = EACH <= 9 && MB * NB <= 4 ? 2 : 1;
    if (slices == 8)
        hipLaunchKernelGGL((gemm_f32_few_rows_kernel<8, 8, MB, NB, XI, U, 1, WIDE>), columns(1), dim3(512), 0, stream, X, W, Y, M, N, K);
    else if (slices == 2)
        hipLaunchKernelGGL((gemm_f32_few_rows_kernel<2, 4, MB, NB, XI, U, SLOTS2, WIDE>), columns(2), dim3(256), 0, stream, X, W, Y, M, N, K);
    else if (N <= 32 * 1024)
        hipLaunchKernelGGL((gemm_f32_few_rows_kernel<1, 4, MB, NB, XI, U, 1, WIDE>), columns(4), dim3(256), 0, stream, X, W, Y, M, N, K);
    else
        hipLaunchKernelGGL((gemm_f32_few_rows_kernel<1, 8, MB, NB, XI, U, SLOTS, WIDE>), columns(8), dim3(512), 0, stream, X, W, Y, M, N, K);
}

// The shape of the few-row kernel: blocks of X's and W's rows, and what it costs: a launch (us), and at what rate its workgroups fetch
// (MB a us).  More blocks share what is read and split of the other operand, where enough workgroups are left.
struct FewRows {
    int mb, nb;
    double launch, rate;
};
static FewRows few_rows_shape(int M, int N, int K) {
    if (M <= 8 && N > 32 * 1024 && K % CHUNK == 0) return {1, 4, 2.5, 12};      // rows of whole cache lines
    if (M <= 16 || K <= 4 * CHUNK) return {1, 1, 4, 16};
    if (N < 8 * 1024) return {2, 1, 4, 13.6};
    if (M > 32 && N > 12 * 1024) return {4, 2, 2.5, 10};
    if (N <= 32 * 1024) return {2, 2, 2.5, 10.8};
    return K % CHUNK == 0 ? FewRows{2, 4, 2.5, 9} : FewRows{2, 2, 2.5, 7};
}

// wide: both operands' rows lie so.
static void few_rows(const float* X, const float* W, float* Y, int M, int N, int K, bool wide, hipStream_t stream) {
    const FewRows few = few_rows_shape(M, N, K);
    if (!wide && M <= 8)
        launch_few_rows<1, 1, 1, false>(X, W, Y, M, N, K, stream);
    else if (!wide && M <= 16)
        launch_few_rows<1, 1, 2, false>(X, W, Y, M, N, K, stream);
    else if (!wide && few.nb == 1)
        launch_few_rows<2, 1, 4, false>(X, W, Y, M, N, K, stream);
    else if (!wide)
        launch_few_rows<2, 2, 4, false>(X, W, Y, M, N, K, stream);
    else if (few.mb == 4)
        launch_few_rows<4, 2, 8, true>(X, W, Y, M, N, K, stream);
    else if (few.mb == 2 && few.nb == 4)
        launch_few_rows<2, 4, 4, true>(X, W, Y, M, N, K, stream);
    else if (few.mb == 2 && few.nb == 2)
        launch_few_rows<2, 2, 4, true>(X, W, Y, M, N, K, stream);
    else if (few.mb == 2)
        launch_few_rows<2, 1, 4, true>(X, W, Y, M, N, K, stream);
    else if (few.nb == 4)
        launch_few_rows<1, 4, 1, true>(X, W, Y, M, N, K, stream);
    else if (M <= 8)
        launch_few_rows<1, 1, 1, true>(X, W, Y, M, N, K, stream);
    else
        launch_few_rows<1, 1, 2, true>(X, W, Y, M, N, K, stream);
}

// ---------------------------------------------------------------------------------------------------------
// tiles
// ---------------------------------------------------------------------------------------------------------

// The parts of X as the matrix cores read them: [chunk][block of 16 rows][part][lane] of 16 bytes, zeros beyond X.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ X, u32x4* __restrict__ parts, int M, int K, int blocks,
                                                         int chunks, bool direct) {
    const long long id = (long long)blockIdx.x * 4 + threadIdx.x / SIA_WAVE;
    const int lane = threadIdx.x % SIA_WAVE, c = (int)(id % chunks);
    const long long b = id / chunks;
    if (b >= blocks) return;
    const long long row = b * 16 + lane % 16;
    const int k = c * CHUNK + lane / 16 * 8;
    u32x4 v[2] = {u32x4{0, 0, 0, 0}, u32x4{0, 0, 0, 0}}, p[PARTS];
    const uint32_t* from = (const uint32_t*)X + row * K + k;
    if (direct) {      // K is a multiple of 4
        if (row < M && k < K) v[0] = *(const u32x4*)from;
        if (row < M && k + 4 < K) v[1] = *(const u32x4*)(from + 4);
    } else
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (row < M && k + e < K) v[e / 4][e % 4] = from[e];
    if (split8(v[0], v[1], p) & 0xffffu) mark_rests(v[0], v[1], p[PARTS - 1]);
    u32x4* at = parts + ((long long)c * blocks + b) * PART_BLOCK + lane;
#pragma unroll
    for (int e = 0; e < PARTS; ++e) at[e * SIA_WAVE] = p[e];
}

// The results that are not finite of a wave's tile, which its lanes have stored themselves, made again.
template <int TM, int TN>
__device__ __forceinline__ void make_again(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K,
                                           int m_first, int n_first) {
    const int lane = threadIdx.x % SIA_WAVE, r = lane % 16, g = lane / 16;
#pragma clang loop unroll(disable)
    for (int i = 0; i < TM * TN; ++i) {
        const int m = m_first + i / TN * 16, n = n_first + i % TN * 16;
        float* at = Y + (size_t)m * N + n;
        unsigned again = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m < M && n + e < N && !finite(*(volatile float*)(at + e))) again |= 1u << e;
        if (!__any(again != 0)) continue;
        const f32x4 v = float_sums(X + (size_t)min(m, M - 1) * K, W + (size_t)min(n - 4 * g + r, N - 1) * K, K);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (again >> e & 1) at[e] = v[e];
    }
}

// A tile of BM rows of W, taken by WM x WN waves.  A ring of D + 1 chunks of both in LDS, asked for D ahead; one
// barrier a chunk: what is read next has come, what was read last may be overwritten.
// apart: a workgroup has one slice of K, whose sums go to `slices` ([slice][M][Ns]) for sum_slices_f32_kernel.  Else it has all of K, and
// adds up the slices, SLICED: in registers, else in Y.
// WIDE: how W is read, see load_chunk.
template <int BM, int BN, int WM, int WN, int D, bool SLICED, bool WIDE>
__global__ __launch_bounds__(WM* WN* SIA_WAVE) void gemm_f32_tile_kernel(
    const u32x4* __restrict__ parts, const float* __restrict__ X, const float* __restrict__ W,
    float* __restrict__ Y, float* __restrict__ slices, int M, int N, int K, int Ns, int n_slices, bool apart, bool four,
    int tiles_m, int n_tiles, int per_die) {
    constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int XT = BM / 16 * PARTS, WT = BN / 8;                 // KiB of a chunk
    constexpr int LX = (XT + WAVES - 1) / WAVES, LW = WT / WAVES;    // loads of a wave
    constexpr int EACH = WIDE ? 1 : 4, STAGE = (XT + WT) * LL_TILE, LOADS = LX + LW * EACH;
    static_assert(TM * WM * 16 == BM && TN * WN * 16 == BN && LW * WAVES == WT && (D + 1) * STAGE <= LL_LDS, "tiles");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    // Workgroups go to the dies in turn: a die gets consecutive tiles, row tiles of X innermost, so that the rows of W
    // that they share are read by one die.
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (tile >= n_tiles) return;
    const int slice = apart ? (tile / tiles_m) % n_slices : 0;
    const int m0 = (tile % tiles_m) * BM, n0 = tile / tiles_m / (apart ? n_slices : 1) * BN;
    const int chunks = (K + CHUNK - 1) / CHUNK, blocks = (M + 15) / 16;
    const int lane = threadIdx.x % SIA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SIA_WAVE);
    const int wm = wave % WM, wn = wave / WM, r = lane % 16, g = lane / 16;

    // X: KiB beyond the tile or the last block repeat the last one (into the same place: the same bytes)
    int x_kib[LX], x_from[LX];
#pragma unroll
    for (int l = 0; l < LX; ++l) {
        x_kib[l] = min(wave * LX + l, XT - 1);
        x_from[l] = min(x_kib[l], (blocks - m0 / 16) * PARTS - 1) * SIA_WAVE + lane;
    }
    const float* const w_tile = W + (size_t)n0 * K;
    unsigned w_from[LW * EACH];      // (f32_plan: K is below 2^22 where the tiles take W)
    int piece[LW * EACH];
#pragma unroll
    for (int l = 0; l < LW; ++l)
#pragma unroll
        for (int q = 0; q < EACH; ++q) {      // rows that do not exist are read as the last one and not stored
            const int row = (wave * LW + l) * 8 + row_of_load<WIDE>(q, lane);
            w_from[l * EACH + q] = (unsigned)(min(n0 + row, N - 1) - n0) * (unsigned)K;
            piece[l * EACH + q] = k_of_load<WIDE>(row & 15, lane);
        }
    const int x_at = wm * TM * PARTS * LL_TILE + lane * 16, w_at = XT * LL_TILE + (wn * (BN / WN) + r) * 128;
    const int place[2] = {((2 * g) ^ turn(r)) * 16, ((2 * g + 1) ^ turn(r)) * 16};

    const int begin = apart ? slice_begin(chunks, slice, n_slices) : 0;
    const int steps = (apart ? slice_begin(chunks, slice + 1, n_slices) : chunks) - begin;
    const u32x4* x_first = parts + ((size_t)begin * blocks + m0 / 16) * PART_BLOCK;
    auto request = [&](int s, int slot) {
        char* to = lds + slot * STAGE;
        const u32x4* from = x_first + (size_t)s * blocks * PART_BLOCK;
#pragma unroll
        for (int l = 0; l < LX; ++l) load_to_lds(from + x_from[l], to + x_kib[l] * LL_TILE);
        to += XT * LL_TILE + wave * LW * LL_TILE;
#pragma unroll
        for (int l = 0; l < LW; ++l)      // (X's parts are zero behind the last k)
#pragma unroll
            for (int q = 0; q < EACH; ++q)
                load_chunk<WIDE>(w_tile + w_from[l * EACH + q], (begin + s) * CHUNK + piece[l * EACH + q], K, to + l * LL_TILE, q);
    };
    f32x4 total[TM][TN], small[TM][TN], sum[SLICED ? TM : 1][SLICED ? TN : 1];      // of the slice, of the slices before it
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            total[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (SLICED) sum[i][j] = total[i][j];
        }
    // total[i][j]: row 16 i + r of the wave's tile, columns 16 j + 4 g .. + 3
    const int m_first = m0 + wm * (BM / WM) + r, n_first = n0 + wn * (BN / WN) + 4 * g, stride = apart ? Ns : N;
    float* const to = apart ? slices + (size_t)slice * M * Ns : Y;
    bool odd = false;
    auto store = [&](bool more) {      // more: Y has the slices before
        int first = m_first;
        asm volatile("" : "+v"(first));      // addresses made here, not in front of the loop and kept through it
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = first + i * 16;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n_first + j * 16;
                float* at = to + (size_t)m * stride + n;
                f32x4 v = total[i][j] + small[i][j];
                if constexpr (SLICED) v = sum[i][j] + v;
                if (four || apart) {
                    if (n >= N) continue;
                    if (more) v = *(const f32x4*)at + v;
                    *(f32x4*)at = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < N) {
                            if (more) v[e] = at[e] + v[e];
                            at[e] = v[e];
                        }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) odd |= !finite(v[e]);
            }
        }
    };
    int ended = 0, end = apart ? chunks : 0;      // slices behind, where this one ends
    while (end == 0) end = slice_begin(chunks, ++ended, n_slices);      // (slices may be empty)
    bool more = false;
#pragma unroll
    for (int s = 0; s < D; ++s)
        if (s < steps) request(s, s);
    int slot = 0;
    for (int s = 0; s < steps; ++s) {
        wait_step<LOADS, D - 1>(steps - 1 - s);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + D < steps) request(s + D, slot == 0 ? D : slot - 1);
        const char* stage = lds + slot * STAGE;
        slot = slot == D ? 0 : slot + 1;
        auto read_w = [&](int j, u32x4& a, u32x4& b) {
            const char* at = stage + w_at + j * 2 * LL_TILE;
            a = *(const u32x4*)(at + place[0]), b = *(const u32x4*)(at + place[1]);
        };
        auto read_x = [&](int i, u32x4 (&x)[PARTS]) {
#pragma unroll
            for (int e = 0; e < PARTS; ++e) x[e] = *(const u32x4*)(stage + x_at + (i * PARTS + e) * LL_TILE);
        };
        u32x4 w[TN][PARTS];
        uint32_t bits = 0;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            u32x4 a, b;
            read_w(j, a, b);
            bits |= or_of(a, b);
            w[j][0] = upper_halves(a, b);
        }
        const bool more_parts = __any((bits & 0xffffu) != 0);
        if (more_parts) {
            uint32_t rest = 0;
            asm volatile("" ::: "memory");      // W is read again, here and below: kept, it would take the registers of the sums
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                u32x4 a, b;
                read_w(j, a, b);
                rest |= split8(a, b, w[j]);
            }
            if (any_rest(rest)) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    u32x4 a, b;
                    read_w(j, a, b);
                    mark_rests(a, b, w[j][PARTS - 1]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            u32x4 x[PARTS];
            read_x(i, x);
            add_chunk(w, x, more_parts, total[i], small[i]);
        }
        if (s + 1 == end && s + 1 < steps) {
            if constexpr (SLICED) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) sum[i][j] += total[i][j] + small[i][j];
            } else {
                store(more);
                more = true;
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) total[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            while (end == s + 1) end = slice_begin(chunks, ++ended, n_slices);
        }
    }
    store(more);
    if (apart || !__any(odd)) return;
    make_again<TM, TN>(X, W, Y, M, N, K, m_first, n_first);
}

// Tiles of BM rows of X by BN of W for whole chunks (K a multiple of CHUNK) of rows on 16 bytes: the sums of 160 x 128 and 160 x 192 results, two each,
// fit, because the parts of W beyond the first are never held for more than 16 rows.  Chunks go by with one part of W until the first that has more; from it on
// X's parts are read again for every 16 rows of W (the eight products of a block need the time anyway).  Half of the waves bring X, half W,
// each with a ring of its own, DX and DW chunks ahead: a wave's loads end in order, and X, which L2 holds, would wait for W behind it.
// Bound by what a compute unit fetches and then reads from LDS, which the matrix cores wait for in part: cycles of a chunk of 160 x 128, each alone: loads
// 1,800, reads 930, products and sums 1,350, all together 2,560 (1.1 us).  Wider tiles fetch less for a result: 303 rows x 128,256 x 2,048, weights of 8 bits,
// 677 us in tiles of 64 x 128, 600 in 160 x 128, 573 in 160 x 192 (650 in a step; 160 x 256 spills: 830);  x 16,384 x 2,048 117 -> 95 (160 x 128), x 3,072 x 2,048 36 -> 30.6 (160 x 192),
// x 2,048 x 8,192 65 -> 54, x 2,048 x 2,048 29 -> 26 (160 x 128);  weights of 24 bits 1,270 -> 1,130, 184 -> 160, 48 -> 43, 107 -> 87, 38 -> 34.
// With the next chunk's first reads in front of the last products of this one nothing changed (600 and 587 us), with four waves of twice the rows and
// 512 registers 660.
template <int BM, int BN, int WM, int WN, int DX, int DW>
__global__ __launch_bounds__(WM* WN* SIA_WAVE) void gemm_f32_tall_kernel(
    const u32x4* __restrict__ parts, const float* __restrict__ X, const float* __restrict__ W,
    float* __restrict__ Y, float* __restrict__ slices, int M, int N, int K, int Ns, int n_slices, bool apart, bool four,
    int tiles_m, int n_tiles, int per_die) {
    constexpr int WAVES = WM * WN, LOADERS = WAVES / 2, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int XT = BM / 16 * PARTS, WT = BN / 8;                   // KiB of a chunk
    constexpr int LX = (XT + LOADERS - 1) / LOADERS, LW = WT / LOADERS, LOADS = LX > LW ? LX : LW;      // loads of a wave
    static_assert(TM * WM * 16 == BM && TN * WN * 16 == BN && LW * LOADERS == WT, "tiles");
    static_assert(((DX + 1) * XT + (DW + 1) * WT) * LL_TILE <= LL_LDS && (DX - 1) * LX < 64 && (DW - 1) * LW < 64, "LDS, loads on their way");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    char* const x_ring = lds;
    char* const w_ring = lds + (DX + 1) * XT * LL_TILE;
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;      // as in gemm_f32_tile_kernel
    if (tile >= n_tiles) return;
    const int slice = apart ? (tile / tiles_m) % n_slices : 0;
    const int m0 = (tile % tiles_m) * BM, n0 = tile / tiles_m / (apart ? n_slices : 1) * BN;
    const int chunks = K / CHUNK, blocks = (M + 15) / 16;
    const int lane = threadIdx.x % SIA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SIA_WAVE);
    const int wm = wave % WM, wn = wave / WM, r = lane % 16, g = lane / 16;
    const int begin = apart ? slice_begin(chunks, slice, n_slices) : 0;
    const int steps = (apart ? slice_begin(chunks, slice + 1, n_slices) : chunks) - begin;

    const bool brings_x = wave < LOADERS;
    const int loader = brings_x ? wave : wave - LOADERS;
    const char* const from = brings_x ? (const char*)(parts + ((size_t)begin * blocks + m0 / 16) * PART_BLOCK)
                                      : (const char*)(W + (size_t)n0 * K + begin * CHUNK);
    const size_t step_bytes = brings_x ? (size_t)blocks * (PART_BLOCK * 16) : (size_t)CHUNK * 4;
    unsigned offset[LOADS];      // KiB of X beyond the tile or the last block repeat the last one, rows of W beyond the last that one (K is below 2^22)
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const int kib = min(loader * LX + l, min(XT, (blocks - m0 / 16) * PARTS) - 1), row = (loader * LW + min(l, LW - 1)) * 8 + lane / 8;
        offset[l] = brings_x ? (unsigned)(kib * SIA_WAVE + lane) * 16
                             : ((unsigned)(min(n0 + row, N - 1) - n0) * (unsigned)K + ((lane & 7) ^ turn(row & 15)) * 4) * 4;
    }
    auto request = [&](int s, int slot) {
        const char* at = from + s * step_bytes;
        if (brings_x) {
#pragma unroll
            for (int l = 0; l < LX; ++l) load_to_lds(at + offset[l], x_ring + (slot * XT + min(loader * LX + l, XT - 1)) * LL_TILE);
        } else {
#pragma unroll
            for (int l = 0; l < LW; ++l) load_to_lds(at + offset[l], w_ring + (slot * WT + loader * LW + l) * LL_TILE);
        }
    };
    f32x4 total[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) total[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < (brings_x ? DX : DW); ++s)
        if (s < steps) request(s, s);
    const int x_at = wm * TM * PARTS * LL_TILE + lane * 16, w_at = (wn * (BN / WN) + r) * 128;
    const int place[2] = {((2 * g) ^ turn(r)) * 16, ((2 * g + 1) ^ turn(r)) * 16};
    int x_slot = 0, w_slot = 0, s = 0;
    const char *xs, *ws;
    // chunk s has come for all waves, and all have read chunk s - 1, whose places are filled again
    auto arrive = [&]() {
        if (brings_x)
            wait_step<LX, DX - 1>(steps - 1 - s);
        else
            wait_step<LW, DW - 1>(steps - 1 - s);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (brings_x) {
            if (s + DX < steps) request(s + DX, x_slot == 0 ? DX : x_slot - 1);
        } else {
            if (s + DW < steps) request(s + DW, w_slot == 0 ? DW : w_slot - 1);
        }
        xs = x_ring + x_slot * XT * LL_TILE + x_at, ws = w_ring + w_slot * WT * LL_TILE + w_at;
        x_slot = x_slot == DX ? 0 : x_slot + 1;
        w_slot = w_slot == DW ? 0 : w_slot + 1;
    };
    auto read_w = [&](int j, u32x4& a, u32x4& b) {
        const char* at = ws + j * 2 * LL_TILE;
        a = *(const u32x4*)(at + place[0]), b = *(const u32x4*)(at + place[1]);
    };
    auto read_x = [&](int i, u32x4 (&x)[PARTS]) {
#pragma unroll
        for (int e = 0; e < PARTS; ++e) x[e] = *(const u32x4*)(xs + (i * PARTS + e) * LL_TILE);
    };
    u32x4 w[TN], x[2][PARTS];
    auto multiply = [&](int i, const u32x4 (&xi)[PARTS]) {      // (written out in the loop it spills)
        f32x4 large[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) large[j] = product(w[j], xi[0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int p = PARTS - 1; p > 0; --p)
#pragma unroll
            for (int j = 0; j < TN; ++j) small[i][j] = product(w[j], xi[p], small[i][j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) total[i][j] += large[j];
    };
    for (; s < steps; ++s) {      // while W has one part
        arrive();
        u32x4 wa[TN], wb[TN];
        read_x(0, x[0]);
#pragma unroll
        for (int j = 0; j < TN; ++j) read_w(j, wa[j], wb[j]);
        uint32_t bits = 0;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bits |= or_of(wa[j], wb[j]);
            w[j] = upper_halves(wa[j], wb[j]);
        }
        if (__any((bits & 0xffffu) != 0)) break;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (i + 1 < TM) read_x(i + 1, x[(i + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);      // no more reads ahead than this: they would take the registers of the sums
            multiply(i, x[i & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    while (s < steps) {      // chunk s has arrived
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            asm volatile("" ::: "memory");      // X's parts are read again, not kept
            u32x4 a, b, part[1][PARTS];
            read_w(j, a, b);
            if (any_rest(split8(a, b, part[0]))) mark_rests(a, b, part[0][PARTS - 1]);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                u32x4 xi[PARTS];
                read_x(i, xi);
                f32x4 t[1] = {total[i][j]}, q[1] = {small[i][j]};
                add_chunk(part, xi, true, t, q);
                total[i][j] = t[0], small[i][j] = q[0];
            }
        }
        if (++s < steps) arrive();
    }
    // total[i][j]: row 16 i + r of the wave's tile, columns 16 j + 4 g .. + 3
    int m_first = m0 + wm * (BM / WM) + r, n_first = n0 + wn * (BN / WN) + 4 * g;
    asm volatile("" : "+v"(m_first), "+v"(n_first));      // addresses made here, not in front of the loop and kept through it
    const int stride = apart ? Ns : N;
    float* const to = apart ? slices + (size_t)slice * M * Ns : Y;
    bool odd = false;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m_first + i * 16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n_first + j * 16;
            float* at = to + (size_t)m * stride + n;
            const f32x4 v = total[i][j] + small[i][j];
            if (four || apart) {
                if (n < N) *(f32x4*)at = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) at[e] = v[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) odd |= n + e < N && !finite(v[e]);
        }
    }
    if (apart || !__any(odd)) return;
    make_again<TM, TN>(X, W, Y, M, N, K, m_first, n_first);
}

// Y = the slices' sums added in order.  A wave has 16 rows and columns, as float_sums gives them, a workgroup 64 columns.
__global__ __launch_bounds__(256) void sum_slices_f32_kernel(const float* __restrict__ slices, const float* __restrict__ X,
                                                             const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int Ns,
                                                             int n_slices, bool four) {
    const int lane = threadIdx.x % SIA_WAVE, r = lane % 16, g = lane / 16;
    const int n0 = blockIdx.y * 64 + threadIdx.x / SIA_WAVE * 16, n = n0 + 4 * g;
    const long long m = (long long)blockIdx.x * 16 + r;
    if (n0 >= N) return;      // a wave leaves as a whole
    const bool live = m < M && n < N;
    const size_t elements = (size_t)M * Ns, i = live ? m * Ns + n : 0;
    f32x4 v = *(const f32x4*)(slices + i);
    for (int s = 1; s < n_slices; ++s) v += *(const f32x4*)(slices + s * elements + i);
    bool odd = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) odd |= live && n + e < N && !finite(v[e]);
    if (__any(odd)) {
        const f32x4 again = float_sums(X + (size_t)(m < M ? m : M - 1) * K, W + (size_t)min(n0 + r, N - 1) * K, K);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = finite(v[e]) ? v[e] : again[e];
    }
    if (!live) return;
    float* at = Y + (size_t)m * N + n;
    if (four)
        *(f32x4*)at = v;
    else
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) at[e] = v[e];
}

// The activation between the two products of a feed-forward: the slices' sums of gate and up added in order, silu(gate) * up, and its parts for the
// product that reads it.  A wave has the 16 rows and 32 columns of a block of parts; lane (r, g) eight columns of row r.  G: [slice][M][2 inter];
// again: sums that are not finite are made from X and W (where no slices are apart, the product has done that).
// Bound by its bytes: 303 rows of 8,192, two slices (40 MB in, 25 out) 12.8 us, where the sums took 11.4, the activation 7.0 and the parts 6.4, each
// a launch behind the other (the float32 step of 303 tokens, four layers, 1,694 -> 1,596).
__global__ __launch_bounds__(256) void sum_swiglu_split_kernel(const float* __restrict__ G, const float* __restrict__ X, const float* __restrict__ W,
                                                               float* __restrict__ act, u32x4* __restrict__ parts, int M, int inter, int K,
                                                               int n_slices, bool again, int blocks) {
    const int chunks = inter / CHUNK;
    const long long id = (long long)blockIdx.x * 4 + threadIdx.x / SIA_WAVE, b = id / chunks;
    const int lane = threadIdx.x % SIA_WAVE, r = lane % 16, g = lane / 16, c = (int)(id % chunks);
    if (b >= blocks) return;      // a wave leaves as a whole
    const long long m = b * 16 + r;
    const int k = c * CHUNK + 8 * g;
    const bool live = m < M;
    const size_t elements = (size_t)M * 2 * inter, at = (live ? m : 0) * 2 * inter + k;
    f32x4 v[2][2];      // gate and up, four columns each
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i / 2][i % 2] = *(const f32x4*)(G + at + i / 2 * inter + i % 2 * 4);
    for (int s = 1; s < n_slices; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i / 2][i % 2] += *(const f32x4*)(G + s * elements + at + i / 2 * inter + i % 2 * 4);
    if (again) {
        bool odd = false;
#pragma unroll
        for (int i = 0; i < 16; ++i) odd |= live && !finite(v[i / 8][i / 4 % 2][i % 4]);
        if (__any(odd)) {
            const float* x = X + (size_t)(live ? m : M - 1) * K;
#pragma clang loop unroll(disable)
            for (int i = 0; i < 4; ++i) {      // place 4 g + e of float_sums is column 8 g + 4 (i % 2) + e
                const f32x4 sums = float_sums(x, W + ((size_t)i / 2 * inter + c * CHUNK + 8 * (r / 4) + 4 * (i % 2) + r % 4) * K, K);
#pragma unroll
                for (int j = 0; j < 4; ++j)      // (registers are not indexed)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (i == j && !finite(v[j / 2][j % 2][e])) v[j / 2][j % 2][e] = sums[e];
            }
        }
    }
    u32x4 a[2], p[PARTS];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float gate = v[0][e / 4][e % 4], up = v[1][e / 4][e % 4], y = gate / (1.f + expf(-gate)) * up;
        a[e / 4][e % 4] = live ? __float_as_uint(y) : 0u;
    }
    if (live) {
        u32x4* out = (u32x4*)(act + m * inter + k);
        out[0] = a[0], out[1] = a[1];
    }
    if (split8(a[0], a[1], p) & 0xffffu) mark_rests(a[0], a[1], p[PARTS - 1]);
    u32x4* to = parts + ((long long)c * blocks + b) * PART_BLOCK + lane;
#pragma unroll
    for (int e = 0; e < PARTS; ++e) to[e * SIA_WAVE] = p[e];
}

// ---------------------------------------------------------------------------------------------------------
// which kernel
// ---------------------------------------------------------------------------------------------------------

// The shapes, how many workgroups of each a compute unit holds at a time, and what a product costs in microseconds, with all of K a
// workgroup or its slices apart: a launch, a round of workgroups over the device, a chunk of a round, what each workgroup on a unit
// adds to that, a MB of the slices' sums written and read (through Y, for tiles of 256 columns).  By least squares over the geometric mean
// of weights of 8 and 24 bits, 2,900 products of 256 to 128,256 columns, k of 256 to 8,192, 17 to 1,024 rows:  median error 2 to 4 %; the choice
// is 2.2 % above the best of seven shapes on average, 11 % in one of twenty.  The tall ones (gemm_f32_tall_kernel) by 695 products of the same sizes and of
// columns to 40,000 (median error 2 to 3 %, one of twenty 10 %; for them only where they are clearly the shorter, see f32_plan), from 65 rows on (fewer not
// measured).
struct F32Cost {
    double launch, round, step, more, sums;
};
struct F32Shape {
    int bm, bn, at_a_time;
    F32Cost whole, apart;
};
constexpr F32Cost NEVER = {1e30, 0, 0, 0, 0};
static const F32Shape F32_SHAPES[] = {{96, 256, 1, {22.6, 13.1, 1.68, 0, 0.109}, {13.3, -2.4, 1.78, 0, 0.287}},
                                      {64, 128, 2, {5.0, 3.2, 0.657, 0.372, 0}, {13.6, -3.9, 0.742, 0.319, 0.305}},
                                      {64, 128, 1, {4.4, 3.2, 0.859, 0, 0}, {11.0, -1.7, 0.891, 0, 0.346}},
                                      {32, 64, 3, {6.8, -0.5, 0.428, 0.127, 0}, NEVER},
                                      {128, 128, 1, {-0.6, 10.1, 1.241, 0, 0}, {12.6, -2.8, 1.282, 0, 0.338}},
                                      {160, 128, 1, {0.8, 5.7, 1.534, 0, 0}, {10.9, 0.8, 1.606, 0, 0.186}},
                                      {160, 192, 1, {5.2, 6.4, 1.978, 0, 0}, {11.7, 1.0, 2.042, 0, 0.175}}};
constexpr int N_F32_SHAPES = sizeof(F32_SHAPES) / sizeof(F32_SHAPES[0]), FIRST_TALL = 5;

struct F32Plan {
    int shape;      // -1: the few-row kernel
    bool apart;
    long long parts, slices;      // bytes of the workspace
};

static bool wide_rows(const float* rows, int K) { return K % 4 == 0 && ((uintptr_t)rows & 15) == 0; }

// wide_x, wide_w: wide_rows of either.  has_parts: the tiles find X's parts made.
static F32Plan f32_plan(int M, int N, int K, bool wide_x, bool wide_w, bool has_parts = false) {
    F32Plan best{-1, false, 0, 0};
    const int cus = compute_units(), n_slices = slices_of(N, K), chunks = (K + CHUNK - 1) / CHUNK;
    if (M <= 16 || K >= 1 << 22) return best;
    // the few-row kernel: what its workgroups fetch (their rows of W and X, from L2 for the most part), or W from memory.
    // Float by float 1.2 to 2 times as long.
    const FewRows few = few_rows_shape(M, N, K);
    const int rows_w = few.nb * 16, rows_x = few.mb * 16;
    const double fetched = (double)((M + rows_x - 1) / rows_x) * ((N + rows_w - 1) / rows_w) * (rows_w + rows_x) * K * 4e-6;
    double least = (few.launch + fmax(fetched / few.rate, (double)N * K * 4e-6 / 5.4)) * (wide_x && wide_w ? 1 : 1.6);
    double others = least;      // the estimate without the tall shapes
    bool two_a_unit = false;
    for (int i = 0; i < N_F32_SHAPES; ++i) {
        const F32Shape& t = F32_SHAPES[i];
        const bool tall = i >= FIRST_TALL;
        if (t.bn == 256 && !wide_w) continue;      // four times the loads' addresses would spill
        if (tall && (!wide_w || K % CHUNK || M <= 64)) continue;
        const long long tiles = (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        for (int apart = tall && n_slices > 1; apart <= (n_slices > 1); ++apart) {      // (a tall one has one slice)
            const F32Cost& c = apart ? t.apart : t.whole;
            const long long workgroups = tiles * (apart ? n_slices : 1), room = (long long)cus * t.at_a_time;
            if (workgroups > 1 << 30 || (apart && (long long)n_slices * M * N > 1LL << 27)) continue;
            const int steps = apart ? (chunks + n_slices - 1) / n_slices : chunks;
            const double full = (double)(workgroups / room), last = (double)((workgroups % room + cus - 1) / cus);      // of `last` workgroups a unit
            double us = c.launch + (full + (last > 0)) * (c.round + c.step * steps) + (full * t.at_a_time + last) * c.more * steps;
            if (apart) us += c.sums * n_slices * M * N * 8e-6;
            else us += c.sums * (n_slices - 1) * M * N * 8e-6;
            // A tall shape's estimate has to be less than others' by what these err: 9 % where two workgroups of 64 x 128 share a unit, else 4 %; it takes
            // no product from the few-row kernel.  (Of 1,560 products of 65 to 4,096 rows that it was estimated the shorter for, 246 took more
            // than 3 % longer with it, up to 24 %;  so it takes 1,247, of which 41 do, and leaves 42 that it has 3 % and more to give.)
            if (tall && ((best.shape < 0 && !has_parts) || us >= (two_a_unit ? 0.91 : 0.96) * others)) continue;
            if (us >= least) continue;
            least = us;
            if (!tall) others = us, two_a_unit = i == 1 && !apart;
            best.shape = i, best.apart = apart;
        }
    }
    if (best.shape < 0) return best;
    best.parts = (long long)((M + 15) / 16) * chunks * PART_BLOCK * 16;
    best.slices = best.apart ? (long long)n_slices * M * ((N + 3) / 4 * 4) * 4 : 0;
    return best;
}

// More LDS than a kernel gets unasked, allowed once per device.
static int allow_lds(const void* kernel, int bytes, bool (&set)[64]) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return (int)hipGetLastError();
    if (device >= 0 && device < 64 && set[device]) return 0;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && device >= 0 && device < 64) set[device] = true;
    return (int)e;
}

template <int BM, int BN, int WM, int WN, int D, bool SLICED, bool WIDE>
static int launch_f32_shape(const float* X, const float* W, float* Y, u32x4* parts, float* slices, int M, int N, int K,
                            bool apart, bool four, hipStream_t stream) {
    constexpr int bytes = (D + 1) * (BM / 16 * PARTS + BN / 8) * LL_TILE;
    const int n_slices = slices_of(N, K), tiles_m = (M + BM - 1) / BM;
    const int n_tiles = tiles_m * ((N + BN - 1) / BN) * (apart ? n_slices : 1), per_die = (n_tiles + 7) / 8;
    const auto kernel = gemm_f32_tile_kernel<BM, BN, WM, WN, D, SLICED, WIDE>;
    static bool set[64];
    const int status = allow_lds((const void*)kernel, bytes, set);
    if (status) return status;
    hipLaunchKernelGGL(kernel, dim3(8 * per_die), dim3(WM * WN * SIA_WAVE), bytes, stream, parts, X, W, Y, slices, M, N, K, (N + 3) / 4 * 4,
                       n_slices, apart, four, tiles_m, n_tiles, per_die);
    return SIA_LAUNCH_CHECK();
}

template <int BM, int BN, int WM, int WN, int D, bool WIDE>
static int launch_f32_tiles(const float* X, const float* W, float* Y, u32x4* parts, float* slices, int M, int N, int K, bool apart, bool four,
                            hipStream_t stream) {
    if (apart || slices_of(N, K) == 1 || BN == 256)      // (registers of the large ones are full)
        return launch_f32_shape<BM, BN, WM, WN, D, false, WIDE>(X, W, Y, parts, slices, M, N, K, apart, four, stream);
    return launch_f32_shape<BM, BN, WM, WN, D, BN != 256, WIDE>(X, W, Y, parts, slices, M, N, K, false, four, stream);
}

template <int BM, int BN, int DX, int DW>
static int launch_f32_tall(const float* X, const float* W, float* Y, u32x4* parts, float* slices, int M, int N, int K, bool apart, bool four,
                           hipStream_t stream) {
    constexpr int bytes = ((DX + 1) * (BM / 16 * PARTS) + (DW + 1) * (BN / 8)) * LL_TILE;
    const int n_slices = slices_of(N, K), tiles_m = (M + BM - 1) / BM;
    const int n_tiles = tiles_m * ((N + BN - 1) / BN) * (apart ? n_slices : 1), per_die = (n_tiles + 7) / 8;
    const auto kernel = gemm_f32_tall_kernel<BM, BN, 2, 4, DX, DW>;
    static bool set[64];
    const int status = allow_lds((const void*)kernel, bytes, set);
    if (status) return status;
    hipLaunchKernelGGL(kernel, dim3(8 * per_die), dim3(8 * SIA_WAVE), bytes, stream, parts, X, W, Y, slices, M, N, K, (N + 3) / 4 * 4, n_slices, apart,
                       four, tiles_m, n_tiles, per_die);
    return SIA_LAUNCH_CHECK();
}

static void split_rows(const float* X, u32x4* parts, int M, int K, bool wide_x, hipStream_t stream) {
    const int blocks = (M + 15) / 16, chunks = (K + CHUNK - 1) / CHUNK;
    hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)(((long long)blocks * chunks + 3) / 4)), dim3(256), 0, stream, X, parts, M, K, blocks, chunks,
                       wide_x);
}

static void sum_slices(const float* slices, const float* X, const float* W, float* Y, int M, int N, int K, bool four, hipStream_t stream) {
    hipLaunchKernelGGL(sum_slices_f32_kernel, dim3((M + 15) / 16, (N + 63) / 64), dim3(256), 0, stream, slices, X, W, Y, M, N, K, (N + 3) / 4 * 4,
                       slices_of(N, K), four);
}

// A product's tiles, from the parts of X: Y, or with plan.apart the slices' sums.
static int f32_tiles(const F32Plan& plan, const float* X, const float* W, float* Y, u32x4* parts, float* slices, int M, int N, int K, bool wide_w,
                     bool four, hipStream_t stream) {
    const bool apart = plan.apart;
    int status = SIA_BAD_ARGUMENT;
#define SHAPE(I, ...)         \
    if (plan.shape == I)     \
    status = wide_w ? launch_f32_tiles<__VA_ARGS__, true>(X, W, Y, parts, slices, M, N, K, apart, four, stream)      \
                    : launch_f32_tiles<__VA_ARGS__, false>(X, W, Y, parts, slices, M, N, K, apart, four, stream)
    if (plan.shape == 0) status = launch_f32_tiles<96, 256, 2, 4, 2, true>(X, W, Y, parts, slices, M, N, K, apart, four, stream);
    SHAPE(1, 64, 128, 2, 2, 1);
    SHAPE(2, 64, 128, 2, 4, 2);
    SHAPE(3, 32, 64, 2, 2, 2);
    SHAPE(4, 128, 128, 2, 4, 2);
#undef SHAPE
    if (plan.shape == 5) status = launch_f32_tall<160, 128, 2, 3>(X, W, Y, parts, slices, M, N, K, apart, four, stream);
    if (plan.shape == 6) status = launch_f32_tall<160, 192, 1, 3>(X, W, Y, parts, slices, M, N, K, apart, four, stream);
    return status;
}

// The way that this product goes, for tests to tell which they reach: 2 * shape + apart of F32_SHAPES, or -(10 mb + nb) of the few-row kernel.
SIA_EXPORT int sia_gemm_f32_way(const float* X, const float* W, int M, int N, int K) {
    const F32Plan plan = f32_plan(M, N, K, wide_rows(X, K), wide_rows(W, K));
    const FewRows few = few_rows_shape(M, N, K);
    return plan.shape < 0 ? -(10 * few.mb + few.nb) : 2 * plan.shape + plan.apart;
}

// Bytes of workspace that this product wants (0: none).
SIA_EXPORT long long sia_gemm_f32_workspace(const float* X, const float* W, int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const F32Plan plan = f32_plan(M, N, K, wide_rows(X, K), wide_rows(W, K));
    return plan.shape < 0 ? 0 : plan.parts + plan.slices;
}

// With `workspace` (of sia_gemm_f32_workspace bytes, on 16) the tiles where they are the faster way; without, the few-row kernel, whatever M
// is, with the same bits.
SIA_EXPORT int sia_gemm_f32(const float* X, const float* W, float* Y, void* workspace, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || ((uintptr_t)workspace & 15)) return SIA_BAD_ARGUMENT;
    const bool wide_x = wide_rows(X, K), wide_w = wide_rows(W, K), four = N % 4 == 0 && ((uintptr_t)Y & 15) == 0;
    const F32Plan plan = workspace ? f32_plan(M, N, K, wide_x, wide_w) : F32Plan{-1, false, 0, 0};
    if (plan.shape < 0) {
        constexpr int MOST = 65535 * 16;      // rows of a launch
        for (; M > MOST; M -= MOST, X += (size_t)MOST * K, Y += (size_t)MOST * N) few_rows(X, W, Y, MOST, N, K, wide_x && wide_w, stream);
        few_rows(X, W, Y, M, N, K, wide_x && wide_w, stream);
        return SIA_LAUNCH_CHECK();
    }
    u32x4* const parts = (u32x4*)workspace;
    float* const slices = (float*)((char*)workspace + plan.parts);
    split_rows(X, parts, M, K, wide_x, stream);
    const int status = f32_tiles(plan, X, W, Y, parts, slices, M, N, K, wide_w, four, stream);
    if (status == 0 && plan.apart) sum_slices(slices, X, W, Y, M, N, K, four, stream);
    return status ? status : SIA_LAUNCH_CHECK();
}

// Y[M, N] = (silu(X Wg^T) * (X Wu^T)) Wd^T, W = [Wg; Wu] of 2 inter rows of K, Wd [N, inter]: the same sums as the two products and the activation by
// themselves.  Where both products are the tiles', with one kernel between them, which makes the second one's parts; else the three one after the
// other, in one call too (the host takes longer for a step of few tokens than the GPU does).
// The workspace has two places, which the fused form uses twice each: `front` has X's parts, then the activation and its parts, `back` the first
// product's result or slices, then the second's slices.  In the other form they hold what a product needs and the activation, the first's result and what
// the second needs, beside one another.
extern "C" int sia_swiglu(const void* gu, void* out, int n_tokens, int inter, int dtype, hipStream_t stream);
struct FeedForwardPlan {
    F32Plan first, second;
    bool fused;
    long long act, front, back;      // bytes
};
static long long on_line(long long bytes) { return (bytes + 255) / 256 * 256; }
static FeedForwardPlan feed_forward_plan(const float* X, const float* W, const float* Wd, int M, int N, int K, int inter) {
    FeedForwardPlan p;
    const bool wide_x = wide_rows(X, K), wide_w = wide_rows(W, K), wide_d = wide_rows(Wd, inter), wide_act = inter % 4 == 0;
    p.first = f32_plan(M, 2 * inter, K, wide_x, wide_w);
    p.fused = p.first.shape >= 0 && inter % CHUNK == 0 && wide_x && wide_w && wide_d;
    p.second = f32_plan(M, N, inter, wide_act, wide_d, p.fused);
    if (p.fused && p.second.shape < 0) p.fused = false, p.second = f32_plan(M, N, inter, wide_act, wide_d);
    const long long gate_up = on_line((long long)M * 2 * inter * 4), first = on_line(p.first.parts + p.first.slices);
    const long long second = on_line(p.second.parts + p.second.slices);
    p.act = on_line((long long)M * inter * 4);
    if (p.fused) {
        p.front = std::max(on_line(p.first.parts), p.act + on_line(p.second.parts));
        p.back = std::max(p.first.apart ? on_line(p.first.slices) : gate_up, on_line(p.second.slices));
    } else {
        p.front = first + p.act;
        p.back = gate_up + second;
    }
    return p;
}
// Bytes of workspace; 0 where the three by themselves are to be called: with it and Y there would be 64 MiB more in use at a time than they have (from about
// 1,000 rows of 14,336 or 2,000 of 8,192 on, where the activation by itself is up to 7 % of the time:  4,096 rows of 8,192 1,774 us, in one 1,656, and 637 MB
// for 403).
SIA_EXPORT long long sia_f32_feed_forward_workspace(const float* X, const float* W, const float* Wd, int M, int N, int K, int inter) {
    if (M <= 0 || N <= 0 || K <= 0 || inter <= 0 || inter > 1 << 29) return 0;
    const FeedForwardPlan p = feed_forward_plan(X, W, Wd, M, N, K, inter);
    const long long y = (long long)M * N * 4, gate_up = (long long)M * 2 * inter * 4, act = gate_up / 2;
    const long long apart = std::max({p.first.parts + p.first.slices + gate_up, gate_up + act, act + p.second.parts + p.second.slices + y});
    return p.front + p.back + y > apart + (64LL << 20) ? 0 : p.front + p.back;
}
SIA_EXPORT int sia_f32_feed_forward(const float* X, const float* W, const float* Wd, float* Y, void* workspace, int M, int N, int K, int inter,
                                    hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || inter <= 0 || inter > 1 << 29 || !workspace || ((uintptr_t)workspace & 15)) return SIA_BAD_ARGUMENT;
    const FeedForwardPlan p = feed_forward_plan(X, W, Wd, M, N, K, inter);
    char* const front = (char*)workspace;
    char* const back = front + p.front;
    if (!p.fused) {
        float* const gate_up = (float*)back;
        float* const act = (float*)(front + p.front - p.act);
        char* const rest = back + on_line((long long)M * 2 * inter * 4);
        int status = sia_gemm_f32(X, W, gate_up, p.first.shape >= 0 ? front : nullptr, M, 2 * inter, K, stream);
        if (!status) status = sia_swiglu(gate_up, act, M, inter, SIA_F32, stream);
        if (!status) status = sia_gemm_f32(act, Wd, Y, p.second.shape >= 0 ? rest : nullptr, M, N, inter, stream);
        return status;
    }
    float* const act = (float*)front;
    u32x4* const parts = (u32x4*)front;
    float* const between = (float*)back;
    u32x4* const act_parts = (u32x4*)(front + p.act);
    float* const slices = (float*)back;
    const bool four = N % 4 == 0 && ((uintptr_t)Y & 15) == 0;
    split_rows(X, parts, M, K, true, stream);
    int status = f32_tiles(p.first, X, W, between, parts, between, M, 2 * inter, K, true, true, stream);
    if (status) return status;
    const int blocks = (M + 15) / 16;
    hipLaunchKernelGGL(sum_swiglu_split_kernel, dim3((unsigned)(((long long)blocks * (inter / CHUNK) + 3) / 4)), dim3(256), 0, stream, between, X, W, act,
                       act_parts, M, inter, K, p.first.apart ? slices_of(2 * inter, K) : 1, p.first.apart, blocks);
    status = f32_tiles(p.second, act, Wd, Y, act_parts, slices, M, N, inter, true, four, stream);
    if (status == 0 && p.second.apart) sum_slices(slices, act, Wd, Y, M, N, inter, four, stream);
    return status ? status : SIA_LAUNCH_CHECK();
}
