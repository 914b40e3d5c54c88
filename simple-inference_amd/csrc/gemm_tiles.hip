// Y[M, N] = X[M, K] * W[N, K]^T in bfloat16 with float accumulation, for steps of some 21 to 1,024 rows: too many to walk along W
// with all of X beside it (gemm_skinny.hip), too few for tiles of whole k to fill the chip, which is where the BLAS library loses
// (3,072 x 8,192: 43 us at 128 rows and 59 at 192, where the weights' bytes take 8).
//
// A workgroup makes a tile of BM rows of X by BN rows of W over a slice of k: k is cut into `splits` slices where the tiles alone
// are fewer than the compute units, each slice's sums are left in float, and whoever reads the result adds the slices in their
// order and rounds once (sia_sum_slices, or the norm behind the product: sia_add_rmsnorm_slices).
//
// Both operands come straight to LDS, 128 bytes of eight rows an instruction (lds_load.h), half of the waves bringing X, half W: a
// wave's loads end in the order in which they were made, so X, which L2 holds, would wait for W from memory behind it; apart,
// W is asked for DW steps ahead and X DX, as deep as its latency wants.  One barrier a step: what is read next has come, what was
// read last may be overwritten.  A wave's tile is 32 to 64 rows each way, with the reads of a step's second half between the
// products of its first.
//
// Bound by what a compute unit fetches, 37 to 50 GB/s of it in every shape: so the tile and the splits are chosen for the least
// (rows of tile) * steps * rounds, the sums of the slices on top.  us, library -> now, the sum in a launch of its own included:
// 2,048 x 8,192 (96, 192, 512 rows) 21.5 -> 18.9, 27.3 -> 20.3, 35.2 -> 32.0;  3,072 x 8,192 (96, 128, 192, 512) 36.4 -> 21.6, 43.3 -> 23.1,
// 59.2 -> 25.8, 46.9 -> 41.0;  4,096 x 14,336 (96, 192, 512, 1,024) 64 -> 32, 106 -> 49, 92 -> 71, 139 -> 115;  5,120 x 3,072 (128, 192) 20.9 -> 18.9,
// 27.3 -> 19.9.  With SwiGLU inside, against library and activation kernel:  8,192 x 2,048 (96, 256, 512, 1,024) 23.0 -> 21.9, 34.8 -> 29.7,
// 44.6 -> 42.4, 75 -> 68;  8,192 x 3,072 (256, 1,024) 46.8 -> 40.2, 100 -> 95.
#include "lds_load.h"

// GLU: W = [gate; up] of N rows each, Y = silu(gate) * up of the sums rounded to bfloat16 (the bits of the product and the
// activation kernel behind it); a wave's columns are half gate, half up, of the same columns of Y, so that a lane holds both.
template <typename TOut, int BM, int BN, int WM, int WN, int DX, int DW, bool GLU>
__global__ __launch_bounds__(WM* WN* SIA_WAVE) void gemm_tiles_kernel(const bf16_t* __restrict__ X,
                                                                     const bf16_t* __restrict__ W, TOut* __restrict__ Y,
                                                                     float* __restrict__ slices, int M, int N, int K,
                                                                     int splits, int row_blocks, int pairs) {
    constexpr int WAVES = WM * WN, LOADERS = WAVES / 2;
    constexpr int LX = BM / 8 / LOADERS, LW = BN / 8 / LOADERS;   // loads of a step, by a wave
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16;           // a wave's tiles of 16 x 16
    constexpr int BNO = GLU ? BN / 2 : BN;                        // columns of Y
    static_assert(LX * 8 * LOADERS == BM && LW * 8 * LOADERS == BN && TM * 16 * WM == BM && TN * 16 * WN == BN, "tiles");
    static_assert(!GLU || TN % 2 == 0, "gate and up rows come in equal numbers");
    constexpr int X_STAGE = BM * LL_STEP * 2, W_STAGE = BN * LL_STEP * 2;
    static_assert((DX + 1) * X_STAGE + (DW + 1) * W_STAGE <= LL_LDS, "a workgroup's LDS");
    __shared__ __attribute__((aligned(1024))) char lds[(DX + 1) * X_STAGE + (DW + 1) * W_STAGE];
    char* const x_ring = lds;
    char* const w_ring = lds + (DX + 1) * X_STAGE;
    // workgroups go round the eight dies: the row blocks of a (column block, slice) pair share its rows of W on one die, one
    // after the other
    const int id = blockIdx.x;
    const int pair = (id / (8 * row_blocks)) * 8 + id % 8, row_block = (id / 8) % row_blocks;
    if (pair >= pairs) return;
    const int slice = pair % splits;
    const int m0 = row_block * BM, n0 = (pair / splits) * BNO;
    const int all = K / LL_STEP;
    const int begin = (int)((long long)all * slice / splits), steps = (int)((long long)all * (slice + 1) / splits) - begin;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SIA_WAVE);
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    // the row of W in row t of the tile; rows beyond the last repeat it
    auto w_row = [&](int t) {
        if (!GLU) return min(n0 + t, N - 1);
        const int of_wave = t / (BN / WN), in = t % (BN / WN), half = BN / WN / 2;
        return min(n0 + of_wave * half + in % half, N - 1) + (in / half) * N;
    };
    const bool brings_x = wave < LOADERS;
    const int loader = brings_x ? wave : wave - LOADERS;
    const char* const from = (const char*)(brings_x ? X : W) + (size_t)begin * LL_STEP * 2;
    constexpr int LOADS = LX > LW ? LX : LW;
    unsigned offset[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const int t = (loader * (brings_x ? LX : LW) + l) * 8 + lane / 8;
        const int row = brings_x ? min(m0 + t, M - 1) : w_row(min(t, BN - 1));
        offset[l] = ((unsigned)row * (unsigned)K + ((lane & 7) ^ turn(t & 15)) * 8) * 2;
    }
    auto request_x = [&](int s, int slot) {
#pragma unroll
        for (int l = 0; l < LX; ++l)
            load_to_lds(from + (size_t)s * LL_STEP * 2 + offset[l], x_ring + slot * X_STAGE + (loader * LX + l) * LL_TILE);
    };
    auto request_w = [&](int s, int slot) {
#pragma unroll
        for (int l = 0; l < LW; ++l)
            load_to_lds(from + (size_t)s * LL_STEP * 2 + offset[l], w_ring + slot * W_STAGE + (loader * LW + l) * LL_TILE);
    };
    if (brings_x) {
        for (int s = 0; s < DX; ++s)
            if (s < steps) request_x(s, s);
    } else {
        for (int s = 0; s < DW; ++s)
            if (s < steps) request_w(s, s);
    }
    const int wm = wave % WM, wn = wave / WM;
    floatx4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // half h of a step: 32 k, lane group g the eight from 8 g on, piece 4 h + g of the row
    const int at[2] = {r * 128 + (g ^ turn(r)) * 16, r * 128 + ((4 + g) ^ turn(r)) * 16};
    int x_slot = 0, w_slot = 0;
    for (int s = 0; s < steps; ++s) {
        if (brings_x)
            wait_step<LX, DX - 1>(steps - 1 - s);
        else
            wait_step<LW, DW - 1>(steps - 1 - s);
        // step s has come for all waves, and all have read step s - 1, whose slots are filled again
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (brings_x) {
            if (s + DX < steps) request_x(s + DX, x_slot == 0 ? DX : x_slot - 1);
        } else {
            if (s + DW < steps) request_w(s + DW, w_slot == 0 ? DW : w_slot - 1);
        }
        const char* xf = x_ring + x_slot * X_STAGE + wm * (BM / WM) * 128;
        const char* wf = w_ring + w_slot * W_STAGE + wn * (BN / WN) * 128;
        x_slot = x_slot == DX ? 0 : x_slot + 1;
        w_slot = w_slot == DW ? 0 : w_slot + 1;
        bf16x8 a[2][TN], b[2][TM];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j = 0; j < TM; ++j) b[h][j] = *(const bf16x8*)(xf + j * 2 * LL_TILE + at[h]);
#pragma unroll
            for (int i = 0; i < TN; ++i) a[h][i] = *(const bf16x8*)(wf + i * 2 * LL_TILE + at[h]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], b[h][j], acc[i][j], 0, 0, 0);
        // the first half's reads, then the second half's one by one between the first half's products
        constexpr int READS = TN + TM, PER_READ = TN * TM / READS > 0 ? TN * TM / READS : 1;
        __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
#pragma unroll
        for (int q = 0; q < READS; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, PER_READ, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * TN * TM - PER_READ * READS, 0);
    }
    // acc[i][j][e]: row m0 + .. + 16 j + r, column n0 + .. + 16 i + 4 g + e (N is a multiple of 4)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = m0 + wm * (BM / WM) + j * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < (GLU ? TN / 2 : TN); ++i) {
            const int n = n0 + wn * (BNO / WN) + i * 16 + g * 4;
            if (n >= N) continue;
            if constexpr (sizeof(TOut) == 4) {   // whole k in one slice
                *(floatx4*)(Y + (size_t)m * N + n) = acc[i][j];
                continue;
            }
            if (!GLU && splits > 1) {
                *(floatx4*)(slices + ((size_t)slice * M + m) * N + n) = acc[i][j];
                continue;
            }
            bf16_t out[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                out[e] = float_to_bf16(acc[i][j][e]);
                if (GLU) {
                    const float gate = bf16_to_float(out[e]), up = bf16_to_float(float_to_bf16(acc[TN / 2 + i][j][e]));
                    out[e] = float_to_bf16(gate / (1.f + expf(-gate)) * up);
                }
            }
            *(uint2*)(Y + (size_t)m * N + n) = *(const uint2*)out;
        }
    }
}

// Y = the slices' sum, in their order, rounded.  Four elements a thread.
__global__ __launch_bounds__(256) void sum_slices_kernel(const float4* __restrict__ slices, uint2* __restrict__ Y, int splits,
                                                         size_t pieces) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    float4 v = slices[i];
    for (int z = 1; z < splits; ++z) {
        const float4 u = slices[z * pieces + i];
        v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
    }
    const bf16_t out[4] = {float_to_bf16(v.x), float_to_bf16(v.y), float_to_bf16(v.z), float_to_bf16(v.w)};
    Y[i] = *(const uint2*)out;
}

// The shapes, and what a compute unit fetches in each (GB/s, as measured).
struct TileShape {
    int bm, bn, rate;
};
static const TileShape TILE_SHAPES[] = {{64, 64, 46}, {96, 64, 42}, {128, 64, 43}, {96, 128, 44}, {128, 128, 50}, {128, 256, 42}, {256, 256, 37}};
constexpr int N_TILE_SHAPES = sizeof(TILE_SHAPES) / sizeof(TILE_SHAPES[0]);

struct TilePlan {
    int shape, splits, workgroups;
    double us;
};

// The shape and the splits that cost least: a launch 1 us; in rounds over the compute units a workgroup's start and end 3 us and
// its steps at its shape's rate; the slices' sum 3 us and its bytes, written and read, at 3.4 TB/s.  At least four steps a
// slice, sixteen slices of 64 MB together at most.
static TilePlan tile_plan(int M, int N, int K, bool glu) {
    const int cus = compute_units(), steps = K / LL_STEP;
    TilePlan best{-1, 1, 0, 0.0};
    for (int i = 0; i < N_TILE_SHAPES; ++i) {
        const TileShape t = TILE_SHAPES[i];
        const int columns = glu ? t.bn / 2 : t.bn;
        const long long row_blocks = (M + t.bm - 1) / t.bm, column_blocks = (N + columns - 1) / columns;
        for (int splits = 1; splits <= (glu ? 1 : 16) && (splits == 1 || (steps / splits >= 4 && (double)splits * M * N <= 1 << 24)); ++splits) {
            // a (column block, slice) pair has its row blocks on one die (of eight, dealt in turn): a die's own rounds count
            const long long workgroups = row_blocks * column_blocks * splits, die = (column_blocks * splits + 7) / 8 * row_blocks;
            const long long rounds = (8 * die + cus - 1) / cus;
            double us = 1.0 + (double)rounds * 3.0 + (double)rounds * ((steps + splits - 1) / splits) * (t.bm + t.bn) * LL_STEP * 2 / (t.rate * 1e3);
            if (splits > 1) us += 3.0 + (double)splits * M * N * 4 / 3.4e6;
            if (best.shape < 0 || us < best.us) best = TilePlan{i, splits, (int)(workgroups < 1 << 30 ? workgroups : 1 << 30), us};
        }
    }
    return best;
}

template <typename TOut, int BM, int BN, int WM, int WN, int DX, int DW, bool GLU>
static void launch_shape(const void* X, const void* W, void* Y, float* slices, int M, int N, int K, int splits, hipStream_t stream) {
    constexpr int COLUMNS = GLU ? BN / 2 : BN;
    const int row_blocks = (M + BM - 1) / BM, pairs = ((N + COLUMNS - 1) / COLUMNS) * splits;
    hipLaunchKernelGGL((gemm_tiles_kernel<TOut, BM, BN, WM, WN, DX, DW, GLU>), dim3((pairs + 7) / 8 * 8 * row_blocks),
                       dim3(WM * WN * SIA_WAVE), 0, stream, (const bf16_t*)X, (const bf16_t*)W, (TOut*)Y, slices, M, N, K,
                       splits, row_blocks, pairs);
}

template <bool GLU>
static int launch_tiles(const void* X, const void* W, void* Y, float* slices, int M, int N, int K, hipStream_t stream) {
    const TilePlan plan = tile_plan(M, N, K, GLU);
    if (plan.splits > 1 && !slices) return SIA_BAD_ARGUMENT;
#define SHAPE(I, ...) \
    if (plan.shape == I) launch_shape<bf16_t, __VA_ARGS__, GLU>(X, W, Y, slices, M, N, K, plan.splits, stream)
    SHAPE(0, 64, 64, 2, 2, 2, 4);
    SHAPE(1, 96, 64, 2, 2, 2, 4);
    SHAPE(2, 128, 64, 2, 2, 2, 3);
    SHAPE(3, 96, 128, 2, 2, 2, 5);
    SHAPE(4, 128, 128, 2, 4, 2, 5);
    SHAPE(5, 128, 256, 2, 4, 2, 2);
    SHAPE(6, 256, 256, 4, 4, 1, 1);
#undef SHAPE
    return SIA_LAUNCH_CHECK();
}

static bool tiles_can(int M, int N, int K) {
    return M > 0 && N > 0 && K > 0 && K % LL_STEP == 0 && N % 4 == 0 && M <= 65535 &&
           (long long)N * K < 1LL << 30 && (long long)M * K < 1LL << 30 && (long long)M * N < 1LL << 30;
}

// Whether a plain product of 21 to 1,024 rows goes to the tiles: long k over few columns (k at least twice the columns), where
// slices of k fill the chip, and other products of some size from 65 to 256 rows.  How large it has to be follows what else there
// is: up to 64 rows the few-row kernels are near for k up to 8,192; from 65 on the library is, and well ahead again at 8,192 columns
// up to some 160 rows (k of 2,048 to 4,096 and 8,192).  us, the better of few-row kernel and library / tiles with the sum of the slices in
// its own launch, of which the norm behind a block's last product saves 3:
//   at 32 rows 4,096 x 14,336 35 / 32, 3,072 x 14,336 29.9 / 25.5, 512 x 14,336 21.0 / 14.6, 64 to 768 x 65,536 0.36 to 0.46 of the
//   other;  4,096 x 9,216 23.6 / 22.4, at 24 22.0 / 24.4 (stays)
//   at 40 rows 2,048 x 8,192 14.4 / 14.7, 2,048 x 5,120 12.4 / 12.5;  1,024 x 8,192 12.5 / 13.3 (stays);  at 57 1,536 x 6,144 16.1 / 13.4
//   at 96 rows 3,072 x 8,192 36.7 / 21.9, 2,560 x 6,144 18.5 / 18.3, 1,024 x 9,216 17.3 / 16.3, 512 x 11,008 33 / 13.5;  512 x 9,216 at 80
//   11.1 / 12.3, 1,536 x 6,144 at 65 to 128 0.84 to 1.15 of the other, 2,048 x 4,096 at 256 16.3 / 20.7 (stay)
//   at 384 rows 1,024 x 8,192 24.8 / 19.4, 2,048 x 5,120 26.3 / 21.3;  1,024 x 5,120 at 512 0.99 to 1.16 of the other, 2,048 x 4,096 at 768
//   24.6 / 28.1 (stay)
//   others:  5,120 x 3,072 at 96 18.6 / 17.3, at 192 27.1 / 20.3;  8,192 x 14,336 at 128 87 / 61;  8,192 x 2,048 at 192 23.2 / 18.4, at 65
//   14.4 / 16.1 (stays);  8,192 x 8,192 at 65 36 / 44, 2,048 x 2,048 at 128 9.0 / 10.7, 12,288 x 3,072 25.9 / 29 (stay)
SIA_EXPORT int sia_gemm_tiles_takes(int M, int N, int K) {
    if (M <= 20 || M > 1024 || !tiles_can(M, N, K)) return 0;
    const long long size = (long long)N * K, MI = 1 << 20;
    if (K >= 2 * N) {
        if (M <= 32) return K > 12 * 1024 && size >= MI / 2;
        if (K > 10 * 1024 && size >= MI / 2) return 1;
        if (M <= 64) return size >= (M > 48 ? 7 : 9) * MI;
        if (M > 256) return K >= 5 * 1024 && size >= 6 * MI;
        return (size >= 12 * MI && (M > 80 || N >= 2048)) || (K >= 9 * 1024 && N >= 1024);
    }
    if (M <= 64 || M > 256 || size < 15 * MI) return 0;
    return N <= 6 * 1024 || (N <= 8 * 1024 && (M > 160 || K > 8 * 1024 || (M <= 128 && K > 4 * 1024 && K % (8 * 1024))));
}

// The same for the gated product: where its tiles come out in one round that fills at least 9/10 of the compute units with
// tiles at least 4/5 full, and the activation kernel is saved.  Their k is in one piece: a longer one pays from 129 to 256 rows
// alone, where the library is at its weakest and the plain tiles, which cut k, do not take the product.  (us, library and activation / tiles, of 8,192 x 2,048: 96 rows
// 22.7 / 21.8, 192 31.2 / 27.0, 256 34.4 / 28.6, 320 35.5 / 39.2 (three quarters of the units: stays), 1,024 72 / 67;  8,192 x 3,072: 256 46.6 / 39.3,
// 512 61.8 / 57.5, 640 66 / 81 (two rounds: stays);  14,336 x 4,096, 224 tiles: 256 74.6 / 82.2 (stays).  x 4,096, the better of
// library and tiles and the activation behind it / tiles with it inside: inter 5,120 at 256 0.79 of the other, 8,192 at 192 52.7 / 51.8;  2,560 at 192
// 26.6 / 27.4, 8,192 at 512 74 / 80, 1,024 at 512 25.1 / 26.4, 1,536 x 14,336 at 320 52 / 83, 2,560 x 14,336 at 192 62 / 87 (stay).)
SIA_EXPORT int sia_gemm_tiles_takes_swiglu(int M, int inter, int K) {
    if (M <= 64 || M > 1024 || !tiles_can(M, inter, K) || (long long)inter * K >= 1LL << 29) return 0;
    const TilePlan plan = tile_plan(M, inter, K, true);
    const long long cus = compute_units();
    const TileShape t = TILE_SHAPES[plan.shape];
    if (K > 3 * 1024 && (M <= 128 || M > 256 || (sia_gemm_tiles_takes(M, 2 * inter, K) && (inter < 4 * 1024 || K > 4 * 1024)))) return 0;
    return plan.workgroups <= cus && 10 * plan.workgroups >= 9 * cus && 5LL * M * 2 * inter >= 4 * cus * t.bm * t.bn;
}

// Slices that sia_gemm_tiles leaves of a product of this size (1: it writes Y).
SIA_EXPORT int sia_gemm_tiles_splits(int M, int N, int K) { return tiles_can(M, N, K) ? tile_plan(M, N, K, false).splits : 0; }

// Y[M, N] = X W^T (bfloat16), or, where sia_gemm_tiles_splits says more than 1, slices[splits][M][N] of floats whose sum it is.
SIA_EXPORT int sia_gemm_tiles(const void* X, const void* W, void* Y, float* slices, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!tiles_can(M, N, K) || !aligned16(X, W) || ((uintptr_t)Y & 7) || ((uintptr_t)slices & 15)) return SIA_BAD_ARGUMENT;
    return launch_tiles<false>(X, W, Y, slices, M, N, K, stream);
}

// An output head of more than 16 rows in float: W's rows are so many that whole tiles fill the chip many times over, and the
// workgroups' rings ask for W the deepest.  Rows of W a multiple of 4 KiB apart lie alike in the memory's channels, which tiles of
// one step's width feel the most: not those.  (us, the better of few-row kernels and library / tiles, of 128,256 x 3,072: 17 rows
// 150 / 141, 27 154 / 145, 33 166 / 148, 64 182 / 159, 65 188 / 158, 128 200 / 177;  x 2,048: 27 rows 108 / 116, 64 127 / 127, 128 142 / 149;
// x 4,096: 201 / 231, 218 / 243, 245 / 257.)
SIA_EXPORT int sia_gemm_tiles_takes_head(int M, int N, int K) {
    return M > 16 && M <= 128 && N >= 32 * 1024 && K % 2048 != 0 && tiles_can(M, N, K);
}

// Y[M, N] = X W^T in float.  Needs M <= 128.
SIA_EXPORT int sia_gemm_tiles_head(const void* X, const void* W, float* Y, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 128 || !tiles_can(M, N, K) || !aligned16(X, W) || ((uintptr_t)Y & 15)) return SIA_BAD_ARGUMENT;
    if (M <= 32)
        launch_shape<float, 32, 128, 1, 4, 2, 3, false>(X, W, Y, nullptr, M, N, K, 1, stream);
    else if (M <= 64)
        launch_shape<float, 64, 128, 2, 2, 1, 3, false>(X, W, Y, nullptr, M, N, K, 1, stream);
    else
        launch_shape<float, 128, 256, 2, 4, 2, 2, false>(X, W, Y, nullptr, M, N, K, 1, stream);
    return SIA_LAUNCH_CHECK();
}

// Y = the sum of `splits` slices of n floats each (n a multiple of 4), rounded to bfloat16.
SIA_EXPORT int sia_sum_slices(const float* slices, void* Y, int splits, long long n, hipStream_t stream) {
    if (n <= 0) return 0;
    if (splits < 1 || n % 4 || !slices || !Y || ((uintptr_t)Y & 7) || ((uintptr_t)slices & 15)) return SIA_BAD_ARGUMENT;
    hipLaunchKernelGGL(sum_slices_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, stream, (const float4*)slices,
                       (uint2*)Y, splits, (size_t)(n / 4));
    return SIA_LAUNCH_CHECK();
}

// Y[M, inter] = silu(X Wg^T) * (X Wu^T) for W = [Wg; Wu] of 2 inter rows.
SIA_EXPORT int sia_gemm_tiles_swiglu(const void* X, const void* W, void* Y, int M, int inter, int K, hipStream_t stream) {
    if (M <= 0 || inter <= 0) return 0;
    if (!tiles_can(M, inter, K) || (long long)inter * K >= 1LL << 29 || !aligned16(X, W) || ((uintptr_t)Y & 7)) return SIA_BAD_ARGUMENT;
    return launch_tiles<true>(X, W, Y, nullptr, M, inter, K, stream);
}
