// Y[M, N] = X[M, K] * W[N, K]^T in float on the matrix cores: the product of the 32-bit path.
//
// v_mfma_f32_16x16x4_f32 multiplies and adds floats as they are (no reduced-precision mode): 157 TFLOP/s where the
// vector units give the plain kernel 24.
//
// One order of sums for every shape, whatever M is, so that a row's result does not depend on the other rows of a
// batch or on which kernel below runs:  K is cut into steps of 64; a step's four pieces of 16 go to four sums
// s0 .. s3, piece by piece in order; within a piece instruction i = 0 .. 3 adds the k = 4 q + i of q = 0 .. 3 at once.
// The result is (s0 + s1) + (s2 + s3).  Shorter chains than k after k: the error against 64 bits is smaller.
//
// * Up to 16 rows: a workgroup owns 16 rows of W; its four waves take a sum each and stream W past the step's rows,
//   eight to sixteen steps of loads in flight a wave.  Bound by reading W.
// * More rows: tiles of Y.  A workgroup has the waves of a tile four times, once per sum; X and W are staged through
//   LDS in steps of 64 k.  Bound by the matrix cores.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SUMS 4            // sums a result is made of
#define PIECE 16          // consecutive k of a sum
#define STEP (SUMS * PIECE)

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 sum_of_piece(f32x4 w, f32x4 x, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = mfma4(w[i], x[i], c);
    return c;
}

// Four consecutive floats at p, a row's floats from k on (p points at float k).  ALIGNED: K is a multiple of four and the
// rows start on 16 bytes, so that the four lie inside or outside the row together; outside, the row's last four are read,
// without a branch, for in_row() to turn into zeros where they are used (not here: a use is a wait for the load).
template <bool ALIGNED>
__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, int k, int K) {
    if (ALIGNED) return *(const f32x4*)(p + min(0, K - 4 - k));
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (k + i < K) v[i] = p[i];
    return v;
}

__device__ __forceinline__ f32x4 in_row(f32x4 v, int k, int K) { return k < K ? v : f32x4{0.f, 0.f, 0.f, 0.f}; }

// The four results of a lane: row `m` of Y, columns n .. n + 3.
__device__ __forceinline__ void store4(float* __restrict__ Y, int m, int n, int M, int N, bool whole, f32x4 v) {
    if (m >= M) return;
    float* at = Y + (size_t)m * N + n;
    if (whole && n + 3 < N) {
        *(f32x4*)at = v;
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < N) at[i] = v[i];
}

// ---------------------------------------------------------------------------------------------------------
// few rows
// ---------------------------------------------------------------------------------------------------------

#define FLIGHT 8   // steps of loads that a wave has issued before it multiplies the eight in front of them

template <bool ALIGNED>
__global__ __launch_bounds__(256) void gemm_f32_few_rows_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                                float* __restrict__ Y, int M, int N, int K, bool whole) {
    __shared__ f32x4 part[SUMS / 2][SIA_WAVE];
    const int lane = threadIdx.x % SIA_WAVE, sum = threadIdx.x / SIA_WAVE;
    const int r = lane % 16, q = lane / 16;
    const int n0 = blockIdx.x * 16;
    const int steps = (K + STEP - 1) / STEP;
    const int k0 = sum * PIECE + 4 * q;
    // rows that do not exist are read as the last one and not stored
    const float* w_row = W + (size_t)min(n0 + r, N - 1) * K + k0;
    const float* x_row = X + (size_t)min(r, M - 1) * K + k0;

    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, w[2][FLIGHT], x[2][FLIGHT];
    auto fetch = [&](int set, int s0) {
#pragma unroll
        for (int s = 0; s < FLIGHT; ++s) {
            const int at = (s0 + s) * STEP;
            w[set][s] = load4<ALIGNED>(w_row + at, k0 + at, K);
            x[set][s] = load4<ALIGNED>(x_row + at, k0 + at, K);
        }
    };
    auto multiply = [&](int set, int s0) {
#pragma unroll
        for (int s = 0; s < FLIGHT; ++s) {
            const int k = k0 + (s0 + s) * STEP;
            acc = sum_of_piece(in_row(w[set][s], k, K), in_row(x[set][s], k, K), acc);
        }
    };
    fetch(0, 0);
    for (int s0 = 0; s0 < steps; s0 += 2 * FLIGHT) {     // steps past the end add zero times zero
        fetch(1, s0 + FLIGHT);
        multiply(0, s0);
        if (s0 + 2 * FLIGHT < steps) fetch(0, s0 + 2 * FLIGHT);
        multiply(1, s0 + FLIGHT);
    }
    // (s0 + s1) + (s2 + s3)
    if (sum & 1) part[sum / 2][lane] = acc;
    __syncthreads();
    if (!(sum & 1)) acc += part[sum / 2][lane];
    if (sum == 2) part[1][lane] = acc;      // its own half of the memory, which it has just read
    __syncthreads();
    if (sum == 0) store4(Y, r, n0 + 4 * q, M, N, whole, acc + part[1][lane]);
}

// ---------------------------------------------------------------------------------------------------------
// tiles
// ---------------------------------------------------------------------------------------------------------

#define STAGES 3

// A tile of BM rows of X by BN rows of W, taken by waves of WM by WN, four times over (once per sum).
template <int BM, int BN, int WM, int WN, bool ALIGNED>
__global__ __launch_bounds__(SUMS * (BM / WM) * (BN / WN) * SIA_WAVE) void gemm_f32_tile_kernel(
    const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int tiles_m,
    int n_tiles, int per_die, bool whole) {
    constexpr int WAVES = (BM / WM) * (BN / WN), THREADS = SUMS * WAVES * SIA_WAVE;
    constexpr int TM = WM / 16, TN = WN / 16;
    constexpr int ROWS = BM + BN, PIECES = ROWS * (STEP / 4), LOADS = (PIECES + THREADS - 1) / THREADS;
    constexpr int STAGE = ROWS * STEP;
    static_assert(STAGES * STAGE >= 2 * BM * BN, "the partial sums are added in the stages' memory");
    extern __shared__ float lds[];

    // Workgroups go to the dies in turn: a die gets consecutive tiles, row tiles of X innermost, so that the rows of W
    // that they share are read by one die.
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (tile >= n_tiles) return;
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;

    const int tid = threadIdx.x, lane = tid % SIA_WAVE, wave = tid / SIA_WAVE;
    const int sum = wave / WAVES, wm = (wave % WAVES) % (BM / WM), wn = (wave % WAVES) / (BM / WM);
    const int r = lane % 16, q = lane / 16;
    const int steps = (K + STEP - 1) / STEP;

    // The loads of a step are issued two steps before they are put into LDS: a step is shorter than the way from memory.
    const float* from[LOADS];
    int k_of[LOADS];
    f32x4 next[2][LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {     // rows that do not exist are read as the last one and not stored
        const int piece = tid + i * THREADS, row = min(piece / (STEP / 4), ROWS - 1);
        k_of[i] = (piece % (STEP / 4)) * 4;
        from[i] = (row < BM ? X + (size_t)min(m0 + row, M - 1) * K : W + (size_t)min(n0 + row - BM, N - 1) * K) + k_of[i];
    }
    auto fetch = [&](int set, int s) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) next[set][i] = load4<ALIGNED>(from[i] + s * STEP, k_of[i] + s * STEP, K);
    };
    // Sixteen pieces of four floats are a row of a stage; piece p of row r lies at place p ^ (r % 16).
    auto put = [&](int set, int s, float* stage) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int piece = tid + i * THREADS, row = piece / (STEP / 4), at = ((piece % (STEP / 4)) ^ (row % 16)) * 4;
            if (PIECES % THREADS == 0 || row < ROWS)
                *(f32x4*)(stage + row * STEP + at) = in_row(next[set][i], k_of[i] + s * STEP, K);
        }
    };

    f32x4 acc[TM][TN], x[2][TM], w[2][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int place = ((sum * 4 + q) ^ r) * 4;
    const int x_at = (wm * WM + r) * STEP + place, w_at = (BM + wn * WN + r) * STEP + place;
    auto read = [&](int set, const float* stage) {
#pragma unroll
        for (int i = 0; i < TM; ++i) x[set][i] = *(const f32x4*)(stage + x_at + i * 16 * STEP);
#pragma unroll
        for (int j = 0; j < TN; ++j) w[set][j] = *(const f32x4*)(stage + w_at + j * 16 * STEP);
    };
    // A step multiplies what lies in registers while the next step's operands are read from LDS, the step after it is
    // written there and the one two further on is on its way from memory.  A wave issues in order, and the waves of a
    // workgroup pass every barrier together: LDS and matrix cores work at the same time only if each wave's own
    // instructions alternate, so the schedule is written down.  Steps past the end move zeros: no branches.
    constexpr int OTHERS = TM + TN + 2 * LOADS, EACH = (4 * TM * TN) / OTHERS > 0 ? (4 * TM * TN) / OTHERS : 1;
    int now = 0;      // s % STAGES
    auto step = [&](int s, int parity) {      // parity: s % 2, known where the loop is unrolled
        const int after = now + 1 == STAGES ? 0 : now + 1, third = after + 1 == STAGES ? 0 : after + 1;
        read(parity ^ 1, lds + after * STAGE);
        put(parity, s + 2, lds + third * STAGE);     // read last in the step before the one before
        fetch(parity, s + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = mfma4(w[parity][j][e], x[parity][i][e], acc[i][j]);
#pragma unroll
        for (int i = 0; i < TM + TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);    // products
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // a read from LDS
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);       // a write to LDS
            __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);       // a load
        }
        __builtin_amdgcn_sched_barrier(0);      // the products stay in front of the barrier
        __syncthreads();
        now = after;
    };
    fetch(0, 0);
    fetch(1, 1);
    put(0, 0, lds);
    fetch(0, 2);
    put(1, 1, lds + STAGE);
    fetch(1, 3);
    __syncthreads();
    read(0, lds);
    for (int s = 0; s < steps; s += 2) {
        step(s, 0);
        step(s + 1, 1);
    }

    // (s0 + s1) + (s2 + s3), through the memory of the stages
    f32x4* part = (f32x4*)lds + (size_t)(sum / 2) * (BM * BN / 4) + (wm + wn * (BM / WM)) * (TM * TN * SIA_WAVE) + lane;
    if (sum & 1)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) part[(i * TN + j) * SIA_WAVE] = acc[i][j];
    __syncthreads();
    if (!(sum & 1))
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += part[(i * TN + j) * SIA_WAVE];
    if (sum == 2)      // its own half of the memory, which it has just read
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) part[(i * TN + j) * SIA_WAVE] = acc[i][j];
    __syncthreads();
    if (sum == 0) {
        const f32x4* other = part + BM * BN / 4;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                store4(Y, m0 + wm * WM + i * 16 + r, n0 + wn * WN + j * 16 + 4 * q, M, N, whole,
                       acc[i][j] + other[(i * TN + j) * SIA_WAVE]);
    }
}

template <int BM, int BN, int WM, int WN>
static int launch_tiles(const float* X, const float* W, float* Y, int M, int N, int K, bool aligned, bool whole, hipStream_t stream) {
    constexpr int threads = SUMS * (BM / WM) * (BN / WN) * SIA_WAVE, bytes = STAGES * (BM + BN) * STEP * (int)sizeof(float);
    const int tiles_m = (M + BM - 1) / BM;
    const long long tiles = (long long)tiles_m * ((N + BN - 1) / BN);
    if (tiles > (1 << 30)) return SIA_BAD_ARGUMENT;
    const int per_die = (int)((tiles + 7) / 8);
    auto kernel = aligned ? gemm_f32_tile_kernel<BM, BN, WM, WN, true> : gemm_f32_tile_kernel<BM, BN, WM, WN, false>;
    static bool set[64][2] = {};      // more LDS than a kernel gets unasked, allowed once per device
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return (int)hipGetLastError();
    if (device < 0 || device >= 64 || !set[device][aligned]) {
        const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return (int)e;
        if (device >= 0 && device < 64) set[device][aligned] = true;
    }
    hipLaunchKernelGGL(kernel, dim3(8 * per_die), dim3(threads), bytes, stream, X, W, Y, M, N, K, tiles_m, (int)tiles, per_die, whole);
    return SIA_LAUNCH_CHECK();
}

// Which kernel: the time of a step of 64 k in microseconds (measured on 256 compute units with operands that come from
// memory; the matrix cores alone would take 0.23, 0.91 and 1.81 for the last three) times the rounds over the device.  The
// two small tiles share a compute unit and need no whole rounds.
//   303 rows x 16384 x 2048:  64x64 211 us (96 TFLOP/s), 64x128 221, 32x32 258;    x 2048 x 8192:  32x32 138, 64x64 153;
//   303 x 128256 x 2048:  64x128 1467 us (109 TFLOP/s), 64x64 1620, 32x32 1808;   24 x 2048 x 8192:  32x16 47, 32x32 58
// where one 4 by 4 block of outputs a thread on the vector units took 596, 904, 5088 and 800.
// 16 rows and fewer: 2048 x 8192 27 us at one row (2.5 TB/s), 34 at 8; 16384 x 2048 30 (4.5 TB/s); 128256 x 2048 209 (5.0).
extern "C" int sia_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K, hipStream_t stream) {
    const bool aligned = K % 4 == 0 && ((uintptr_t)X | (uintptr_t)W) % 16 == 0;
    const bool whole = N % 4 == 0 && (uintptr_t)Y % 16 == 0;
    if (M <= 16) {
        auto kernel = aligned ? gemm_f32_few_rows_kernel<true> : gemm_f32_few_rows_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3((N + 15) / 16), dim3(256), 0, stream, X, W, Y, M, N, K, whole);
        return SIA_LAUNCH_CHECK();
    }
    auto rounds = [&](int bm, int bn) { return (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn) / 256; };
    const double shared[2] = {0.37 * fmax(1.0, rounds(32, 16)), 0.44 * fmax(1.0, rounds(32, 32))};
    const double alone[2] = {1.17 * ceil(rounds(64, 64)), 2.15 * ceil(rounds(64, 128))};
    const double best = fmin(fmin(shared[0], shared[1]), fmin(alone[0], alone[1]));
    if (best == alone[1]) return launch_tiles<64, 128, 64, 64>(X, W, Y, M, N, K, aligned, whole, stream);
    if (best == alone[0]) return launch_tiles<64, 64, 32, 64>(X, W, Y, M, N, K, aligned, whole, stream);
    if (best == shared[1]) return launch_tiles<32, 32, 32, 16>(X, W, Y, M, N, K, aligned, whole, stream);
    return launch_tiles<32, 16, 32, 16>(X, W, Y, M, N, K, aligned, whole, stream);
}
