// Y[M, N] = X[M, K] * W[N, K]^T in bfloat16 with float accumulation, for few rows (M <= 64): the matrix products of a
// decode step and of a short prompt, where every weight is read once and the time is the time to stream W from HBM.
//
// One workgroup of 4 or 8 waves per RB blocks of up to 16 rows of W.  K is cut into chunks of 128, and chunk c
// belongs to *share* c % 16: a share's chunks are summed front to back into one accumulator, and the 16 shares'
// sums are added as (s0 + s8) + (s1 + s9) + ... + (s7 + s15), left to right.  Wave w has the shares w, w + WAVES, ...,
// one accumulator each, and the workgroup walks its rows front to back.  A wave's step covers 64 k of its blocks with
// MFMAs 16x16x32:
//   A = W[row of lane r in block rb][k0 + 16g .. + 15],   B = X[r of block mb][same k]
// (an MFMA's k index only has to mean the same element in A and B, so lane group g may take the 16
// consecutive k that start at 16g and feed them to two MFMAs.)
//
// A step's rows of W and X come to LDS directly (global_load_lds), into a ring of SLOTS steps that the wave has for
// itself: nobody waits at a barrier before the sums meet, and what is on its way takes no registers.  A load
// instruction brings the 128 bytes of 8 rows, whole cache lines in lane order.  (Loaded straight into the MFMAs' registers,
// neighbouring lanes hold different rows, so an instruction touches 16 lines in pieces of 16 bytes, and the address unit,
// not the memory, sets the pace.  us a launch, everything from memory, before -> now:  gate/up with SwiGLU of 8,192 x 2,048
// 17.7 -> 14.4, x 3,072 21.0 -> 19.8, 14,336 x 4,096 50 -> 42.5;  2,048 x 8,192 11.1 -> 8.2, 3,072 x 8,192 12.3 -> 10.7;  a read of
// the same bytes that does nothing else takes 12.1, 19.2, 42; 7.6, 10.2.  A second copy of W in the order of the loads gains nothing
// over this at these widths; over k of 11,008 it took 18.5 for 4,096 columns where this takes 21.5, over 8,192 14.3 and 15.6.)
//   Inside a 1 KiB tile of 8 rows the 16-byte pieces of a row are permuted by the row's number (the lane that writes place p
// of row r fetches piece p ^ turn(r)), so that the 16 lanes that a 128-bit LDS read serves at a time meet no bank twice.
//
// X is fetched once per workgroup (L2 serves it); a workgroup whose rows are few against X's takes more of them at once.
// A product is as fast as the busiest compute unit: a block holds `bh` <= 16 rows, chosen on the host so that
// the workgroups come out as whole rounds over the compute units, of as many at a time as LDS holds (3,072 rows on
// 256 units: 256 blocks of 12, not 192 of 16).  Rows beyond the block, and rows m >= M of X, are the last live one again (the same cache
// lines, no further traffic), or not fetched where a whole tile of 8 is beyond; what the MFMAs make of them is never stored.
//
// The result element (m, n) is summed over k in an order that depends on K only, not on M, the other rows,
// the number of waves, the row blocks of a workgroup or their height: whichever shape a launch takes, a row's
// result is the same bit for bit.
#include "lds_load.h"

#include <algorithm>
#include <initializer_list>

constexpr int SK_STEP = LL_STEP;
constexpr int SK_CHUNK = 128;    // k per chunk: two steps
constexpr int SK_SHARES = 16;    // chunk c is summed into share c % 16
constexpr int SK_MAX_ROWS = 64;
constexpr int SK_TILE = LL_TILE;

enum SkinnyEpilogue { EPI_STORE = 0, EPI_SWIGLU = 1, EPI_ROPE = 2, EPI_RESIDUAL = 3, EPI_ACT = 4, EPI_GROUPED = 5 };

// What the q/k/v product needs to rotate its result and to put keys and values into the cache pages.
struct RopeOut {
    const float* cos_table;      // [positions][head_dim / 2]
    const float* sin_table;
    const int* positions;        // [M]
    const int* seq_of_token;     // [M]
    const int* block_table;      // [sequences][table_width]
    bf16_t* k_pages;             // [page][kv_head][offset][dim]
    bf16_t* v_pages;             // [page][kv_head][dim][offset]
    int table_width, n_heads, n_kv, head_dim, page_size;
};

// The product adds its result into the float residual and leaves what the norm after it needs.
struct ResidualOut {
    float* residual;      // [M][N], updated in place
    const float* gain;    // [N], the norm's weight
    bf16_t* scaled;       // [M][N] = residual * gain, not yet divided by the row's root mean square
    float* partials;      // [column blocks][16]: sum over a block's columns of residual^2, by row (M <= 16)
};

// X is such a `scaled` matrix (M <= 16): row m of the result is to be multiplied by rsqrt(sum_p partials[p][m] / K + eps).
struct RowScale {
    const float* partials;
    int n_partials;
    float eps;
};

struct Epilogue {
    RopeOut rope;
    ResidualOut res;
    RowScale scale;
    int activation;   // EPI_ACT: which (SiaActivation)
    const bf16_t* table;     // EPI_ACT: if given, the activation is multiplied by table[ids[m] * table_width + n] for
    const int* ids;          //          n < table_dim and by 0 beyond
    int table_width, table_dim;
    int glu;          // EPI_SWIGLU: which gated activation (SiaGlu; 0 is silu(gate) * up)
    float limit;      // EPI_SWIGLU: the clamp of the gated activations that have one
    const float* glu_bias;   // EPI_SWIGLU: if given, [2 * N] floats added to gate and up in front of the activation
    int groups, group_rows, last_rows, group_blocks;   // EPI_GROUPED: see below
};

// RB: blocks of bh rows of W per workgroup; MB: blocks of 16 rows of X; WAVES: 4 or 8 waves that split K; SLOTS: steps in
// a wave's ring; WI: tiles of 8 rows that a block of W has (1 where bh <= 8); XI: tiles of X (1 where M <= 8, else 2 MB).
//   EPI_STORE:   row block rb holds bh rows of W and gives as many columns of Y (TOut)
//   EPI_ACT:     as EPI_STORE, with an activation without a gate applied to the float sums, rounded once
//   EPI_SWIGLU:  W = [gate; up] of N rows each; the first RB / 2 row blocks are gate rows, the others the up rows of
//                the same columns: Y = silu(gate) * up (or another gated activation of common.h), in float, rounded once
//   EPI_ROPE:    RB = 2, W = [q heads | k heads | v heads] of head_dim rows each; a workgroup owns 16 columns of
//                the first half of a head and the 16 that the rotation pairs them with (head_dim / 2 further).
//                q and k are rotated in float on the float sums (one rounding; the rotation kernel rotates the
//                rounded product, so the two paths differ by a rounding); q goes to Y, k and v into the pages.
//   EPI_RESIDUAL: the result, rounded as EPI_STORE rounds it, is added to the float residual; Y is not written.
//                RMSNorm(x) W^T = rsqrt(mean x^2 + eps) * ((x * gain) W^T): the kernel leaves x * gain and the sums
//                of squares of its own column blocks, and the product after it (SCALED) adds those up, in an
//                order that depends on their number only, and scales its rows: no kernel of its own for the norm.
//   EPI_GROUPED: as EPI_STORE, for W = groups of rows one behind the other that read inputs of their own: X is
//                [groups][M][K], group g has group_rows rows of W (the last one last_rows) and gives the matrix
//                Y + g * M * group_rows, [M][its rows]; a workgroup's blocks lie in one group (group_blocks workgroups
//                each).
// With MB > 1 (more than 16 rows) the epilogues that change the sums, EPI_SWIGLU and EPI_ROPE, round them to bfloat16 first, as
// EPI_STORE does: steps of that many rows give the bits of the product and the kernel behind it.
// Output columns come in *units*: a column of Y (EPI_STORE, EPI_RESIDUAL, EPI_SWIGLU, where unit u needs row u of
// the gate half and row u of the up half of W), or a pair of columns that the rotation mixes (EPI_ROPE: unit u is
// column u % (head_dim / 2) of head u / (head_dim / 2) together with the column head_dim / 2 further).  A workgroup
// owns UNIT_BLOCKS blocks of bh consecutive units from blockIdx.x * UNIT_BLOCKS * bh on.
// DIRECT: X and W begin at multiples of 16 bytes, as the way straight to LDS needs.  Else every lane loads its own operands, which
// may begin at any element, into registers, a chunk at a time (the same sums, in one shape; us of 3,072 x 3,072, 8 rows, W 6 bytes
// beside such a multiple: 13.4, by lines of 128 bytes through registers and LDS 18.3, with a copy of W first 15.4).
template <typename TOut, int EPI, bool SCALED, int RB, int MB, int WAVES, int SLOTS, int WI, int XI, bool DIRECT>
__global__ __launch_bounds__(WAVES* SIA_WAVE) void gemm_skinny_kernel(const bf16_t* __restrict__ X,
                                                                     const bf16_t* __restrict__ W,
                                                                     TOut* __restrict__ Y, int M, int N, int K,
                                                                     int bh, const Epilogue ep) {
    static_assert(WAVES == 4 || WAVES == 8, "4 or 8 waves share the 16 shares of K");
    static_assert(EPI != EPI_ROPE || RB == 2, "the rotation pairs two row blocks");
    static_assert(EPI != EPI_SWIGLU || RB % 2 == 0, "gate and up rows come in equal numbers");
    static_assert((WI == 1 || WI == 2) && (XI == 2 * MB || (MB == 1 && XI == 1)), "tiles of 8 rows");
    static_assert(DIRECT || (SLOTS == 1 && MB == 1), "a form of up to 16 rows, without a ring");
    static_assert(MB == 1 || (!SCALED && EPI != EPI_RESIDUAL && EPI != EPI_ACT), "forms of up to 16 rows");
    constexpr bool ROUND_FIRST = MB > 1;
    constexpr int THREADS = WAVES * SIA_WAVE;
    constexpr int SPW = SK_SHARES / WAVES;  // shares per wave
    constexpr int UNIT_BLOCKS = EPI == EPI_SWIGLU ? RB / 2 : EPI == EPI_ROPE ? 1 : RB;
    constexpr int LOADS = RB * WI + XI;     // of a step
    constexpr int ROWS = MB * 16;
    // the ring, and when the weights have been read the sums of pairs of shares and a row's sums of squares in its place
    constexpr int RING = DIRECT ? WAVES * SLOTS * LOADS * SK_TILE : 0;
    constexpr int PART = 8 * RB * ROWS * 17 * 4, SQUARES = SCALED ? SK_SHARES * 16 * 4 : 0;
    constexpr int LDS = RING > PART + SQUARES ? RING : PART + SQUARES;
    static_assert(LDS <= LL_LDS, "a workgroup's LDS");
    __shared__ __attribute__((aligned(1024))) char lds[LDS];
    float(*part)[RB][ROWS][17] = reinterpret_cast<float(*)[RB][ROWS][17]>(lds);
    float(*squares)[16] = reinterpret_cast<float(*)[16]>(lds + PART);
    const RopeOut& rope = ep.rope;
    int bx = blockIdx.x;
    if (EPI == EPI_GROUPED) {
        const int group = min(bx / ep.group_blocks, ep.groups - 1);
        bx -= group * ep.group_blocks;
        N = group + 1 < ep.groups ? ep.group_rows : ep.last_rows;
        X += (size_t)group * M * K;
        W += (size_t)group * ep.group_rows * K;
        Y += (size_t)group * M * ep.group_rows;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SIA_WAVE);  // a scalar, and the compiler knows
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int rope_half = EPI == EPI_ROPE ? rope.head_dim / 2 : 0;
    const int units = EPI == EPI_ROPE ? (rope.n_heads + 2 * rope.n_kv) * rope_half : N;
    const int u0 = bx * UNIT_BLOCKS * bh;
    // the unit of place n of unit block jb; places beyond the block or beyond the last unit repeat a unit before
    auto unit_at = [&](int jb, int n) { return min(u0 + jb * bh + min(n, bh - 1), units - 1); };
    auto is_live = [&](int jb, int n) { return n < bh && u0 + jb * bh + n < units; };
    auto row_of = [&](int rb, int n) {
        const int u = unit_at(rb % UNIT_BLOCKS, n);
        if (EPI == EPI_ROPE)  // the second row block holds the rotation's partners
            return (u / rope_half) * rope.head_dim + u % rope_half + rb * rope_half;
        return u + (rb / UNIT_BLOCKS) * N;  // rb / UNIT_BLOCKS: 0 gate (or all), 1 up
    };
    // load l of a step: its first row, the same in all lanes, and this lane's 16 bytes from there at k = 0.  Lane p of a row's
    // eight fetches the piece that belongs at place p.  (Units ascend with n and rows with units: the offset is not negative.)
    const bf16_t* base[LOADS];
    unsigned offset[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const bool of_w = l < RB * WI;
        const int n = 8 * (of_w ? l % WI : l - RB * WI) + lane / 8;
        const int first = of_w ? __builtin_amdgcn_readfirstlane(row_of(l / WI, 0)) : 0;
        const int row = of_w ? row_of(l / WI, n) : min(n, M - 1);
        base[l] = (of_w ? W : X) + (size_t)first * K;
        offset[l] = ((unsigned)(row - first) * (unsigned)K + ((lane & 7) ^ turn(n & 15)) * 8) * 2;
    }

    // requested before the weights, used after them.  The sums of squares of a row are added up the way the
    // products are: 64 runners (16 shares of 4 lane groups), runner l taking partials l, l + 64, ...
    constexpr int SQ_RUNNERS = SK_SHARES * 4;
    const int sq_m = lane & 15;
    float sq[SPW][4];
    if (SCALED) {
#pragma unroll
        for (int j = 0; j < SPW; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int p = (wave + j * WAVES) * 4 + (lane >> 4) + i * SQ_RUNNERS;
                sq[j][i] = p < ep.scale.n_partials ? ep.scale.partials[p * 16 + sq_m] : 0.f;
            }
    }
    constexpr int RES_ITER = EPI == EPI_RESIDUAL ? (RB * 256 + THREADS - 1) / THREADS : 1;
    float res_old[RES_ITER], res_gain[RES_ITER];
    if (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int it = 0; it < RES_ITER; ++it) {
            const int idx = threadIdx.x + it * THREADS;
            const int j = idx / 256, m = (idx / 16) % 16, n = idx % 16;
            const bool live = idx < RB * 256 && m < M && is_live(j, n);
            res_old[it] = live ? ep.res.residual[(size_t)m * N + u0 + j * bh + n] : 0.f;
            res_gain[it] = live ? ep.res.gain[u0 + j * bh + n] : 0.f;
        }
    }
    constexpr int ROPE_ITER = EPI == EPI_ROPE ? (ROWS * 16 + THREADS - 1) / THREADS : 1;
    int position[ROPE_ITER], sequence[ROPE_ITER];
    if (EPI == EPI_ROPE) {
#pragma unroll
        for (int it = 0; it < ROPE_ITER; ++it) {
            const int m = (threadIdx.x + it * THREADS) / 16;   // (waves beyond the rows wait for their weights alone)
            position[it] = m < M ? rope.positions[m] : 0;
            sequence[it] = m < M ? rope.seq_of_token[m] : 0;
        }
    }

    // Step s of the wave: half s % 2 of its chunk s / 2, chunk wave + (s / 2) * WAVES of the row, whose share has the
    // accumulator (s / 2) % SPW.  Only the row's last chunk may be half a chunk (K is a multiple of 64).
    const int row_steps = K / SK_STEP;
    const int turns = row_steps / (2 * WAVES), rest = row_steps % (2 * WAVES) - 2 * wave;
    const int steps = 2 * turns + min(max(rest, 0), 2);
    // Rows a multiple of 4 KiB apart lie alike in the memory's channels: workgroups that walk them in step would all be in the
    // same half of the channels.  Every other workgroup (of a die) takes the chunks of shares s and s + 8 in the other order:
    // each share's own order stays, and the two are added to each other.  (us: 128,256 x 2,048 91.5 -> 87.0 for one row, 120 -> 108 for
    // 27, 14,336 x 4,096 gated 43.0 -> 42.2 for 16 and 48.7 -> 45.4 for 27, 6,144 x 4,096 11.3 -> 10.6, 8,192 x 2,048 gated 20.6 -> 18.4 for 64;
    // but 13.7 -> 14.6 for one row, whose two turns are all on their way at once: not that.)
    const bool alike = K % (SK_SHARES * SK_CHUNK) == 0 && (EPI != EPI_SWIGLU || XI > 1 || K > SK_SHARES * SK_CHUNK);
    constexpr int HOP = WAVES * SK_CHUNK;  // from one chunk of the wave to its next
    const int swap = alike && (blockIdx.x >> 3 & 1) ? SPW / 2 * HOP : 0;
    char* ring = lds + wave * (SLOTS * LOADS * SK_TILE);
    // step s0 + u, s0 a multiple of 2 SPW and u known to the compiler
    auto request = [&](int s0, int u, int slot) {
        const size_t k = (size_t)(wave * SK_CHUNK + (s0 / 2 + u / 2) * HOP + u % 2 * SK_STEP + (u / 2 % SPW < SPW / 2 ? swap : -swap));
        char* to = ring + slot * (LOADS * SK_TILE);
#pragma unroll
        for (int l = 0; l < LOADS; ++l) load_to_lds((const char*)(base[l] + k) + offset[l], to + l * SK_TILE);
    };
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
        if (DIRECT && s < steps) request(0, s, s);

    // what the rotation and the cache write need is on its way beside the weights
    float rope_cos[ROPE_ITER], rope_sin[ROPE_ITER];
    int rope_page[ROPE_ITER];
    if (EPI == EPI_ROPE) {
        const int u = unit_at(0, threadIdx.x % 16), head = u / rope_half, j = u % rope_half;
#pragma unroll
        for (int it = 0; it < ROPE_ITER; ++it) {
            if ((int)(threadIdx.x + it * THREADS) / 16 >= M) break;
            const bool rotates = head < rope.n_heads + rope.n_kv, cached = head >= rope.n_heads;
            const size_t at = (size_t)position[it] * rope_half + j;
            rope_cos[it] = rotates ? rope.cos_table[at] : 1.f;
            rope_sin[it] = rotates ? rope.sin_table[at] : 0.f;
            rope_page[it] = cached ? rope.block_table[(size_t)sequence[it] * rope.table_width + position[it] / rope.page_size] : 0;
        }
    }

    const int wr = WI == 1 ? r & 7 : r, xr = XI == 1 ? r & 7 : r;
    const int w_at[2] = {wr * 128 + ((2 * g) ^ turn(wr)) * 16, wr * 128 + ((2 * g + 1) ^ turn(wr)) * 16};
    const int x_at[2] = {xr * 128 + ((2 * g) ^ turn(xr)) * 16, xr * 128 + ((2 * g + 1) ^ turn(xr)) * 16};
    floatx4 acc[SPW][RB][MB];
#pragma unroll
    for (int j = 0; j < SPW; ++j)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) acc[j][rb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (!DIRECT) {
        const bf16_t* own[RB + 1];   // the lane's rows of W, and of X
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) own[rb] = W + (size_t)row_of(rb, r) * K + g * 16;
        own[RB] = X + (size_t)min(r, M - 1) * K + g * 16;
        for (int s0 = 0; s0 < steps; s0 += 2 * SPW)
#pragma unroll
            for (int j = 0; j < SPW; ++j) {
                bf16x8 held[2][RB + 1][2];
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (s0 + 2 * j + u < steps) {
                        const int k = wave * SK_CHUNK + (s0 / 2 + j) * HOP + u * SK_STEP;
#pragma unroll
                        for (int l = 0; l <= RB; ++l) __builtin_memcpy(held[u][l], own[l] + k, 32);
                    }
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (s0 + 2 * j + u < steps) {
#pragma unroll
                        for (int rb = 0; rb < RB; ++rb) {
                            acc[j][rb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(held[u][rb][0], held[u][RB][0], acc[j][rb][0], 0, 0, 0);
                            acc[j][rb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(held[u][rb][1], held[u][RB][1], acc[j][rb][0], 0, 0, 0);
                        }
                    }
            }
    }
    int slot = 0;
    for (int s0 = 0; DIRECT && s0 < steps; s0 += 2 * SPW) {
#pragma unroll
        for (int t = 0; t < 2 * SPW; ++t) {
            const int s = s0 + t, j = t / 2;
            // s is the same in all lanes of the wave (a scalar): a step beyond the last is skipped by a branch
            if (s < steps) {
                wait_step<LOADS, SLOTS - 1>(steps - 1 - s);
                const char* from = ring + slot * (LOADS * SK_TILE);
                bf16x8 a[RB][2], b[MB][2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) b[mb][h] = *(const bf16x8*)(from + (RB * WI + 2 * mb) * SK_TILE + x_at[h]);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) a[rb][h] = *(const bf16x8*)(from + rb * WI * SK_TILE + w_at[h]);
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read: it may be filled again
                if (s + SLOTS < steps) request(s0, t + SLOTS, slot);
                slot = slot + 1 < SLOTS ? slot + 1 : 0;
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        acc[j][rb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rb][0], b[mb][0], acc[j][rb][mb], 0, 0, 0);
                        acc[j][rb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rb][1], b[mb][1], acc[j][rb][mb], 0, 0, 0);
                    }
            }
        }
    }
    __syncthreads();  // every wave has read its ring
    // acc[j][rb][mb][i] = share wave + j * WAVES of row m = 16 mb + r, column 4g + i of row block rb; part[w]: shares w and w + 8
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < SPW / 2; ++j)
                    part[wave + j * WAVES][rb][mb * 16 + r][g * 4 + i] = acc[j][rb][mb][i] + acc[j + SPW / 2][rb][mb][i];
    // the sum over all of k of element (j, m, n)
    auto total = [&](int j, int m, int n) -> float {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += part[w][j][m][n];
        return s;
    };
    auto rounded = [](float x) { return ROUND_FIRST ? bf16_to_float(float_to_bf16(x)) : x; };
    if (SCALED) {
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            float ss = (sq[j][0] + sq[j][1]) + (sq[j][2] + sq[j][3]);
            for (int p = (wave + j * WAVES) * 4 + (lane >> 4) + 4 * SQ_RUNNERS; p < ep.scale.n_partials; p += SQ_RUNNERS)
                ss += ep.scale.partials[p * 16 + sq_m];
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (lane < 16) squares[wave + j * WAVES][lane] = ss;
        }
    }
    __syncthreads();
    // the row's scale: every thread that finishes an element of row m adds the waves' sums in the same order
    auto row_scale = [&](int m) -> float {
        if (!SCALED) return 1.f;
        float ss = 0.f;
#pragma unroll
        for (int w = 0; w < SK_SHARES; ++w) ss += squares[w][m];
        return rsqrtf(ss / (float)K + ep.scale.eps);
    };
    if (EPI == EPI_ROPE) {
        const int n = threadIdx.x % 16;
        if (!is_live(0, n)) return;
        const int u = u0 + n, head = u / rope_half, j = u % rope_half;
        const bool is_v = head >= rope.n_heads + rope.n_kv;
#pragma unroll
        for (int it = 0; it < ROPE_ITER; ++it) {
            const int m = (threadIdx.x + it * THREADS) / 16;
            if (m >= M) return;
            float a = total(0, m, n), b = total(1, m, n);  // columns j and j + half of the head
            const float rs = row_scale(m);
            a = rounded(a * rs);
            b = rounded(b * rs);
            if (!is_v) {
                const float c = rope_cos[it], sn = rope_sin[it];
                float ra, rb_;
                rotate_pair(a, b, c, sn, ra, rb_);
                a = ra;
                b = rb_;
            }
            if (head < rope.n_heads) {
                TOut* y = Y + (size_t)m * N + head * rope.head_dim;
                y[j] = from_float<TOut>(a);
                y[j + rope_half] = from_float<TOut>(b);
                continue;
            }
            const int page = rope_page[it];
            if (page < 0) continue;  // never for a token the step owns
            const int off = position[it] % rope.page_size, D = rope.head_dim, ps = rope.page_size;
            if (!is_v) {
                const int hk = head - rope.n_heads;
                bf16_t* dst = rope.k_pages + (((size_t)page * rope.n_kv + hk) * ps + off) * D;
                dst[j] = float_to_bf16(a);
                dst[j + rope_half] = float_to_bf16(b);
            } else {
                const int hk = head - rope.n_heads - rope.n_kv;
                bf16_t* dst = rope.v_pages + ((size_t)page * rope.n_kv + hk) * D * ps + off;
                dst[(size_t)j * ps] = float_to_bf16(a);
                dst[(size_t)(j + rope_half) * ps] = float_to_bf16(b);
            }
        }
        return;
    }
    if (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int it = 0; it < RES_ITER; ++it) {
            const int idx = threadIdx.x + it * THREADS;
            const int j = idx / 256, m = (idx / 16) % 16, n = idx % 16;
            if (idx >= RB * 256 || m >= M) continue;  // a whole 16-lane group leaves or stays
            const bool live = is_live(j, n);
            float x = 0.f;
            if (live) {
                x = res_old[it] + bf16_to_float(float_to_bf16(total(j, m, n) * row_scale(m)));
                const size_t at = (size_t)m * N + u0 + j * bh + n;
                ep.res.residual[at] = x;
                ep.res.scaled[at] = float_to_bf16(x * res_gain[it]);
            }
            float xx = x * x;
            xx += __shfl_xor(xx, 1);
            xx += __shfl_xor(xx, 2);
            xx += __shfl_xor(xx, 4);
            xx += __shfl_xor(xx, 8);
            if (n == 0) ep.res.partials[(blockIdx.x * RB + j) * 16 + m] = xx;  // 0 for a block beyond the last column
        }
        return;
    }
    for (int idx = threadIdx.x; idx < UNIT_BLOCKS * ROWS * 16; idx += THREADS) {
        const int j = idx / (ROWS * 16), m = (idx / 16) % ROWS, n = idx % 16;
        if (m >= M || !is_live(j, n)) continue;
        const float rs = row_scale(m);
        TOut* y = Y + (size_t)m * N + u0 + j * bh + n;
        if (EPI == EPI_SWIGLU) {
            float gate = rounded(total(j, m, n) * rs), up = rounded(total(UNIT_BLOCKS + j, m, n) * rs);
            if (ep.glu_bias) {
                gate += ep.glu_bias[u0 + j * bh + n];
                up += ep.glu_bias[N + u0 + j * bh + n];
            }
            *y = from_float<TOut>(ep.glu == SIA_GLU_SILU ? gate / (1.f + expf(-gate)) * up
                                                         : gated_activation(gate, up, ep.glu, ep.limit));
        } else if (EPI == EPI_ACT) {
            float a = activate(total(j, m, n) * rs, ep.activation);
            if (ep.table) {
                const int c = u0 + j * bh + n;
                a = c < ep.table_dim ? a * bf16_to_float(ep.table[(size_t)ep.ids[m] * ep.table_width + c]) : 0.f;
            }
            *y = from_float<TOut>(a);
        } else {
            *y = from_float<TOut>(total(j, m, n) * rs);
        }
    }
}

// The rows up to which every epilogue has a kernel; EPI_STORE, EPI_SWIGLU and EPI_ROPE go up to SK_MAX_ROWS.
SIA_EXPORT int sia_gemm_skinny_max_rows() { return 16; }
SIA_EXPORT int sia_gemm_skinny_most_rows() { return SK_MAX_ROWS; }

extern "C" int sia_gemm_tiles_takes(int M, int N, int K);

// Whether a product goes to this file's kernels rather than to the tiles of gemm_tiles.hip or to the BLAS library.  Up to 16 rows all
// do.  Beyond, X's rows weigh as much as W's in what a workgroup fetches, and k is in one piece: the tiles are ahead over long k,
// the library where the columns are many, or few and k so long that few workgroups walk it for long (k of 5,120 to 10,240, which the tiles
// do not take).  A multiple of 8,192 columns comes to a unit as 32 rows of W that start a large power of two apart, which the channels
// of the memory feel; the library's shapes do not.  us, own / the library's best candidate:
//   at 27 rows 2,048 x 2,048 4.5 / 8.4, 5,120 x 3,072 11.1 / 12.4;  at 32 8,192 x 5,120 21.7 / 20.8, 8,192 x 8,192 33.3 / 30.4 (stays), 28,672 x
//   3,072 38.3 / 35.0 (stays), x 4,096 0.86 of the other, 18,432 x 1,024 0.95
//   at 40 rows 2,048 x 4,096 0.78, 1,024 x 5,120 0.60, 512 x 6,144 1.08, 1,024 x 8,192 14.6 / 12.5, 2,560 x 8,192 17.5 / 16.5 (these three
//   stay), 9,216 x 3,072 0.89, 12,288 x 3,072 1.02 (stays)
//   at 57 rows 3,072 x 4,096 0.95, 5,120 x 5,120 0.99, 6,144 x 4,096 1.00, 6,144 x 5,120 1.08 (stays), 9,216 x 8,192 1.01 (stays), 8,192 x 3,072 0.95,
//   8,192 x 4,096 21.4 / 19.1 (stays)
SIA_EXPORT int sia_gemm_skinny_takes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 || M > SK_MAX_ROWS) return 0;
    if (M <= 16) return 1;
    if (sia_gemm_tiles_takes(M, N, K)) return 0;
    if (N % (8 * 1024) == 0 && (M > 48 ? K >= 4 * 1024 : M > 20 && K % (8 * 1024) == 0)) return 0;
    if (M <= 32) return N <= 20 * 1024 || K % 2048 == 0;
    if (N > 10 * 1024 || (K > 5 * 1024 && N < 1536) || (K > 6 * 1024 && N < 3 * 1024)) return 0;
    return M <= 48 || (K <= 8 * 1024 && (N < 6 * 1024 || K < 5 * 1024));
}

// Whether the product with SwiGLU inside goes to this file's kernel.  Up to 16 rows always.  More rows weigh in every workgroup,
// and k is in one piece: where the columns are few and k long, too few workgroups walk too long; where the columns are many
// and k short, the library's tiles fill the chip, unless the rows of W are a multiple of 4 KiB apart, where it loses.  us, library or
// tiles and activation / this kernel:
//   inter 1,024 x 3,072 at 27 rows 15.0 / 11.3, at 57 13.3 / 16.4;  x 5,120 at 27 20.7 / 17.3, at 48 17.5 / 22.0;  x 14,336 at 57 29.0 / 53.4
//   inter 2,560 x 4,096 at 48 25.3 / 17.8, at 64 20.4 / 20.6;  x 8,192 at 64 32.2 / 35.6
//   inter 4,096 x 3,072 at 64 23.0 / 20.2;  x 5,120 at 48 29.1 / 27.4;  x 8,192 at 32 34.1 / 35.7, at 64 37.6 / 41.7
//   inter 5,120 x 8,192 at 64 46.5 / 44.6;  inter 8,192 x 3,072 at 64 28.5 / 27.0;  inter 9,216 x 3,072 at 57 37.4 / 38.6;  inter 14,336 at 57 x 3,072 41.3 / 47.2, x 4,096 57.7 / 55.4
SIA_EXPORT int sia_gemm_skinny_takes_swiglu(int M, int inter, int K) {
    if (M <= 0 || inter <= 0 || K <= 0 || K % 64 || M > SK_MAX_ROWS) return 0;
    if (M <= 16) return 1;
    if (K % 2048 && (M > 48 ? inter > 8704 && (K > 2048 || inter > 10 * 1024) : M > 32 && inter > 10 * 1024)) return 0;
    return inter >= 4608 || K <= 2048 || (inter >= 2560 ? K <= 3 * 1024 || (K <= 5 * 1024 && M <= 48) : K <= 5 * 1024 && M <= 32);
}

// How a product is cut into workgroups: `unit_blocks` blocks of `bh` units each, `grid` workgroups.
struct Cut {
    int unit_blocks, bh, grid;
    double cost;
};

// The block height for workgroups of `unit_blocks` blocks (each unit costs `rows_per_unit` rows of W, a workgroup `x_rows`
// rows of X on top): 16 when the workgroups are many; else the height from `least` to 16 that gives the busiest compute
// unit the least to fetch.
static Cut cut_for(int units, int unit_blocks, int rows_per_unit, int least, int x_rows) {
    const int cus = compute_units();
    auto with = [&](int bh) {
        const int grid = (units + unit_blocks * bh - 1) / (unit_blocks * bh);
        return Cut{unit_blocks, bh, grid, (double)((grid + cus - 1) / cus) * (bh * unit_blocks * rows_per_unit + x_rows)};
    };
    Cut best = with(16);
    if (best.grid > 4 * cus) return best;
    for (int bh = 15; bh >= least; --bh) {
        const Cut c = with(bh);
        if (c.cost < best.cost) best = c;
    }
    return best;
}

// Of the cuts an epilogue has kernels for, the cheapest; of equals the one with the higher blocks (fewer rows that
// repeat one), then the one with more blocks per workgroup (fewer workgroups fetch X).
static Cut cheapest(int units, int rows_per_unit, std::initializer_list<int> unit_blocks, int x_rows = 0) {
    Cut best{0, 0, 0, 0};
    for (int ub : unit_blocks) {
        const Cut c = cut_for(units, ub, rows_per_unit, 8, x_rows);
        if (!best.grid || c.cost < best.cost || (c.cost == best.cost && c.bh > best.bh)) best = c;
    }
    return best;
}

// A kernel for up to 16 rows: blocks of columns a workgroup, waves, steps in a wave's ring, and whether it has a form with
// half a tile for blocks of up to 8.
struct Shape {
    int blocks, waves, slots;
    bool low;
};

// Workgroups of a shape that LDS has room for on a compute unit.
static int room_for(const Shape& s, int bh, int M) {
    const int tiles = s.blocks * (s.low && bh <= 8 ? 1 : 2) + (M <= 8 ? 1 : 2);
    return std::max(1, LL_LDS / (s.waves * s.slots * tiles * SK_TILE));
}

// us that `grid` workgroups of blocks of `bh` rows of W take beside M <= 16 rows of X.  As many as have room in LDS run on a
// compute unit at a time, and each such round costs a start and an end: the ring fills, the sums meet.  A unit fetches at a
// rate that what it has on its way allows: 30 GB/s of its own and 1.5 us a trip.  Rows of X (L2 serves them) and repeated
// rows of W (the same lines) cost half.
static double few_rows_us(int M, int K, int grid, int bh, const Shape& s) {
    const int cus = compute_units(), w_rows = s.blocks * (s.low && bh <= 8 ? 8 : 16), x_rows = M <= 8 ? 8 : 16;
    const int ring = s.waves * s.slots * (w_rows + x_rows) / 8;   // KiB
    const int room = room_for(s, bh, M), on_unit = (grid + cus - 1) / cus, at_a_time = std::min(on_unit, room);
    const double rate = 30.0 / (1.0 + 1.5 * 30.0 / (at_a_time * ring));
    const double rows = s.blocks * bh + 0.5 * (w_rows - s.blocks * bh) + 0.5 * x_rows;
    return 3.0 * ((on_unit + room - 1) / room) + on_unit * rows * K * 2e-3 / rate;
}

// The shapes that launch_columns has: up to 8 rows, and up to 16.  (Four blocks a workgroup for 9 to 16 rows: LDS holds two such
// workgroups of one step a wave, but only one of two blocks and three steps.  us of 16 rows without -> with them: 9,216 x 3,072
// 17.0 -> 12.4, 12,352 x 3,072 24.5 -> 16.0, 28,672 x 4,096 49.6 -> 42.3, a head of 128,256 x 3,072 156 -> 147.5.  For up to 8 rows two
// blocks leave room for two workgroups as well: a head of 128,256 x 2,048 89 us, with four blocks 95.)
static const Shape FEW_ROWS_SHAPES[2][3] = {{{2, 8, 2, false}, {1, 8, 4, true}}, {{4, 8, 1, false}, {2, 8, 3, false}, {1, 8, 4, true}}};

// Of those and the heights of their blocks, what takes the shortest; of equals the higher blocks, then more of them.
// grid_of(columns): workgroups of that many columns that the result takes.  (By the rows alone, which cheapest goes by, 12,352
// columns got five rounds of blocks of 10: 8 rows x 1,024 11.3 us, now 6.6, x 3,072 20.5, now 15.1.  From 120 rows of W a unit on the
// rounds of up to 8 rows run into each other, and the rows do decide: 32,000 x 4,096, one row, 45 us, by rounds 51.)
// Without ``direct`` operands there is one shape, of one block.
template <typename GridOf> static Cut few_rows_cut(int M, int K, bool direct, GridOf grid_of) {
    if (!direct) {
        Cut cut = cheapest(grid_of(1), 1, {1});
        cut.grid = grid_of(cut.bh);
        return cut;
    }
    const int columns = grid_of(1);
    if (M <= 8 && columns > 120 * compute_units()) {
        Cut cut = cheapest(columns, 1, {2, 1});
        cut.grid = grid_of(cut.unit_blocks * cut.bh);   // (groups end in workgroups of their own)
        return cut;
    }
    Cut best{0, 0, 0, 0};
    for (const Shape& s : FEW_ROWS_SHAPES[M > 8])
        for (int bh = 16; s.blocks && bh >= (s.low ? 8 : 9); --bh) {
            const int grid = grid_of(s.blocks * bh);
            const double us = few_rows_us(M, K, grid, bh, s);
            if (!best.grid || us < best.cost || (us == best.cost && bh > best.bh)) best = Cut{s.blocks, bh, grid, us};
        }
    return best;
}

static Cut few_rows_cut(int M, int K, int N, bool direct = true) {
    return few_rows_cut(M, K, direct, [&](int columns) { return (N + columns - 1) / columns; });
}

// How a plain product of up to 16 rows is cut: cut[0] blocks of cut[1] columns a workgroup, cut[2] workgroups, cut[3] of them at a
// time on a compute unit.  0, or SIA_BAD_ARGUMENT.
SIA_EXPORT int sia_gemm_skinny_cut(int M, int N, int K, int* cut) {
    if (M <= 0 || M > 16 || N <= 0 || K <= 0 || !cut) return SIA_BAD_ARGUMENT;
    const Cut c = few_rows_cut(M, K, N);
    cut[0] = c.unit_blocks, cut[1] = c.bh, cut[2] = c.grid, cut[3] = 1;
    for (const Shape& s : FEW_ROWS_SHAPES[M > 8])
        if (s.blocks == c.unit_blocks) cut[3] = room_for(s, c.bh, M);
    return 0;
}

struct Product {
    const bf16_t* X;
    const bf16_t* W;
    void* Y;
    int M, N, K;
    hipStream_t stream;
};

template <typename TOut, int EPI, bool SCALED, int RB, int MB, int WAVES, int SLOTS, int WI = 2, int XI = 2 * MB, bool DIRECT = true>
static void launch(const Product& p, const Cut& cut, const Epilogue& ep) {
    hipLaunchKernelGGL((gemm_skinny_kernel<TOut, EPI, SCALED, RB, MB, WAVES, SLOTS, WI, XI, DIRECT>), dim3(cut.grid),
                       dim3(WAVES * SIA_WAVE), 0, p.stream, p.X, p.W, (TOut*)p.Y, p.M, p.N, p.K, cut.bh, ep);
}

// The one shape for up to 16 rows of operands that begin anywhere: RB blocks of weight rows a workgroup.
template <typename TOut, int EPI, bool SCALED, int RB> static void launch_anywhere(const Product& p, const Cut& cut, const Epilogue& ep) {
    launch<TOut, EPI, SCALED, RB, 1, 8, 1, 2, 2, false>(p, cut, ep);
}

// The kernel of a cut whose blocks are columns of Y, up to 16 rows.  Eight waves; the ring as deep as leaves a compute unit one
// or two workgroups, four steps at most: 64 to 160 KB are then on their way.
template <typename TOut, int EPI>
static void launch_columns(const Product& p, const Cut& cut, const Epilogue& ep) {
    if (!aligned16(p.X, p.W)) {
        if constexpr (EPI == EPI_RESIDUAL)
            if (cut.unit_blocks == 2) return launch_anywhere<TOut, EPI, false, 2>(p, cut, ep);
        return launch_anywhere<TOut, EPI, false, 1>(p, cut, ep);
    }
    const bool low = cut.bh <= 8;
    if constexpr (EPI != EPI_RESIDUAL)   // (whose cut is by the columns alone, in one block or two)
        if (cut.unit_blocks == 4) return launch<TOut, EPI, false, 4, 1, 8, 1>(p, cut, ep);
    if (p.M <= 8) {
        if (cut.unit_blocks == 2) launch<TOut, EPI, false, 2, 1, 8, 2, 2, 1>(p, cut, ep);
        else if (low) launch<TOut, EPI, false, 1, 1, 8, 4, 1, 1>(p, cut, ep);
        else launch<TOut, EPI, false, 1, 1, 8, 4, 2, 1>(p, cut, ep);
    } else if (p.M <= 16) {
        if (cut.unit_blocks == 2) launch<TOut, EPI, false, 2, 1, 8, 3>(p, cut, ep);
        else if (low) launch<TOut, EPI, false, 1, 1, 8, 4, 1>(p, cut, ep);
        else launch<TOut, EPI, false, 1, 1, 8, 4>(p, cut, ep);
    }
}

// 17 to 64 rows: the same, and four blocks a workgroup where the columns are many.
template <typename TOut, int MB>
static void launch_more_rows(const Product& p, const Cut& cut) {
    constexpr int TWO = MB == 4 ? 1 : 2, ONE = MB == 2 ? 3 : 2;   // steps in the ring of two blocks, and of one
    const Epilogue ep{};
    if (cut.unit_blocks == 4) launch<TOut, EPI_STORE, false, 4, MB, 8, 1>(p, cut, ep);
    else if (cut.unit_blocks == 2) launch<TOut, EPI_STORE, false, 2, MB, 8, TWO>(p, cut, ep);
    else if (cut.bh <= 8) launch<TOut, EPI_STORE, false, 1, MB, 8, ONE, 1>(p, cut, ep);
    else launch<TOut, EPI_STORE, false, 1, MB, 8, ONE>(p, cut, ep);
}

template <typename TOut> static void launch_store(const Product& p) {
    if (p.M <= 16) return launch_columns<TOut, EPI_STORE>(p, few_rows_cut(p.M, p.K, p.N, aligned16(p.X, p.W)), Epilogue{});
    const int mb = (p.M + 15) / 16;
    const Cut cut = cheapest(p.N, 1, {4, 2, 1}, mb * 16);
    if (mb == 2) launch_more_rows<TOut, 2>(p, cut);
    else if (mb == 3) launch_more_rows<TOut, 3>(p, cut);
    else launch_more_rows<TOut, 4>(p, cut);
}

// out_float: 1 -> Y is float, 0 -> bfloat16.  Needs K % 64 == 0 and M <= 16, or M <= 64 for operands that begin at multiples of
// 16 bytes.
SIA_EXPORT int sia_gemm_skinny(const void* X, const void* W, void* Y, int M, int N, int K, int out_float,
                               hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > SK_MAX_ROWS || K % 64 || K <= 0 || (M > 16 && !aligned16(X, W))) return SIA_BAD_ARGUMENT;
    const Product p{(const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, stream};
    if (out_float)
        launch_store<float>(p);
    else
        launch_store<bf16_t>(p);
    return SIA_LAUNCH_CHECK();
}

// Y[M, N] = act(X W^T) in bfloat16, act one of SiaActivation.  Needs M <= 16, K % 64 == 0.
SIA_EXPORT int sia_gemm_skinny_act(const void* X, const void* W, void* Y, int M, int N, int K, int activation,
                                   hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K % 64 || K <= 0 || (activation != SIA_RELU2 && activation != SIA_GELU_TANH && activation != SIA_GELU)) return SIA_BAD_ARGUMENT;
    Epilogue ep{};
    ep.activation = activation;
    launch_columns<bf16_t, EPI_ACT>(Product{(const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, stream}, few_rows_cut(M, K, N, aligned16(X, W)), ep);
    return SIA_LAUNCH_CHECK();
}

// Y[M, N] = act(X W^T) * table[ids[m], first + n] for n < dim, 0 beyond (N >= dim): the gate on a token's own input.
SIA_EXPORT int sia_gemm_skinny_embedding_gate(const void* X, const void* W, void* Y, int M, int N, int K, int activation,
                                              const void* table, int table_width, int first, int dim, const int* ids,
                                              hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K % 64 || K <= 0 || (activation != SIA_RELU2 && activation != SIA_GELU_TANH && activation != SIA_GELU) ||
        !table || !ids || dim <= 0 || dim > N || first < 0 || first + dim > table_width)
        return SIA_BAD_ARGUMENT;
    Epilogue ep{};
    ep.activation = activation;
    ep.table = (const bf16_t*)table + first;
    ep.ids = ids;
    ep.table_width = table_width;
    ep.table_dim = dim;
    launch_columns<bf16_t, EPI_ACT>(Product{(const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, stream}, few_rows_cut(M, K, N, aligned16(X, W)), ep);
    return SIA_LAUNCH_CHECK();
}

// The products of groups of rows of W with inputs of their own (EPI_GROUPED): Y[g] = X[g] W[g]^T in bfloat16, group g's
// matrix at Y + g * M * group_rows.  Needs M <= 16, K % 64 == 0.
SIA_EXPORT int sia_gemm_skinny_grouped(const void* X, const void* W, void* Y, int M, int K, int groups, int group_rows,
                                       int last_rows, hipStream_t stream) {
    if (M <= 0) return 0;
    if (M > 16 || K % 64 || K <= 0 || groups <= 0 || group_rows <= 0 || last_rows <= 0 || !X || !W || !Y) return SIA_BAD_ARGUMENT;
    const Cut best = few_rows_cut(M, K, aligned16(X, W), [&](int columns) {
        return (groups - 1) * ((group_rows + columns - 1) / columns) + (last_rows + columns - 1) / columns;
    });
    const int columns = best.unit_blocks * best.bh;
    Epilogue ep{};
    ep.groups = groups;
    ep.group_rows = group_rows;
    ep.last_rows = last_rows;
    ep.group_blocks = (group_rows + columns - 1) / columns;
    launch_columns<bf16_t, EPI_GROUPED>(Product{(const bf16_t*)X, (const bf16_t*)W, Y, M, group_rows, K, stream}, best, ep);
    return SIA_LAUNCH_CHECK();
}

// Blocks of columns whose sums of squares sia_gemm_skinny_residual leaves for a result of N columns.
SIA_EXPORT int sia_gemm_skinny_residual_blocks(int N) {
    if (N <= 0) return 0;
    const Cut cut = cheapest(N, 1, {2, 1});
    return cut.grid * cut.unit_blocks;
}

// residual[M, N] += round_bf16(X W^T); scaled = residual * gain (bfloat16); partials[blocks][16] = sums of squares of
// the residual over blocks of columns, by row (rows >= M are not written), blocks = sia_gemm_skinny_residual_blocks(N).
// Needs M <= 16, K % 64 == 0.
SIA_EXPORT int sia_gemm_skinny_residual(const void* X, const void* W, int M, int N, int K, float* residual,
                                        const float* gain, void* scaled, float* partials, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K % 64 || K <= 0 || !residual || !gain || !scaled || !partials) return SIA_BAD_ARGUMENT;
    Epilogue ep{};
    ep.res = ResidualOut{residual, gain, (bf16_t*)scaled, partials};
    launch_columns<bf16_t, EPI_RESIDUAL>(Product{(const bf16_t*)X, (const bf16_t*)W, nullptr, M, N, K, stream}, cheapest(N, 1, {2, 1}), ep);
    return SIA_LAUNCH_CHECK();
}

// Y[M, I] = silu(X Wg^T) * (X Wu^T) for W = [Wg; Wu] of 2 I rows.  Needs K % 64 == 0 and M <= 16, or M <= 64 for operands that
// begin at multiples of 16 bytes, without partials or bias and with silu.  Up to 16 rows the activation is of the float sums; with
// more they are rounded to bfloat16 first (the bits of the product and the activation kernel).
// With `partials` (else null) X is a `scaled` matrix of sia_gemm_skinny_residual and the rows are divided by their
// root mean square first.
// glu, limit: another gated activation than silu(gate) * up (SiaGlu of common.h); bias: [2 I] floats or null.
SIA_EXPORT int sia_gemm_skinny_glu(const void* X, const void* W, void* Y, int M, int inter, int K,
                                   const float* partials, int n_partials, float eps, int glu, float limit,
                                   const float* bias, hipStream_t stream) {
    if (M <= 0 || inter <= 0) return 0;
    if (M > SK_MAX_ROWS || (M > 16 && (partials || glu != SIA_GLU_SILU || bias || !aligned16(X, W))) || K % 64 || K <= 0 ||
        (partials && n_partials <= 0) || glu < SIA_GLU_SILU || glu > SIA_GLU_GELU_TANH)
        return SIA_BAD_ARGUMENT;
    Epilogue ep{};
    ep.glu_bias = bias;
    ep.scale = RowScale{partials, n_partials, eps};
    ep.glu = glu;
    ep.limit = limit;
    const Product p{(const bf16_t*)X, (const bf16_t*)W, Y, M, inter, K, stream};
    if (M <= 16) {
        // two workgroups a compute unit: one's sums meet while the other's rows come.  Where there is one a unit, it has eight
        // waves (9 rows, four waves / eight: 4,096 x 2,048 7.5 / 6.4 us, 8,192 x 8,192 32 / 29).
        const Cut cut = cheapest(inter, 2, {1});
        const bool alone = cut.grid <= compute_units(), direct = aligned16(X, W);
        if (!direct && partials) launch_anywhere<bf16_t, EPI_SWIGLU, true, 2>(p, cut, ep);
        else if (!direct) launch_anywhere<bf16_t, EPI_SWIGLU, false, 2>(p, cut, ep);
        else if (M <= 8 && partials) launch<bf16_t, EPI_SWIGLU, true, 2, 1, 8, 2, 2, 1>(p, cut, ep);
        else if (M <= 8) launch<bf16_t, EPI_SWIGLU, false, 2, 1, 8, 2, 2, 1>(p, cut, ep);
        else if (alone && partials) launch<bf16_t, EPI_SWIGLU, true, 2, 1, 8, 3>(p, cut, ep);
        else if (alone) launch<bf16_t, EPI_SWIGLU, false, 2, 1, 8, 3>(p, cut, ep);
        else if (partials) launch<bf16_t, EPI_SWIGLU, true, 2, 1, 4, 3>(p, cut, ep);
        else launch<bf16_t, EPI_SWIGLU, false, 2, 1, 4, 3>(p, cut, ep);
        return SIA_LAUNCH_CHECK();
    }
    // More rows: 64 rows of W a workgroup, against which X's weigh less; two workgroups of 32 where the rows are short and
    // one's few steps would stand alone (8,192 x 2,048, 27 rows 18.0 -> 15.7 us, 45 18.2 -> 17.7, 64 19.4 -> 20.8; x 3,072 20.9 -> 21.6,
    // 23.5 -> 25.0, 24.9 -> 29.4)
    const int mb = (M + 15) / 16;
    const bool wide = mb == 4 || K > 2048;
    const Cut cut = cheapest(inter, 2, {wide ? 2 : 1}, mb * 16);
    if (mb == 4) launch<bf16_t, EPI_SWIGLU, false, 4, 4, 8, 1>(p, cut, ep);
    else if (mb == 3 && wide) launch<bf16_t, EPI_SWIGLU, false, 4, 3, 8, 1>(p, cut, ep);
    else if (mb == 3) launch<bf16_t, EPI_SWIGLU, false, 2, 3, 4, 2>(p, cut, ep);
    else if (wide) launch<bf16_t, EPI_SWIGLU, false, 4, 2, 8, 1>(p, cut, ep);
    else launch<bf16_t, EPI_SWIGLU, false, 2, 2, 4, 2>(p, cut, ep);
    return SIA_LAUNCH_CHECK();
}

SIA_EXPORT int sia_gemm_skinny_swiglu(const void* X, const void* W, void* Y, int M, int inter, int K,
                                      const float* partials, int n_partials, float eps, hipStream_t stream) {
    return sia_gemm_skinny_glu(X, W, Y, M, inter, K, partials, n_partials, eps, SIA_GLU_SILU, 0.f, nullptr, stream);
}

// The q/k/v product of few tokens with the rotation and the cache write in its epilogue:
// W = [q heads | k heads | v heads], head_dim even, every dim of a head rotates (tables of head_dim / 2 floats
// a position).  Rotated q goes to Y[M][(n_heads + 2 n_kv) head_dim] (its k and v columns are not written); rotated
// k and v go to the pages at each token's position.  Needs K % 64 == 0 and M <= 16, or M <= 64 for operands that begin at
// multiples of 16 bytes and without partials.  Up to 16 rows the float sums are rotated; with more they are rounded to bfloat16
// first (the bits of the product and the rotation kernel).  `partials` as above.
SIA_EXPORT int sia_gemm_skinny_rope(const void* X, const void* W, void* Y, int M, int K, const float* cos_table,
                                    const float* sin_table, const int* positions, const int* seq_of_token,
                                    const int* block_table, int table_width, void* k_pages, void* v_pages,
                                    int n_heads, int n_kv, int head_dim, int page_size, const float* partials,
                                    int n_partials, float eps, hipStream_t stream) {
    if (M <= 0) return 0;
    if (M > SK_MAX_ROWS || (M > 16 && (partials || !aligned16(X, W))) || K % 64 || K <= 0 || head_dim % 2 || head_dim <= 0 || n_heads <= 0 || n_kv <= 0 || page_size <= 0 ||
        table_width <= 0 || !cos_table || !sin_table || !positions || !seq_of_token || !block_table || !k_pages ||
        !v_pages || (partials && n_partials <= 0))
        return SIA_BAD_ARGUMENT;
    const int heads = n_heads + 2 * n_kv, N = heads * head_dim;
    Epilogue ep{};
    ep.rope = RopeOut{cos_table, sin_table, positions, seq_of_token, block_table, (bf16_t*)k_pages, (bf16_t*)v_pages,
                      table_width, n_heads, n_kv, head_dim, page_size};
    ep.scale = RowScale{partials, n_partials, eps};
    const Product p{(const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, stream};
    const Cut cut = cut_for(heads * (head_dim / 2), 1, 2, 4, 0);
    const bool low = cut.bh <= 8;
    if (M > 16) {
        const int mb = (M + 15) / 16;
        if (mb == 2 && low) launch<bf16_t, EPI_ROPE, false, 2, 2, 8, 2, 1>(p, cut, ep);
        else if (mb == 2) launch<bf16_t, EPI_ROPE, false, 2, 2, 8, 2>(p, cut, ep);
        else if (mb == 3 && low) launch<bf16_t, EPI_ROPE, false, 2, 3, 8, 2, 1>(p, cut, ep);
        else if (mb == 3) launch<bf16_t, EPI_ROPE, false, 2, 3, 8, 2>(p, cut, ep);
        else if (low) launch<bf16_t, EPI_ROPE, false, 2, 4, 8, 2, 1>(p, cut, ep);
        else launch<bf16_t, EPI_ROPE, false, 2, 4, 8, 1>(p, cut, ep);
        return SIA_LAUNCH_CHECK();
    }
    // up to 8 rows: two steps leave a compute unit room for two workgroups, three for one (us of 9,216 x 3,072, one row: 13.7 / 14.9)
    const bool pairs = cut.grid > compute_units();
    const bool direct = aligned16(X, W);
#define LAUNCH(SCALED)                                                                        \
    do {                                                                                      \
        if (!direct) launch_anywhere<bf16_t, EPI_ROPE, SCALED, 2>(p, cut, ep);                \
        else if (M <= 8 && low) launch<bf16_t, EPI_ROPE, SCALED, 2, 1, 8, 3, 1, 1>(p, cut, ep);    \
        else if (M <= 8) launch<bf16_t, EPI_ROPE, SCALED, 2, 1, 8, 3, 2, 1>(p, cut, ep);      \
        else if (low) launch<bf16_t, EPI_ROPE, SCALED, 2, 1, 8, 3, 1>(p, cut, ep);            \
        else launch<bf16_t, EPI_ROPE, SCALED, 2, 1, 8, 3>(p, cut, ep);                        \
    } while (0)
    if (partials) LAUNCH(true);
    else LAUNCH(false);
#undef LAUNCH
    return SIA_LAUNCH_CHECK();
}
