// Linear attention with a decaying matrix state per head (gated linear attention), token by token.
//
// For every sequence and head, with a state S [D, Dv] of floats that a request keeps in its slot:
//
//   z_t     = A2 a_t + b                       a_t: the token's low-rank decay input [rank]; A2 [H * D, rank]
//   alpha_t = exp(logsigmoid(z_t) / tau)       one decay per key channel, in (0, 1)
//   S_t     = diag(alpha_t) S_(t-1) + k_t v_t^T
//   o_t     = S_t^T (q_t * q_scale)
//   y_t     = o_t * rsqrt(mean(o_t^2) + eps) * w  *  silu(g_t)         w [Dv], shared by the heads
//
// q, k [H * D], v, g [H * Dv] and a [rank] are columns of one projected row (row_stride apart, at the given column
// offsets); y is written as [tokens, H * Dv].  Products' results come in the compute type; decays, their logarithms,
// the state, the sums over channels, the norm and the gate are float, with one rounding of y.
//
// The decays of all tokens and channels are computed first, by a kernel of their own (they do not depend on the
// state, and a step's tokens are thousands of independent little products), into a float workspace.
// A workgroup owns one (sequence, head) and walks the sequence's tokens of this step in order; an entry of the state
// is written by the request's own tokens in their order.
// Thread (j, r) keeps rows r, r + R, r + 2R, ... of column j of S in registers (R a power of two: the lanes of a
// column are neighbours and add their shares of o by lane exchanges).  Blocks of a few tokens are staged through
// LDS (q, k, alpha, v, g as floats), walked, and their outputs normed and gated a token a wave.
//
// A step with few (sequence, head) pairs and runs of many tokens (a prompt) would leave most of the chip idle, and
// the walk along a sequence cannot be shortened.  Such a step gives every pair several workgroups, each with a
// slice of the state's columns (they are independent of one another), more lanes per column and fewer rows per
// lane; the outputs go to a float workspace and a second kernel norms and gates them, since a norm spans a head.
// A long prompt in bfloat16 is cut into segments that are walked at the same time, each from zero: what the state S
// in front of a segment adds to its outputs is (q_t * P_t)^T S with P_t the products of the decays since the segment began,
// and S itself follows from segment to segment by S <- diag(P_last) S + (the segment's own).  Only products of decays,
// which lie in (0, 1), are taken ahead: nothing is divided by them.
//
// What a request's numbers depend on beside its own tokens: the number of sequences and the longest run choose how many lanes
// share a column, and with it the order of an output's sum over the state's rows, in float32 too (states keep their bits
// there).  In bfloat16 the step's tokens, sequences and longest run also say whether and how prompts are cut, and with a cut the last
// bits of float of a state depend on where its segments began.
#include "common.h"

#include <type_traits>

// sigmoid(z) to the power of ``tau_inv`` as 2^whole 2^part, from log2(sigmoid(z)) = min(z, 0) log2(e) - log2(1 + 2^(-|z| log2(e)))
// with the hardware's exponent and logarithm.  The part keeps its bits: the product by log2(e) / tau is rounded once, less its
// whole number, log2(e) and the quotient come with what float leaves of them, and what rounding 1 + u drops is added again.
// Against 64 bits, z normal times four, largest relative error, tau 16 and 1: 8.3e-8 and 1.4e-7 (exp and log1p of the
// mathematics library: 1.0e-7 and 5.4e-7); for tau 16 and 4 the means are 1.7e-8 and 1.9e-8 (1.8e-8 and 2.2e-8).
__device__ __forceinline__ float sigmoid_power(float z, float tau_inv) {
    constexpr float LOG2E = 1.44269502f, LOG2E_REST = 1.92596299e-8f;
    const float scale = LOG2E * tau_inv, rest = fmaf(LOG2E_REST, tau_inv, fmaf(LOG2E, tau_inv, -scale));
    const float u = __builtin_amdgcn_exp2f(-fabsf(z) * LOG2E), w = 1.f + u;
    const float l = fmaf((u - (w - 1.f)) * LOG2E, __builtin_amdgcn_rcpf(w), __builtin_amdgcn_logf(w));
    const float m = fmaxf(fminf(z, 0.f), -160.f / fabsf(tau_inv));      // e^-160 is zero; an infinity has no whole number
    const float whole = rintf(m * scale);
    return ldexpf(__builtin_amdgcn_exp2f(fmaf(m, scale, -whole) + fmaf(m, rest, -l * tau_inv)), (int)whole);
}

// BONUS: the query reads the state before this token's write, and the write itself weighed per key channel by ``bonus``
// [heads, D] for this token only:  o_t = (S_(t-1) + diag(bonus) k_t v_t^T)^T q_t.  Where the outputs go to ``raw_out`` the
// weighed write is left to the finishing kernel.  The norm's weights are then [heads, Dv], not shared.
template <typename T, int ROWS, bool BONUS>
__global__ __launch_bounds__(512) void gla_recurrent_kernel(
    const T* __restrict__ proj, int row_stride, int q_col, int k_col, int v_col, int g_col,
    const float* __restrict__ alpha, const float* __restrict__ norm_w, float* __restrict__ state, const int* __restrict__ cu_q, const int* __restrict__ slots, T* __restrict__ out,
    int n_heads, int D, int Dv, int R, int block_tokens, float q_scale, float eps, int slice,
    float* __restrict__ raw_out, const float* __restrict__ k_f32, int q_share, long long state_stride,
    const float* __restrict__ bonus) {
    extern __shared__ float lds[];
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int j0 = blockIdx.z * slice;     // this workgroup's columns: j0 .. j0 + slice - 1
    const int first = cu_q[seq], last = cu_q[seq + 1];
    if (first >= last) return;
    const int TB = block_tokens;
    float* q_s = lds;                  // [TB][D]
    float* k_s = q_s + TB * D;         // [TB][D]
    float* al_s = k_s + TB * D;        // [TB][D]
    float* v_s = al_s + TB * D;        // [TB][Dv]
    float* g_s = v_s + TB * Dv;        // [TB][Dv]
    float* o_s = g_s + TB * Dv;        // [TB][Dv]
    float* u_s = o_s + TB * Dv;        // [D], BONUS only
    if (BONUS)      // (read behind the first block's barrier)
        for (int d = tid; d < D; d += blockDim.x) u_s[d] = raw_out ? 0.f : bonus[(size_t)head * D + d];

    const int j = j0 + tid / R, r = tid % R;
    const bool owns = tid / R < slice && j < Dv;
    float* S_mem = state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv;
    float S[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = i * R + r;
        S[i] = (owns && d < D) ? S_mem[(size_t)d * Dv + j] : 0.f;
    }
    const int wave = tid / SIA_WAVE, lane = tid % SIA_WAVE, n_waves = blockDim.x / SIA_WAVE;
    const int q_head = head / q_share;      // q (and a k read from the rows) may be shared by q_share neighbouring heads

    for (int t0 = first; t0 < last; t0 += TB) {
        const int nt = min(TB, last - t0);
        for (int idx = tid; idx < nt * Dv; idx += blockDim.x) {
            const int t = idx / Dv, c = idx % Dv;
            const T* row = proj + (size_t)(t0 + t) * row_stride;
            v_s[t * Dv + c] = to_float(row[v_col + head * Dv + c]);
            g_s[t * Dv + c] = g_col >= 0 ? to_float(row[g_col + head * Dv + c]) : 0.f;
        }
        for (int idx = tid; idx < nt * D; idx += blockDim.x) {
            const int t = idx / D, c = idx % D;
            const T* row = proj + (size_t)(t0 + t) * row_stride;
            q_s[t * D + c] = to_float(row[q_col + q_head * D + c]) * q_scale;
            k_s[t * D + c] = k_f32 ? k_f32[((size_t)(t0 + t) * n_heads + head) * D + c]
                                   : to_float(row[k_col + q_head * D + c]);
            al_s[t * D + c] = alpha[((size_t)(t0 + t) * n_heads + head) * D + c];
        }
        __syncthreads();
        for (int t = 0; t < nt; ++t) {
            float acc = 0.f;
            const float v = owns ? v_s[t * Dv + j] : 0.f;
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int d = i * R + r;
                if (d < D) {
                    const float write = k_s[t * D + d] * v;
                    if (BONUS) acc += q_s[t * D + d] * (S[i] + u_s[d] * write);
                    S[i] = al_s[t * D + d] * S[i] + write;
                    if (!BONUS) acc += q_s[t * D + d] * S[i];
                }
            }
            for (int o = R / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, SIA_WAVE);
            if (owns && r == 0) {
                if (raw_out) raw_out[((size_t)(t0 + t) * n_heads + head) * Dv + j] = acc;
                else o_s[t * Dv + j] = acc;
            }
        }
        __syncthreads();
        if (raw_out) continue;   // uniform: the norm is another kernel's
        for (int t = wave; t < nt; t += n_waves) {
            float ss = 0.f;
            for (int c = lane; c < Dv; c += SIA_WAVE) ss += o_s[t * Dv + c] * o_s[t * Dv + c];
            const float inv = rsqrtf(wave_sum(ss) / (float)Dv + eps);
            T* dst = out + ((size_t)(t0 + t) * n_heads + head) * Dv;
            for (int c = lane; c < Dv; c += SIA_WAVE) {
                const float g = g_s[t * Dv + c];
                dst[c] = from_float<T>(o_s[t * Dv + c] * inv * norm_w[(BONUS ? head * Dv : 0) + c] * (g_col >= 0 ? g / (1.f + expf(-g)) : 1.f));
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = i * R + r;
        if (owns && d < D) S_mem[(size_t)d * Dv + j] = S[i];
    }
}

// A step of one token a sequence in bfloat16: a workgroup a (sequence, head), whose state of D x Dv floats is read and
// written once, 16 bytes a lane in rows of the matrix, all of it under way at once.  Bound by those bytes and the way to
// memory and back; what the kernel above does for such a step reads 4 bytes a lane, four rows an instruction.
// Thread (group, quad) has four columns of rows group, group + G, ...; the groups' shares of the outputs are added by lane
// exchanges and through LDS.  Dv a power of two from 16 to 256, D up to ROWS * G.
// LOW_RANK: the decays exp(logsigmoid(a2 a + bias) / tau) are taken here, four lanes a channel, while the state is on
// its way; else they come as floats.
// 8 sequences of 24 heads of 128 x 128 (25 MB), rank 64: 15.5 us and 9.4 for the decays -> 10.9 for both; 10.4 with the gates and gains asked for first.
struct LowRank {
    const bf16_t* a2;
    const float* bias;
    int a_col, rank;
    float tau_inv;
};
template <int ROWS, bool BONUS, bool LOW_RANK>
__global__ __launch_bounds__(512) void state_decode_kernel(
    const bf16_t* __restrict__ proj, int row_stride, int q_col, int k_col, int v_col, int g_col,
    const float* __restrict__ alpha, const LowRank low, const float* __restrict__ norm_w, float* __restrict__ state,
    long long state_stride, const int* __restrict__ cu_q, const int* __restrict__ slots, bf16_t* __restrict__ out, int n_heads,
    int D, int Dv, float q_scale, float eps, float* __restrict__ raw_out, const float* __restrict__ k_f32, int q_share,
    const float* __restrict__ bonus) {
    constexpr int WAVES = 8;
    __shared__ float part[WAVES][256];
    __shared__ float decay[LOW_RANK ? 512 : 1];
    __shared__ float squares[WAVES];
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int n = cu_q[seq];
    if (cu_q[seq + 1] <= n) return;
    const int quads = Dv / 4, G = 512 / quads, quad = tid % quads, group = tid / quads;
    float* S_mem = state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv + 4 * quad;
    float4 S[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) S[i] = *reinterpret_cast<const float4*>(S_mem + (size_t)min(group + i * G, D - 1) * Dv);
    const bf16_t* row = proj + (size_t)n * row_stride;
    const size_t at = ((size_t)n * n_heads + head) * D;
    const bf16_t *q_row = row + q_col + head / q_share * D, *k_row = row + k_col + head / q_share * D;
    float q[ROWS], k[ROWS], a[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = min(group + i * G, D - 1);
        q[i] = bf16_to_float(q_row[d]) * q_scale;
        k[i] = k_f32 ? k_f32[at + d] : bf16_to_float(k_row[d]);
        if (!LOW_RANK) a[i] = alpha[at + d];
    }
    const uint2 v2 = *reinterpret_cast<const uint2*>(row + v_col + head * Dv + 4 * quad);
    const float v[4] = {__uint_as_float(v2.x << 16), __uint_as_float(v2.x & 0xffff0000u), __uint_as_float(v2.y << 16),
                        __uint_as_float(v2.y & 0xffff0000u)};
    // what the end needs, asked for here: a trip to memory less behind the sums
    const int column = min(tid, Dv - 1);
    const float g = !raw_out && g_col >= 0 ? bf16_to_float(row[g_col + head * Dv + column]) : 0.f;
    const float gain = !raw_out ? norm_w[(BONUS ? head * Dv : 0) + column] : 0.f;
    if (LOW_RANK) {
        const uint4* in = reinterpret_cast<const uint4*>(row + low.a_col);
        for (int c = tid / 4; c < D; c += 512 / 4) {      // four lanes a channel, pieces of eight in turn
            const uint4* w = reinterpret_cast<const uint4*>(low.a2 + (size_t)(head * D + c) * low.rank);
            const float bias = low.bias ? low.bias[head * D + c] : 0.f;
            float z = 0.f;
            for (int m = tid % 4; m < low.rank / 8; m += 4) {
                Vec8<bf16_t> x, y;
                x.u = in[m];
                y.u = w[m];
                float xs[8], ys[8];
                x.get(xs);
                y.get(ys);
#pragma unroll
                for (int e = 0; e < 8; ++e) z += xs[e] * ys[e];
            }
            z += __shfl_xor(z, 1, SIA_WAVE);
            z += __shfl_xor(z, 2, SIA_WAVE);
            if (tid % 4 == 0) decay[c] = sigmoid_power(z + bias, low.tau_inv);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ROWS; ++i) a[i] = decay[min(group + i * G, D - 1)];
    }
    float o[4] = {};
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = group + i * G;
        if (d >= D) continue;
        const float u = BONUS && !raw_out ? bonus[(size_t)head * D + d] : 0.f;
        float s[4] = {S[i].x, S[i].y, S[i].z, S[i].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float write = k[i] * v[e];
            if (BONUS) o[e] += q[i] * (s[e] + u * write);
            s[e] = a[i] * s[e] + write;
            if (!BONUS) o[e] += q[i] * s[e];
        }
        *reinterpret_cast<float4*>(S_mem + (size_t)d * Dv) = make_float4(s[0], s[1], s[2], s[3]);
    }
    for (int off = quads; off < SIA_WAVE; off <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], off, SIA_WAVE);
    const int wave = tid / SIA_WAVE, lane = tid % SIA_WAVE;
    if (lane < quads) *reinterpret_cast<float4*>(&part[wave][4 * quad]) = make_float4(o[0], o[1], o[2], o[3]);
    __syncthreads();
    float y = 0.f;
    if (tid < Dv)
#pragma unroll
        for (int w = 0; w < WAVES; ++w) y += part[w][tid];
    if (raw_out) {
        if (tid < Dv) raw_out[((size_t)n * n_heads + head) * Dv + tid] = y;
        return;
    }
    const float ss = wave_sum(y * y);
    if (lane == 0) squares[wave] = ss;
    __syncthreads();
    if (tid >= Dv) return;
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total += squares[w];      // of threads beyond the columns: zeros
    out[((size_t)n * n_heads + head) * Dv + tid] =
        float_to_bf16(y * rsqrtf(total / (float)Dv + eps) * gain * (g_col >= 0 ? g / (1.f + expf(-g)) : 1.f));
}

// Sum over the 16 lanes of a row of a wave by lane exchanges inside the vector unit (no trip through LDS's crossbar):
// neighbours, pairs of a quad, the mirrored half, the mirrored row.  Every lane of the row gets the sum.
__device__ __forceinline__ float row16_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));   // row_mirror
    return v;
}

// The sums over the 16 lanes of a row of four values, lane r getting that of value r % 4: neighbours, then pairs, swap the
// values that the other is to add up, so that five additions serve the four.
__device__ __forceinline__ float row16_sum_of_four(const float (&v)[4], int r) {
    auto moved = [](float x, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    using neighbour = std::integral_constant<int, 0xB1>;     // quad_perm [1,0,3,2]
    using pair = std::integral_constant<int, 0x4E>;          // quad_perm [2,3,0,1]
    using by4 = std::integral_constant<int, 0x124>;          // row_ror:4
    using by8 = std::integral_constant<int, 0x128>;          // row_ror:8
    const bool odd = r & 1, high = r & 2;
    const float a = (odd ? v[1] : v[0]) + moved(odd ? v[0] : v[1], neighbour());
    const float b = (odd ? v[3] : v[2]) + moved(odd ? v[2] : v[3], neighbour());
    float c = (high ? b : a) + moved(high ? a : b, pair());
    c += moved(c, by4());
    return c + moved(c, by8());
}

// How a step's runs of tokens are cut into segments: of ``len`` tokens (0: not at all), the last of a sequence perhaps shorter.
struct Segments {
    int len;
    bool by_sequence;      // of the two ways to place their states below, whichever needs fewer places
};

// Where a segment's state lies among those of the step.  By sequence: from one segment to the next either its first
// token moves on by a whole length or the sequence is the next one.  Else: segments of full length, which do not overlap,
// begin in different multiples of it; the last ones of their sequences have the odd places (two of them lie at least a
// whole segment apart).
__device__ __forceinline__ int segment_place(int first, int end, int seq, Segments cut) {
    const int multiple = first / cut.len;
    return cut.by_sequence ? multiple + seq : 2 * multiple + (first + cut.len >= end ? 1 : 0);
}

// The walk alone, of sizes that do not go by blocks (below), for a prompt's step in bfloat16 whose heads' columns are shared out (D a multiple of 8, rows and
// columns aligned to 16 bytes).  What bounds it: one prompt alone, a wave's chain of tokens (0.36 us each); cut into
// segments, the vector units (three instructions an element of the state and token, 78 us at 2,048 tokens of 24 heads of 128).  The 16 lanes of one row of a wave share two or four columns of the state, lane r
// keeping rows r * ROWS .. r * ROWS + ROWS - 1 of each (what a lane reads of q, k and the decays serves all its
// columns: LDS bandwidth, which every lane's reads of the same numbers would exhaust, is spent once per
// those columns); a token's outputs are sums over the row.  q, k and the decays lie in LDS so that the 16
// lanes' 16-byte pieces of a read are one contiguous run (no bank meets twice).  Blocks of 32 tokens: their q, k
// (16-byte pieces), decays (float4) and values are requested into registers while the block before is walked, so
// that the walk never waits for memory (16 tokens where four columns are shared, so that four workgroups fit a unit).
// Outputs go to the float workspace; the norm is the finishing kernel's.
#define GLA_WALK_THREADS 256
constexpr int gla_walk_tokens(int columns) { return columns == 4 ? 16 : 32; }
// KF: what is written (k) comes as floats [tokens, heads, D] from ``k_f32``, as the decays do, not as columns of the
// rows.  ``q_share`` neighbouring heads read the same q columns; a sequence's matrices begin ``state_stride`` floats
// after the sequence before it.
// BEFORE: the query reads the state before this token's write.
//
// Segments (cut.len > 0): a sequence of more than so many tokens is cut into segments of that length, walked by workgroups of
// their own at the same time: the first from the request's state, the others from zero.  Every segment leaves its last
// state in ``seg_state``; the kernels behind this one add what the states in front of the segments contribute.
template <int ROWS, int GLA_WALK_COLS, bool KF, bool BEFORE>
__global__ __launch_bounds__(GLA_WALK_THREADS) void gla_walk_kernel(
    const bf16_t* __restrict__ proj, int row_stride, int q_col, int k_col, int v_col, const float* __restrict__ alpha,
    const float* __restrict__ k_f32, int q_share, float* __restrict__ state, long long state_stride,
    const int* __restrict__ cu_q, const int* __restrict__ slots, int n_heads, int D, int Dv, float q_scale,
    float* __restrict__ raw_out, Segments cut, float* __restrict__ seg_state) {
    extern __shared__ float lds[];
    constexpr int C = GLA_WALK_COLS, TB = gla_walk_tokens(C), threads = GLA_WALK_THREADS;
    constexpr int slice = threads / 16 * C;      // columns a workgroup
    constexpr int Dp = 16 * ROWS;                // D filled up to the rows the lanes hold: what lies beyond D is zero
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int n_slices = (Dv + slice - 1) / slice;
    const int j0 = blockIdx.z % n_slices * slice, seg = blockIdx.z / n_slices;
    const int first = cu_q[seq] + seg * cut.len, end = cu_q[seq + 1];
    if (first >= end) return;
    const bool is_cut = cut.len > 0 && end - cu_q[seq] > cut.len;
    const int last = is_cut ? min(first + cut.len, end) : end;
    float* q_s = lds;               // [TB][Dp], row d = r * ROWS + i at (i / 4) * 64 + r * 4 + i % 4
    float* k_s = q_s + TB * Dp;
    float* al_s = k_s + TB * Dp;
    float* v_s = al_s + TB * Dp;    // [TB][slice]
    float* o_s = v_s + TB * slice;  // [TB][slice]: a block's outputs, written out together
    auto place = [](int d) { const int r = d / ROWS, i = d % ROWS; return (i / 4) * 64 + r * 4 + i % 4; };
    for (int i = tid; i < 3 * TB * Dp; i += threads) lds[i] = 0.f;
    const int jl = (tid / 16) * C, r = tid % 16;      // this lane's first column inside the slice, and its rows
    float* S_mem = state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv;
    float S[C][ROWS];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int d = r * ROWS + i, j = j0 + jl + c;
            S[c][i] = (seg == 0 && j < Dv && d < D) ? S_mem[(size_t)d * Dv + j] : 0.f;
        }
    if (is_cut) S_mem = seg_state + ((size_t)segment_place(first, end, seq, cut) * n_heads + head) * D * Dv;
    const int d8 = D / 8, d4 = D / 4;
    const int q_at = q_col + (head / q_share) * D, k_at = k_col + (head / q_share) * D;
    // What is on its way from memory is held in named registers, and the two steps below are written out piece by
    // piece: arrays indexed in loops ended up in scratch memory here, and a wave then waited for every piece twice.
    static_assert(TB * slice / threads == 4, "four values a thread and block");
    constexpr int NQ = (TB * Dp / 8 + threads - 1) / threads, NA = 2 * NQ;      // pieces of 16 bytes a thread and block
    static_assert(NQ <= 4, "pieces in named registers");
    uint4 rq0, rq1, rq2, rq3, rk0, rk1, rk2, rk3;
    float4 ra0, ra1, ra2, ra3, ra4, ra5, ra6, ra7;
    float4 rf0, rf1, rf2, rf3, rf4, rf5, rf6, rf7;
    float rv0, rv1, rv2, rv3;
    // pieces beyond the block's end repeat its last piece (every load is issued, none is conditional)
#define GLA_REQ_QK(i, Q, K)                                                                          \
    if constexpr ((i) < NQ) {                                                                        \
        const int idx = min(tid + (i) * threads, rnt * d8 - 1);                                       \
        const bf16_t* row = proj + (size_t)(rt0 + idx / d8) * row_stride + (idx % d8) * 8;            \
        Q = *reinterpret_cast<const uint4*>(row + q_at);                                             \
        if constexpr (!KF) K = *reinterpret_cast<const uint4*>(row + k_at);                          \
    }
#define GLA_REQ_F(i, A, SRC)                                                                         \
    if constexpr ((i) < NA) {                                                                        \
        const int idx = min(tid + (i) * threads, rnt * d4 - 1);                                       \
        A = *reinterpret_cast<const float4*>(SRC + ((size_t)(rt0 + idx / d4) * n_heads + head) * D + (idx % d4) * 4); \
    }
#define GLA_REQ_A(i, A) GLA_REQ_F(i, A, alpha)
#define GLA_REQ_V(i, V)                                                                              \
    do {                                                                                             \
        const int idx = min(tid + (i) * threads, rnt * slice - 1);                                    \
        V = bf16_to_float(proj[(size_t)(rt0 + idx / slice) * row_stride + v_col + head * Dv +         \
                               min(j0 + idx % slice, Dv - 1)]);                                      \
    } while (0)
#define GLA_REQUEST(T0)                                                                              \
    do {                                                                                             \
        const int rt0 = (T0), rnt = min(TB, last - rt0);                                                \
        GLA_REQ_QK(0, rq0, rk0); GLA_REQ_QK(1, rq1, rk1); GLA_REQ_QK(2, rq2, rk2); GLA_REQ_QK(3, rq3, rk3); \
        GLA_REQ_A(0, ra0); GLA_REQ_A(1, ra1); GLA_REQ_A(2, ra2); GLA_REQ_A(3, ra3);                  \
        GLA_REQ_A(4, ra4); GLA_REQ_A(5, ra5); GLA_REQ_A(6, ra6); GLA_REQ_A(7, ra7);                  \
        if constexpr (KF) {                                                                          \
            GLA_REQ_F(0, rf0, k_f32); GLA_REQ_F(1, rf1, k_f32); GLA_REQ_F(2, rf2, k_f32); GLA_REQ_F(3, rf3, k_f32); \
            GLA_REQ_F(4, rf4, k_f32); GLA_REQ_F(5, rf5, k_f32); GLA_REQ_F(6, rf6, k_f32); GLA_REQ_F(7, rf7, k_f32); \
        }                                                                                            \
        GLA_REQ_V(0, rv0); GLA_REQ_V(1, rv1); GLA_REQ_V(2, rv2); GLA_REQ_V(3, rv3);                  \
    } while (0)
    // two 16-bit halves of a word are rows d and d + 1
#define GLA_PUT(word_q, word_k, d)                                                                   \
    do {                                                                                             \
        const int p0 = base + place(d), p1 = base + place((d) + 1);                                  \
        q_s[p0] = __uint_as_float((word_q) << 16) * q_scale;                                         \
        q_s[p1] = __uint_as_float((word_q) & 0xffff0000u) * q_scale;                                 \
        if constexpr (!KF) {                                                                         \
            k_s[p0] = __uint_as_float((word_k) << 16);                                               \
            k_s[p1] = __uint_as_float((word_k) & 0xffff0000u);                                       \
        }                                                                                            \
    } while (0)
#define GLA_DEP_QK(i, Q, K)                                                                          \
    if constexpr ((i) < NQ) {                                                                        \
        const int idx = tid + (i) * threads;                                                         \
        if (idx < dnt * d8) {                                                                         \
            const int base = (idx / d8) * Dp, d0 = (idx % d8) * 8;                                   \
            GLA_PUT(Q.x, K.x, d0);                                                                   \
            GLA_PUT(Q.y, K.y, d0 + 2);                                                               \
            GLA_PUT(Q.z, K.z, d0 + 4);                                                               \
            GLA_PUT(Q.w, K.w, d0 + 6);                                                               \
        }                                                                                            \
    }
#define GLA_DEP_F(i, A, DST)                                                                         \
    if constexpr ((i) < NA) {   /* four rows of one lane (ROWS is a multiple of 4) */                 \
        const int idx = tid + (i) * threads;                                                         \
        if (idx < dnt * d4) *reinterpret_cast<float4*>(DST + (idx / d4) * Dp + place((idx % d4) * 4)) = A; \
    }
#define GLA_DEP_A(i, A) GLA_DEP_F(i, A, al_s)
#define GLA_DEP_V(i, V)                                                                              \
    do {                                                                                             \
        const int idx = tid + (i) * threads;                                                         \
        if (idx < dnt * slice) v_s[idx] = (j0 + idx % slice < Dv) ? V : 0.f;                          \
    } while (0)
#define GLA_DEPOSIT(T0)                                                                              \
    do {                                                                                             \
        const int dnt = min(TB, last - (T0));                                                         \
        GLA_DEP_QK(0, rq0, rk0); GLA_DEP_QK(1, rq1, rk1); GLA_DEP_QK(2, rq2, rk2); GLA_DEP_QK(3, rq3, rk3); \
        GLA_DEP_A(0, ra0); GLA_DEP_A(1, ra1); GLA_DEP_A(2, ra2); GLA_DEP_A(3, ra3);                  \
        GLA_DEP_A(4, ra4); GLA_DEP_A(5, ra5); GLA_DEP_A(6, ra6); GLA_DEP_A(7, ra7);                  \
        if constexpr (KF) {                                                                          \
            GLA_DEP_F(0, rf0, k_s); GLA_DEP_F(1, rf1, k_s); GLA_DEP_F(2, rf2, k_s); GLA_DEP_F(3, rf3, k_s); \
            GLA_DEP_F(4, rf4, k_s); GLA_DEP_F(5, rf5, k_s); GLA_DEP_F(6, rf6, k_s); GLA_DEP_F(7, rf7, k_s); \
        }                                                                                            \
        GLA_DEP_V(0, rv0); GLA_DEP_V(1, rv1); GLA_DEP_V(2, rv2); GLA_DEP_V(3, rv3);                  \
    } while (0)
    // One round before the first block only requests it (each of the two steps is written once, so that the pieces
    // on their way stay in registers).
    for (int t0 = first - TB; t0 < last; t0 += TB) {
        const int nt = min(TB, last - t0);
        if (t0 >= first) GLA_DEPOSIT(t0);
        __syncthreads();   // in the first round: the zeros are in place before the first pieces land on them
        if (t0 + TB < last) GLA_REQUEST(t0 + TB);
        if (t0 < first) continue;   // uniform
        // a token's q, k and decays are read from LDS while the token before is worked on
        float4 qn[ROWS / 4], kn[ROWS / 4], an[ROWS / 4];
        auto fetch = [&](int t) {
#pragma unroll
            for (int i = 0; i < ROWS / 4; ++i) {
                const int at = t * Dp + i * 64 + r * 4;
                qn[i] = *reinterpret_cast<const float4*>(q_s + at);
                kn[i] = *reinterpret_cast<const float4*>(k_s + at);
                an[i] = *reinterpret_cast<const float4*>(al_s + at);
            }
        };
        fetch(0);
        for (int t = 0; t < nt; ++t) {
            float4 qv[ROWS / 4], kv[ROWS / 4], av[ROWS / 4];
            float vv[C];
#pragma unroll
            for (int i = 0; i < ROWS / 4; ++i) { qv[i] = qn[i]; kv[i] = kn[i]; av[i] = an[i]; }
            if constexpr (C == 4) {
                const float4 v4 = *reinterpret_cast<const float4*>(v_s + t * slice + jl);
                vv[0] = v4.x; vv[1] = v4.y; vv[2] = v4.z; vv[3] = v4.w;
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) vv[c] = v_s[t * slice + jl + c];
            }
            fetch(min(t + 1, TB - 1));
            float sums[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float v = vv[c];
                float acc = 0.f;
#pragma unroll
                for (int i = 0; i < ROWS / 4; ++i) {
                    if (BEFORE) {
                        acc += qv[i].x * S[c][4 * i];
                        acc += qv[i].y * S[c][4 * i + 1];
                        acc += qv[i].z * S[c][4 * i + 2];
                        acc += qv[i].w * S[c][4 * i + 3];
                    }
                    S[c][4 * i] = av[i].x * S[c][4 * i] + kv[i].x * v;
                    S[c][4 * i + 1] = av[i].y * S[c][4 * i + 1] + kv[i].y * v;
                    S[c][4 * i + 2] = av[i].z * S[c][4 * i + 2] + kv[i].z * v;
                    S[c][4 * i + 3] = av[i].w * S[c][4 * i + 3] + kv[i].w * v;
                    if (!BEFORE) {
                        acc += qv[i].x * S[c][4 * i];
                        acc += qv[i].y * S[c][4 * i + 1];
                        acc += qv[i].z * S[c][4 * i + 2];
                        acc += qv[i].w * S[c][4 * i + 3];
                    }
                }
                sums[c] = acc;
            }
            if constexpr (C == 4) {
                const float sum = row16_sum_of_four(sums, r);
                if (r < 4) o_s[t * slice + jl + r] = sum;
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const float sum = row16_sum(sums[c]);
                    if (r == 0) o_s[t * slice + jl + c] = sum;
                }
            }
        }
        __syncthreads();
        for (int idx = tid; idx < nt * slice; idx += threads)
            if (j0 + idx % slice < Dv)
                raw_out[((size_t)(t0 + idx / slice) * n_heads + head) * Dv + j0 + idx % slice] = o_s[idx];
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int d = r * ROWS + i, j = j0 + jl + c;
            if (j < Dv && d < D) S_mem[(size_t)d * Dv + j] = S[c][i];
        }
}

#undef GLA_REQ_QK
#undef GLA_REQ_A
#undef GLA_REQ_F
#undef GLA_DEP_F
#undef GLA_REQ_V
#undef GLA_REQUEST
#undef GLA_PUT
#undef GLA_DEP_QK
#undef GLA_DEP_A
#undef GLA_DEP_V
#undef GLA_DEPOSIT

// The products of the decays from a segment's beginning on, in place of the decays (segments behind a sequence's first).
// A thread a channel.
__global__ __launch_bounds__(256) void segment_decays_kernel(float* __restrict__ alpha, const int* __restrict__ cu_q,
                                                             int channels, int seg_len) {
    const int seq = blockIdx.z, c = blockIdx.y * 256 + threadIdx.x;
    const int first = cu_q[seq] + (blockIdx.x + 1) * seg_len, end = cu_q[seq + 1];
    if (first >= end || c >= channels) return;
    const int n = min(seg_len, end - first);
    float* a = alpha + (size_t)first * channels + c;
    float p = 1.f;
    constexpr int AHEAD = 16;
    float next[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) next[i] = a[(size_t)min(i, n - 1) * channels];
    for (int t = 0; t < n; t += AHEAD) {
        float now[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) now[i] = next[i];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) next[i] = a[(size_t)min(t + AHEAD + i, n - 1) * channels];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            p *= now[i];
            if (t + i < n) a[(size_t)(t + i) * channels] = p;
        }
    }
}

// The state in front of every segment, in place of the segment's own last state; the state behind the last goes to the
// request's slot.  A thread four neighbouring elements of a matrix.
__global__ __launch_bounds__(256) void segment_states_kernel(const float* __restrict__ decays, float* __restrict__ seg_state,
                                                             float* __restrict__ state, long long state_stride,
                                                             const int* __restrict__ cu_q, const int* __restrict__ slots,
                                                             int n_heads, int D, int Dv, Segments cut) {
    const int seq = blockIdx.z, head = blockIdx.y, at = (blockIdx.x * 256 + threadIdx.x) * 4;
    const int begin = cu_q[seq], end = cu_q[seq + 1], seg_len = cut.len;
    if (end - begin <= seg_len || at >= D * Dv) return;
    const int d = at / Dv;
    auto matrix = [&](int first) {
        return reinterpret_cast<float4*>(seg_state + ((size_t)segment_place(first, end, seq, cut) * n_heads + head) * D * Dv + at);
    };
    auto decay = [&](int first) { return decays[((size_t)(min(first + seg_len, end) - 1) * n_heads + head) * D + d]; };
    float4 S = *matrix(begin), local = *matrix(begin + seg_len);
    float a = decay(begin + seg_len);
    for (int first = begin + seg_len; first < end; first += seg_len) {
        const int next = first + seg_len < end ? first + seg_len : first;
        float4* here = matrix(first);
        const float4 now = local;
        const float now_a = a;
        if (next != first) {      // before the store below, which the compiler must not assume to lie elsewhere
            local = *matrix(next);
            a = decay(next);
        }
        *here = S;
        S = make_float4(now_a * S.x + now.x, now_a * S.y + now.y, now_a * S.z + now.z, now_a * S.w + now.w);
    }
    *reinterpret_cast<float4*>(state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv + at) = S;
}

// o_t += (q_t * P_t)^T S for the tokens of a segment, with the state S in front of it and the products P of the decays up
// to the token: a product [tokens, D] x [D, Dv] in float on the matrix cores (v_mfma_f32_16x16x4_f32).  A wave has 32
// tokens and 64 columns, a lane four neighbouring columns (one of each of four tiles), so that S and o move 16 bytes a
// lane; instruction i of a step of 16 channels takes the channels 4 * (lane / 16) + i.
typedef float segf32x4 __attribute__((ext_vector_type(4)));
template <bool BEFORE>
__global__ __launch_bounds__(256) void segment_outputs_kernel(const bf16_t* __restrict__ proj, int row_stride, int q_col, int q_share,
                                                              const float* __restrict__ decays, const float* __restrict__ seg_state,
                                                              const int* __restrict__ cu_q, int n_heads, int D, int Dv, float q_scale,
                                                              float* __restrict__ raw, Segments cut) {
    const int seq = blockIdx.z, head = blockIdx.y % n_heads, j0 = blockIdx.y / n_heads * 64, seg_len = cut.len;
    const int first = cu_q[seq] + (blockIdx.x + 1) * seg_len, end = cu_q[seq + 1];
    const int t0 = first + threadIdx.x / SIA_WAVE * 32;
    if (t0 >= end) return;      // a wave leaves as a whole; no barriers below
    const int last = min(first + seg_len, end);
    const int lane = threadIdx.x % SIA_WAVE, r = lane % 16, g = lane / 16;
    const int j = j0 + 4 * r;
    const bool has_j = j < Dv;      // Dv is a multiple of four
    const float* S = seg_state + ((size_t)segment_place(first, end, seq, cut) * n_heads + head) * D * Dv + (has_j ? j : 0);
    const int q_at = q_col + head / q_share * D;

    segf32x4 acc[2][4];      // [tile of 16 tokens][column of the four] = tokens 4 g .. 4 g + 3
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + 16 * m + 4 * g + i;
            float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
            if (t < last && has_j) o = *reinterpret_cast<const float4*>(raw + ((size_t)t * n_heads + head) * Dv + j);
            acc[m][0][i] = o.x; acc[m][1][i] = o.y; acc[m][2][i] = o.z; acc[m][3][i] = o.w;
        }
    for (int d0 = 0; d0 < D; d0 += 16) {
        const int d = d0 + 4 * g;
        const bool has_d = d < D;      // D is a multiple of eight
        float a[2][4];
        float4 b[4];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int t = min(t0 + 16 * m + r, last - 1);      // rows past the end repeat the last and are not stored
            const uint2 q = *reinterpret_cast<const uint2*>(proj + (size_t)t * row_stride + q_at + (has_d ? d : 0));
            float4 p = make_float4(1.f, 1.f, 1.f, 1.f);
            if (!BEFORE || t > first)
                p = *reinterpret_cast<const float4*>(decays + ((size_t)(BEFORE ? t - 1 : t) * n_heads + head) * D + (has_d ? d : 0));
            const float z = has_d ? q_scale : 0.f;
            a[m][0] = __uint_as_float(q.x << 16) * z * p.x;
            a[m][1] = __uint_as_float(q.x & 0xffff0000u) * z * p.y;
            a[m][2] = __uint_as_float(q.y << 16) * z * p.z;
            a[m][3] = __uint_as_float(q.y & 0xffff0000u) * z * p.w;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = *reinterpret_cast<const float4*>(S + (size_t)(has_d ? d + i : 0) * Dv);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                acc[m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][i], b[i].x, acc[m][0], 0, 0, 0);
                acc[m][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][i], b[i].y, acc[m][1], 0, 0, 0);
                acc[m][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][i], b[i].z, acc[m][2], 0, 0, 0);
                acc[m][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][i], b[i].w, acc[m][3], 0, 0, 0);
            }
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + 16 * m + 4 * g + i;
            if (t < last && has_j)
                *reinterpret_cast<float4*>(raw + ((size_t)t * n_heads + head) * Dv + j) =
                    make_float4(acc[m][0][i], acc[m][1][i], acc[m][2][i], acc[m][3][i]);
        }
}

// The recurrence by blocks of 16 tokens on the matrix cores, for runs of a prompt in bfloat16: the chunked form of Yang and others, "Gated linear
// attention transformers with hardware-efficient training" (2023).
// With P_t the products of a block's decays up to token t, R_s those behind token s and S the state in front of the block:
//   o_t = (q_t * P_t)^T S + sum_(s <= t) A_ts v_s,   A_ts = sum_d q_td k_sd prod_(s < r <= t) alpha_rd,   S <- diag(P_15) S + sum_s (k_s * R_s) v_s^T
// A = (q P) (k / P)^T where no channel of 64 has decayed to 2^-40 within the block; else its part of A is made pair by pair on the vector units,
// from products of decays alone, lane (s, four channels) carrying k_s prod alpha from token to token.
// A workgroup of BLOCK_D / 16 waves has a (segment, head) and BLOCK_D columns of its state, a wave 16 of them, D x 16 floats in the registers in which
// the matrix cores leave them: lane (r, g) has S[16 b + 4 g + i][r], which is also how S^T is read as a left operand when instruction i of a
// block of channels takes the channels 4 g + i.  S and A are multiplied as floats (v_mfma_f32_16x16x4_f32); k R goes into the state's
// product as the three bfloat16 numbers that it is the sum of, values as they are (v_mfma_f32_16x16x16_bf16, float sums).
// All but the values is staged in LDS a block at a time, requested a block ahead.
// A run or segment with a number of more than 2^32 among its q, k and v, or one that is not finite, is then taken again, token by token on
// the vector units (one NaN among 2,048 tokens of 24 heads of 128 x 128 127 -> 630 us, beside 63 tokens in a run of 449 458 -> 600): a product by zero carries such a number to the tokens of its block in front of it, and k / P or q k
// may leave the range of floats where the recurrence does not.
// Segments behind one another: with OUT false only what a segment adds to the state (all but a sequence's last), and the product of its
// decays; block_states_kernel makes the states in front of the segments; with OUT true the outputs, from there.
// What bounds it: the barriers between staging, A and products, LDS (a wave reads 13 KiB a block) and the float products (36 of 32
// cycles), by reading the code, about in equal parts; 128 registers leave two workgroups a unit.
// us, a layer's recurrence with its decays and the finishing kernel, by the walk (with two or four columns a lane group) -> by blocks:  24 heads
// of 128 x 128, one run of 64 tokens 38 -> 31, 128 60 -> 49, 200 83 -> 52, 512 103 -> 62, 2,048 222 -> 131;  8 runs of 64 84 -> 42, 16 of 200 259 -> 135,
// one run of 449 beside 63 tokens 740 -> 466;  24 of 64 x 64, 2,048 117 -> 70, 16 of 200 132 -> 72;  8 of 128 x 64, 2,048 109 -> 65.  With decays that go
// pair by pair, lower-bounded gates, keys as floats:  24 of 128 x 128, 128 57 -> 60, 2,048 210 -> 147, 16 of 200 241 -> 168.
// D up to BLOCK_D and a multiple of 16.  KF, q_share, state_stride, BEFORE and the segments as in the walk above.
constexpr int BLOCK_TOKENS = 16, BLOCK_COLUMN = BLOCK_TOKENS + 4;
constexpr float BLOCK_LEAST = 9.094947e-13f;      // 2^-40
constexpr float BLOCK_MOST = 4294967296.f;        // 2^32
constexpr float BLOCK_SCALE = 1099511627776.f;    // 2^40: k R, which may be as small as floats get, goes into its parts that much larger
constexpr int BLOCK_MOST_V = 0x4f80;              // the same in bfloat16
typedef short segshort4 __attribute__((ext_vector_type(4)));
template <int BLOCK_D, bool OUT, bool KF, bool BEFORE>
__global__ __launch_bounds__(BLOCK_D / 16 * SIA_WAVE, 4) void gla_blocks_kernel(
    const bf16_t* __restrict__ proj, int row_stride, int q_col, int k_col, int v_col, const float* __restrict__ alpha,
    const float* __restrict__ k_f32, int q_share, float* __restrict__ state, long long state_stride,
    const int* __restrict__ cu_q, const int* __restrict__ slots, int n_heads, int D, int Dv, float q_scale,
    float* __restrict__ raw_out, Segments cut, float* __restrict__ seg_state, float* __restrict__ seg_decay) {
    constexpr int T = BLOCK_TOKENS, TILES = BLOCK_D / 16, BLOCK_WAVES = BLOCK_D / 16, BLOCK_ROW = BLOCK_D + 4, PARTS = 3;
    __shared__ __attribute__((aligned(16))) float qp_s[OUT ? T * BLOCK_ROW : 4];      // q P, by token
    __shared__ __attribute__((aligned(16))) float kx_s[OUT ? T * BLOCK_ROW : 4];      // k / P, or k
    __shared__ __attribute__((aligned(16))) float q_s[OUT ? T * BLOCK_ROW : 4], al_s[OUT ? T * BLOCK_ROW : 4];
    __shared__ __attribute__((aligned(16))) uint2 kr_s[PARTS][BLOCK_D][4 + 1];       // parts of k R, by channel: four tokens a piece
    __shared__ __attribute__((aligned(16))) float end_s[BLOCK_D];                     // P of the block's last token
    __shared__ __attribute__((aligned(16))) float a_s[OUT ? BLOCK_WAVES * T * BLOCK_COLUMN : 4];      // [wave's channels][t][s]
    __shared__ int by_pairs[2];      // of 64 channels each
    __shared__ int any_odd;
    const int n_slices = (Dv + BLOCK_D - 1) / BLOCK_D;
    const int seq = blockIdx.x, head = blockIdx.y, slice = blockIdx.z % n_slices, seg = blockIdx.z / n_slices;
    const int begin = cu_q[seq], first = begin + seg * cut.len, end = cu_q[seq + 1];
    if (first >= end) return;
    const bool is_cut = cut.len > 0 && end - begin > cut.len;
    const int last = is_cut ? min(first + cut.len, end) : end;
    if (!is_cut && seg > 0) return;
    if (!OUT && (!is_cut || last == end)) return;
    const int tid = threadIdx.x, lane = tid % SIA_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / SIA_WAVE), r = lane % 16, g = lane / 16;
    const int j = slice * BLOCK_D + wave * 16 + r;
    const bool has_j = slice * BLOCK_D + wave * 16 < Dv;      // Dv is a multiple of 16: a wave has columns or has none
    const int matrix = D * Dv, from = 4 * g * Dv + j;      // a tile's rows 4 g .. 4 g + 3 begin there
    float* const own = state + (size_t)slots[seq] * state_stride + (size_t)head * matrix;
    float* const segment = seg_state + ((size_t)(is_cut ? segment_place(first, end, seq, cut) : 0) * n_heads + head) * matrix;
    segf32x4 S[TILES];
#pragma unroll
    for (int b = 0; b < TILES; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            S[b][i] = 0.f;
            if (OUT && has_j && 16 * b < D) S[b][i] = (is_cut ? segment : own)[(16 * b + i) * Dv + from];
        }
    // Staging: a thread has a channel.  What it makes of the block:  0 q P;  1 k R;  2 k / P
    const int role = __builtin_amdgcn_readfirstlane(tid / BLOCK_D), ch = tid % BLOCK_D;
    const bool has_ch = ch < D, stages = OUT ? role < 3 : role == 1;
    const int at = head / q_share * D + (has_ch ? ch : 0), at_f = head * D + (has_ch ? ch : 0);
    float x[T], al[T];
    uint16_t v_next[4];
    const unsigned x_at = (unsigned)((role == 0 ? q_col : k_col) + at), f_at = (unsigned)at_f, v_at = (unsigned)(v_col + head * Dv + j);
    auto request = [&](int t0) {      // tokens behind the last repeat it
        auto row = [&](int t) { return (size_t)__builtin_amdgcn_readfirstlane(min(t0 + t, last - 1)); };      // it begins at a scalar
        if (stages) {
            if (KF && role != 0)      // one branch, nothing converted in it: a conversion waits for its load
#pragma unroll
                for (int t = 0; t < T; ++t) x[t] = (k_f32 + row(t) * n_heads * D)[f_at];
            else
#pragma unroll
                for (int t = 0; t < T; ++t) x[t] = __uint_as_float((uint32_t)(proj + row(t) * row_stride)[x_at]);
#pragma unroll
            for (int t = 0; t < T; ++t) al[t] = (alpha + row(t) * n_heads * D)[f_at];
        }
        if (has_j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v_next[i] = (proj + (size_t)min(t0 + 4 * g + i, last - 1) * row_stride)[v_at];
    };
    request(first);
    float seg_product = 1.f;
    if (tid == 0) any_odd = 0;
    bool odd = false;
    for (int t0 = first; t0 < last; t0 += T) {
        const int nt = min(T, last - t0);
        if (stages && (!KF || role == 0))
#pragma unroll
            for (int t = 0; t < T; ++t) x[t] = __uint_as_float(__float_as_uint(x[t]) << 16);
        if (nt < T || !has_ch)
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (!has_ch || t >= nt) x[t] = 0.f, al[t] = 1.f;
        const segshort4 v = {(short)v_next[0], (short)v_next[1], (short)v_next[2], (short)v_next[3]};      // of no weight behind the last token: k is zero there
        if (stages) {
            float most[2] = {0.f, 0.f};      // NaN and infinities stay
#pragma unroll
            for (int t = 0; t < T; ++t) most[t & 1] += fabsf(x[t]);
            odd |= !(most[0] + most[1] <= BLOCK_MOST);
        }
        if (role == 1) {
            float p = BLOCK_SCALE;
#pragma unroll
            for (int t = T - 1; t >= 0; --t) {
                x[t] *= p;
                p *= al[t];
            }
            p *= 1.f / BLOCK_SCALE;
            end_s[ch] = p;
            seg_product *= p;
            odd |= !(p <= BLOCK_MOST);      // (decays are at most one)
#pragma unroll
            for (int e = 0; e < PARTS; ++e)
#pragma unroll
                for (int t = 0; t < T; t += 4) {
                    uint2 u;
                    u.x = bf16_pair(x[t], x[t + 1]), u.y = bf16_pair(x[t + 2], x[t + 3]);
                    kr_s[e][ch][t / 4] = u;
                    x[t] -= __uint_as_float(u.x << 16), x[t + 1] -= __uint_as_float(u.x & 0xffff0000u);
                    x[t + 2] -= __uint_as_float(u.y << 16), x[t + 3] -= __uint_as_float(u.y & 0xffff0000u);
                }
        } else if (OUT && stages) {
            float p = 1.f;
#pragma unroll
            for (int t = 0; t < T; ++t) p *= al[t];
            const bool pairs = __any(!(p >= BLOCK_LEAST));
            p = 1.f;
            if (role == 0) {
                if (lane == 0) by_pairs[wave % (BLOCK_D / 64)] = pairs;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if (!BEFORE) p *= al[t];
                    qp_s[t * BLOCK_ROW + ch] = x[t] * q_scale * p;
                    if (BEFORE) p *= al[t];
                }
                if (pairs)
#pragma unroll
                    for (int t = 0; t < T; ++t) q_s[t * BLOCK_ROW + ch] = x[t] * q_scale, al_s[t * BLOCK_ROW + ch] = al[t];
            } else {
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    p *= al[t];
                    kx_s[t * BLOCK_ROW + ch] = pairs ? x[t] : x[t] / p;
                }
            }
        }
        __syncthreads();
        if (t0 + T < last) request(t0 + T);
        if (OUT) {
            const int c = wave * 16 + 4 * g;      // the lane's four of the wave's 16 channels
            const float4 k4 = *reinterpret_cast<const float4*>(kx_s + r * BLOCK_ROW + c);
            segf32x4 A = {0.f, 0.f, 0.f, 0.f};      // A_ts of t = 4 g + i, s = r
            if (!by_pairs[wave / 4]) {
                const float4 q4 = *reinterpret_cast<const float4*>(qp_s + r * BLOCK_ROW + c);
                A = __builtin_amdgcn_mfma_f32_16x16x4f32(q4.x, k4.x, A, 0, 0, 0);
                A = __builtin_amdgcn_mfma_f32_16x16x4f32(q4.y, k4.y, A, 0, 0, 0);
                A = __builtin_amdgcn_mfma_f32_16x16x4f32(q4.z, k4.z, A, 0, 0, 0);
                A = __builtin_amdgcn_mfma_f32_16x16x4f32(q4.w, k4.w, A, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (BEFORE ? 4 * g + i <= r : 4 * g + i < r) A[i] = 0.f;
            } else {
                // a token's sums of the four lane groups go to its row by a product with a row of ones
                float4 ck = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 2
                for (int t = 0; t < T; ++t) {
                    const float4 q4 = *reinterpret_cast<const float4*>(q_s + t * BLOCK_ROW + c);
                    const float4 a4 = *reinterpret_cast<const float4*>(al_s + t * BLOCK_ROW + c);
                    if (!BEFORE) ck = t == r ? k4 : make_float4(ck.x * a4.x, ck.y * a4.y, ck.z * a4.z, ck.w * a4.w);
                    const float sum = (q4.x * ck.x + q4.y * ck.y) + (q4.z * ck.z + q4.w * ck.w);
                    A = __builtin_amdgcn_mfma_f32_16x16x4f32(t == r ? 1.f : 0.f, sum, A, 0, 0, 0);
                    if (BEFORE) ck = t == r ? k4 : make_float4(ck.x * a4.x, ck.y * a4.y, ck.z * a4.z, ck.w * a4.w);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) a_s[(wave * T + 4 * g + i) * BLOCK_COLUMN + r] = A[i];
            __syncthreads();
        }
        if (has_j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) odd |= (v[i] & 0x7fff) > BLOCK_MOST_V;
            if (OUT) {
                segf32x4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                float4 a4 = make_float4(0.f, 0.f, 0.f, 0.f);      // A_ts of t = r, s = 4 g .. 4 g + 3
#pragma unroll 2
                for (int w = 0; w < BLOCK_WAVES; ++w) {
                    const float4 part = *reinterpret_cast<const float4*>(a_s + (w * T + r) * BLOCK_COLUMN + 4 * g);
                    a4.x += part.x, a4.y += part.y, a4.z += part.z, a4.w += part.w;
                }
#pragma unroll
                for (int b = 0; b < TILES; ++b) {
                    const float4 qp = *reinterpret_cast<const float4*>(qp_s + r * BLOCK_ROW + 16 * b + 4 * g);
                    o[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[b][0], qp.x, o[b & 1], 0, 0, 0);
                    o[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[b][1], qp.y, o[b & 1], 0, 0, 0);
                    o[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[b][2], qp.z, o[b & 1], 0, 0, 0);
                    o[b & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[b][3], qp.w, o[b & 1], 0, 0, 0);
                    if (b % 2) __builtin_amdgcn_sched_barrier(0);      // operands of two steps in registers, not of all
                }
                segf32x4 av = {0.f, 0.f, 0.f, 0.f};
                av = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_to_float((uint16_t)v[0]), a4.x, av, 0, 0, 0);
                av = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_to_float((uint16_t)v[1]), a4.y, av, 0, 0, 0);
                av = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_to_float((uint16_t)v[2]), a4.z, av, 0, 0, 0);
                av = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_to_float((uint16_t)v[3]), a4.w, av, 0, 0, 0);
                // columns 4 g .. 4 g + 3 of token r
                const segf32x4 sum = (o[0] + o[1]) + av;
                if (r < nt)
                    *reinterpret_cast<segf32x4*>(raw_out + ((size_t)(t0 + r) * n_heads + head) * Dv + slice * BLOCK_D + wave * 16 + 4 * g) = sum;
            }
#pragma unroll
            for (int b = 0; b < TILES; ++b) {
                const float4 p = *reinterpret_cast<const float4*>(end_s + 16 * b + 4 * g);
                segf32x4 added = {0.f, 0.f, 0.f, 0.f};      // small parts first
#pragma unroll
                for (int e = PARTS - 1; e >= 0; --e)
                    added = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(segshort4, kr_s[e][16 * b + r][g]), v, added, 0, 0, 0);
                added *= 1.f / BLOCK_SCALE;
                S[b][0] = fmaf(S[b][0], p.x, added[0]), S[b][1] = fmaf(S[b][1], p.y, added[1]);
                S[b][2] = fmaf(S[b][2], p.z, added[2]), S[b][3] = fmaf(S[b][3], p.w, added[3]);
                if (b % 2) __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    if (odd) any_odd = 1;
    __syncthreads();
    if (!OUT && role == 1 && has_ch && slice == 0)
        seg_decay[((size_t)segment_place(first, end, seq, cut) * n_heads + head) * D + ch] = seg_product;
    if (!has_j) return;
    if (any_odd) {
        const size_t per_token = (size_t)n_heads * D;
        const int shared = head / q_share * D + 4 * g, own_at = head * D + 4 * g;
        float s[TILES][4];      // (S itself, in the registers of the products, would spill)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // what is written again has been written
#pragma unroll
        for (int b = 0; b < TILES; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[b][i] = OUT && 16 * b < D ? (is_cut ? segment : own)[(16 * b + i) * Dv + from] : 0.f;
#pragma clang loop unroll(disable)
        for (int n = first; n < last; ++n) {
            const bf16_t* row = proj + (size_t)n * row_stride;
            const float vj = bf16_to_float(row[v_at]);
            float o = 0.f;
#pragma unroll
            for (int b = 0; b < TILES; ++b)
                if (16 * b < D) {
                    const float4 a = *reinterpret_cast<const float4*>(alpha + n * per_token + own_at + 16 * b);
                    float4 k, q;
                    if constexpr (KF)
                        k = *reinterpret_cast<const float4*>(k_f32 + n * per_token + own_at + 16 * b);
                    else {
                        const ushort4 u = *reinterpret_cast<const ushort4*>(row + k_col + shared + 16 * b);
                        k = make_float4(bf16_to_float(u.x), bf16_to_float(u.y), bf16_to_float(u.z), bf16_to_float(u.w));
                    }
                    if constexpr (OUT) {
                        const ushort4 u = *reinterpret_cast<const ushort4*>(row + q_col + shared + 16 * b);
                        q = make_float4(bf16_to_float(u.x), bf16_to_float(u.y), bf16_to_float(u.z), bf16_to_float(u.w));
                    }
                    const float ai[4] = {a.x, a.y, a.z, a.w}, ki[4] = {k.x, k.y, k.z, k.w}, qi[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float moved = fmaf(ki[i], vj, ai[i] * s[b][i]);
                        if constexpr (OUT) o = fmaf(qi[i] * q_scale, BEFORE ? s[b][i] : moved, o);
                        s[b][i] = moved;
                    }
                }
            if constexpr (OUT) {
                o += __shfl_xor(o, 16, SIA_WAVE);
                o += __shfl_xor(o, 32, SIA_WAVE);
                if (g == 0) raw_out[((size_t)n * n_heads + head) * Dv + j] = o;
            }
        }
        if (!OUT || last == end)
#pragma unroll
            for (int b = 0; b < TILES; ++b)
                if (16 * b < D)
#pragma unroll
                    for (int i = 0; i < 4; ++i) (OUT ? own : segment)[(16 * b + i) * Dv + from] = s[b][i];
        return;
    }
    if (!OUT || last == end)
#pragma unroll
        for (int b = 0; b < TILES; ++b)
            if (16 * b < D)      // a multiple of 16
#pragma unroll
                for (int i = 0; i < 4; ++i) (OUT ? own : segment)[(16 * b + i) * Dv + from] = S[b][i];
}

// The state in front of every segment of a sequence that is cut, in place of what the segment adds to it.  A thread four neighbouring
// elements of a matrix.
__global__ __launch_bounds__(256) void block_states_kernel(const float* __restrict__ seg_decay, float* __restrict__ seg_state,
                                                           const float* __restrict__ state, long long state_stride,
                                                           const int* __restrict__ cu_q, const int* __restrict__ slots, int n_heads,
                                                           int D, int Dv, Segments cut) {
    const int seq = blockIdx.z, head = blockIdx.y, at = (blockIdx.x * 256 + threadIdx.x) * 4;
    const int begin = cu_q[seq], end = cu_q[seq + 1];
    if (end - begin <= cut.len || at >= D * Dv) return;
    const int d = at / Dv;
    float4 S = *reinterpret_cast<const float4*>(state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv + at);
    auto place = [&](int first) { return (size_t)segment_place(first, end, seq, cut) * n_heads + head; };
    auto matrix = [&](int first) { return reinterpret_cast<float4*>(seg_state + place(first) * D * Dv + at); };
    float4 added = *matrix(begin);
    float a = seg_decay[place(begin) * D + d];
    for (int first = begin; first < end; first += cut.len) {
        const bool more = first + 2 * cut.len < end;      // the segment behind this one is not the last
        const float4 now = added;
        const float now_a = a;
        if (more) added = *matrix(first + cut.len), a = seg_decay[place(first + cut.len) * D + d];
        *matrix(first) = S;
        if (first + cut.len < end) S = make_float4(now_a * S.x + now.x, now_a * S.y + now.y, now_a * S.z + now.z, now_a * S.w + now.w);
    }
}

// alpha[n, c] = exp(logsigmoid(a2_bias[c] + sum_m a[n, m] * A2[c, m]) / tau) for every token n and key channel c of all
// heads: a thread a channel, eight tokens a workgroup (their low-rank inputs staged in LDS, a channel's row of A2
// read once for the eight).
#define GLA_DECAY_TOKENS 8
template <typename T>
__global__ __launch_bounds__(256) void gla_decay_kernel(const T* __restrict__ proj, int row_stride, int a_col,
                                                        const T* __restrict__ a2, const float* __restrict__ a2_bias,
                                                        float* __restrict__ alpha, int n_tokens, int channels, int rank,
                                                        float tau_inv) {
    extern __shared__ float a_s[];   // [GLA_DECAY_TOKENS][rank]
    const int n0 = blockIdx.x * GLA_DECAY_TOKENS, nt = min(GLA_DECAY_TOKENS, n_tokens - n0);
    for (int idx = threadIdx.x; idx < nt * rank; idx += blockDim.x)
        a_s[idx] = to_float(proj[(size_t)(n0 + idx / rank) * row_stride + a_col + idx % rank]);
    __syncthreads();
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= channels) return;
    const T* w = a2 + (size_t)c * rank;
    float z[GLA_DECAY_TOKENS];
    const float b = a2_bias ? a2_bias[c] : 0.f;
#pragma unroll
    for (int t = 0; t < GLA_DECAY_TOKENS; ++t) z[t] = b;
    for (int m = 0; m < rank; ++m) {
        const float wm = to_float(w[m]);
#pragma unroll
        for (int t = 0; t < GLA_DECAY_TOKENS; ++t) z[t] += a_s[min(t, nt - 1) * rank + m] * wm;
    }
#pragma unroll
    for (int t = 0; t < GLA_DECAY_TOKENS; ++t)
        if (t < nt) alpha[(size_t)(n0 + t) * channels + c] = sigmoid_power(z[t], tau_inv);
}

// The same on the matrix cores (v_mfma_f32_16x16x32_bf16, float sums) where the rank is a multiple of 32 and rows lie on 16
// bytes: a wave has 64 channels of 32 tokens, A2's rows as the left operand, so that a lane holds four neighbouring
// channels of a token.  A thread a channel reads A2 two bytes a lane and a token's inputs from LDS once per channel.
// 2,048 tokens, 3,072 channels, rank 64: 65 -> 31 us, and 16 with sigmoid_power in place of exp and log1p, whose arithmetic
// then bound it (the decays are 25 MB).
typedef __bf16 recbf16x8 __attribute__((ext_vector_type(8)));
__global__ __launch_bounds__(256) void gla_decay_mfma_kernel(const bf16_t* __restrict__ proj, int row_stride, int a_col,
                                                             const bf16_t* __restrict__ a2, const float* __restrict__ a2_bias,
                                                             float* __restrict__ alpha, int n_tokens, int channels, int rank,
                                                             float tau_inv) {
    const int lane = threadIdx.x % SIA_WAVE, r = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * 32, c0 = (blockIdx.y * 4 + threadIdx.x / SIA_WAVE) * 64;
    if (c0 >= channels) return;      // a wave leaves as a whole; no barriers below
    // rows that do not exist are read as the last one and not stored
    const bf16_t *w[4], *a[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = a2 + (size_t)min(c0 + 16 * i + r, channels - 1) * rank + 8 * g;
#pragma unroll
    for (int t = 0; t < 2; ++t) a[t] = proj + (size_t)min(n0 + 16 * t + r, n_tokens - 1) * row_stride + a_col + 8 * g;
    segf32x4 z[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) z[t][i] = segf32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < rank; k += 32) {
        recbf16x8 wk[4], ak[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) wk[i] = __builtin_bit_cast(recbf16x8, *reinterpret_cast<const uint4*>(w[i] + k));
#pragma unroll
        for (int t = 0; t < 2; ++t) ak[t] = __builtin_bit_cast(recbf16x8, *reinterpret_cast<const uint4*>(a[t] + k));
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) z[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk[i], ak[t], z[t][i], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int n = n0 + 16 * t + r;
        if (n >= n_tokens) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = c0 + 16 * i + 4 * g;
            if (c >= channels) continue;      // channels are a multiple of four
            float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
            if (a2_bias) b = *reinterpret_cast<const float4*>(a2_bias + c);
            *reinterpret_cast<float4*>(alpha + (size_t)n * channels + c) =
                make_float4(sigmoid_power(z[t][i][0] + b.x, tau_inv), sigmoid_power(z[t][i][1] + b.y, tau_inv),
                            sigmoid_power(z[t][i][2] + b.z, tau_inv), sigmoid_power(z[t][i][3] + b.w, tau_inv));
        }
    }
}

// y = o * rsqrt(mean(o^2) + eps) * w * silu(g) for outputs left in a float workspace: a wave one (token, head) pair or four,
// whose loads are under way together (a workgroup of one wave a pair was bound by the dispatch of workgroups: 2,048 tokens of
// 24 heads of 128 25 -> 20 us).
#define GLA_FINISH_WAVES 4
template <typename T, int PAIRS>
__global__ __launch_bounds__(GLA_FINISH_WAVES * SIA_WAVE) void gla_finish_kernel(
    const float* __restrict__ raw, const T* __restrict__ proj, int row_stride, int g_col, const float* __restrict__ norm_w,
    T* __restrict__ out, int n_pairs, int n_heads, int Dv, float eps) {
    const int lane = threadIdx.x % SIA_WAVE;
    const int first = ((int)blockIdx.x * GLA_FINISH_WAVES + (int)threadIdx.x / SIA_WAVE) * PAIRS;
    if (first >= n_pairs) return;      // a wave leaves as a whole
    // a lane has every 64th pair of neighbouring elements (the last one alone where Dv is odd); Dv is at most 512
    constexpr int TURNS = 4;
    float2 o[TURNS][PAIRS];
    float ss[PAIRS] = {};
    int at[PAIRS], g_at[PAIRS];
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
        const int pair = min(first + i, n_pairs - 1), n = pair / n_heads;
        at[i] = pair;
        g_at[i] = n;
    }
#pragma unroll
    for (int k = 0; k < TURNS; ++k) {
        const int c = 2 * (lane + k * SIA_WAVE);
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) {
            const float* p = raw + (size_t)at[i] * Dv + c;
            o[k][i] = make_float2(0.f, 0.f);
            if (c + 1 < Dv) o[k][i] = make_float2(p[0], p[1]);
            else if (c < Dv) o[k][i].x = p[0];
        }
    }
#pragma unroll
    for (int k = 0; k < TURNS; ++k)
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) ss[i] += o[k][i].x * o[k][i].x + o[k][i].y * o[k][i].y;
    float inv[PAIRS];
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) inv[i] = rsqrtf(wave_sum(ss[i]) / (float)Dv + eps);
#pragma unroll
    for (int k = 0; k < TURNS; ++k) {
        const int c = 2 * (lane + k * SIA_WAVE);
        if (c >= Dv) break;
        const bool two = c + 1 < Dv;
        const float w0 = norm_w[c], w1 = two ? norm_w[c + 1] : 0.f;
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) {
            float f0 = 1.f, f1 = 1.f;
            if (g_col >= 0) {
                const T* g_row = proj + (size_t)g_at[i] * row_stride + g_col + (at[i] - g_at[i] * n_heads) * Dv + c;
                const float g0 = to_float(g_row[0]), g1 = two ? to_float(g_row[1]) : 0.f;
                f0 = g0 / (1.f + expf(-g0));
                f1 = g1 / (1.f + expf(-g1));
            }
            if (first + i >= n_pairs) continue;
            T* y = out + (size_t)at[i] * Dv + c;
            y[0] = from_float<T>(o[k][i].x * inv[i] * w0 * f0);
            if (two) y[1] = from_float<T>(o[k][i].y * inv[i] * w1 * f1);
        }
    }
}

// The same in bfloat16 for Dv a multiple of 8 and rows aligned to 16 bytes: a lane has eight neighbouring elements, 2^group_log lanes
// (Dv / 8 or the next power of two; the lanes behind Dv add zeros) share a pair, so that a wave has up to 64 pairs and all of a lane's loads,
// 16 bytes each, are on their way before the sum.  Bound by memory: 2,048 tokens of 24 heads of 128 move 50 MB, at 4.5 TB/s.
// us, the kernel above -> this one:  24 heads of 128, 33 tokens 3.9 -> 3.9, 64 4.3 -> 4.6, 128 4.7 -> 4.1, 512 6.4 -> 4.9, 1,024 10.2 -> 7.2, 2,048 17.6 -> 11.2, 4,096
// 34.4 -> 18.8;  24 of 64, 33 3.9 -> 4.0, 1,024 9.4 -> 5.0, 4,096 28.2 -> 11.0;  16 of 256, 64 4.6 -> 4.6, 2,048 19.0 -> 13.6;  4 of 512, 512 5.6 -> 4.0;  80 of
// 16, 2,048 41.7 -> 6.6.
__global__ __launch_bounds__(GLA_FINISH_WAVES * SIA_WAVE) void gla_finish_vec_kernel(
    const float* __restrict__ raw, const bf16_t* __restrict__ proj, int row_stride, int g_col, const float* __restrict__ norm_w,
    bf16_t* __restrict__ out, int n_pairs, int n_heads, int Dv, int group_log, float eps) {
    const long long id = (long long)blockIdx.x * (GLA_FINISH_WAVES * SIA_WAVE) + threadIdx.x;
    const int pair = (int)(id >> group_log), c = ((int)id & ((1 << group_log) - 1)) * 8;
    const bool live = pair < n_pairs && c < Dv;      // lanes without elements take part in the sums' exchanges
    Vec8<float> vo, vw;
    Vec8<bf16_t> vg;
    float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, w[8], f[8];
    if (live) {
        vo.load(raw + (size_t)pair * Dv + c);
        vw.load(norm_w + c);
        if (g_col >= 0) vg.load(proj + (size_t)(pair / n_heads) * row_stride + g_col + pair % n_heads * Dv + c);
        vo.get(o);
    }
    float ss = ((o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3])) + ((o[4] * o[4] + o[5] * o[5]) + (o[6] * o[6] + o[7] * o[7]));
    for (int lanes = 1 << group_log >> 1; lanes > 0; lanes >>= 1) ss += __shfl_xor(ss, lanes, SIA_WAVE);
    if (!live) return;
    const float inv = rsqrtf(ss / (float)Dv + eps);
    vw.get(w);
    if (g_col >= 0) vg.get(f);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = o[i] * inv * w[i] * (g_col >= 0 ? f[i] / (1.f + expf(-f[i])) : 1.f);
    Vec8<bf16_t> y;
    y.set(o);
    y.store(out + (size_t)pair * Dv + c);
}

// The form with eight elements a lane where bfloat16 rows allow it, from the smallest step on (figures there; the 32-bit path keeps one order
// of sums whatever the step's addresses are).  Else four pairs a wave where there are many narrow ones, as the 32-bit path and rows that
// begin anywhere have them;  one and four, a layer's recurrence as it was walked in bfloat16, us:  24 heads of 128, 512 tokens 75.1 and 75.9,
// 1,024 91.5 and 91.2, 2,048 138.9 and 137.7;  16 of 256, 2,048 149.0 and 151.6.
template <typename T>
static void launch_finish(const float* raw, const void* proj, int row_stride, int g_col, const float* norm_w, void* out, int n_tokens,
                          int n_heads, int Dv, float eps, hipStream_t stream) {
    const int n_pairs = n_tokens * n_heads;
    auto launch = [&](auto kernel, int pairs) {
        const int each = GLA_FINISH_WAVES * pairs;
        hipLaunchKernelGGL(kernel, dim3((n_pairs + each - 1) / each), dim3(GLA_FINISH_WAVES * SIA_WAVE), 0, stream, raw, (const T*)proj,
                           row_stride, g_col, norm_w, (T*)out, n_pairs, n_heads, Dv, eps);
    };
    if constexpr (std::is_same<T, bf16_t>::value) {
        const bool gate = g_col < 0 || (g_col % 8 == 0 && row_stride % 8 == 0 && (uintptr_t)proj % 16 == 0);
        if (gate && Dv % 8 == 0 && Dv <= 8 * SIA_WAVE && ((uintptr_t)raw | (uintptr_t)norm_w | (uintptr_t)out) % 16 == 0) {
            int group_log = 0;
            while (8 << group_log < Dv) ++group_log;
            const int each = GLA_FINISH_WAVES * SIA_WAVE >> group_log;
            hipLaunchKernelGGL(gla_finish_vec_kernel, dim3((n_pairs + each - 1) / each), dim3(GLA_FINISH_WAVES * SIA_WAVE), 0, stream, raw,
                               (const bf16_t*)proj, row_stride, g_col, norm_w, (bf16_t*)out, n_pairs, n_heads, Dv, group_log, eps);
            return;
        }
    }
    if (n_pairs >= 20000 && Dv <= 128) launch(gla_finish_kernel<T, 4>, 4);
    else launch(gla_finish_kernel<T, 1>, 1);
}

SIA_EXPORT int sia_gla_max_dims() { return 512; }

// Whether a step shares a head's columns out between workgroups (and needs the outputs' part of the workspace).
static bool gla_slices(int n_seqs, int max_q_len, int n_heads) {
    (void)n_seqs; (void)n_heads;
    return max_q_len > 1;
}

// The shortest segment that a prompt is cut into, and the shortest run of tokens that the walk with four columns a lane
// group is taken for.
#define SEG_MIN 64
#define WALK_MIN_RUN 128

// Whether runs go by blocks on the matrix cores, from BLOCKS_MIN_RUN tokens on.  us for one run, by the walk, by blocks, by blocks whose decays make
// them go pair by pair:  24 heads of 128 x 128 with a bonus, 33 tokens 29, 28, 33;  48 33.6, 28.3, 33.5;  64 38.7, 32.7, 39.8;  128 62, 52, 66;  200 82,
// 57, 63;  24 of 64 x 64 22.7, 21.2, 26.3;  25.5, 21.3, 26.7;  28.6, 24, 31;  45, 37, 51;  56, 39, 46.
// A workgroup has room for 64 channels and columns where the state has 64 channels, else for 128: with 128, half of the products
// of 64 channels multiplied nothing (us, walk, 128, 64:  16 of 64 x 128, 449 tokens beside 63 254, 295, 225, 16 runs of 200 123, 88, 69;  8 of 64 x 144,
// 449 beside 63 197, 259, 165).  80 to 112 channels fill 128 by halves and more, and are faster so than walked (8 of 80 x 192, 2,048 tokens 128 -> 87).
#define BLOCKS_MIN_RUN 48
static bool by_blocks(int D, int Dv) { return D % 16 == 0 && D >= 64 && D <= 128 && Dv % 16 == 0 && Dv >= 64; }

static long long segment_places(int n_tokens, int n_seqs, Segments cut) {
    if (cut.len == 0) return 0;
    const long long multiples = (n_tokens - 1) / cut.len + 1;
    return cut.by_sequence ? multiples + n_seqs - 1 : 2 * multiples;
}

// Whether runs that are not cut are walked with four columns a lane group (a longer chain a token, but LDS serves twice
// the columns) or two: where the workgroups are many, and where two would not fit into LDS.  Four against two, us (128 x 128 and 64 x 64 from
// before they went by blocks):
//   24 heads of 128 x 128, 128 tokens:  one run 83 against 62, 4 runs 96 against 88, 8 runs 118 against 133; one run beside 63
//   single tokens 268 against 405;   24 of 64 x 64, 16 runs 82 against 80, one beside 63 104 against 120;   80 of 64 x 128, 4
//   runs 120 against 135;   16 of 256 x 256, one run of 128 133 against 205 by the kernel that takes every size.
static bool four_columns(int n_seqs, int n_heads, int D, int Dv) {
    return D > 128 || (long long)n_seqs * n_heads * ((Dv + 63) / 64) * D >= 256 * 128;
}

// How a step is cut, from its sizes alone, so that whoever makes the workspace and whoever launches agree.
// A step of few and long sequences leaves most of the chip idle behind the walk's chain of tokens: it is cut into
// segments, long ones where there are enough of them.  (Workgroups the step keeps busy without: the tokens
// over the longest run, times heads and slices.)  2,048 tokens of 24 heads of 128: one walk of 96 workgroups 740 us; 16
// segments 177 with two columns a lane group, 121 with four (LDS serves twice the columns, 140 registers), and 53 for
// the decays' products, the states and the outputs behind it (100 MB of states and outputs).
// A cut costs three kernels and the more traffic the more heads and rows; a run saves its chain: `shortest` follows where
// both are even, in tokens of the longest run (walked; measured with one run, 4, 8 and 16):  24 heads of 128 x 128 at 190, 210, -, -;  4 of them at
// 172, 175, 192, 200;  24 of 64 x 64 at 165, 180, 200, 300;  8 of 128 x 64 at 172, 185, 190, 210;  32 of 16 x 64 at 148, 160,
// 150, -.  States of more than 128 rows (no walk with two columns):  16 of 256 x 256 one run of 128 122 us against 133, 4
// runs of 128 152 against 148 and of 256 257 against 257, 8 runs of 192 323 against 261;  4 of 256 x 128 are cut from 128 on with up to 16.
// The same rule for states that go by blocks, whose cut costs two kernels and less traffic: us, whole and cut,  24 heads of 128 x 128, one run of 136 53
// and 49, of 168 62 and 49, of 200 72 and 52, of 2,048 573 and 130;  4 runs of 168 74 and 73, of 2,048 637 and 412;  16 runs of 320 205 and 288 (not cut);
// 24 of 64 x 64, one run of 168 42 and 34, 4 of 200 54 and 48;  8 of 128 x 64, 16 of 256 82 and 69.  (Both are even earlier than the rule
// cuts, at 120 tokens for one run, and shorter segments would be faster there: 32 tokens, one run of 136, 40.)
static Segments segments_of(int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, int Dv, int dtype) {
    const Segments none{0, false};
    const int slices = (Dv + 63) / 64;
    if (dtype != SIA_BF16 || max_q_len < WALK_MIN_RUN || D % 8 || D > 256 || Dv % 4 || n_seqs > 65535 ||
        (long long)n_heads * slices > 65535)
        return none;
    const long long busy = (long long)(n_tokens / max_q_len) * n_heads * slices;
    const int shortest = D <= 128 ? 136 + 5 * D / 16 + (int)(busy / 4) : (long long)n_seqs * n_heads * slices * D <= 256 * 128 ? 128 : 512;
    if (busy >= 768 || max_q_len < shortest) return none;
    const int len = (long long)n_tokens * n_heads * slices / (2 * SEG_MIN) >= 768 ? 2 * SEG_MIN : SEG_MIN;
    if ((long long)slices * ((max_q_len + len - 1) / len) > 65535) return none;      // a grid's third number
    const Segments by_sequence{len, true}, apart{len, false};
    return segment_places(n_tokens, n_seqs, by_sequence) <= segment_places(n_tokens, n_seqs, apart) ? by_sequence : apart;
}

// The raw outputs [tokens, heads, Dv] as floats, and behind them the states of the step's segments.
static long long recurrence_space(int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, int Dv, int dtype) {
    const long long states = segment_places(n_tokens, n_seqs, segments_of(n_tokens, n_seqs, max_q_len, n_heads, D, Dv, dtype));
    return (long long)n_tokens * n_heads * Dv + states * n_heads * D * Dv;
}

// Floats of workspace a step of n_tokens needs: the decays [tokens, heads, D], and the space above.
SIA_EXPORT long long sia_gla_workspace(int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, int Dv, int dtype) {
    return (long long)n_tokens * n_heads * D + recurrence_space(n_tokens, n_seqs, max_q_len, n_heads, D, Dv, dtype);
}

// A step of one token a sequence, if the kernel for it takes these sizes and addresses; false with nothing done if not.
static bool launch_state_decode(const void* proj, int row_stride, int q_col, int k_col, int v_col, int g_col, const float* k_f32,
                                int q_share, const float* alpha, const LowRank* low, const float* norm_w, float* state,
                                long long state_stride, const int* cu_q, const int* slots, void* out, int n_seqs, int max_q_len,
                                int n_heads, int D, int Dv, float q_scale, float eps, int dtype, float* raw, hipStream_t stream,
                                const float* bonus) {
    const int rows = (D * (Dv / 4) + 511) / 512;      // of the state a thread has
    if (max_q_len != 1 || dtype != SIA_BF16 || Dv < 16 || Dv > 256 || (Dv & (Dv - 1)) || rows > 16 || D > 512 || row_stride % 4 ||
        v_col % 4 || state_stride % 4 || ((uintptr_t)proj % 8) || ((uintptr_t)state % 16) || n_heads > 65535)
        return false;
    if (low && (low->rank % 8 || low->a_col % 8 || row_stride % 8 || ((uintptr_t)proj % 16) || ((uintptr_t)low->a2 % 16))) return false;
    const dim3 grid(n_seqs, n_heads), block(512);
    const LowRank none{};
#define DECODE_AS(ROWS, BONUS, LOW)                                                                                      \
    hipLaunchKernelGGL((state_decode_kernel<ROWS, BONUS, LOW>), grid, block, 0, stream, (const bf16_t*)proj, row_stride, q_col, \
                       k_col, v_col, g_col, alpha, low ? *low : none, norm_w, state, state_stride, cu_q, slots, (bf16_t*)out,   \
                       n_heads, D, Dv, q_scale, eps, raw, k_f32, q_share, bonus)
#define DECODE(ROWS)                                                                                                     \
    do {                                                                                                                 \
        if (bonus) DECODE_AS(ROWS, true, false);                                                                         \
        else if (low) DECODE_AS(ROWS, false, true);                                                                      \
        else DECODE_AS(ROWS, false, false);                                                                              \
    } while (0)
    if (rows <= 2) DECODE(2);
    else if (rows <= 4) DECODE(4);
    else if (rows <= 8) DECODE(8);
    else DECODE(16);
#undef DECODE
#undef DECODE_AS
    return true;
}

// The recurrence itself for a step's runs of tokens, whoever prepared its inputs: S <- diag(alpha) S + k v^T, o = S^T q.
// q and v (and k, unless k_f32 gives it as floats [tokens, heads, D]) are columns of rows of the compute type; head h
// reads the q (and such a k) of head h / q_share.  A sequence's matrices lie state_stride floats apart from the next
// slot's.  The outputs go to ``raw`` [tokens, heads, Dv] as floats if the caller wants them there (want_raw) or if a
// head's columns are shared out between workgroups; otherwise they are normed over the head (norm_w, eps), gated by
// silu of the columns at g_col (none if negative) and written to ``out``.  Returns through ``raw_used`` whether ``raw``
// holds the outputs.  With ``bonus`` [heads, D] the query reads the state before the token's write and, unless the outputs are
// raw, that write weighed by it; the norm's weights are then [heads, Dv].  ``alpha`` is working space: it may hold other
// numbers afterwards.
static int launch_recurrence(const void* proj, int row_stride, int q_col, int k_col, int v_col, int g_col,
                             const float* k_f32, int q_share, float* alpha, const float* norm_w, float* state,
                             long long state_stride, const int* cu_q, const int* slots, void* out, int n_tokens, int n_seqs,
                             int max_q_len, int n_heads, int D, int Dv, float q_scale, float eps, int dtype,
                             float* raw_space, bool want_raw, bool* raw_used, hipStream_t stream,
                             const float* bonus = nullptr) {
    if (launch_state_decode(proj, row_stride, q_col, k_col, v_col, g_col, k_f32, q_share, alpha, nullptr, norm_w, state, state_stride,
                            cu_q, slots, out, n_seqs, max_q_len, n_heads, D, Dv, q_scale, eps, dtype, want_raw ? raw_space : nullptr,
                            stream, bonus)) {
        if (raw_used) *raw_used = want_raw;
        return 0;
    }
    // columns a workgroup: all of a head's, or with a workspace a slice of them, as narrow as it takes to fill the chip
    int slice = Dv;
    const bool prompt = gla_slices(n_seqs, max_q_len, n_heads);
    if (prompt)
        while (slice > 8 && (long long)n_seqs * n_heads * ((Dv + slice - 1) / slice) < 256) slice = (slice + 1) / 2;
    // lanes a column: the largest power of two that keeps the workgroup within 512 threads and a wave's columns whole;
    // a state too tall for the rows a lane can keep is shared out over more workgroups, whatever the step
    int R = 1, rows = D;
    for (;;) {
        R = 1;
        while (R * 2 <= SIA_WAVE && slice * R * 2 <= 512 && R * 2 <= D) R *= 2;
        rows = (D + R - 1) / R;
        if (rows <= 128 || slice <= 1) break;
        slice = (slice + 1) / 2;
    }
    if (rows > 128) return SIA_BAD_ARGUMENT;
    const bool sliced = slice < Dv;
    const int threads = ((slice * R + SIA_WAVE - 1) / SIA_WAVE) * SIA_WAVE;
    int TB = max_q_len >= 16 ? 16 : (max_q_len >= 4 ? 4 : 1);
    auto bytes = [&](int tb) { return ((size_t)tb * (3 * D + 3 * Dv) + (bonus ? D : 0)) * sizeof(float); };
    while (TB > 1 && bytes(TB) > 60 * 1024) TB /= 2;
    if (bytes(TB) > 60 * 1024) return SIA_BAD_ARGUMENT;
    dim3 grid(n_seqs, n_heads, (Dv + slice - 1) / slice), block(threads);
    // the walk with requests a block ahead, where its pieces are aligned and fit its registers.  (Its workgroups take
    // as many columns as their threads hold whatever the step: the waves of a workgroup share the staged tokens, and
    // what bounds the walk is a wave's own chain of tokens, not the number of workgroups.)
    const bool blocks = by_blocks(D, Dv) && max_q_len >= BLOCKS_MIN_RUN;
    const bool long_runs = (max_q_len >= WALK_MIN_RUN || blocks) && Dv % 4 == 0 && n_seqs <= 65535 && n_heads * ((Dv + 63) / 64) <= 65535 &&
                           ((uintptr_t)raw_space % 16) == 0 && ((uintptr_t)state % 16) == 0 && state_stride % 4 == 0;
    Segments cut{0, false};
    if (long_runs) cut = segments_of(n_tokens, n_seqs, max_q_len, n_heads, D, Dv, dtype);
    const int w_cols = long_runs && (cut.len || four_columns(n_seqs, n_heads, D, Dv)) ? 4 : 2;
    const int w_slice = GLA_WALK_THREADS / 16 * w_cols;
    const int w_rows = (D + 15) / 16;
    const int w_rows_t = w_rows <= 4 ? 4 : w_rows <= 8 ? 8 : w_rows <= 16 ? 16 : 32;
    const size_t w_lds = (size_t)gla_walk_tokens(w_cols) * (3 * 16 * w_rows_t + 2 * w_slice) * sizeof(float);
    const bool ahead = prompt && dtype == SIA_BF16 && D % 8 == 0 && row_stride % 8 == 0 && q_col % 8 == 0 &&
                       (k_f32 ? ((uintptr_t)k_f32 % 16) == 0 : k_col % 8 == 0) && ((uintptr_t)alpha % 16) == 0 &&
                       ((uintptr_t)proj % 16) == 0 &&
                       w_lds <= 60 * 1024 && w_rows_t <= 16;
    float* raw = (sliced || ahead || want_raw) ? raw_space : nullptr;
    if (raw_used) *raw_used = raw != nullptr;
    if (ahead) {
        const int w_slices = (Dv + w_slice - 1) / w_slice;
        const int seg_len = cut.len, n_segs = seg_len ? (max_q_len + seg_len - 1) / seg_len : 1;
        float* seg_state = raw_space + (size_t)n_tokens * n_heads * Dv;
        if (blocks && long_runs) {
            float* seg_decay = raw;      // behind the states nobody reads them, and the outputs come after
            const int width = D <= 64 ? 64 : 128;
            const dim3 bgrid(n_seqs, n_heads, (Dv + width - 1) / width * n_segs), bblock(width / 16 * SIA_WAVE);
#define BLOCKS_AS(WIDTH, OUT, KF, BEFORE)                                                                                    \
    hipLaunchKernelGGL((gla_blocks_kernel<WIDTH, OUT, KF, BEFORE>), bgrid, bblock, 0, stream, (const bf16_t*)proj, row_stride,   \
                       q_col, k_col, v_col, alpha, k_f32, q_share, state, state_stride, cu_q, slots, n_heads, D, Dv, q_scale,   \
                       raw, cut, seg_state, seg_decay)
#define BLOCKS_OF(WIDTH, OUT)                                                                                                \
    do {                                                                                                                     \
        if (bonus) BLOCKS_AS(WIDTH, OUT, false, true);                                                                       \
        else if (k_f32) BLOCKS_AS(WIDTH, OUT, true, false);                                                                  \
        else BLOCKS_AS(WIDTH, OUT, false, false);                                                                            \
    } while (0)
#define BLOCKS(OUT)                                                                                                          \
    do {                                                                                                                     \
        if (width == 64) BLOCKS_OF(64, OUT);                                                                                 \
        else BLOCKS_OF(128, OUT);                                                                                            \
    } while (0)
            if (n_segs > 1) {
                BLOCKS(false);
                hipLaunchKernelGGL(block_states_kernel, dim3((D * Dv / 4 + 255) / 256, n_heads, n_seqs), dim3(256), 0, stream, seg_decay,
                                   seg_state, state, state_stride, cu_q, slots, n_heads, D, Dv, cut);
            }
            BLOCKS(true);
#undef BLOCKS
#undef BLOCKS_OF
#undef BLOCKS_AS
            return 0;
        }
        dim3 wgrid(n_seqs, n_heads, w_slices * n_segs), wblock(GLA_WALK_THREADS);
#define WALK_AS(ROWS, COLS, KF, BEFORE)                                                                                      \
    hipLaunchKernelGGL((gla_walk_kernel<ROWS, COLS, KF, BEFORE>), wgrid, wblock, w_lds, stream, (const bf16_t*)proj,         \
                       row_stride, q_col, k_col, v_col, alpha, k_f32, q_share, state, state_stride, cu_q, slots,     \
                       n_heads, D, Dv, q_scale, raw, cut, seg_state)
#define WALK(ROWS, COLS)                                                                                             \
    do {                                                                                                             \
        if (bonus) WALK_AS(ROWS, COLS, false, true);                                                                 \
        else if (k_f32) WALK_AS(ROWS, COLS, true, false);                                                            \
        else WALK_AS(ROWS, COLS, false, false);                                                                      \
    } while (0)
        if (w_cols == 4) {
            if (w_rows_t == 4) WALK(4, 4);
            else if (w_rows_t == 8) WALK(8, 4);
            else WALK(16, 4);
        } else if (w_rows_t == 4) WALK(4, 2);
        else WALK(8, 2);      // a state of more than 128 rows would need more LDS for 32 tokens than is asked for
#undef WALK
#undef WALK_AS
        if (n_segs > 1) {
            const int channels = n_heads * D;
            hipLaunchKernelGGL(segment_decays_kernel, dim3(n_segs - 1, (channels + 255) / 256, n_seqs), dim3(256), 0, stream, alpha,
                               cu_q, channels, seg_len);
            hipLaunchKernelGGL(segment_states_kernel, dim3((D * Dv / 4 + 255) / 256, n_heads, n_seqs), dim3(256), 0, stream, alpha,
                               seg_state, state, state_stride, cu_q, slots, n_heads, D, Dv, cut);
            const dim3 ogrid(n_segs - 1, n_heads * ((Dv + 63) / 64), n_seqs), oblock(seg_len / 32 * SIA_WAVE);
            if (bonus)
                hipLaunchKernelGGL(segment_outputs_kernel<true>, ogrid, oblock, 0, stream, (const bf16_t*)proj, row_stride, q_col,
                                   q_share, alpha, seg_state, cu_q, n_heads, D, Dv, q_scale, raw, cut);
            else
                hipLaunchKernelGGL(segment_outputs_kernel<false>, ogrid, oblock, 0, stream, (const bf16_t*)proj, row_stride, q_col,
                                   q_share, alpha, seg_state, cu_q, n_heads, D, Dv, q_scale, raw, cut);
        }
    } else {
#define LAUNCH_AS(T, ROWS, BONUS)                                                                                    \
    hipLaunchKernelGGL((gla_recurrent_kernel<T, ROWS, BONUS>), grid, block, bytes(TB), stream, (const T*)proj,       \
                       row_stride, q_col, k_col, v_col, g_col, alpha, norm_w, state, cu_q, slots, (T*)out, n_heads, D, \
                       Dv, R, TB, q_scale, eps, slice, raw, k_f32, q_share, state_stride, bonus)
#define LAUNCH(T, ROWS)                                                                                              \
    do {                                                                                                             \
        if (bonus) LAUNCH_AS(T, ROWS, true);                                                                         \
        else LAUNCH_AS(T, ROWS, false);                                                                              \
    } while (0)
#define PICK(T)                                                                                                      \
    do {                                                                                                             \
        if (rows <= 4) LAUNCH(T, 4);                                                                                 \
        else if (rows <= 8) LAUNCH(T, 8);                                                                            \
        else if (rows <= 16) LAUNCH(T, 16);                                                                          \
        else if (rows <= 32) LAUNCH(T, 32);                                                                          \
        else if (rows <= 64) LAUNCH(T, 64);                                                                          \
        else LAUNCH(T, 128);                                                                                         \
    } while (0)
    if (dtype == SIA_F32) PICK(float);
    else if (dtype == SIA_BF16) PICK(bf16_t);
    else return SIA_BAD_ARGUMENT;
#undef PICK
#undef LAUNCH
#undef LAUNCH_AS
    }
    return 0;
}

// y = o * rsqrt(mean(o^2) + eps) * w * silu(g) with o = raw + (sum_d q_d bonus_d k_d) v: what the walk left in the float
// workspace and the token's own weighed write.  A wave a (token, head); q, k, v and g are columns of rows row_stride apart,
// weights and bonus a head's own.
template <typename T>
__global__ __launch_bounds__(4 * SIA_WAVE) void bonus_finish_kernel(const float* __restrict__ raw, const T* __restrict__ proj,
                                                                int row_stride, int q_col, int k_col, int v_col, int g_col,
                                                                const float* __restrict__ bonus,
                                                                const float* __restrict__ norm_w, T* __restrict__ out,
                                                                int n_heads, int D, int Dv, float eps) {
    const int n = blockIdx.x, head = blockIdx.y * 4 + threadIdx.x / SIA_WAVE, lane = threadIdx.x % SIA_WAVE;
    if (head >= n_heads) return;      // a wave leaves as a whole
    const T* row = proj + (size_t)n * row_stride;
    const T *q = row + q_col + head * D, *k = row + k_col + head * D, *v = row + v_col + head * Dv, *g = row + g_col + head * Dv;
    float own = 0.f;
    for (int d = lane; d < D; d += SIA_WAVE) own += to_float(q[d]) * bonus[(size_t)head * D + d] * to_float(k[d]);
    own = wave_sum(own);
    const float* o = raw + ((size_t)n * n_heads + head) * Dv;
    float ss = 0.f;
    for (int c = lane; c < Dv; c += SIA_WAVE) {
        const float x = o[c] + own * to_float(v[c]);
        ss += x * x;
    }
    const float inv = rsqrtf(wave_sum(ss) / (float)Dv + eps);
    T* dst = out + ((size_t)n * n_heads + head) * Dv;
    for (int c = lane; c < Dv; c += SIA_WAVE) {
        const float x = o[c] + own * to_float(v[c]), z = to_float(g[c]);
        dst[c] = from_float<T>(x * inv * norm_w[(size_t)head * Dv + c] * (z / (1.f + expf(-z))));
    }
}

// floats of workspace behind the decays
SIA_EXPORT long long sia_bonus_recurrence_workspace(int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, int dtype) {
    return recurrence_space(n_tokens, n_seqs, max_q_len, n_heads, D, D, dtype);
}

// The recurrence with a bonus for the current token: rkvg is four matrices [tokens, heads * D] one behind the other (r, k, v
// and the output gate), decays [tokens, heads, D] float (working space from here on), bonus and norm_w [heads, D].
SIA_EXPORT int sia_bonus_recurrence(const void* rkvg, float* decays, const float* bonus, const float* norm_w,
                                    float* state, long long state_stride, const int* cu_q, const int* slots, void* out,
                                    int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, float eps, int dtype,
                                    float* workspace, hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    const long long plane = (long long)n_tokens * n_heads * D;
    if (D <= 0 || D > 512 || n_heads <= 0 || n_heads > 65535 || !rkvg || !decays || !bonus || !norm_w || !state || !out ||
        !workspace || state_stride < (long long)n_heads * D * D || 4 * plane > 0x7fffffffLL)
        return SIA_BAD_ARGUMENT;
    const int width = n_heads * D, k_col = (int)plane, v_col = (int)(2 * plane), g_col = (int)(3 * plane);
    bool raw = false;
    const int code = launch_recurrence(rkvg, width, 0, k_col, v_col, g_col, nullptr, 1, decays, norm_w, state, state_stride,
                                       cu_q, slots, out, n_tokens, n_seqs, max_q_len, n_heads, D, D, 1.f, eps, dtype, workspace,
                                       false, &raw, stream, bonus);
    if (code) return code;
    if (raw) {
        dim3 grid(n_tokens, (n_heads + 3) / 4), block(4 * SIA_WAVE);
        if (dtype == SIA_F32)
            hipLaunchKernelGGL(bonus_finish_kernel<float>, grid, block, 0, stream, workspace, (const float*)rkvg, width, 0,
                               k_col, v_col, g_col, bonus, norm_w, (float*)out, n_heads, D, D, eps);
        else
            hipLaunchKernelGGL(bonus_finish_kernel<bf16_t>, grid, block, 0, stream, workspace, (const bf16_t*)rkvg, width,
                               0, k_col, v_col, g_col, bonus, norm_w, (bf16_t*)out, n_heads, D, D, eps);
    }
    return SIA_LAUNCH_CHECK();
}

SIA_EXPORT int sia_gla_recurrent(const void* proj, int row_stride, int q_col, int k_col, int v_col, int g_col, int a_col,
                                 const void* a2, const float* a2_bias, const float* norm_w, float* state,
                                 const int* cu_q, const int* slots, void* out, int n_seqs, int max_q_len, int n_heads,
                                 int D, int Dv, int rank, float tau, float q_scale, float eps, int dtype,
                                 float* workspace, int n_tokens, hipStream_t stream) {
    if (n_seqs <= 0) return 0;
    if (D <= 0 || Dv <= 0 || D > 512 || Dv > 512 || rank <= 0 || rank > 1024 || n_heads <= 0 || n_heads > 65535 ||
        !(tau > 0.f) || !state || !norm_w || !workspace || n_tokens <= 0)
        return SIA_BAD_ARGUMENT;
    float* alpha = workspace;
    float* raw_space = workspace + (size_t)n_tokens * n_heads * D;
    const LowRank low{(const bf16_t*)a2, a2_bias, a_col, rank, 1.f / tau};
    if (launch_state_decode(proj, row_stride, q_col, k_col, v_col, g_col, nullptr, 1, nullptr, &low, norm_w, state,
                            (long long)n_heads * D * Dv, cu_q, slots, out, n_seqs, max_q_len, n_heads, D, Dv, q_scale, eps, dtype,
                            nullptr, stream, nullptr))
        return SIA_LAUNCH_CHECK();
    {
        const int channels = n_heads * D;
        dim3 dgrid((n_tokens + GLA_DECAY_TOKENS - 1) / GLA_DECAY_TOKENS, (channels + 255) / 256), dblock(256);
        const size_t lds = (size_t)GLA_DECAY_TOKENS * rank * sizeof(float);
        // The matrix cores where there is work for them: a wave has 64 channels of 32 tokens to itself, and few waves take
        // longer than a thread a channel does.  A layer's whole recurrence, us, without and with:  rank 64, 3,072 channels, 32
        // tokens 31 / 37, 128: 63 / 67, 256: 89 / 91, 384: 102 / 98, 2,048: 232 / 202;  512 channels, 512: 80 / 85, 2,048: 106 / 105;
        // rank 32, 3,072 channels, 512: 98 / 101, 1,024: 128 / 129;  rank 128, 128: 66 / 69, 256: 95 / 92.
        const bool many = (long long)n_tokens * channels * rank >= 1LL << 26;
        if (many && dtype == SIA_BF16 && rank % 32 == 0 && channels % 4 == 0 && row_stride % 8 == 0 && a_col % 8 == 0 &&
            ((uintptr_t)proj | (uintptr_t)a2 | (uintptr_t)a2_bias | (uintptr_t)alpha) % 16 == 0)
            hipLaunchKernelGGL(gla_decay_mfma_kernel, dim3((n_tokens + 31) / 32, (channels + 255) / 256), dblock, 0, stream,
                               (const bf16_t*)proj, row_stride, a_col, (const bf16_t*)a2, a2_bias, alpha, n_tokens, channels,
                               rank, 1.f / tau);
        else if (dtype == SIA_F32)
            hipLaunchKernelGGL(gla_decay_kernel<float>, dgrid, dblock, lds, stream, (const float*)proj, row_stride, a_col,
                               (const float*)a2, a2_bias, alpha, n_tokens, channels, rank, 1.f / tau);
        else if (dtype == SIA_BF16)
            hipLaunchKernelGGL(gla_decay_kernel<bf16_t>, dgrid, dblock, lds, stream, (const bf16_t*)proj, row_stride,
                               a_col, (const bf16_t*)a2, a2_bias, alpha, n_tokens, channels, rank, 1.f / tau);
        else
            return SIA_BAD_ARGUMENT;
    }
    bool raw = false;
    const int code = launch_recurrence(proj, row_stride, q_col, k_col, v_col, g_col, nullptr, 1, alpha, norm_w, state,
                                       (long long)n_heads * D * Dv, cu_q, slots, out, n_tokens, n_seqs, max_q_len, n_heads, D, Dv,
                                       q_scale, eps, dtype, raw_space, false, &raw, stream);
    if (code) return code;
    if (raw) {
        if (dtype == SIA_F32) launch_finish<float>(raw_space, proj, row_stride, g_col, norm_w, out, n_tokens, n_heads, Dv, eps, stream);
        else launch_finish<bf16_t>(raw_space, proj, row_stride, g_col, norm_w, out, n_tokens, n_heads, Dv, eps, stream);
    }
    return SIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------------------------
// The gated linear recurrence whose forget gate also decides what is written:
//   f = l + (1 - l) * sigmoid(z_f + b),  S <- diag(f) S + (1 - f) v^T,  o = S^T silu(z_q),  y = o * rsqrt(mean(o^2) + eps) * w
// Rows are [z_q (H * D) | z_f (H * D) | v (H * Dv)].  A first kernel leaves f and 1 - f in the float workspace and
// silu(z_q) in the rows' own q columns; then the recurrence above, without an output gate.
template <typename T>
__global__ __launch_bounds__(256) void hgrn2_prepare_kernel(T* __restrict__ proj, int row_stride,
                                                            const float* __restrict__ f_bias,
                                                            const float* __restrict__ lower, float* __restrict__ alpha,
                                                            float* __restrict__ k_f32, int channels) {
    const int n = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= channels) return;
    T* row = proj + (size_t)n * row_stride;
    const float zq = to_float(row[c]);
    row[c] = from_float<T>(zq / (1.f + expf(-zq)));
    const float z = to_float(row[channels + c]) + (f_bias ? f_bias[c] : 0.f);
    const float l = lower ? lower[c] : 0.f;
    const float f = l + (1.f - l) * (1.f / (1.f + expf(-z)));
    alpha[(size_t)n * channels + c] = f;
    k_f32[(size_t)n * channels + c] = 1.f - f;
}

// floats of workspace: the gates and their complements [tokens, heads, D] each, the recurrence's own
SIA_EXPORT long long sia_hgrn2_workspace(int n_tokens, int n_seqs, int max_q_len, int n_heads, int D, int Dv, int dtype) {
    return 2LL * n_tokens * n_heads * D + recurrence_space(n_tokens, n_seqs, max_q_len, n_heads, D, Dv, dtype);
}

SIA_EXPORT int sia_hgrn2_scan(void* proj, int row_stride, const float* f_bias, const float* lower, const float* norm_w,
                              float* state, const int* cu_q, const int* slots, void* out, int n_tokens, int n_seqs,
                              int max_q_len, int n_heads, int D, int Dv, float eps, int dtype, float* workspace,
                              hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    if (D <= 0 || Dv <= 0 || D > 512 || Dv > 512 || n_heads <= 0 || n_heads > 65535 || !state || !norm_w || !workspace ||
        row_stride < n_heads * (2 * D + Dv))
        return SIA_BAD_ARGUMENT;
    const int channels = n_heads * D;
    float* alpha = workspace;
    float* kf = alpha + (size_t)n_tokens * channels;
    float* raw_space = kf + (size_t)n_tokens * channels;
    dim3 pgrid(n_tokens, (channels + 255) / 256), pblock(256);
    if (dtype == SIA_F32)
        hipLaunchKernelGGL(hgrn2_prepare_kernel<float>, pgrid, pblock, 0, stream, (float*)proj, row_stride, f_bias, lower,
                           alpha, kf, channels);
    else if (dtype == SIA_BF16)
        hipLaunchKernelGGL(hgrn2_prepare_kernel<bf16_t>, pgrid, pblock, 0, stream, (bf16_t*)proj, row_stride, f_bias,
                           lower, alpha, kf, channels);
    else
        return SIA_BAD_ARGUMENT;
    bool raw = false;
    const int code = launch_recurrence(proj, row_stride, 0, 0, 2 * channels, -1, kf, 1, alpha, norm_w, state,
                                       (long long)n_heads * D * Dv, cu_q, slots, out, n_tokens, n_seqs, max_q_len, n_heads, D, Dv,
                                       1.f, eps, dtype, raw_space, false, &raw, stream);
    if (code) return code;
    if (raw) {
        if (dtype == SIA_F32) launch_finish<float>(raw_space, proj, row_stride, -1, norm_w, out, n_tokens, n_heads, Dv, eps, stream);
        else launch_finish<bf16_t>(raw_space, proj, row_stride, -1, norm_w, out, n_tokens, n_heads, Dv, eps, stream);
    }
    return SIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------------------------
// The state-space recurrence with one decay per head:
//   dt = softplus(z_dt + dt_bias),  S <- exp(-exp(A_log) dt) S + (dt B) x^T,  y = S^T C + D x        S [N, P] per head
//   out = y * silu(z), divided by the root mean square of each of norm_groups equal parts of the row, times w
// z and z_dt are columns of the projected rows ([z (H * P) | ... | z_dt (H)], the step sizes last); x, B, C are the
// convolved rows [x (H * P) | B (G * N) | C (G * N)], head h reading the B and C of group h / (H / G).  A first kernel
// leaves the decays and dt * B in the float workspace, the recurrence leaves y there, a last kernel adds D x, gates
// and norms.
template <typename T>
__global__ __launch_bounds__(256) void ssd_prepare_kernel(const T* __restrict__ proj, int row_stride, int dt_col,
                                                          const T* __restrict__ xbc, int xbc_stride, int b_col,
                                                          const float* __restrict__ dt_bias,
                                                          const float* __restrict__ a_log, float* __restrict__ alpha,
                                                          float* __restrict__ k_f32, int n_heads, int N, int share) {
    const int n = blockIdx.x, idx = blockIdx.y * blockDim.x + threadIdx.x;
    if (idx >= n_heads * N) return;
    const int h = idx / N, c = idx % N;
    const float z = to_float(proj[(size_t)n * row_stride + dt_col + h]) + (dt_bias ? dt_bias[h] : 0.f);
    const float dt = fmaxf(z, 0.f) + log1pf(expf(-fabsf(z)));
    alpha[(size_t)n * n_heads * N + idx] = expf(-expf(a_log[h]) * dt);
    k_f32[(size_t)n * n_heads * N + idx] = dt * to_float(xbc[(size_t)n * xbc_stride + b_col + (h / share) * N + c]);
}

template <typename T>
__global__ __launch_bounds__(256) void ssd_finish_kernel(const float* __restrict__ raw, const T* __restrict__ proj,
                                                         int row_stride, const T* __restrict__ xbc, int xbc_stride,
                                                         const float* __restrict__ d_skip,
                                                         const float* __restrict__ norm_w, T* __restrict__ out,
                                                         int inner, int P, int part, float eps) {
    __shared__ float scratch[16];
    const int n = blockIdx.x, c0 = blockIdx.y * part;
    const float* y = raw + (size_t)n * inner;
    const T* z = proj + (size_t)n * row_stride;
    const T* x = xbc + (size_t)n * xbc_stride;
    float ss = 0.f;
    for (int c = c0 + threadIdx.x; c < c0 + part; c += blockDim.x) {
        const float g = to_float(z[c]);
        const float v = (y[c] + (d_skip ? d_skip[c / P] : 0.f) * to_float(x[c])) * (g / (1.f + expf(-g)));
        ss += v * v;
    }
    const float inv = rsqrtf(block_sum(ss, scratch) / (float)part + eps);
    for (int c = c0 + threadIdx.x; c < c0 + part; c += blockDim.x) {
        const float g = to_float(z[c]);
        const float v = (y[c] + (d_skip ? d_skip[c / P] : 0.f) * to_float(x[c])) * (g / (1.f + expf(-g)));
        out[(size_t)n * inner + c] = from_float<T>(v * inv * norm_w[c]);
    }
}

SIA_EXPORT long long sia_ssd_workspace(int n_tokens, int n_seqs, int max_q_len, int n_heads, int N, int P, int dtype) {
    return 2LL * n_tokens * n_heads * N + recurrence_space(n_tokens, n_seqs, max_q_len, n_heads, N, P, dtype);
}

SIA_EXPORT int sia_ssd_scan(const void* proj, int row_stride, const void* xbc, int xbc_stride, const float* dt_bias,
                            const float* a_log, const float* d_skip, const float* norm_w, float* state,
                            long long state_stride, const int* cu_q, const int* slots, void* out, int n_tokens,
                            int n_seqs, int max_q_len, int n_heads, int P, int N, int groups, int norm_groups, float eps,
                            int dtype, float* workspace, hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    const int inner = n_heads * P;
    if (N <= 0 || P <= 0 || N > 512 || P > 512 || n_heads <= 0 || n_heads > 65535 || groups <= 0 || n_heads % groups ||
        norm_groups <= 0 || inner % norm_groups || norm_groups > 65535 || !state || !norm_w || !a_log || !workspace ||
        row_stride < inner + n_heads || xbc_stride < inner + 2 * groups * N ||
        state_stride < (long long)n_heads * N * P)
        return SIA_BAD_ARGUMENT;
    const int channels = n_heads * N, share = n_heads / groups;
    float* alpha = workspace;
    float* kf = alpha + (size_t)n_tokens * channels;
    float* raw_space = kf + (size_t)n_tokens * channels;
    const int dt_col = row_stride - n_heads, b_col = inner, c_col = inner + groups * N;
    dim3 pgrid(n_tokens, (channels + 255) / 256), pblock(256), fgrid(n_tokens, norm_groups), fblock(256);
    bool raw = false;
#define RUN(T)                                                                                                          \
    do {                                                                                                                \
        hipLaunchKernelGGL(ssd_prepare_kernel<T>, pgrid, pblock, 0, stream, (const T*)proj, row_stride, dt_col,         \
                           (const T*)xbc, xbc_stride, b_col, dt_bias, a_log, alpha, kf, n_heads, N, share);             \
        const int code = launch_recurrence(xbc, xbc_stride, c_col, 0, 0, -1, kf, share, alpha, norm_w, state,           \
                                           state_stride, cu_q, slots, nullptr, n_tokens, n_seqs, max_q_len, n_heads, N, P, 1.f, \
                                           eps, dtype, raw_space, true, &raw, stream);                                  \
        if (code) return code;                                                                                          \
        hipLaunchKernelGGL(ssd_finish_kernel<T>, fgrid, fblock, 0, stream, raw_space, (const T*)proj, row_stride,       \
                           (const T*)xbc, xbc_stride, d_skip, norm_w, (T*)out, inner, P, inner / norm_groups, eps);     \
    } while (0)
    if (dtype == SIA_F32) RUN(float);
    else if (dtype == SIA_BF16) RUN(bf16_t);
    else return SIA_BAD_ARGUMENT;
#undef RUN
    return SIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------------------------
// Linear attention with a constant decay per head, behind activations:
//   q, k, v = silu(z_q), silu(z_k), silu(z_v);  S <- decay_h S + k v^T;  o = S^T q                  S [D, Dv] per head
//   out = o / sqrt(mean over the whole row of o^2 + eps) * w * sigmoid(z_g)                          w [H * Dv]
// Rows are [z_q (H * D) | z_k (H * D) | z_v (H * Dv) | z_g (H * Dv)].  A first kernel leaves the activations in the
// rows' own columns and the decays, one per head, in the float workspace as the recurrence reads them; then the
// recurrence above with raw outputs, and a kernel that norms a row over all its heads and gates it.
template <typename T>
__global__ __launch_bounds__(256) void decay_prepare_kernel(T* __restrict__ proj, int row_stride,
                                                            const float* __restrict__ decays,
                                                            float* __restrict__ alpha, int n_heads, int D, int active) {
    const int n = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c < active) {
        T* row = proj + (size_t)n * row_stride;
        const float z = to_float(row[c]);
        row[c] = from_float<T>(z / (1.f + expf(-z)));
    }
    if (c < n_heads * D) alpha[(size_t)n * n_heads * D + c] = decays[c / D];
}

template <typename T>
__global__ __launch_bounds__(256) void decay_finish_kernel(const float* __restrict__ raw, const T* __restrict__ proj,
                                                           int row_stride, int g_col,
                                                           const float* __restrict__ norm_w, T* __restrict__ out,
                                                           int inner, float eps) {
    __shared__ float scratch[16];
    const int n = blockIdx.x;
    const float* o = raw + (size_t)n * inner;
    const T* g = proj + (size_t)n * row_stride + g_col;
    float ss = 0.f;
    for (int c = threadIdx.x; c < inner; c += blockDim.x) ss += o[c] * o[c];
    const float inv = rsqrtf(block_sum(ss, scratch) / (float)inner + eps);
    for (int c = threadIdx.x; c < inner; c += blockDim.x) {
        const float z = to_float(g[c]);
        out[(size_t)n * inner + c] = from_float<T>(o[c] * inv * norm_w[c] * (1.f / (1.f + expf(-z))));
    }
}

SIA_EXPORT int sia_decay_attention(void* proj, int row_stride, const float* decays, const float* norm_w, float* state,
                                   const int* cu_q, const int* slots, void* out, int n_tokens, int n_seqs,
                                   int max_q_len, int n_heads, int D, int Dv, float eps, int dtype, float* workspace,
                                   hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    if (D <= 0 || Dv <= 0 || D > 512 || Dv > 512 || n_heads <= 0 || n_heads > 65535 || !state || !norm_w || !decays ||
        !workspace || row_stride < n_heads * (2 * D + 2 * Dv))
        return SIA_BAD_ARGUMENT;
    const int qk = n_heads * D, inner = n_heads * Dv, active = 2 * qk + inner;
    float* alpha = workspace;
    float* raw_space = alpha + (size_t)n_tokens * qk;
    dim3 pgrid(n_tokens, (active + 255) / 256), pblock(256), fgrid(n_tokens), fblock(256);
    bool raw = false;
#define RUN(T)                                                                                                          \
    do {                                                                                                                \
        hipLaunchKernelGGL(decay_prepare_kernel<T>, pgrid, pblock, 0, stream, (T*)proj, row_stride, decays, alpha,      \
                           n_heads, D, active);                                                                         \
        const int code = launch_recurrence(proj, row_stride, 0, qk, 2 * qk, -1, nullptr, 1, alpha, norm_w, state,       \
                                           (long long)n_heads * D * Dv, cu_q, slots, nullptr, n_tokens, n_seqs, max_q_len, \
                                           n_heads, D, Dv, 1.f, eps, dtype, raw_space, true, &raw, stream);             \
        if (code) return code;                                                                                          \
        hipLaunchKernelGGL(decay_finish_kernel<T>, fgrid, fblock, 0, stream, raw_space, (const T*)proj, row_stride,     \
                           active, norm_w, (T*)out, inner, eps);                                                        \
    } while (0)
    if (dtype == SIA_F32) RUN(float);
    else if (dtype == SIA_BF16) RUN(bf16_t);
    else return SIA_BAD_ARGUMENT;
#undef RUN
    return SIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------------------------
// The gated delta rule, token by token:
//   q <- q / sqrt(sum(q^2) + 1e-6) * D^(-1/2),  k <- k / sqrt(sum(k^2) + 1e-6)            per query/key head
//   beta = sigmoid(z_b),  g = exp(-exp(A_log_h) * softplus(z_a + dt_bias_h))              per value head
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q                          S [D, Dv] per value head
//   out = o * rsqrt(mean(o^2) + eps) * w * silu(z_g)                                      per head, w [Dv]
// q, k [G * D] and v [H * Dv] are columns of the convolved rows (value head h reads query/key head h / (H / G)); z_g
// [H * Dv], z_b and z_a [H] are columns of the projected rows.  A workgroup owns a (sequence, value head) or, in a
// step of few such pairs and many tokens, a slice of the head's columns (a column of S is corrected and read alone:
// S^T k and S^T q are sums down a column).  Thread (j, r) keeps rows r, r + R, ... of column j in registers; a token
// costs two sums over the R lanes of a column, one before the write and one after.  Blocks of tokens are staged
// through LDS as floats, where the unit norms, the write strengths and the decays of the block are taken, by every
// workgroup for itself.  The raw outputs go to the float workspace; the head's norm and gate are a second kernel.
// CHANNELS: every key channel has a decay of its own, g [H, D] acting on the rows of S, and the output gate comes as a
// factor: both were computed before (``decays`` [tokens, H, D] and ``gates`` [tokens, H * Dv], float), and a_log,
// dt_bias and the columns a_col and g_col are not read.
template <typename T, int ROWS, bool CHANNELS>
__global__ __launch_bounds__(512) void delta_rule_kernel(
    const T* __restrict__ qkv, int qkv_stride, const T* __restrict__ proj, int proj_stride, int b_col, int a_col,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias, float* __restrict__ state,
    long long state_stride, const int* __restrict__ cu_q, const int* __restrict__ slots, float* __restrict__ raw_out,
    int n_heads, int n_kv, int D, int Dv, int R, int block_tokens, int slice, int g_col,
    const float* __restrict__ norm_w, T* __restrict__ out, float eps, const float* __restrict__ decays,
    const float* __restrict__ gates) {
    // raw_out absent: the workgroup owns all of the head's columns (slice == Dv) and norms and gates its outputs itself
    extern __shared__ float lds[];
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int j0 = blockIdx.z * slice;
    const int first = cu_q[seq], last = cu_q[seq + 1];
    if (first >= last) return;
    const int TB = block_tokens;
    float* q_s = lds;                  // [TB][D]
    float* k_s = q_s + TB * D;         // [TB][D]
    float* v_s = k_s + TB * D;         // [TB][slice]
    float* be_s = v_s + TB * slice;    // [TB]
    float* de_s = be_s + TB;           // [TB]
    float* al_s = de_s + TB;           // [TB][D], CHANNELS only
    float* o_s = al_s + (CHANNELS ? TB * D : 0);   // [TB][slice], without raw_out only
    const int j = j0 + tid / R, r = tid % R;
    const bool owns = tid / R < slice && j < Dv;
    float* S_mem = state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv;
    float S[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = i * R + r;
        S[i] = (owns && d < D) ? S_mem[(size_t)d * Dv + j] : 0.f;
    }
    const int wave = tid / SIA_WAVE, lane = tid % SIA_WAVE, n_waves = blockDim.x / SIA_WAVE;
    const int kv_head = head / (n_heads / n_kv);
    const int q_col = kv_head * D, k_col = n_kv * D + kv_head * D, v_col = 2 * n_kv * D + head * Dv;
    const float rate = CHANNELS ? 0.f : expf(a_log[head]), bias = !CHANNELS && dt_bias ? dt_bias[head] : 0.f;
    const float q_scale = rsqrtf((float)D);

    for (int t0 = first; t0 < last; t0 += TB) {
        const int nt = min(TB, last - t0);
        for (int idx = tid; idx < nt * slice; idx += blockDim.x) {
            const int t = idx / slice, c = idx % slice;
            v_s[idx] = j0 + c < Dv ? to_float(qkv[(size_t)(t0 + t) * qkv_stride + v_col + j0 + c]) : 0.f;
        }
        for (int idx = tid; idx < nt * D; idx += blockDim.x) {
            const int t = idx / D, c = idx % D;
            const T* row = qkv + (size_t)(t0 + t) * qkv_stride;
            q_s[idx] = to_float(row[q_col + c]);
            k_s[idx] = to_float(row[k_col + c]);
            if (CHANNELS) al_s[idx] = decays[((size_t)(t0 + t) * n_heads + head) * D + c];
        }
        if (tid < nt) {
            const T* row = proj + (size_t)(t0 + tid) * proj_stride;
            be_s[tid] = 1.f / (1.f + expf(-to_float(row[b_col + head])));
            if (!CHANNELS) {
                const float za = to_float(row[a_col + head]) + bias;
                de_s[tid] = expf(-rate * (fmaxf(za, 0.f) + log1pf(expf(-fabsf(za)))));
            }
        }
        __syncthreads();
        for (int t = wave; t < nt; t += n_waves) {      // unit vectors, a wave a token
            float sq = 0.f, sk = 0.f;
            for (int c = lane; c < D; c += SIA_WAVE) {
                sq += q_s[t * D + c] * q_s[t * D + c];
                sk += k_s[t * D + c] * k_s[t * D + c];
            }
            const float iq = rsqrtf(wave_sum(sq) + 1e-6f) * q_scale, ik = rsqrtf(wave_sum(sk) + 1e-6f);
            for (int c = lane; c < D; c += SIA_WAVE) {
                q_s[t * D + c] *= iq;
                k_s[t * D + c] *= ik;
            }
        }
        __syncthreads();
        for (int t = 0; t < nt; ++t) {
            const float g = CHANNELS ? 1.f : de_s[t], b = be_s[t];
            const float v = owns ? v_s[t * slice + (j - j0)] : 0.f;
            float kept = 0.f;
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int d = i * R + r;
                if (d < D) {
                    S[i] *= CHANNELS ? al_s[t * D + d] : g;
                    kept += k_s[t * D + d] * S[i];
                }
            }
            for (int o = R / 2; o > 0; o >>= 1) kept += __shfl_xor(kept, o, SIA_WAVE);
            const float u = b * (v - kept);
            float acc = 0.f;
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int d = i * R + r;
                if (d < D) {
                    S[i] += k_s[t * D + d] * u;
                    acc += q_s[t * D + d] * S[i];
                }
            }
            for (int o = R / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, SIA_WAVE);
            if (owns && r == 0) {
                if (raw_out) raw_out[((size_t)(t0 + t) * n_heads + head) * Dv + j] = acc;
                else o_s[t * slice + (j - j0)] = acc;
            }
        }
        __syncthreads();
        if (raw_out) continue;   // uniform: the norm is another kernel's
        for (int t = wave; t < nt; t += n_waves) {
            float ss = 0.f;
            for (int c = lane; c < Dv; c += SIA_WAVE) ss += o_s[t * slice + c] * o_s[t * slice + c];
            const float inv = rsqrtf(wave_sum(ss) / (float)Dv + eps);
            T* dst = out + ((size_t)(t0 + t) * n_heads + head) * Dv;
            if (CHANNELS) {
                const float* factor = gates + ((size_t)(t0 + t) * n_heads + head) * Dv;
                for (int c = lane; c < Dv; c += SIA_WAVE)
                    dst[c] = from_float<T>(o_s[t * slice + c] * inv * norm_w[c] * factor[c]);
                continue;
            }
            const T* g_row = proj + (size_t)(t0 + t) * proj_stride + g_col + head * Dv;
            for (int c = lane; c < Dv; c += SIA_WAVE) {
                const float z = to_float(g_row[c]);
                dst[c] = from_float<T>(o_s[t * slice + c] * inv * norm_w[c] * (z / (1.f + expf(-z))));
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = i * R + r;
        if (owns && d < D) S_mem[(size_t)d * Dv + j] = S[i];
    }
}

// The same walk for a prompt's step in bfloat16, laid out as the linear attention's walk above: the 16 lanes of one
// row of a wave share C columns of the state, lane r keeping rows r * ROWS .. r * ROWS + ROWS - 1 of each, so that what
// a lane reads of q and k from LDS serves all its columns and the two sums of a token (S^T k before the write, S^T q
// after it) are exchanges inside the vector unit.  q and k lie in LDS as floats so that the 16 lanes' 16-byte pieces
// of a read are one contiguous run; rows beyond D are zero.  Blocks of 32 tokens; a block's unit norms, write
// strengths and decays are taken in LDS before it is walked, and its outputs leave together.
#define DELTA_WALK_TOKENS 32
#define DELTA_WALK_THREADS 256
template <int ROWS, int C, bool CHANNELS>
__global__ __launch_bounds__(DELTA_WALK_THREADS) void delta_walk_kernel(
    const bf16_t* __restrict__ qkv, int qkv_stride, const bf16_t* __restrict__ proj, int proj_stride, int b_col,
    int a_col, const float* __restrict__ a_log, const float* __restrict__ dt_bias, float* __restrict__ state,
    long long state_stride, const int* __restrict__ cu_q, const int* __restrict__ slots, float* __restrict__ raw_out,
    int n_heads, int n_kv, int D, int Dv, const float* __restrict__ decays) {
    extern __shared__ float lds[];
    constexpr int TB = DELTA_WALK_TOKENS, threads = DELTA_WALK_THREADS;
    constexpr int slice = threads / 16 * C;      // columns a workgroup
    constexpr int Dp = 16 * ROWS;
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int j0 = blockIdx.z * slice;
    const int first = cu_q[seq], last = cu_q[seq + 1];
    if (first >= last) return;
    float* q_s = lds;               // [TB][Dp], row d = r * ROWS + i at (i / 4) * 64 + r * 4 + i % 4
    float* k_s = q_s + TB * Dp;
    float* al_s = k_s + TB * Dp;    // [TB][Dp] in the same order, CHANNELS only
    float* v_s = al_s + (CHANNELS ? TB * Dp : 0);     // [TB][slice]
    float* o_s = v_s + TB * slice;  // [TB][slice]
    float* be_s = o_s + TB * slice; // [TB]
    float* de_s = be_s + TB;        // [TB]
    auto place = [](int d) { const int r = d / ROWS, i = d % ROWS; return (i / 4) * 64 + r * 4 + i % 4; };
    for (int i = tid; i < (CHANNELS ? 3 : 2) * TB * Dp; i += threads) lds[i] = 0.f;
    const int jl = (tid / 16) * C, r = tid % 16;
    float* S_mem = state + (size_t)slots[seq] * state_stride + (size_t)head * D * Dv;
    float S[C][ROWS];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int d = r * ROWS + i, j = j0 + jl + c;
            S[c][i] = (j < Dv && d < D) ? S_mem[(size_t)d * Dv + j] : 0.f;
        }
    const int wave = tid / SIA_WAVE, lane = tid % SIA_WAVE;
    const int kv_head = head / (n_heads / n_kv);
    const int q_col = kv_head * D, k_col = n_kv * D + kv_head * D, v_col = 2 * n_kv * D + head * Dv;
    const float rate = CHANNELS ? 0.f : expf(a_log[head]), bias = !CHANNELS && dt_bias ? dt_bias[head] : 0.f;
    const float q_scale = rsqrtf((float)D);
    __syncthreads();
    for (int t0 = first; t0 < last; t0 += TB) {
        const int nt = min(TB, last - t0);
        for (int idx = tid; idx < nt * D; idx += threads) {
            const int t = idx / D, d = idx % D;
            const bf16_t* row = qkv + (size_t)(t0 + t) * qkv_stride;
            q_s[t * Dp + place(d)] = bf16_to_float(row[q_col + d]);
            k_s[t * Dp + place(d)] = bf16_to_float(row[k_col + d]);
            if (CHANNELS) al_s[t * Dp + place(d)] = decays[((size_t)(t0 + t) * n_heads + head) * D + d];
        }
        for (int idx = tid; idx < nt * slice; idx += threads) {
            const int t = idx / slice, c = idx % slice;
            v_s[idx] = j0 + c < Dv ? bf16_to_float(qkv[(size_t)(t0 + t) * qkv_stride + v_col + j0 + c]) : 0.f;
        }
        if (tid < nt) {
            const bf16_t* row = proj + (size_t)(t0 + tid) * proj_stride;
            be_s[tid] = 1.f / (1.f + expf(-bf16_to_float(row[b_col + head])));
            if (!CHANNELS) {
                const float za = bf16_to_float(row[a_col + head]) + bias;
                de_s[tid] = expf(-rate * (fmaxf(za, 0.f) + log1pf(expf(-fabsf(za)))));
            }
        }
        __syncthreads();
        for (int t = wave; t < nt; t += threads / SIA_WAVE) {      // unit vectors, a wave a token (the padding is zero)
            float sq = 0.f, sk = 0.f;
            for (int c = lane; c < Dp; c += SIA_WAVE) {
                sq += q_s[t * Dp + c] * q_s[t * Dp + c];
                sk += k_s[t * Dp + c] * k_s[t * Dp + c];
            }
            const float iq = rsqrtf(wave_sum(sq) + 1e-6f) * q_scale, ik = rsqrtf(wave_sum(sk) + 1e-6f);
            for (int c = lane; c < Dp; c += SIA_WAVE) {
                q_s[t * Dp + c] *= iq;
                k_s[t * Dp + c] *= ik;
            }
        }
        __syncthreads();
        float4 qn[ROWS / 4], kn[ROWS / 4], an[CHANNELS ? ROWS / 4 : 1];
        auto fetch = [&](int t) {
#pragma unroll
            for (int i = 0; i < ROWS / 4; ++i) {
                const int at = t * Dp + i * 64 + r * 4;
                qn[i] = *reinterpret_cast<const float4*>(q_s + at);
                kn[i] = *reinterpret_cast<const float4*>(k_s + at);
                if (CHANNELS) an[i] = *reinterpret_cast<const float4*>(al_s + at);
            }
        };
        fetch(0);
        for (int t = 0; t < nt; ++t) {
            float4 qv[ROWS / 4], kv[ROWS / 4], av[CHANNELS ? ROWS / 4 : 1];
            float vv[C];
#pragma unroll
            for (int i = 0; i < ROWS / 4; ++i) {
                qv[i] = qn[i];
                kv[i] = kn[i];
                if (CHANNELS) av[i] = an[i];
            }
#pragma unroll
            for (int c = 0; c < C; ++c) vv[c] = v_s[t * slice + jl + c];
            const float g = CHANNELS ? 1.f : de_s[t], b = be_s[t];
            fetch(min(t + 1, TB - 1));
            float kept[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                float acc = 0.f;
#pragma unroll
                for (int i = 0; i < ROWS / 4; ++i) {
                    S[c][4 * i] *= CHANNELS ? av[CHANNELS ? i : 0].x : g;
                    S[c][4 * i + 1] *= CHANNELS ? av[CHANNELS ? i : 0].y : g;
                    S[c][4 * i + 2] *= CHANNELS ? av[CHANNELS ? i : 0].z : g;
                    S[c][4 * i + 3] *= CHANNELS ? av[CHANNELS ? i : 0].w : g;
                    acc += kv[i].x * S[c][4 * i];
                    acc += kv[i].y * S[c][4 * i + 1];
                    acc += kv[i].z * S[c][4 * i + 2];
                    acc += kv[i].w * S[c][4 * i + 3];
                }
                kept[c] = acc;
            }
#pragma unroll
            for (int c = 0; c < C; ++c) kept[c] = row16_sum(kept[c]);
            float out[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float u = b * (vv[c] - kept[c]);
                float acc = 0.f;
#pragma unroll
                for (int i = 0; i < ROWS / 4; ++i) {
                    S[c][4 * i] += kv[i].x * u;
                    S[c][4 * i + 1] += kv[i].y * u;
                    S[c][4 * i + 2] += kv[i].z * u;
                    S[c][4 * i + 3] += kv[i].w * u;
                    acc += qv[i].x * S[c][4 * i];
                    acc += qv[i].y * S[c][4 * i + 1];
                    acc += qv[i].z * S[c][4 * i + 2];
                    acc += qv[i].w * S[c][4 * i + 3];
                }
                out[c] = acc;
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                out[c] = row16_sum(out[c]);
                if (r == 0) o_s[t * slice + jl + c] = out[c];
            }
        }
        __syncthreads();
        for (int idx = tid; idx < nt * slice; idx += threads)
            if (j0 + idx % slice < Dv)
                raw_out[((size_t)(t0 + idx / slice) * n_heads + head) * Dv + j0 + idx % slice] = o_s[idx];
        // (the next block's staging touches q_s, k_s, v_s and the gates, which nobody reads any more; o_s is written
        // again only behind two more barriers)
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int d = r * ROWS + i, j = j0 + jl + c;
            if (j < Dv && d < D) S_mem[(size_t)d * Dv + j] = S[c][i];
        }
}

// floats of workspace: the raw outputs [tokens, heads, Dv]
SIA_EXPORT long long sia_delta_rule_workspace(int n_tokens, int n_heads, int Dv) {
    return (long long)n_tokens * n_heads * Dv;
}

// y = o * rsqrt(mean(o^2) + eps) * w * factor for outputs left in a float workspace: a wave a (token, head).
template <typename T>
__global__ __launch_bounds__(SIA_WAVE) void delta_finish_kernel(const float* __restrict__ raw,
                                                                const float* __restrict__ gates,
                                                                const float* __restrict__ norm_w, T* __restrict__ out,
                                                                int n_heads, int Dv, float eps) {
    const size_t at = ((size_t)blockIdx.x * n_heads + blockIdx.y) * Dv;
    const int lane = threadIdx.x;
    float ss = 0.f;
    for (int c = lane; c < Dv; c += SIA_WAVE) ss += raw[at + c] * raw[at + c];
    const float inv = rsqrtf(wave_sum(ss) / (float)Dv + eps);
    for (int c = lane; c < Dv; c += SIA_WAVE) out[at + c] = from_float<T>(raw[at + c] * inv * norm_w[c] * gates[at + c]);
}

template <bool CHANNELS>
static int launch_delta_rule(const void* qkv, int qkv_stride, const void* proj, int proj_stride, int g_col, int b_col,
                             int a_col, const float* a_log, const float* dt_bias, const float* norm_w, float* state,
                             long long state_stride, const int* cu_q, const int* slots, void* out, int n_tokens,
                             int n_seqs, int max_q_len, int n_heads, int n_kv, int D, int Dv, float eps, int dtype,
                             float* workspace, const float* decays, const float* gates, hipStream_t stream) {
    // columns a workgroup: all of a head's, or in a step of runs of tokens a slice of them, as narrow as it takes to
    // fill the chip; lanes a column: the largest power of two that keeps the workgroup within 512 threads
    int slice = Dv;
    if (max_q_len > 1)
        while (slice > 8 && (long long)n_seqs * n_heads * ((Dv + slice - 1) / slice) < 256) slice = (slice + 1) / 2;
    int R = 1, rows = D;
    for (;;) {
        R = 1;
        while (R * 2 <= SIA_WAVE && slice * R * 2 <= 512 && R * 2 <= D) R *= 2;
        rows = (D + R - 1) / R;
        if (rows <= 128 || slice <= 1) break;
        slice = (slice + 1) / 2;
    }
    if (rows > 128) return SIA_BAD_ARGUMENT;
    const int threads = ((slice * R + SIA_WAVE - 1) / SIA_WAVE) * SIA_WAVE;
    int TB = max_q_len >= 16 ? 16 : (max_q_len >= 4 ? 4 : 1);
    // a workgroup that owns a whole head norms and gates its outputs itself (a decode step: one launch less)
    const bool whole = slice == Dv;
    auto bytes = [&](int tb) {
        return (size_t)tb * ((CHANNELS ? 3 : 2) * D + (whole ? 2 : 1) * slice + 2) * sizeof(float);
    };
    while (TB > 1 && bytes(TB) > 60 * 1024) TB /= 2;
    if (bytes(TB) > 60 * 1024) return SIA_BAD_ARGUMENT;
    float* raw = whole ? nullptr : workspace;
    dim3 grid(n_seqs, n_heads, (Dv + slice - 1) / slice), block(threads), fgrid(n_tokens, n_heads), fblock(SIA_WAVE);
    // a prompt's step in bfloat16: the walk whose lanes share columns, where its rows fit a lane's registers and LDS
    constexpr int w_cols = 2, w_slice = DELTA_WALK_THREADS / 16 * w_cols;
    const int w_rows = (D + 15) / 16;
    const int w_rows_t = w_rows <= 4 ? 4 : w_rows <= 8 ? 8 : w_rows <= 16 ? 16 : 32;
    const size_t w_lds = (size_t)(DELTA_WALK_TOKENS * ((CHANNELS ? 3 : 2) * 16 * w_rows_t + 2 * w_slice + 2)) * sizeof(float);
    if (max_q_len > 1 && dtype == SIA_BF16 && w_rows_t <= 16 && w_lds <= 60 * 1024) {
        dim3 wgrid(n_seqs, n_heads, (Dv + w_slice - 1) / w_slice), wblock(DELTA_WALK_THREADS);
#define WALK(ROWS)                                                                                                   \
    hipLaunchKernelGGL((delta_walk_kernel<ROWS, w_cols, CHANNELS>), wgrid, wblock, w_lds, stream, (const bf16_t*)qkv, \
                       qkv_stride, (const bf16_t*)proj, proj_stride, b_col, a_col, a_log, dt_bias, state,            \
                       state_stride, cu_q, slots, workspace, n_heads, n_kv, D, Dv, decays)
        if (w_rows_t == 4) WALK(4);
        else if (w_rows_t == 8) WALK(8);
        else WALK(16);
#undef WALK
        if (CHANNELS)
            hipLaunchKernelGGL(delta_finish_kernel<bf16_t>, fgrid, fblock, 0, stream, workspace, gates, norm_w, (bf16_t*)out,
                               n_heads, Dv, eps);
        else
            launch_finish<bf16_t>(workspace, proj, proj_stride, g_col, norm_w, out, n_tokens, n_heads, Dv, eps, stream);
        return SIA_LAUNCH_CHECK();
    }
#define LAUNCH(T, ROWS)                                                                                              \
    hipLaunchKernelGGL((delta_rule_kernel<T, ROWS, CHANNELS>), grid, block, bytes(TB), stream, (const T*)qkv, qkv_stride,      \
                       (const T*)proj, proj_stride, b_col, a_col, a_log, dt_bias, state, state_stride, cu_q, slots,   \
                       raw, n_heads, n_kv, D, Dv, R, TB, slice, g_col, norm_w, (T*)out, eps, decays, gates)
#define RUN(T)                                                                                                       \
    do {                                                                                                             \
        if (rows <= 4) LAUNCH(T, 4);                                                                                 \
        else if (rows <= 8) LAUNCH(T, 8);                                                                            \
        else if (rows <= 16) LAUNCH(T, 16);                                                                          \
        else if (rows <= 32) LAUNCH(T, 32);                                                                          \
        else if (rows <= 64) LAUNCH(T, 64);                                                                          \
        else LAUNCH(T, 128);                                                                                         \
        if (raw && CHANNELS)                                                                                         \
            hipLaunchKernelGGL(delta_finish_kernel<T>, fgrid, fblock, 0, stream, workspace, gates, norm_w, (T*)out,  \
                               n_heads, Dv, eps);                                                                    \
        else if (raw)                                                                                                \
            launch_finish<T>(workspace, proj, proj_stride, g_col, norm_w, out, n_tokens, n_heads, Dv, eps, stream);  \
    } while (0)
    if (dtype == SIA_F32) RUN(float);
    else if (dtype == SIA_BF16) RUN(bf16_t);
    else return SIA_BAD_ARGUMENT;
#undef RUN
#undef LAUNCH
    return SIA_LAUNCH_CHECK();
}

SIA_EXPORT int sia_delta_rule(const void* qkv, int qkv_stride, const void* proj, int proj_stride, int g_col, int b_col,
                              int a_col, const float* a_log, const float* dt_bias, const float* norm_w, float* state,
                              long long state_stride, const int* cu_q, const int* slots, void* out, int n_tokens,
                              int n_seqs, int max_q_len, int n_heads, int n_kv, int D, int Dv, float eps, int dtype,
                              float* workspace, hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    if (D <= 0 || Dv <= 0 || D > 512 || Dv > 512 || n_heads <= 0 || n_heads > 65535 || n_kv <= 0 || n_heads % n_kv ||
        !state || !norm_w || !a_log || !workspace || qkv_stride < 2 * n_kv * D + n_heads * Dv || g_col < 0 ||
        b_col < 0 || a_col < 0 || g_col + n_heads * Dv > proj_stride || b_col + n_heads > proj_stride ||
        a_col + n_heads > proj_stride || state_stride < (long long)n_heads * D * Dv)
        return SIA_BAD_ARGUMENT;
    return launch_delta_rule<false>(qkv, qkv_stride, proj, proj_stride, g_col, b_col, a_col, a_log, dt_bias, norm_w, state,
                                    state_stride, cu_q, slots, out, n_tokens, n_seqs, max_q_len, n_heads, n_kv, D, Dv, eps,
                                    dtype, workspace, nullptr, nullptr, stream);
}

// The same rule with a decay per key channel (decays [tokens, n_heads, D]) and the output gate's factors (gates
// [tokens, n_heads * Dv]) computed before, both float; b_col names the write strengths' logits in the rows of proj.
SIA_EXPORT int sia_channel_delta_rule(const void* qkv, int qkv_stride, const void* proj, int proj_stride, int b_col,
                                      const float* decays, const float* gates, const float* norm_w, float* state,
                                      long long state_stride, const int* cu_q, const int* slots, void* out, int n_tokens,
                                      int n_seqs, int max_q_len, int n_heads, int n_kv, int D, int Dv, float eps,
                                      int dtype, float* workspace, hipStream_t stream) {
    if (n_seqs <= 0 || n_tokens <= 0) return 0;
    if (D <= 0 || Dv <= 0 || D > 512 || Dv > 512 || n_heads <= 0 || n_heads > 65535 || n_kv <= 0 || n_heads % n_kv ||
        !state || !norm_w || !decays || !gates || !workspace || qkv_stride < 2 * n_kv * D + n_heads * Dv || b_col < 0 ||
        b_col + n_heads > proj_stride || state_stride < (long long)n_heads * D * Dv)
        return SIA_BAD_ARGUMENT;
    return launch_delta_rule<true>(qkv, qkv_stride, proj, proj_stride, 0, b_col, 0, nullptr, nullptr, norm_w, state,
                                   state_stride, cu_q, slots, out, n_tokens, n_seqs, max_q_len, n_heads, n_kv, D, Dv, eps,
                                   dtype, workspace, decays, gates, stream);
}
