// Attention of the 32-bit path over the paged cache, for head sizes up to 128: the arithmetic of the plain kernel
// (attention_generic.hip), operation for operation, on the float matrix cores.
//
// v_mfma_f32_16x16x4_f32 adds its four products one after the other, each with one rounding (the bits of four fmaf in order, denormal
// numbers among them: 640,000 results compared), so that a dot product by it has the plain kernel's bits if the elements come in
// their order.  What came before gave a lane a key and read queries and weights from LDS for every key, which LDS could not keep up with.
//
// A workgroup of four waves takes 16 rows: the heads of one key/value head for some consecutive tokens.  Of a chunk of 64 absolute
// positions a wave brings 16 keys, of which it makes the scores, and then the values' dimensions that are its own for all 64: nothing is
// loaded twice, and only the rows' maxima and weights go through LDS, behind a barrier each.  (A wave for 16 rows and a whole chunk
// needs no barriers, but has four times the chain, which is what a step of few hundred tokens waits for.)
// A token that is its sequence's only one (decode) has a workgroup of its own.
// What bounds it is the chain of a chunk: 16 dependent products of 32 cycles a wave each for scores and values (heads of 64), and two barriers, 5,000 cycles
// in all; 600 and more tokens fill the chip with chains.  us, before (a lane a key) and now: 303 tokens (three decoded over 200 keys, a prompt of 300), 32 heads of 64 on 8
// 57 -> 16.2 (19.4 in a step), 24 of 128 on 8 101 -> 22.8;  a prompt of 2,048 956 -> 308 (56 TFLOP/s of 157), 2,160 -> 443;  one token over 16,000 keys 1,358 -> 535;
// 64 over 2,048 211 -> 115 (537 MB: 4.7 TB/s);  256 over 17 with a query head for each of 16 key/value heads of 64 33 -> 23 (by the plain kernel).
#include <algorithm>
#include <cmath>

#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

#define CHUNK SIA_WAVE      // keys at a time
#define WAVES 4
#define ROWS 16             // (token, head) pairs of a workgroup
#define P_ROW (CHUNK + 4)

// Lane (r, g) = 16 g + r holds elements 4 g .. 4 g + 3 of its row; afterwards element e of it is element 4 e + g of the row: the order in which
// four steps of the matrix instruction take them.  And the other way round.
__device__ __forceinline__ void across_groups(f32x4& x) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const u32x2 v = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[e]), __float_as_uint(x[e + 2]), false, false);
        x[e] = __uint_as_float(v[0]), x[e + 2] = __uint_as_float(v[1]);
    }
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
        const u32x2 v = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[e]), __float_as_uint(x[e + 1]), false, false);
        x[e] = __uint_as_float(v[0]), x[e + 1] = __uint_as_float(v[1]);
    }
}

// x of this lane and x of the lane OFF away (16 or 32), one way round or the other
template <int OFF>
__device__ __forceinline__ u32x2 beside(float x) {
    const unsigned u = __float_as_uint(x);
    return OFF == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false) : __builtin_amdgcn_permlane16_swap(u, u, false, false);
}
template <int OFF>
__device__ __forceinline__ float max_beside(float x) {
    const u32x2 v = beside<OFF>(x);
    return fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
}
template <int OFF>
__device__ __forceinline__ float sum_beside(float x) {
    const u32x2 v = beside<OFF>(x);
    return __uint_as_float(v[0]) + __uint_as_float(v[1]);
}

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// all waves have come here, and what they have written to LDS is there; loads from memory stay on their way
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// DP: 32, 64 or 128, the head sizes' upper bound.  (Of 32 dimensions two of the waves have the values.)
template <int DP>
__global__ __launch_bounds__(WAVES * SIA_WAVE) void attention_f32_kernel(
    const float* __restrict__ q, int q_row_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_width, const int* __restrict__ seq_of_token,
    const int* __restrict__ positions, float* __restrict__ out, int n_tokens, int n_single, int n_heads, int n_kv,
    int head_dim, int value_dim, int page_size, float scale, int window, int chunk, const float* __restrict__ sinks,
    float cap, int keep_first, int tile_rows) {
    constexpr int PIECES = DP / 16, BLOCKS = DP < 64 ? 1 : DP / 64;      // a lane's fours of a row of keys; blocks of 16 dimensions of a wave's values
    __shared__ float most[WAVES][ROWS];
    __shared__ __attribute__((aligned(16))) float weight[ROWS * P_ROW];      // [row][position: 16 (j % 4) + j / 4]

    const int lane = threadIdx.x % SIA_WAVE, wave = threadIdx.x / SIA_WAVE, r = lane % 16, g = lane / 16;
    const bool has_values = DP >= 64 || wave < DP / 16;
    const int group = n_heads / n_kv, hk = blockIdx.x % n_kv, page_log2 = __ffs(page_size) - 1, in_page = page_size - 1;
    // The rows: token * group + head, those of a single token in tiles of their own, which come first; then the others', tile_rows a tile, from the
    // last on, whose tokens see the most keys.
    const int tile = blockIdx.x / n_kv, per_single = (group + ROWS - 1) / ROWS, single_tiles = n_single * per_single;
    long long row0, row_end;
    if (tile < single_tiles) {
        row0 = (long long)(tile / per_single) * group + tile % per_single * ROWS;
        row_end = (long long)(tile / per_single + 1) * group;
    } else {
        row_end = (long long)n_tokens * group;
        row0 = (long long)n_single * group + (long long)((int)(gridDim.x / n_kv) - 1 - tile) * tile_rows;
    }
    const int n_rows = (int)min((long long)(tile < single_tiles ? ROWS : tile_rows), row_end - row0);
    const int token = (int)((row0 + min(r, n_rows - 1)) / group), head = hk * group + (int)((row0 + min(r, n_rows - 1)) % group);
    const int my_seq = seq_of_token[token], my_pos = positions[token];
    auto oldest = [&](int pos) {
        int lo = window > 0 ? max(0, pos - window + 1) : 0;
        return chunk > 0 ? max(lo, pos - pos % chunk) : lo;
    };
    const int my_lo = oldest(my_pos), my_keep = min(keep_first, my_lo);

    f32x4 qf[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int d = 16 * i + 4 * g;
        qf[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (d < head_dim) qf[i] = *(const f32x4*)(q + (size_t)token * q_row_stride + head * head_dim + d);
        across_groups(qf[i]);
    }

    float m = -INFINITY, l = 0.f;
    f32x4 acc[BLOCKS];
#pragma unroll
    for (int a = 0; a < BLOCKS; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int begin = 0; begin < n_rows;) {      // the rows of one sequence after those of another
        const int seq = __builtin_amdgcn_readlane(my_seq, begin);
        const unsigned same = (unsigned)(__ballot(r < n_rows && my_seq == seq) & 0xffff) >> begin;
        const int end = begin + __builtin_ctz(~same);
        const bool mine = r >= begin && r < end;
        const int* table = block_table + (size_t)seq * table_width;
        int first = mine ? my_pos : 0x7fffffff, last = mine ? my_pos : -1;
#pragma unroll
        for (int off = 1; off < 16; off *= 2) {
            first = min(first, __shfl_xor(first, off, SIA_WAVE));
            last = max(last, __shfl_xor(last, off, SIA_WAVE));
        }
        first = __builtin_amdgcn_readfirstlane(first), last = __builtin_amdgcn_readfirstlane(last);
        // chunks that some row of the run may see, in order: those of the kept positions, then from the window's on
        const int lo0 = oldest(first), lo_last = oldest(last), keep0 = min(keep_first, lo_last), c_lo = lo0 / CHUNK * CHUNK;
        auto next_chunk = [&](int c0) { return c0 + CHUNK < keep0 ? c0 + CHUNK : max(c0 + CHUNK, c_lo); };
        auto page_of = [&](int c0) {
            const int j = c0 + lane;
            return j <= last && (j >> page_log2) < table_width ? table[j >> page_log2] : -1;
        };
        // Keys 16 wave + r of the chunk, and dimensions of the values, four positions at a time.  Where there is no page (nor is there behind the
        // last position), or no such dimension, something near is read and not used:  a branch instead of that makes every chunk wait for its
        // loads (one token over 16,000 keys, 32 heads of 64 on 8: 543 us, 695 so).
        f32x4 kr[PIECES], vr[BLOCKS][4];
        auto fetch_keys = [&](int c0, int page) {
            const int j = 16 * wave + r, pg0 = __shfl(page, j, SIA_WAVE), pg = max(pg0, 0), in = pg0 < 0 ? 0 : (c0 + j) & in_page;
            const float* at = k_pages + ((((size_t)pg * n_kv + hk) << page_log2) + in) * head_dim;
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const int d = 16 * i + 4 * g;
                kr[i] = *(const f32x4*)(at + (d < head_dim ? d : 0));
            }
        };
        auto fetch_values = [&](int c0, int page) {
            if (!has_values) return;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int j = 16 * b + 4 * g, pg0 = __shfl(page, j, SIA_WAVE), pg = max(pg0, 0), in = pg0 < 0 ? 0 : (c0 + j) & in_page;
#pragma unroll
                for (int a = 0; a < BLOCKS; ++a) {
                    const int d = (wave * BLOCKS + a) * 16 + r;
                    vr[a][b] = *(const f32x4*)(v_pages + ((((size_t)pg * n_kv + hk) * value_dim + (d < value_dim ? d : 0)) << page_log2) + in);
                }
            }
        };

        int c0 = keep0 > 0 ? 0 : c_lo;
        int page = page_of(c0), page_next = page_of(next_chunk(c0));
        fetch_keys(c0, page);
        fetch_values(c0, page);
        while (c0 <= last) {
            const int c1 = next_chunk(c0);
            f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};      // of keys 16 wave + 4 g + e, row r
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                if (16 * i + 4 * g >= head_dim) kr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                across_groups(kr[i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) s = mfma(kr[i][e], qf[i][e], s);
            }
            if (c1 <= last) fetch_keys(c1, page_next);
            const bool has_page = __shfl(page, 16 * wave + 4 * g, SIA_WAVE) >= 0;
            const bool sees = mine && c0 <= my_pos && (c0 + CHUNK > my_lo || c0 < my_keep);      // a key of this chunk
            bool visible[4];
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = c0 + 16 * wave + 4 * g + e;
                visible[e] = mine && (j >= my_lo || j < my_keep) && j <= my_pos && has_page;
                x[e] = s[e] * scale;
                if (cap > 0.f) x[e] = cap * tanhf(x[e] / cap);
                if (!visible[e]) x[e] = -INFINITY;
            }
            float top = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
            top = max_beside<32>(max_beside<16>(top));
            if (g == 0) most[wave][r] = top;
            lds_barrier();
            const float m_new = fmaxf(m, fmaxf(fmaxf(most[0][r], most[1][r]), fmaxf(most[2][r], most[3][r])));
#pragma unroll
            for (int e = 0; e < 4; ++e) weight[r * P_ROW + e * 16 + wave * 4 + g] = visible[e] ? expf(x[e] - m_new) : 0.f;
            const float alpha = sees ? expf(m - m_new) : 1.f;
            m = m_new;
            lds_barrier();
            f32x4 p[4];      // element e of p[b]: position 16 b + 4 e + g
#pragma unroll
            for (int b = 0; b < 4; ++b) p[b] = *(const f32x4*)(weight + r * P_ROW + g * 16 + b * 4);
            const f32x4 pair = (p[0] + p[2]) + (p[1] + p[3]);      // the order of a wave's sum over 64 positions
            const float sum = sum_beside<16>(sum_beside<32>((pair[0] + pair[2]) + (pair[1] + pair[3])));
            if (sees) l = l * alpha + sum;
#pragma unroll
            for (int a = 0; a < BLOCKS; ++a) acc[a] *= alpha;
            if (has_values) {
                // Values of keys that a row does not see may be anything: where they are finite a weight of 0 leaves them out.  Those that no
                // row of the run sees are replaced; if one of the others is not finite, and rows differ in what they see, every row gets its own values.
                bool apart = false;
                if (c0 + CHUNK - 1 > first || c0 < lo_last || end - begin < n_rows || __any(page < 0)) {
                    const int j = c0 + lane;
                    const unsigned long long seen = __ballot(page >= 0 && (j >= lo0 || j < keep0)) >> (4 * g);      // bit 16 b + e
                    const unsigned half[2] = {(unsigned)seen, (unsigned)(seen >> 32)};
#pragma unroll
                    for (int b = 0; b < 4; ++b)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
#pragma unroll
                            for (int a = 0; a < BLOCKS; ++a) vr[a][b][e] = half[b / 2] >> (16 * (b % 2) + e) & 1 ? vr[a][b][e] : 0.f;
                    if (first < last || end - begin < n_rows) {
                        float odd = 0.f;
#pragma unroll
                        for (int b = 0; b < 4; ++b)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
#pragma unroll
                                for (int a = 0; a < BLOCKS; ++a) odd = fmaf(vr[a][b][e], 0.f, odd);
                        apart = __any(!(odd == 0.f));
                    }
                }
#pragma unroll
                for (int a = 0; a < BLOCKS; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) across_groups(vr[a][b]);
                if (!apart) {
#pragma unroll
                    for (int b = 0; b < 4; ++b)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
#pragma unroll
                            for (int a = 0; a < BLOCKS; ++a) acc[a] = mfma(vr[a][b][e], p[b][e], acc[a]);
                } else {
#pragma clang loop unroll(disable)
                    for (int row = begin; row < end; ++row) {
                        const int pos = __builtin_amdgcn_readlane(my_pos, row), lo = __builtin_amdgcn_readlane(my_lo, row);
                        const int keep = min(keep_first, lo);
#pragma unroll
                        for (int a = 0; a < BLOCKS; ++a) {
                            f32x4 own = acc[a];
#pragma unroll
                            for (int b = 0; b < 4; ++b)
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const int j = c0 + 16 * b + 4 * e + g;
                                    own = mfma(j <= pos && (j >= lo || j < keep) ? vr[a][b][e] : 0.f, p[b][e], own);
                                }
                            if (r == row) acc[a] = own;
                        }
                    }
                }
            }
            page = page_next;
            if (c1 <= last) fetch_values(c1, page);
            page_next = page_of(next_chunk(c1));
            c0 = c1;
        }
        begin = end;
    }
    if (r >= n_rows) return;
    if (sinks) l += expf(sinks[head] - m);
    const float inv = 1.f / l;
    float* o = out + ((size_t)token * n_heads + head) * value_dim;
#pragma unroll
    for (int a = 0; a < BLOCKS; ++a) {
        const int d = (wave * BLOCKS + a) * 16 + 4 * g;
        if (value_dim % 4 == 0) {
            if (d < value_dim) *(f32x4*)(o + d) = acc[a] * inv;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (d + e < value_dim) o[d + e] = acc[a][e] * inv;
        }
    }
}

static long long tiles_of(long long n_tokens, long long n_single, long long group, int tile_rows) {
    return n_single * ((group + ROWS - 1) / ROWS) + ((n_tokens - n_single) * group + tile_rows - 1) / tile_rows;
}

template <int DP>
static int launch(const float* q, int q_row_stride, const float* k_pages, const float* v_pages, const int* block_table,
                  int table_width, const int* seq_of_token, const int* positions, float* out, int n_tokens, int n_single,
                  int n_heads, int n_kv, int head_dim, int value_dim, int page_size, float scale,
                  int window, int chunk, const float* sinks, float cap, int keep_first, int tile_rows, hipStream_t stream) {
    const long long tiles = tiles_of(n_tokens, n_single, n_heads / n_kv, tile_rows);
    if (tiles * n_kv > 0x7fffffff) return SIA_BAD_ARGUMENT;
    hipLaunchKernelGGL(attention_f32_kernel<DP>, dim3((unsigned)(tiles * n_kv)), dim3(WAVES * SIA_WAVE), 0, stream, q, q_row_stride, k_pages,
                       v_pages, block_table, table_width, seq_of_token, positions, out, n_tokens, n_single, n_heads, n_kv, head_dim,
                       value_dim, page_size, scale, window, chunk, sinks, cap, keep_first, tile_rows);
    return SIA_LAUNCH_CHECK();
}

extern "C" int sia_attention_generic(const void*, int, const void*, const void*, const int*, int, const int*, const int*, void*,
                                     int, int, int, int, int, int, float, int, int, const float*, float, int, int, hipStream_t);

// The arguments of the plain kernel, and n_single: that many tokens, the first ones, are their sequences' only ones; n_seqs;
// max_kv: no sequence holds more keys.
// Rows of other sizes, and rows and pages that do not lie in sixteens of bytes, go to the plain kernel; so do steps whose sequences hold so few keys
// that one of its waves is through before this kernel's barriers are, as long as those waves find room:  32 heads of 64 on 8, one token, us, plain:  over 4 keys
// 5.2, 17: 7.3, here 5.5 (7.0 when the border of 16 was set);  45 tokens over 45 14.5 and 5.8;  24 heads of 128 on 8:  4: 6.5, 17: 11.6, here 7.2.  And so
// do those whose workgroups here would have one row of 16 each (a query head for every key/value head) in more than a round over the chip, with keys that
// fill no chunk:  256 tokens over 17 and 33 keys, plain and here, 16 heads of 64 on 16 22.9 / 38.9 and 28.5 / 39.8 (64 keys: 58 / 40), 40 of 96 on 40 70 / 161
// and 152 / 185;  64 tokens, 16 of 64 7.7 / 11.5 and 11.3 / 11.7.
SIA_EXPORT int sia_attention_f32(const float* q, int q_row_stride, const float* k_pages, const float* v_pages,
                                 const int* block_table, int table_width, const int* seq_of_token, const int* positions,
                                 float* out, int n_tokens, int n_single, int n_seqs, int max_kv, int n_heads, int n_kv,
                                 int head_dim, int value_dim, int page_size, float scale, int window, int chunk, const float* sinks, float cap,
                                 int keep_first, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    const bool takes = head_dim > 0 && head_dim <= 128 && head_dim % 4 == 0 && value_dim > 0 && value_dim <= 128 &&
                       q_row_stride % 4 == 0 && page_size >= 4 && (page_size & (page_size - 1)) == 0 && n_kv > 0 &&
                       n_heads % n_kv == 0 && n_heads <= 65535 && cap >= 0.f && keep_first >= 0 && n_single >= 0 && n_seqs >= 0 &&
                       !(max_kv <= 16 && (long long)n_tokens * n_heads <= 4096) &&
                       ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0;
    auto plain = [&]() {
        return sia_attention_generic(q, q_row_stride, k_pages, v_pages, block_table, table_width, seq_of_token, positions, out,
                                     n_tokens, n_heads, n_kv, head_dim, value_dim, page_size, scale, window, chunk, sinks,
                                     cap, keep_first, SIA_F32, stream);
    };
    if (!takes) return plain();
    n_single = min(n_single, n_tokens);
    // A workgroup whose 16 rows belong to several sequences takes one after the other: where runs are short, a workgroup for every token instead, if the
    // chip has room (two or three workgroups a unit, 640 in all, take little longer than one), or 8 or 4 rows a workgroup.  16 sequences of 3 tokens over
    // 300 keys, us, together and a token each:  16 heads of 64 on 16 98 / 24, 32 on 8 33 / 18.5, 24 of 128 on 8 68 / 29;  200 of 4 over 64, 6 heads of 32
    // on 6, 16 and 8 rows:  21 / 13 (10.7 with the kernel for heads of 32).
    const double room = 640, group = n_heads / n_kv, many = n_tokens - n_single, runs = n_seqs - n_single;
    const long long per_token = (n_heads / n_kv + ROWS - 1) / ROWS;
    int tile_rows = ROWS;
    if (runs > 1 && many > 0) {
        const double together = (1.0 + (runs - 1) * ROWS / (many * group)) * std::max(room, many * n_heads / ROWS);
        auto most = [&](int rows) {      // with the sequences that a workgroup's rows may be of
            return (1.0 + std::ceil((rows - 1) * runs / (many * group))) * std::max(room, many * n_heads / rows);
        };
        if (5 * std::max(room, many * per_token * n_kv) <= 4 * together)
            n_single = n_tokens;
        else
            for (int rows = ROWS / 2; rows >= 4; rows /= 2)
                if (5 * most(rows) <= 4 * most(tile_rows)) tile_rows = rows;
    }
    const long long workgroups = tiles_of(n_tokens, n_single, n_heads / n_kv, tile_rows) * n_kv;
    if (max_kv <= (workgroups >= 1536 ? 40 : 20) && workgroups >= 768 && 2LL * n_tokens * n_heads < 3 * workgroups) return plain();
    const int widest = max(head_dim, value_dim);
    return (widest <= 32 ? launch<32> : widest <= 64 ? launch<64> : launch<128>)(
        q, q_row_stride, k_pages, v_pages, block_table, table_width, seq_of_token, positions, out, n_tokens, n_single, n_heads, n_kv,
        head_dim, value_dim, page_size, scale, window, chunk, sinks, cap, keep_first, tile_rows, stream);
}
