// Attention of the 32-bit path over the paged cache, for head sizes up to 128: the arithmetic of the plain kernel
// (attention_generic.hip), operation for operation, with keys and values that several rows share.
//
// What bounds the plain kernel is its loads: a wave per (token, head) reads every key alone, a lane a key row, and the
// values 4 bytes in every 64.  Here a workgroup of four waves takes the heads of one key/value head (up to four at a
// time) of eight consecutive tokens, and brings each chunk of 64 absolute positions into LDS once, 16 bytes a
// lane in the order of the pages; the next chunk is on its way from memory meanwhile, its pages looked up a chunk
// earlier.  A token that is its sequence's only one (decode) has a workgroup of its own, and so has every token of a step
// that leaves the chip room for that.  Everything a row's result is made of (chunks, order of sums, exponentials) is as in the
// plain kernel, so it depends on the row's own keys only, not on which of the forms it goes through.
//   303 tokens (three decoded over 200 keys, a prompt of 300), 32 heads of 64 on 8: 240 -> 58 us;  one token over 16,000 keys 3,895 ->
//   1,365, 64 over 2,048 810 -> 215.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define CHUNK SIA_WAVE      // keys at a time, a lane each
#define WAVES 4
#define TOKENS 8            // tokens a workgroup; a wave takes every fourth
#define TURNS (TOKENS / WAVES)

// DP: 64 or 128, the head sizes' upper bound.  HB: heads a wave takes together.
// KEEP: with kept first positions; what tells them from the window costs the others 3 to 5 % (one token over 550 keys beside seven
// more, 32 heads of 64 on 8: 64.8 us with, 61.1 without;  600 tokens 138.7 and 131.0).
template <int DP, int HB, bool KEEP>
__global__ __launch_bounds__(WAVES * SIA_WAVE) void attention_f32_kernel(
    const float* __restrict__ q, int q_row_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_width, const int* __restrict__ seq_of_token,
    const int* __restrict__ positions, float* __restrict__ out, int n_tokens, int n_single, int n_heads, int n_kv,
    int head_dim, int value_dim, int page_size, float scale, int window, int chunk, const float* __restrict__ sinks,
    float cap, int keep_first) {
    constexpr int K_ROW = DP + 4, V_ROW = CHUNK + 4;      // 16 bytes more than the data: rows begin in other banks
    constexpr int K_LOADS = CHUNK * DP / 4 / (WAVES * SIA_WAVE), V_LOADS = K_LOADS;
    extern __shared__ float lds[];
    float* k_s = lds;                            // [CHUNK][K_ROW]
    float* v_s = k_s + CHUNK * K_ROW;            // [DP][V_ROW]
    float* q_s = v_s + DP * V_ROW;               // [TOKENS][HB][DP]
    float* p_s = q_s + TOKENS * HB * DP;         // [WAVES][HB][CHUNK]

    const int tid = threadIdx.x, lane = tid % SIA_WAVE, wave = tid / SIA_WAVE;
    const int h0 = blockIdx.y * HB, hk = h0 / (n_heads / n_kv);
    const bool single = (int)blockIdx.x < n_single;
    int t0 = single ? blockIdx.x : n_single + (blockIdx.x - n_single) * TOKENS;
    const int t_end = single ? t0 + 1 : min(t0 + TOKENS, n_tokens);
    const int d4 = head_dim / 4, in_page = page_size - 1, page_log2 = __ffs(page_size) - 1;
    const int run4 = min(page_size, CHUNK) / 4;  // pieces of four positions that lie together in a page
    float* p_w = p_s + wave * HB * CHUNK;

    // The pieces of four floats that this thread brings in: key and dimension, in the order of a key's row, and
    // dimension and first position, in the order of a page.  -1: none.
    int kj[K_LOADS], kd[K_LOADS], vj[V_LOADS], vd[V_LOADS];
#pragma unroll
    for (int i = 0; i < K_LOADS; ++i) {
        const int at = tid + i * WAVES * SIA_WAVE;
        kj[i] = at < CHUNK * d4 ? at / d4 : -1;
        kd[i] = at % d4 * 4;
        vj[i] = at < CHUNK / 4 * value_dim ? (at / (run4 * value_dim) * run4 + at % run4) * 4 : -1;
        vd[i] = at / run4 % value_dim;
    }

    while (t0 < t_end) {      // the tokens of one sequence after those of another
        const int seq = seq_of_token[t0];
        int n = 1;
        while (t0 + n < t_end && seq_of_token[t0 + n] == seq) ++n;
        const int* table = block_table + (size_t)seq * table_width;
        int first = positions[t0], last = first;
        for (int i = 1; i < n; ++i) {
            first = min(first, positions[t0 + i]);
            last = max(last, positions[t0 + i]);
        }
        auto oldest = [&](int pos) {
            int lo = window > 0 ? max(0, pos - window + 1) : 0;
            return chunk > 0 ? max(lo, pos - pos % chunk) : lo;
        };
        // chunks that some row of the run may see, in order: those of the kept positions, then from the window's on
        const int lo0 = oldest(first), keep0 = KEEP ? min(keep_first, oldest(last)) : 0, c_lo = lo0 / CHUNK * CHUNK;
        auto next_chunk = [&](int c0) { return KEEP && c0 + CHUNK < keep0 ? c0 + CHUNK : max(c0 + CHUNK, c_lo); };
        auto page_of = [&](int c0) {
            const int j = c0 + lane;
            return j <= last && (j >> page_log2) < table_width ? table[j >> page_log2] : -1;
        };

        for (int i = tid; i < n * HB * d4; i += WAVES * SIA_WAVE) {
            const int row = i / d4, piece = i % d4;
            *(f32x4*)(q_s + row * DP + piece * 4) =
                *(const f32x4*)(q + (size_t)(t0 + row / HB) * q_row_stride + (h0 + row % HB) * head_dim + piece * 4);
        }

        f32x4 kr[K_LOADS], vr[V_LOADS];
        auto fetch = [&](int c0, int page) {
#pragma unroll
            for (int i = 0; i < K_LOADS; ++i) {
                const int pg = __shfl(page, max(kj[i], 0), SIA_WAVE);
                kr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (kj[i] >= 0 && pg >= 0)
                    kr[i] = *(const f32x4*)(k_pages + ((((size_t)pg * n_kv + hk) << page_log2) + ((c0 + kj[i]) & in_page)) * head_dim + kd[i]);
            }
#pragma unroll
            for (int i = 0; i < V_LOADS; ++i) {
                const int pg = __shfl(page, max(vj[i], 0), SIA_WAVE);
                vr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (vj[i] >= 0 && pg >= 0)
                    vr[i] = *(const f32x4*)(v_pages + ((((size_t)pg * n_kv + hk) * value_dim + vd[i]) << page_log2) + ((c0 + vj[i]) & in_page));
            }
        };
        auto put = [&]() {
#pragma unroll
            for (int i = 0; i < K_LOADS; ++i)
                if (kj[i] >= 0) *(f32x4*)(k_s + kj[i] * K_ROW + kd[i]) = kr[i];
#pragma unroll
            for (int i = 0; i < V_LOADS; ++i)
                if (vj[i] >= 0) *(f32x4*)(v_s + vd[i] * V_ROW + vj[i]) = vr[i];
        };

        float m[TURNS][HB], l[TURNS][HB], acc[TURNS][HB][DP / SIA_WAVE];
#pragma unroll
        for (int t = 0; t < TURNS; ++t)
#pragma unroll
            for (int h = 0; h < HB; ++h) {
                m[t][h] = -INFINITY;
                l[t][h] = 0.f;
#pragma unroll
                for (int a = 0; a < DP / SIA_WAVE; ++a) acc[t][h][a] = 0.f;
            }

        int c0 = KEEP && keep0 > 0 ? 0 : c_lo;
        int page = page_of(c0), page_next = page_of(next_chunk(c0));
        fetch(c0, page);
        while (c0 <= last) {
            const int c1 = next_chunk(c0);
            const bool has_page = page >= 0;
            __syncthreads();      // the readers of the chunk before are through
            put();
            __syncthreads();
            page = page_next;
            if (c1 <= last) fetch(c1, page);
            page_next = page_of(next_chunk(c1));
#pragma unroll
            for (int t = 0; t < TURNS; ++t) {
                const int i = wave + t * WAVES;
                if (i >= n) continue;
                const int pos = positions[t0 + i], lo = oldest(pos), keep = KEEP ? min(keep_first, lo) : 0;
                if (c0 > pos || (c0 + CHUNK <= lo && !(KEEP && c0 < keep))) continue;      // no visible key in this chunk
                const int j = c0 + lane;
                const bool visible = (j >= lo || (KEEP && j < keep)) && j <= pos && has_page;
                float s[HB];
#pragma unroll
                for (int h = 0; h < HB; ++h) s[h] = 0.f;
                const float* q_row = q_s + i * HB * DP;
                for (int d = 0; d < head_dim; d += 4) {
                    const f32x4 kk = *(const f32x4*)(k_s + lane * K_ROW + d);
#pragma unroll
                    for (int h = 0; h < HB; ++h) {
                        const f32x4 qq = *(const f32x4*)(q_row + h * DP + d);
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[h] += qq[e] * kk[e];
                    }
                }
#pragma unroll
                for (int h = 0; h < HB; ++h) {
                    float x = s[h] * scale;
                    if (cap > 0.f) x = cap * tanhf(x / cap);
                    if (!visible) x = -INFINITY;
                    const float m_new = fmaxf(m[t][h], wave_max(x));
                    const float p = visible ? expf(x - m_new) : 0.f;
                    const float alpha = expf(m[t][h] - m_new);
                    l[t][h] = l[t][h] * alpha + wave_sum(p);
                    m[t][h] = m_new;
#pragma unroll
                    for (int a = 0; a < DP / SIA_WAVE; ++a) acc[t][h][a] *= alpha;
                    p_w[h * CHUNK + lane] = p;
                }
                __builtin_amdgcn_wave_barrier();      // the wave's LDS accesses run in order: no more than that is needed
                // values of keys that the row does not see may be anything: they are left out, not weighted with 0.  In a
                // chunk with kept positions the loop is run for those, and again for what the window holds of the chunk.
                const int j_last = min(pos, c0 + CHUNK - 1) - c0;
                const bool kept = KEEP && c0 < keep;
                int j_from = kept ? 0 : max(lo, c0) - c0, j_to = kept ? min(keep, c0 + CHUNK) - 1 - c0 : j_last;
                for (;;) {
                    for (int jj = j_from & ~3; jj <= j_to; jj += 4) {
                        const bool whole = jj >= j_from && jj + 3 <= j_to;
                        f32x4 pp[HB];
#pragma unroll
                        for (int h = 0; h < HB; ++h) pp[h] = *(const f32x4*)(p_w + h * CHUNK + jj);
#pragma unroll
                        for (int a = 0; a < DP / SIA_WAVE; ++a) {
                            f32x4 vv = *(const f32x4*)(v_s + (lane + a * SIA_WAVE) * V_ROW + jj);
                            if (!whole)
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    if (jj + e < j_from || jj + e > j_to) vv[e] = 0.f;
#pragma unroll
                            for (int h = 0; h < HB; ++h)
#pragma unroll
                                for (int e = 0; e < 4; ++e) acc[t][h][a] += pp[h][e] * vv[e];
                        }
                    }
                    if (!KEEP || j_to >= j_last) break;
                    j_from = max(lo - c0, j_to + 1);
                    j_to = j_last;
                }
            }
            c0 = c1;
        }
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            const int i = wave + t * WAVES;
            if (i >= n) continue;
#pragma unroll
            for (int h = 0; h < HB; ++h) {
                float sum = l[t][h];
                if (sinks) sum += expf(sinks[h0 + h] - m[t][h]);
                const float inv = 1.f / sum;
                float* o = out + ((size_t)(t0 + i) * n_heads + h0 + h) * value_dim;
#pragma unroll
                for (int a = 0; a < DP / SIA_WAVE; ++a)
                    if (lane + a * SIA_WAVE < value_dim) o[lane + a * SIA_WAVE] = acc[t][h][a] * inv;
            }
        }
        __syncthreads();      // before the next sequence's queries
        t0 += n;
    }
}

template <int DP, int HB>
static int launch(const float* q, int q_row_stride, const float* k_pages, const float* v_pages, const int* block_table,
                  int table_width, const int* seq_of_token, const int* positions, float* out, int n_tokens, int n_single,
                  int n_seqs, int max_kv, int max_run_kv, int n_heads, int n_kv, int head_dim, int value_dim, int page_size, float scale,
                  int window, int chunk, const float* sinks, float cap, int keep_first, hipStream_t stream) {
    constexpr int bytes = (CHUNK * (DP + 4) + DP * (CHUNK + 4) + TOKENS * HB * DP + WAVES * HB * CHUNK) * (int)sizeof(float);
    // Eight tokens a workgroup share what is loaded, but follow one another in a wave, and their sequences one another in the
    // workgroup: a token each where one round of two workgroups a unit (one, if LDS holds no more) takes them all, or, if an eight
    // holds several sequences, three rounds for four of them.  32 heads of 64 on 8, us, the plain kernel, eight, one:  8 tokens over 72 keys
    // 20, 25, 14.5;  16 over 216 53, 49, 27;  64 over 264 87, 59, 36;  128 over 328 182, 71, 80 (two rounds);  24 heads of
    // 128 on 8, 16 sequences of 3 over 300 (two rounds) 164, 170, 90.  Where single tokens see more keys than the others do, the step
    // takes as long as theirs, which a second workgroup on the unit makes longer: 45 tokens beside six over up to 145 keys 19.0 eight, 20.3 one;
    // 60 beside three over up to 234 24.9 and 25.5;  with the others' keys more, 45 beside one over 30 15.2 and 9.6.
    const long long many = n_tokens - n_single, runs = n_seqs - n_single;
    const long long at_once = 256 * (n_single > 0 && max_run_kv < max_kv ? 1 : min(2, 160 * 1024 / bytes));
    if (many > 0 && 4 * many * n_tokens * (n_heads / HB) <= at_once * max(4 * many, 3 * TOKENS * runs)) n_single = n_tokens;
    const dim3 grid(n_single + (n_tokens - n_single + TOKENS - 1) / TOKENS, n_heads / HB);
    const bool keeps = keep_first > 0;
    auto kernel = keeps ? attention_f32_kernel<DP, HB, true> : attention_f32_kernel<DP, HB, false>;
    static bool set[64][2] = {};      // more LDS than a kernel gets unasked, allowed once per device
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return (int)hipGetLastError();
    if (device < 0 || device >= 64 || !set[device][keeps]) {
        const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return (int)e;
        if (device >= 0 && device < 64) set[device][keeps] = true;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(WAVES * SIA_WAVE), bytes, stream, q, q_row_stride, k_pages, v_pages, block_table,
                       table_width, seq_of_token, positions, out, n_tokens, n_single, n_heads, n_kv, head_dim, value_dim,
                       page_size, scale, window, chunk, sinks, cap, keep_first);
    return SIA_LAUNCH_CHECK();
}

extern "C" int sia_attention_generic(const void*, int, const void*, const void*, const int*, int, const int*, const int*, void*,
                                     int, int, int, int, int, int, float, int, int, const float*, float, int, int, hipStream_t);

// The arguments of the plain kernel, and n_single: that many tokens, the first ones, are their sequences' only ones; n_seqs;
// max_kv: no sequence holds more keys, max_run_kv: nor does one of more than a token (max_kv if that is not known).
// Rows of other sizes, and rows and pages that do not lie in sixteens of bytes, go to the plain kernel; so do steps whose sequences hold so few keys that bringing them into LDS first takes longer than a wave a row and head
// does, as long as those waves find room:  32 heads of 64 on 8, plain against this, us:  one token over 4 keys 6.1 / 8.2, 16: 7.4 / 8.6, 40:
// 12.1 / 9.4, 16 tokens over 16 7.4 / 14.5;  24 heads of 128 on 8:  4: 6.6 / 10.4, 16: 11.3 / 10.9, 64 sequences over 16 13.4 / 20.8.
SIA_EXPORT int sia_attention_f32(const float* q, int q_row_stride, const float* k_pages, const float* v_pages,
                                 const int* block_table, int table_width, const int* seq_of_token, const int* positions,
                                 float* out, int n_tokens, int n_single, int n_seqs, int max_kv, int max_run_kv, int n_heads, int n_kv,
                                 int head_dim, int value_dim, int page_size, float scale, int window, int chunk, const float* sinks, float cap,
                                 int keep_first, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    const bool takes = head_dim > 0 && head_dim <= 128 && head_dim % 4 == 0 && value_dim > 0 && value_dim <= 128 &&
                       q_row_stride % 4 == 0 && page_size >= 4 && (page_size & (page_size - 1)) == 0 && n_kv > 0 &&
                       n_heads % n_kv == 0 && n_heads <= 65535 && cap >= 0.f && keep_first >= 0 && n_single >= 0 && n_seqs >= 0 &&
                       !(max_kv <= 16 && (long long)n_tokens * n_heads <= 4096) &&
                       ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0;
    if (!takes)
        return sia_attention_generic(q, q_row_stride, k_pages, v_pages, block_table, table_width, seq_of_token, positions, out,
                                     n_tokens, n_heads, n_kv, head_dim, value_dim, page_size, scale, window, chunk, sinks,
                                     cap, keep_first, SIA_F32, stream);
    n_single = min(n_single, n_tokens);
    const int group = n_heads / n_kv;
    auto run = [&](auto narrow, auto wide) {
        return (head_dim <= 64 && value_dim <= 64 ? narrow : wide)(
            q, q_row_stride, k_pages, v_pages, block_table, table_width, seq_of_token, positions, out, n_tokens, n_single,
            n_seqs, max_kv, max_run_kv, n_heads, n_kv, head_dim, value_dim, page_size, scale, window, chunk, sinks, cap, keep_first,
            stream);
    };
    if (group % 4 == 0) return run(launch<64, 4>, launch<128, 4>);
    if (group % 3 == 0) return run(launch<64, 3>, launch<128, 3>);
    if (group % 2 == 0) return run(launch<64, 2>, launch<128, 2>);
    return run(launch<64, 1>, launch<128, 1>);
}
