// Sampling of one token per row of float logits [rows, vocab]: argmax, or temperature with
// optional top-k and top-p and a draw by inverting the cumulative distribution at a uniform
// number that the caller supplies (so that a request's draws do not depend on its batch).
//
// Order of operations (reference: sampling.py:141-173): temperature 0 -> argmax, all else
// ignored.  Otherwise x = logits / T; top-k keeps the values not below the k-th largest
// (ties with it stay; reference: sampling.py:69-84); top-p, over what top-k kept, drops a
// token iff the probability mass of the tokens above it already exceeds p (reference:
// sampling.py:96-129; tokens of equal value are kept or dropped together here, where the
// reference's sort splits them arbitrarily); p <= 0 keeps the top value only.  Then softmax
// over what is left, and the token is the first, in index order, whose cumulative
// probability exceeds u * total.
//
// Every row is spread over SP_CHUNKS workgroups, and the work is a short series of launches:
//   1. the maximum (and its index) of each chunk; the row's histograms are set to zero beside it;
//   2. top-k: the k-th largest value by radix selection over the order-preserving integer image
//      of the floats, 11 + 11 + 10 bits, one counting pass per digit;
//   3. top-p: the lowest kept value the same way, with the probability mass per digit in place of
//      the count;
//   4. the mass of what is kept, for SP_PIECES pieces of consecutive tokens of the row (a piece a wave), and then
//      one wave per row that finds the piece in which the cumulative mass passes u * total and the token in it.
// Probabilities enter every sum as fixed-point integers (exp(x - max) * 2^s with the largest s that keeps
// a row's sum below 2^63: 46 bits for 128,256 entries): integer sums do not depend on their order, so
// histograms can be built with atomics and every workgroup that recomputes a sum gets the same bits.  A
// token whose probability is below 2^-s of the most likely one's counts as zero.  A launch starts by reading
// the digit that the histogram of the launch before it decides, and leaves what has been decided so far in the
// row's workspace for the next (every workgroup of a row computes the same bits and writes them to the same
// place).  Launches whose filter no row asks for are skipped by the caller's hint.
//
// Where every row that is sampled keeps few tokens by its top-k (the caller's hint too), two launches do, with the same
// integers and so the same token:
//   1. a chunk's workgroup holds the chunk in registers and leaves, in index order, every token that may be among the
//      row's k largest: those not below the chunk's own k-th largest, or a little more where the digits found so far
//      tell few enough apart;
//   2. a workgroup a row takes top-k, top-p and the draw among those alone, its histograms in LDS; a row of so many equal
//      values that a chunk's would not fit their places is read whole instead.
// What bounds the series above is the launches: each waits for the digit of the one before.  top-k 50 and top-p 0.9 over
// 128,256 entries: 47 -> 22 us for one row, 76 -> 26 for 27, 136 -> 38 for 64.
#include "common.h"
#include "no_alloc.h"

#include <cstddef>
#include <mutex>

#define SP_CHUNKS 16
#define SP_THREADS 1024
#define SP_WAVES (SP_THREADS / SIA_WAVE)
#define SP_PASSES 3
#define SP_MAX_BINS 2048
#define SP_COUNT_COPIES 4  // histograms of a workgroup in LDS: lanes that meet in a bin add to different copies
#define SP_MASS_COPIES 3
#define SP_PIECES (SP_CHUNKS * SP_WAVES)  // of a row when the kept mass is summed: one for each wave of each chunk

typedef unsigned long long u64;

__host__ __device__ constexpr int sp_shift(int pass) { return pass == 0 ? 21 : pass == 1 ? 10 : 0; }
__host__ __device__ constexpr int sp_bins(int pass) { return pass == 2 ? 1024 : 2048; }

// What one more digit decided: of the k-th largest key (prefix, k_rem) or of the lowest kept key (the rest).
struct Decided {
    uint32_t prefix;  // the digits found so far
    int k_rem;        // rank of the k-th largest among the keys that share them
    u64 carried;      // mass above the keys that share them
    u64 limit;        // p * total mass
};

// What the launches of one row share.  `mass` and `count` are zero before the first counting launch.
struct SampleRow {
    u64 mass[SP_PASSES][SP_MAX_BINS];
    int count[SP_PASSES][SP_MAX_BINS];
    Decided after_k[SP_PASSES], after_p[SP_PASSES];
    u64 piece_mass[SP_PIECES];  // of the kept tokens
    float chunk_max[SP_CHUNKS];
    int chunk_arg[SP_CHUNKS];
};

__device__ __forceinline__ uint32_t ordered_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The float with a given key.
__device__ __forceinline__ float key_value(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

__device__ __forceinline__ u64 fixed_mass(float x, float mx, float one) { return (u64)(expf(x - mx) * one); }

__device__ __forceinline__ void take_better(float& bv, int& bi, float v, int i) {
    if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}

// Sum over the lanes above this one.
template <typename T>
__device__ __forceinline__ T lanes_above_sum(T v) {
    const int lane = threadIdx.x & 63;
    T inc = v;
#pragma unroll
    for (int off = 1; off < SIA_WAVE; off <<= 1) {
        const T other = __shfl_down(inc, off, SIA_WAVE);
        if (lane + off < SIA_WAVE) inc += other;
    }
    return inc - v;
}

// Sum over this lane and the lanes below it.
__device__ __forceinline__ u64 lanes_up_to_sum(u64 v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < SIA_WAVE; off <<= 1) {
        const u64 other = __shfl_up(v, off, SIA_WAVE);
        if (lane >= off) v += other;
    }
    return v;
}

// What the passes so far have decided for a row; computed by wave 0 of a workgroup.
struct RowState {
    float T, mx;          // temperature, maximum of x = logit / T
    uint32_t cut_k;       // keep keys >= cut_k (0: all); final after SP_PASSES top-k passes
    uint32_t prefix_k;    // digits of the k-th largest key found so far
    uint32_t cut_p;       // keep keys >= cut_p; final after SP_PASSES top-p passes
    uint32_t prefix_p;    // digits of the lowest kept key found so far
    int wants_k, wants_p; // the row has a top-k / a top-p filter to search for
};

// k-th largest: one more digit.  Lane l owns PER bins from l * PER on; lane 63 the highest.
template <int PER>
__device__ __forceinline__ void refine_top_k(const int* __restrict__ count, int shift, Decided& d) {
    const int lane = threadIdx.x & 63, base = lane * PER;
    int c[PER];
    const int4* src = (const int4*)(count + base);
#pragma unroll
    for (int i = 0; i < PER / 4; ++i) {
        const int4 v = src[i];
        c[4 * i] = v.x; c[4 * i + 1] = v.y; c[4 * i + 2] = v.z; c[4 * i + 3] = v.w;
    }
    int local = 0;
#pragma unroll
    for (int b = 0; b < PER; ++b) local += c[b];
    const int above = lanes_above_sum(local);
    int digit = -1, rank = 0;
    if (above < d.k_rem && d.k_rem <= above + local) {  // the lane that holds the k-th
        int seen = above;
#pragma unroll
        for (int b = PER - 1; b >= 0; --b) {
            if (digit < 0 && seen + c[b] >= d.k_rem) { digit = base + b; rank = d.k_rem - seen; }
            seen += c[b];
        }
    }
    const u64 owner = __ballot(digit >= 0);
    if (!owner) return;  // fewer keys than k under these digits (cannot be: k < vocab)
    const int src_lane = __ffsll((long long)owner) - 1;
    digit = __shfl(digit, src_lane, SIA_WAVE);
    rank = __shfl(rank, src_lane, SIA_WAVE);
    d.prefix |= (uint32_t)digit << shift;
    d.k_rem = rank;
}

// Lowest kept key: one more digit.  A bin holds a kept key iff it is not empty and the mass above it
// (carried + the bins above it) does not exceed the limit; the lowest such bin is taken.  With `first` the
// histogram is the whole row's, and the limit is taken from its total.
template <int PER>
__device__ __forceinline__ void refine_top_p(const u64* __restrict__ mass, int shift, Decided& d, float p, bool first) {
    const int lane = threadIdx.x & 63, base = lane * PER;
    u64 m[PER];
    const ulonglong2* src = (const ulonglong2*)(mass + base);
#pragma unroll
    for (int i = 0; i < PER / 2; ++i) {
        const ulonglong2 v = src[i];
        m[2 * i] = v.x; m[2 * i + 1] = v.y;
    }
    u64 local = 0;
#pragma unroll
    for (int b = 0; b < PER; ++b) local += m[b];
    const u64 higher = lanes_above_sum(local);
    if (first) {
        const u64 total = __shfl(higher + local, 0, SIA_WAVE);  // lane 0 has every other lane above it
        d.limit = (u64)((double)p * (double)total);
    }
    u64 above = d.carried + higher;
    int digit = -1;
    u64 above_digit = 0;
#pragma unroll
    for (int b = PER - 1; b >= 0; --b) {
        if (m[b] > 0 && above <= d.limit) { digit = base + b; above_digit = above; }
        above += m[b];
    }
    const u64 owners = __ballot(digit >= 0);
    if (!owners) return;  // no mass at all under these digits (cannot be: the row's maximum has the mass of one)
    const int src_lane = __ffsll((long long)owners) - 1;  // the lowest lane with a kept bin holds the lowest kept bin
    digit = __shfl(digit, src_lane, SIA_WAVE);
    above_digit = __shfl(above_digit, src_lane, SIA_WAVE);
    d.prefix |= (uint32_t)digit << shift;
    d.carried = above_digit;
}

// The row's state when `k_done` top-k and `p_done` top-p histograms are complete.  The digit of the latest
// histogram is decided here and left in the workspace; the digits before it were left there by the launches
// before.  With negative numbers nothing is decided: every digit is in the workspace.  One whole wave calls it.
__device__ __forceinline__ RowState row_state(SampleRow* __restrict__ ws, float T, int k, float p, int vocab,
                                              int filters, int k_done, int p_done) {
    const int lane = threadIdx.x & 63;
    RowState s;
    s.T = T;
    const float mx = wave_max(lane < SP_CHUNKS ? ws->chunk_max[lane] : -INFINITY);
    s.mx = T > 0.f ? mx / T : mx;
    s.wants_k = (filters & 1) && T > 0.f && k > 0 && k < vocab;
    s.wants_p = (filters & 2) && T > 0.f && p > 0.f && p < 1.f;
    s.cut_k = s.prefix_k = 0;
    if (s.wants_k && k_done != 0) {
        Decided d;
        if (k_done < 0 || (s.wants_p && p_done > 0)) {
            d = ws->after_k[SP_PASSES - 1];  // final since the first launch after the last top-k histogram
        } else {
            if (k_done >= 2) d = ws->after_k[k_done - 2];
            else { d.prefix = 0; d.k_rem = k; }
            d.carried = d.limit = 0;
            const int pass = k_done - 1;
            if (pass == 2) refine_top_k<sp_bins(2) / SIA_WAVE>(ws->count[2], sp_shift(2), d);
            else refine_top_k<sp_bins(0) / SIA_WAVE>(ws->count[pass], sp_shift(pass), d);
            if (lane == 0) ws->after_k[pass] = d;
        }
        s.prefix_k = d.prefix;
        if (k_done < 0 || k_done == SP_PASSES) s.cut_k = d.prefix;
    }
    s.cut_p = s.prefix_p = 0;
    if (T > 0.f && p <= 0.f) s.cut_p = ordered_key(s.mx);  // the top value only
    if (s.wants_p && p_done != 0) {
        Decided d;
        if (p_done < 0) {
            d = ws->after_p[SP_PASSES - 1];
        } else {
            if (p_done >= 2) d = ws->after_p[p_done - 2];
            else { d.prefix = 0; d.k_rem = 0; d.carried = d.limit = 0; }
            const int pass = p_done - 1;
            if (pass == 2) refine_top_p<sp_bins(2) / SIA_WAVE>(ws->mass[2], sp_shift(2), d, p, false);
            else refine_top_p<sp_bins(0) / SIA_WAVE>(ws->mass[pass], sp_shift(pass), d, p, pass == 0);
            if (lane == 0) ws->after_p[pass] = d;
        }
        s.prefix_p = d.prefix;
        if (p_done < 0 || p_done == SP_PASSES) s.cut_p = d.prefix;
    }
    return s;
}

// Every thread of the workgroup gets the state that wave 0 computed.
__device__ __forceinline__ RowState shared_row_state(SampleRow* __restrict__ ws, float T, int k, float p, int vocab,
                                                     int filters, int k_done, int p_done) {
    __shared__ RowState shared;
    if (threadIdx.x < SIA_WAVE) {
        const RowState s = row_state(ws, T, k, p, vocab, filters, k_done, p_done);
        if (threadIdx.x == 0) shared = s;
    }
    __syncthreads();
    return shared;
}

__device__ __forceinline__ void chunk_range(int chunk, int vocab, int& begin, int& end) {
    const int per = (vocab + SP_CHUNKS - 1) / SP_CHUNKS;
    begin = min(vocab, chunk * per);
    end = min(vocab, begin + per);
}

// The logits at i0, i0 + stride, ... below `end`, asked for together so that their latencies overlap; -inf, which
// has no probability mass and is nobody's maximum, where there is none.
#define SP_AT_ONCE 8
__device__ __forceinline__ void load_together(const float* __restrict__ row, int i0, int stride, int end,
                                              float (&v)[SP_AT_ONCE]) {
#pragma unroll
    for (int u = 0; u < SP_AT_ONCE; ++u) v[u] = i0 + u * stride < end ? row[i0 + u * stride] : -INFINITY;
}

#define SP_CLEAR_BYTES (sizeof(u64) * SP_PASSES * SP_MAX_BINS + sizeof(int) * SP_PASSES * SP_MAX_BINS)
static_assert(offsetof(SampleRow, after_k) == SP_CLEAR_BYTES, "the histograms lead the row and are contiguous");
static_assert(SP_CLEAR_BYTES % (sizeof(uint4) * SP_CHUNKS) == 0 && sizeof(SampleRow) % sizeof(uint4) == 0,
              "cleared in 16-byte pieces, a share by each chunk's workgroup");

// 1. maximum and its (lowest) index of each chunk, on the raw logits.  With `clear` each chunk's workgroup also
// sets its share of the row's histograms to zero: the counting launches come after this one.
// Of many rows by workgroups of four waves: a compute unit then has the loads of eight on their way while others reduce, where it had two of
// 16 waves that did both in step.  us with the pick behind it, 16 waves and 4:  rows of 128,256: 64 14.0 and 10.8, 303 42.7 and 29.1
// (155 MB: 6 TB/s while it reads);  17 8.4 and 8.1, 32 8.9 and 8.4;  rows of 512:  17 6.9 and 5.7, 64 9.7 and 6.1;  300 of 32,000 33 and 12.7.  Up to 16 rows,
// whose chunks (SP_CHUNKS each) are a workgroup a unit, 16 waves, whose threads ask for a chunk's logits at once: one row of 128,256 7.3 and 7.8, 8 7.6 and 8.2.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void sample_max_kernel(const float* __restrict__ logits, int vocab,
                                                                    SampleRow* __restrict__ ws, int clear) {
    constexpr int WAVES = THREADS / SIA_WAVE;
    __shared__ float vals[WAVES];
    __shared__ int idxs[WAVES];
    const int chunk = blockIdx.x, r = blockIdx.y;
    const float* row = logits + (size_t)r * vocab;
    int begin, end;
    chunk_range(chunk, vocab, begin, end);
    float bv = -INFINITY;
    int bi = vocab;
    for (int i0 = begin + threadIdx.x; i0 < end; i0 += SP_AT_ONCE * THREADS) {
        float v[SP_AT_ONCE];
        load_together(row, i0, THREADS, end, v);
#pragma unroll
        for (int u = 0; u < SP_AT_ONCE; ++u)
            if (i0 + u * THREADS < end) take_better(bv, bi, v[u], i0 + u * THREADS);
    }
    if (clear) {
        constexpr int share = (int)(SP_CLEAR_BYTES / sizeof(uint4) / SP_CHUNKS);
        uint4* mine = (uint4*)(ws + r) + chunk * share;
        for (int i = threadIdx.x; i < share; i += THREADS) mine[i] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int off = SIA_WAVE / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, SIA_WAVE);
        const int oi = __shfl_xor(bi, off, SIA_WAVE);
        take_better(bv, bi, ov, oi);
    }
    if (threadIdx.x % SIA_WAVE == 0) { vals[threadIdx.x / SIA_WAVE] = bv; idxs[threadIdx.x / SIA_WAVE] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < WAVES; ++w) take_better(bv, bi, vals[w], idxs[w]);
        ws[r].chunk_max[chunk] = bv;
        ws[r].chunk_arg[chunk] = bi;
    }
}

// A workgroup's histogram in LDS: COPIES of it, each one element longer than its bins so that the same bin of two
// copies lies in different banks.  A thread adds to the copy of its number.
template <typename T, int COPIES>
struct LocalHistogram {
    T bins[COPIES][SP_MAX_BINS + 1];
    __device__ __forceinline__ void clear(int n_bins) {
        for (int c = 0; c < COPIES; ++c)
            for (int b = threadIdx.x; b < n_bins; b += SP_THREADS) bins[c][b] = 0;
    }
    __device__ __forceinline__ void add(int bin, T v) { atomicAdd(&bins[threadIdx.x % COPIES][bin], v); }
    // adds what the workgroup has counted to the row's histogram
    __device__ __forceinline__ void add_to(T* __restrict__ row_bins, int n_bins) {
        for (int b = threadIdx.x; b < n_bins; b += SP_THREADS) {
            T sum = 0;
#pragma unroll
            for (int c = 0; c < COPIES; ++c) sum += bins[c][b];
            if (sum) atomicAdd(&row_bins[b], sum);
        }
    }
};

// 2. one digit of the k-th largest key: counts of the keys that share the digits found so far
__global__ __launch_bounds__(SP_THREADS) void sample_top_k_kernel(const float* __restrict__ logits,
                                                                  const float* __restrict__ temperature,
                                                                  const int* __restrict__ top_k, int vocab,
                                                                  SampleRow* __restrict__ ws, int filters, int pass) {
    __shared__ LocalHistogram<int, SP_COUNT_COPIES> hist;
    const int chunk = blockIdx.x, r = blockIdx.y;
    const float T = temperature[r];
    const int k = top_k[r];
    if (!(T > 0.f && k > 0 && k < vocab)) return;  // the whole workgroup
    const int bins = sp_bins(pass), shift = sp_shift(pass);
    const float* row = logits + (size_t)r * vocab;
    int begin, end;
    chunk_range(chunk, vocab, begin, end);
    int i0 = begin + threadIdx.x;
    float v[SP_AT_ONCE];
    load_together(row, i0, SP_THREADS, end, v);  // on their way while the row's state is made up
    hist.clear(bins);
    const RowState s = shared_row_state(ws + r, T, k, 1.f, vocab, filters, pass, 0);  // with a barrier
    const uint32_t high_mask = pass == 0 ? 0u : ~((1u << (shift + (pass == 1 ? 11 : 10))) - 1u);
    while (i0 < end) {
#pragma unroll
        for (int u = 0; u < SP_AT_ONCE; ++u) {
            const uint32_t key = ordered_key(v[u] / T);
            if (i0 + u * SP_THREADS < end && (key & high_mask) == s.prefix_k) hist.add((key >> shift) & (bins - 1), 1);
        }
        i0 += SP_AT_ONCE * SP_THREADS;
        if (i0 < end) load_together(row, i0, SP_THREADS, end, v);
    }
    __syncthreads();
    hist.add_to(ws[r].count[pass], bins);
}

// 3. one digit of the lowest kept key: mass of the keys (that top-k kept) that share the digits found so far
__global__ __launch_bounds__(SP_THREADS) void sample_top_p_kernel(const float* __restrict__ logits,
                                                                  const float* __restrict__ temperature,
                                                                  const int* __restrict__ top_k,
                                                                  const float* __restrict__ top_p, int vocab,
                                                                  SampleRow* __restrict__ ws, int filters, int pass,
                                                                  float one) {
    __shared__ LocalHistogram<u64, SP_MASS_COPIES> hist;
    const int chunk = blockIdx.x, r = blockIdx.y;
    const float T = temperature[r], p = top_p[r];
    if (!(T > 0.f && p > 0.f && p < 1.f)) return;  // the whole workgroup
    const int bins = sp_bins(pass), shift = sp_shift(pass);
    const float* row = logits + (size_t)r * vocab;
    int begin, end;
    chunk_range(chunk, vocab, begin, end);
    int i0 = begin + threadIdx.x;
    float v[SP_AT_ONCE];
    load_together(row, i0, SP_THREADS, end, v);  // on their way while the row's state is made up
    hist.clear(bins);
    const RowState s = shared_row_state(ws + r, T, top_k[r], p, vocab, filters, (filters & 1) ? SP_PASSES : 0, pass);
    const uint32_t high_mask = pass == 0 ? 0u : ~((1u << (shift + (pass == 1 ? 11 : 10))) - 1u);
    while (i0 < end) {
#pragma unroll
        for (int u = 0; u < SP_AT_ONCE; ++u) {
            const float x = v[u] / T;
            const uint32_t key = ordered_key(x);
            if (key >= s.cut_k && (key & high_mask) == s.prefix_p) {
                const u64 q = fixed_mass(x, s.mx, one);  // none where there is no token
                if (q) hist.add((key >> shift) & (bins - 1), q);
            }
        }
        i0 += SP_AT_ONCE * SP_THREADS;
        if (i0 < end) load_together(row, i0, SP_THREADS, end, v);
    }
    __syncthreads();
    hist.add_to(ws[r].mass[pass], bins);
}

// The tokens of piece `piece` of a row: a chunk is cut into one piece for each wave of its workgroup.
__device__ __forceinline__ void piece_range(int piece, int vocab, int& begin, int& end) {
    int chunk_begin, chunk_end;
    chunk_range(piece / SP_WAVES, vocab, chunk_begin, chunk_end);
    const int per = (chunk_end - chunk_begin + SP_WAVES - 1) / SP_WAVES;
    begin = min(chunk_end, chunk_begin + (piece % SP_WAVES) * per);
    end = min(chunk_end, begin + per);
}

// Mass of the token with logit `v` if it is kept, else 0 (-inf, which stands for "no token", has none).
__device__ __forceinline__ u64 kept_mass(float v, const RowState& s, uint32_t cut, float one) {
    const float x = v / s.T;
    return ordered_key(x) >= cut ? fixed_mass(x, s.mx, one) : 0;
}

// 4a. mass of each piece's kept tokens
__global__ __launch_bounds__(SP_THREADS) void sample_kept_kernel(const float* __restrict__ logits,
                                                                 const float* __restrict__ temperature,
                                                                 const int* __restrict__ top_k,
                                                                 const float* __restrict__ top_p, int vocab,
                                                                 SampleRow* __restrict__ ws, int filters, float one) {
    const int chunk = blockIdx.x, r = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x / SIA_WAVE;
    const float T = temperature[r];
    if (!(T > 0.f)) return;  // the whole workgroup: a greedy row
    const float* row = logits + (size_t)r * vocab;
    const int piece = chunk * SP_WAVES + wave;
    int begin, end;
    piece_range(piece, vocab, begin, end);
    int i0 = begin + lane;
    float v[SP_AT_ONCE];
    load_together(row, i0, SIA_WAVE, end, v);  // on their way while the row's state is made up
    const RowState s = shared_row_state(ws + r, T, top_k[r], top_p[r], vocab, filters, (filters & 1) ? SP_PASSES : 0,
                                        (filters & 2) ? SP_PASSES : 0);
    const uint32_t cut = max(s.cut_k, s.cut_p);
    u64 sum = 0;
    while (i0 < end) {
#pragma unroll
        for (int u = 0; u < SP_AT_ONCE; ++u) sum += kept_mass(v[u], s, cut, one);
        i0 += SP_AT_ONCE * SIA_WAVE;
        if (i0 < end) load_together(row, i0, SIA_WAVE, end, v);
    }
    sum += lanes_above_sum(sum);  // lane 0 holds the piece's
    if (lane == 0) ws[r].piece_mass[piece] = sum;
}

// 4b. the token: argmax for a greedy row; else the first token, in index order, at which the cumulative mass of
// what is kept exceeds u * total: first the piece, then the token in it.  One wave per row.
__global__ __launch_bounds__(SIA_WAVE) void sample_pick_kernel(const float* __restrict__ logits,
                                                               const float* __restrict__ temperature,
                                                               const int* __restrict__ top_k,
                                                               const float* __restrict__ top_p,
                                                               const float* __restrict__ uniform,
                                                               int* __restrict__ out, int vocab,
                                                               SampleRow* __restrict__ ws, int filters, float one) {
    const int r = blockIdx.x, lane = threadIdx.x;
    const float T = temperature ? temperature[r] : 0.f;
    int pick = -1;
    if (T > 0.f) {
        const RowState s = row_state(ws + r, T, top_k[r], top_p[r], vocab, filters, -1, -1);
        const uint32_t cut = max(s.cut_k, s.cut_p);
        constexpr int each = SP_PIECES / SIA_WAVE;  // lane l looks at pieces each * l onwards
        u64 mine = 0;
#pragma unroll
        for (int j = 0; j < each; ++j) mine += ws[r].piece_mass[lane * each + j];
        u64 up_to = lanes_up_to_sum(mine);
        const u64 total = __shfl(up_to, SIA_WAVE - 1, SIA_WAVE);
        u64 target = (u64)((double)uniform[r] * (double)total);
        if (total > 0 && target >= total) target = total - 1;
        u64 passes = __ballot(up_to > target);
        if (passes) {  // else nothing kept has mass in fixed point
            const int owner = __ffsll((long long)passes) - 1;
            int piece = lane * each;
            u64 before = up_to - mine;
            for (int j = 0; j < each - 1 && before + ws[r].piece_mass[piece] <= target; ++j)
                before += ws[r].piece_mass[piece++];
            piece = __shfl(piece, owner, SIA_WAVE);
            before = __shfl(before, owner, SIA_WAVE);
            const float* row = logits + (size_t)r * vocab;
            int begin, end;
            piece_range(piece, vocab, begin, end);
            for (int i0 = begin; i0 < end && pick < 0; i0 += SP_AT_ONCE * SIA_WAVE) {
                float v[SP_AT_ONCE];
                load_together(row, i0 + lane, SIA_WAVE, end, v);
#pragma unroll
                for (int u = 0; u < SP_AT_ONCE; ++u) {
                    if (pick < 0) {  // the same in every lane
                        up_to = before + lanes_up_to_sum(kept_mass(v[u], s, cut, one));
                        passes = __ballot(up_to > target);
                        if (passes) pick = i0 + u * SIA_WAVE + __ffsll((long long)passes) - 1;
                        before = __shfl(up_to, SIA_WAVE - 1, SIA_WAVE);
                    }
                }
            }
        }
    }
    if (lane == 0) {
        if (pick < 0) {  // a greedy row, or nothing but the row's maximum itself has mass in fixed point: that one
            float bv = -INFINITY;
            int bi = vocab;
            for (int c = 0; c < SP_CHUNKS; ++c) take_better(bv, bi, ws[r].chunk_max[c], ws[r].chunk_arg[c]);
            pick = bi < vocab ? bi : 0;
        }
        out[r] = pick;
    }
}

// ---- few tokens kept by top-k ---------------------------------------------------------------------------------
#define SP_MAX_K 256          // the largest k of this way
#define SP_PLACES 512         // for a chunk's candidates
#define SP_FEW 512            // tokens kept by top-k that one wave takes alone
#define SP_CHUNK_TOKENS (SP_AT_ONCE * SP_THREADS)      // that a workgroup holds in registers

// The candidates of a row, in place of its histograms.
struct Candidates {
    float logit[SP_CHUNKS][SP_PLACES];
    int index[SP_CHUNKS][SP_PLACES];
    int number[SP_CHUNKS];      // of a chunk's candidates; more than SP_PLACES: they are not there
};
static_assert(sizeof(Candidates) <= SP_CLEAR_BYTES, "in the histograms' place");

// How many of the workgroup's threads a wave's `mine` counts together: the waves' counts meet in one of two rows of LDS in
// turn, so that one barrier a call is enough.
__device__ __forceinline__ int counted_together(int mine, int (&counts)[2][SP_WAVES], int turn) {
    if (threadIdx.x % SIA_WAVE == 0) counts[turn & 1][threadIdx.x / SIA_WAVE] = mine;
    __syncthreads();
    int sum = 0;
#pragma unroll
    for (int w = 0; w < SP_WAVES; ++w) sum += counts[turn & 1][w];
    return sum;
}

// The q-th largest of the lanes' keys (0 if a wave has not that many above 0); no barrier.
__device__ __forceinline__ uint32_t largest_of_lanes(uint32_t key, int q) {
    uint32_t found = 0;
#pragma unroll 1
    for (int bit = 31; bit >= 0; --bit) {
        const uint32_t t = found | (1u << bit);
        if (__popcll(__ballot(key >= t)) >= q) found = t;
    }
    return found;
}

// 1. maximum of each chunk, and its candidates
__global__ __launch_bounds__(SP_THREADS, 8) void sample_candidates_kernel(const float* __restrict__ logits,
                                                                          const float* __restrict__ temperature,
                                                                          const int* __restrict__ top_k, int vocab,
                                                                          SampleRow* __restrict__ ws) {
    __shared__ float vals[SP_WAVES];
    __shared__ int idxs[SP_WAVES];
    __shared__ int found[SP_AT_ONCE * SP_WAVES];
    __shared__ int counts[2][SP_WAVES];
    __shared__ int total;
    const int chunk = blockIdx.x, r = blockIdx.y, lane = threadIdx.x % SIA_WAVE, wave = threadIdx.x / SIA_WAVE;
    const float* row = logits + (size_t)r * vocab;
    const float T = temperature[r];
    const int k = top_k[r];
    int begin, end;
    chunk_range(chunk, vocab, begin, end);
    const int i0 = begin + threadIdx.x;
    float v[SP_AT_ONCE];
    load_together(row, i0, SP_THREADS, end, v);
    float bv = -INFINITY;
    int bi = vocab;
#pragma unroll
    for (int u = 0; u < SP_AT_ONCE; ++u)
        if (i0 + u * SP_THREADS < end) take_better(bv, bi, v[u], i0 + u * SP_THREADS);
#pragma unroll
    for (int off = SIA_WAVE / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, SIA_WAVE);
        const int oi = __shfl_xor(bi, off, SIA_WAVE);
        take_better(bv, bi, ov, oi);
    }
    if (lane == 0) { vals[wave] = bv; idxs[wave] = bi; }
    __syncthreads();
    bv = vals[0];
    bi = idxs[0];
    for (int w = 1; w < SP_WAVES; ++w) take_better(bv, bi, vals[w], idxs[w]);
    if (threadIdx.x == 0) {
        ws[r].chunk_max[chunk] = bv;
        ws[r].chunk_arg[chunk] = bi;
    }
    if (!(T > 0.f)) return;  // the whole workgroup: a greedy row

    uint32_t key[SP_AT_ONCE], top = 0;
#pragma unroll
    for (int u = 0; u < SP_AT_ONCE; ++u) {
        key[u] = i0 + u * SP_THREADS < end ? ordered_key(v[u]) : 0;
        top = max(top, key[u]);
    }
    // A bound that at least k tokens are not below: each wave's share of k of its lanes' largest keys, and of those the waves'
    // smallest.  Hardly more tokens than that are not below it either.  Where the tokens are laid out so that too many are,
    // the k-th largest of the threads' largest keys, bit by bit, which takes a barrier a bit.  (Logits as they are: to divide
    // all of them by T costs more than the rest, and keeps their order but for values that become equal; a little
    // room below the bound takes those in.  A very large T could make many equal: then nothing is left out here.)
    uint32_t cut = 0;
    if (end - begin > SP_PLACES && T < 1e6f) {
        const uint32_t bound = largest_of_lanes(top, (k + SP_WAVES - 1) / SP_WAVES);
        if (lane == 0) found[wave] = (int)bound;
        __syncthreads();
        cut = (uint32_t)found[0];
        for (int w = 1; w < SP_WAVES; ++w) cut = min(cut, (uint32_t)found[w]);
        int mine = 0, turn = 0;
#pragma unroll
        for (int u = 0; u < SP_AT_ONCE; ++u) mine += __popcll(__ballot(key[u] >= cut));
        if (counted_together(mine, counts, turn++) > SP_PLACES) {
            cut = 0;
#pragma unroll 1
            for (int bit = 31; bit >= 0; --bit, ++turn) {
                const uint32_t t = cut | (1u << bit);
                if (counted_together(__popcll(__ballot(top >= t)), counts, turn) >= k) cut = t;
            }
        }
    }
    // in index order: the loads of a thread are SP_THREADS apart.  A token without mass below the chunk's own maximum (more
    // than 32 T below it; 45 to be safe) has none below the row's: it is never drawn, and whether it counts among the k
    // changes nothing for those that are (only for tokens below it, which have no mass either).  A value that is no number
    // is not below anything: it counts, as it does above.
    const float least = cut ? key_value(cut) : -INFINITY;
    const float low = fmaxf(least - fabsf(least) * 2e-6f, bv - 45.f * T);
    uint32_t mine = 0;
#pragma unroll
    for (int u = 0; u < SP_AT_ONCE; ++u) {
        const bool is = i0 + u * SP_THREADS < end && !(v[u] < low);
        if (is) mine |= 1u << u;
        const u64 all = __ballot(is);
        if (lane == 0) found[u * SP_WAVES + wave] = __popcll(all);
    }
    __syncthreads();
    if (wave == 0) {      // how many come before each wave's
        constexpr int each = SP_AT_ONCE * SP_WAVES / SIA_WAVE;
        int n[each], sum = 0;
#pragma unroll
        for (int i = 0; i < each; ++i) {
            n[i] = found[lane * each + i];
            sum += n[i];
        }
        int before = (int)lanes_up_to_sum((u64)sum) - sum;
        if (lane == SIA_WAVE - 1) total = before + sum;
#pragma unroll
        for (int i = 0; i < each; ++i) {
            found[lane * each + i] = before;
            before += n[i];
        }
    }
    __syncthreads();
    Candidates* list = (Candidates*)(ws + r);
    const int number = total;
    if (threadIdx.x == 0) list->number[chunk] = number;
    if (number > SP_PLACES) return;      // the whole workgroup
#pragma unroll
    for (int u = 0; u < SP_AT_ONCE; ++u) {
        const u64 all = __ballot((mine >> u) & 1);
        if ((mine >> u) & 1) {
            const int at = found[u * SP_WAVES + wave] + __popcll(all & ((1ull << lane) - 1ull));
            list->logit[chunk][at] = v[u];
            list->index[chunk][at] = i0 + u * SP_THREADS;
        }
    }
}

// 2. the token of a row from its candidates: wave w has those of chunk w.
__global__ __launch_bounds__(SP_THREADS) void sample_few_kernel(const float* __restrict__ logits, const float* __restrict__ temperature,
                                                                const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                                const float* __restrict__ uniform, int* __restrict__ out, int vocab,
                                                                SampleRow* __restrict__ ws, int filters, float one) {
    constexpr int PER_LANE = SP_PLACES / SIA_WAVE;
    __shared__ __align__(16) LocalHistogram<u64, 1> hist;
    __shared__ float value[SP_CHUNKS][SP_PLACES];
    __shared__ u64 few_mass[SP_THREADS];
    __shared__ uint32_t few_key[SP_THREADS];
    __shared__ int few_index[SP_THREADS];
    __shared__ int counts[2][SP_WAVES];
    __shared__ int n_few;
    __shared__ Decided decided;
    __shared__ u64 wave_mass[SP_WAVES];
    static_assert(SP_WAVES == SP_CHUNKS, "a wave a chunk");
    const int r = blockIdx.x, lane = threadIdx.x % SIA_WAVE, wave = threadIdx.x / SIA_WAVE;
    const float T = temperature[r], p = top_p[r], u_row = uniform[r];
    const int k = top_k[r];
    SampleRow* mine = ws + r;
    const Candidates* list = (const Candidates*)mine;
    // everything is asked for at once, the places that hold no candidate too: each round trip to memory is 1.5 us
    float listed_logit[PER_LANE];
    int listed_index[PER_LANE];
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        listed_logit[j] = list->logit[wave][j * SIA_WAVE + lane];
        listed_index[j] = list->index[wave][j * SIA_WAVE + lane];
    }
    const int my_chunk = lane % SP_CHUNKS;
    float bv = mine->chunk_max[my_chunk];
    int bi = mine->chunk_arg[my_chunk], number = list->number[my_chunk];
#pragma unroll
    for (int off = SP_CHUNKS / 2; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, SIA_WAVE);
        const int oi = __shfl_xor(bi, off, SIA_WAVE);
        take_better(bv, bi, ov, oi);
    }
    if (!(T > 0.f)) {  // the whole workgroup: a greedy row
        if (threadIdx.x == 0) out[r] = bi < vocab ? bi : 0;
        return;
    }
    const bool listed = __ballot(number > SP_PLACES) == 0;
    const int here = __shfl(number, wave, SIA_WAVE);
    int candidates = number;
#pragma unroll
    for (int off = SP_CHUNKS / 2; off > 0; off >>= 1) candidates += __shfl_xor(candidates, off, SIA_WAVE);
    const float* row = logits + (size_t)r * vocab;
    int begin, end;
    chunk_range(wave, vocab, begin, end);
    const int n = listed ? here : end - begin;      // tokens of this wave
    if (listed) {
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j) value[wave][j * SIA_WAVE + lane] = listed_logit[j];
    } else {
        candidates = vocab;
    }
    auto logit = [&](int i) { return i >= n ? -INFINITY : listed ? value[wave][i] : row[begin + i]; };

    const float mx = bv / T;
    uint32_t cut = 0;
    const bool wants_k = (filters & 1) && k > 0 && k < vocab && k <= candidates;
    if (listed) {
        uint32_t key[PER_LANE], top = 0;
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j) {
            key[j] = j * SIA_WAVE + lane < n ? ordered_key(listed_logit[j] / T) : 0;
            top = max(top, key[j]);
        }
        // a bound below the k-th largest, as in the launch before, if the candidates would not fit otherwise
        if (wants_k && candidates > SP_THREADS) {
            const uint32_t bound = largest_of_lanes(top, (k + SP_WAVES - 1) / SP_WAVES);
            if (lane == 0) few_index[wave] = (int)bound;
            __syncthreads();
            cut = (uint32_t)few_index[0];
            for (int w = 1; w < SP_WAVES; ++w) cut = min(cut, (uint32_t)few_index[w]);
        }
        int mine = 0, at = 0;
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j)
            if (j * SIA_WAVE < n) mine += __popcll(__ballot(j * SIA_WAVE + lane < n && key[j] >= cut));
        int kept = counted_together(mine, counts, 0);
        if (kept <= SP_THREADS) {      // they meet in LDS, in index order
            for (int w = 0; w < wave; ++w) at += counts[0][w];
#pragma unroll
            for (int j = 0; j < PER_LANE; ++j) {
                const bool is = j * SIA_WAVE + lane < n && key[j] >= cut;
                const u64 all = __ballot(is);
                if (is) {
                    const int to = at + __popcll(all & ((1ull << lane) - 1ull));
                    few_key[to] = key[j];
                    few_mass[to] = fixed_mass(listed_logit[j] / T, mx, one);
                    few_index[to] = listed_index[j];
                }
                at += __popcll(all);
            }
            __syncthreads();
            if (wave == 0) {      // a wave alone needs no barriers: the k-th largest, bit by bit, and what is not below it
                const int groups = (kept + SIA_WAVE - 1) / SIA_WAVE;
                cut = 0;
                if (wants_k) {
                    // from the first bit in which the keys differ on, until the keys that are not below are k, or the last bit
                    uint32_t high = 0, low = 0xffffffffu, own[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int e = j * SIA_WAVE + lane;
                        own[j] = e < kept ? few_key[e] : 0;
                        if (e < kept) { high = max(high, own[j]); low = min(low, own[j]); }
                    }
                    for (int e = 4 * SIA_WAVE + lane; e < kept; e += SIA_WAVE) {
                        high = max(high, few_key[e]);
                        low = min(low, few_key[e]);
                    }
#pragma unroll
                    for (int off = SIA_WAVE / 2; off > 0; off >>= 1) {
                        high = max(high, (uint32_t)__shfl_xor((int)high, off, SIA_WAVE));
                        low = min(low, (uint32_t)__shfl_xor((int)low, off, SIA_WAVE));
                    }
                    const int same = high == low ? 32 : __clz((int)(high ^ low));
                    cut = same == 32 ? high : same == 0 ? 0 : high & ~(0xffffffffu >> same);
#pragma unroll 1
                    for (int bit = 31 - same; bit >= 0; --bit) {
                        const uint32_t t = cut | (1u << bit);
                        int not_below = 0;
#pragma unroll
                        for (int j = 0; j < 4; ++j) not_below += __popcll(__ballot(own[j] >= t));
                        for (int j = 4; j < groups; ++j) {
                            const int e = j * SIA_WAVE + lane;
                            not_below += __popcll(__ballot(e < kept && few_key[e] >= t));
                        }
                        if (not_below >= k) cut = t;
                        if (not_below == k) break;
                    }
                }
                if (p <= 0.f) cut = max(cut, ordered_key(mx));  // the top value only
                int to = 0;
#pragma unroll 1
                for (int j = 0; j < groups; ++j) {
                    const int e = j * SIA_WAVE + lane;
                    const bool is = e < kept && few_key[e] >= cut;
                    const u64 all = __ballot(is);
                    if (is) {      // to places that this wave has read already
                        const uint32_t moved_key = few_key[e];
                        const u64 moved_mass = few_mass[e];
                        const int moved_index = few_index[e], place = to + __popcll(all & ((1ull << lane) - 1ull));
                        __builtin_amdgcn_wave_barrier();
                        few_key[place] = moved_key;
                        few_mass[place] = moved_mass;
                        few_index[place] = moved_index;
                    }
                    to += __popcll(all);
                }
                if (lane == 0) n_few = to;
            }
            __syncthreads();
            kept = n_few;
            if (kept <= SP_FEW) {
                if (wave > 0) return;      // what follows is one wave's, without barriers
                uint32_t lowest = 0;
                if ((filters & 2) && p > 0.f && p < 1.f) {
                    u64 all = 0;
                    for (int e = lane; e < kept; e += SIA_WAVE) all += few_mass[e];
                    all = __shfl(lanes_up_to_sum(all), SIA_WAVE - 1, SIA_WAVE);
                    const u64 limit = (u64)((double)p * (double)all);
                    // the smallest key that top-p keeps: what is above it does not exceed the limit
                    lowest = 0xffffffffu;
                    for (int i0 = 0; i0 < kept; i0 += SIA_WAVE) {
                        const int e = i0 + lane;
                        const uint32_t own = e < kept ? few_key[e] : 0;
                        u64 above = 0;
#pragma unroll 4
                        for (int j = 0; j < kept; ++j) above += few_key[j] > own ? few_mass[j] : 0;
                        if (e < kept && few_mass[e] > 0 && above <= limit) lowest = min(lowest, own);
                    }
#pragma unroll
                    for (int off = SIA_WAVE / 2; off > 0; off >>= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, off, SIA_WAVE));
                }
                auto drawn = [&](int e) { return e < kept && few_key[e] >= lowest ? few_mass[e] : 0; };
                u64 total = 0, before = 0;
                for (int e = lane; e < kept; e += SIA_WAVE) total += drawn(e);
                total = __shfl(lanes_up_to_sum(total), SIA_WAVE - 1, SIA_WAVE);
                u64 target = (u64)((double)u_row * (double)total);
                if (total > 0 && target >= total) target = total - 1;
                int pick = bi < vocab ? bi : 0;      // nothing has mass in fixed point but, perhaps, the maximum itself: that one
                for (int i0 = 0; total > 0 && i0 < kept; i0 += SIA_WAVE) {
                    const u64 up_to = before + lanes_up_to_sum(drawn(i0 + lane));
                    const u64 passes = __ballot(up_to > target);
                    if (passes) {
                        pick = few_index[i0 + __ffsll((long long)passes) - 1];
                        break;
                    }
                    before = __shfl(up_to, SIA_WAVE - 1, SIA_WAVE);
                }
                if (lane == 0) out[r] = pick;
                return;
            }
        }
        cut = 0;      // many equal values: the long way, from the list
    }
    if (wants_k) {
        int* count = (int*)hist.bins[0];
        Decided d;
        d.prefix = 0;
        d.k_rem = k;
        d.carried = d.limit = 0;
        for (int pass = 0; pass < SP_PASSES; ++pass) {
            const int bins = sp_bins(pass), shift = sp_shift(pass);
            const uint32_t high_mask = pass == 0 ? 0u : ~((1u << (shift + (pass == 1 ? 11 : 10))) - 1u);
            for (int b = threadIdx.x; b < bins; b += SP_THREADS) count[b] = 0;
            __syncthreads();
            for (int i = lane; i < n; i += SIA_WAVE) {
                const uint32_t key = ordered_key(logit(i) / T);
                if ((key & high_mask) == cut) atomicAdd(&count[(key >> shift) & (bins - 1)], 1);
            }
            __syncthreads();
            if (wave == 0) {
                if (pass == 2) refine_top_k<sp_bins(2) / SIA_WAVE>(count, shift, d);
                else refine_top_k<sp_bins(0) / SIA_WAVE>(count, shift, d);
                if (lane == 0) decided = d;
            }
            __syncthreads();
            cut = decided.prefix;
        }
    }
    if (p <= 0.f) {
        cut = max(cut, ordered_key(mx));  // the top value only
    } else if ((filters & 2) && p < 1.f) {
        const uint32_t cut_k = cut;
        uint32_t prefix = 0;
        Decided d;
        d.prefix = 0;
        d.k_rem = 0;
        d.carried = d.limit = 0;
        for (int pass = 0; pass < SP_PASSES; ++pass) {
            const int bins = sp_bins(pass), shift = sp_shift(pass);
            const uint32_t high_mask = pass == 0 ? 0u : ~((1u << (shift + (pass == 1 ? 11 : 10))) - 1u);
            __syncthreads();
            for (int b = threadIdx.x; b < bins; b += SP_THREADS) hist.bins[0][b] = 0;
            __syncthreads();
            for (int i = lane; i < n; i += SIA_WAVE) {
                const float x = logit(i) / T;
                const uint32_t key = ordered_key(x);
                if (key >= cut_k && (key & high_mask) == prefix) {
                    const u64 q = fixed_mass(x, mx, one);
                    if (q) atomicAdd(&hist.bins[0][(key >> shift) & (bins - 1)], q);
                }
            }
            __syncthreads();
            if (wave == 0) {
                if (pass == 2) refine_top_p<sp_bins(2) / SIA_WAVE>(hist.bins[0], shift, d, p, false);
                else refine_top_p<sp_bins(0) / SIA_WAVE>(hist.bins[0], shift, d, p, pass == 0);
                if (lane == 0) decided = d;
            }
            __syncthreads();
            prefix = decided.prefix;
        }
        cut = max(cut, prefix);
    }
    // the first token, in index order, at which the cumulative mass of what is kept exceeds u * total
    auto kept = [&](int i) {
        const float x = logit(i) / T;
        return ordered_key(x) >= cut ? fixed_mass(x, mx, one) : 0;
    };
    u64 sum = 0;
    for (int i = lane; i < n; i += SIA_WAVE) sum += kept(i);
    sum += lanes_above_sum(sum);
    if (lane == 0) wave_mass[wave] = sum;
    __syncthreads();
    u64 total = 0, before = 0;
    for (int w = 0; w < SP_WAVES; ++w) {
        if (w == wave) before = total;
        total += wave_mass[w];
    }
    if (total == 0) {  // nothing has mass in fixed point but, perhaps, the maximum itself: that one
        if (threadIdx.x == 0) out[r] = bi < vocab ? bi : 0;
        return;
    }
    u64 target = (u64)((double)u_row * (double)total);
    if (target >= total) target = total - 1;
    if (target < before || target >= before + wave_mass[wave]) return;  // another wave's
    for (int i0 = 0; i0 < n; i0 += SIA_WAVE) {
        const u64 up_to = before + lanes_up_to_sum(kept(i0 + lane));
        const u64 passes = __ballot(up_to > target);
        if (passes) {
            const int i = i0 + __ffsll((long long)passes) - 1;
            if (lane == 0) out[r] = listed ? list->index[wave][i] : begin + i;
            return;
        }
        before = __shfl(up_to, SIA_WAVE - 1, SIA_WAVE);
    }
}

SIA_EXPORT int sia_sample_few_max_k(void) { return SP_MAX_K; }

SIA_EXPORT long long sia_sample_workspace_bytes(int rows) { return (long long)rows * (long long)sizeof(SampleRow); }

// The launches of one call.
static int launch_sampling(const float* logits, const float* temperature, const int* top_k, const float* top_p,
                           const float* uniform, int* out, SampleRow* ws, int rows, int vocab, int filters,
                           hipStream_t stream) {
    const dim3 grid(SP_CHUNKS, rows), block(SP_THREADS);
    int bits = 62;  // fixed point: vocab * 2^bits < 2^63
    while (bits > 0 && ((long long)vocab << bits) >> bits != (long long)vocab) --bits;
    while (bits > 0 && (double)vocab * (double)(1ull << bits) >= 9.2e18) --bits;
    const float one = (float)(1ull << bits);
    if ((filters & 8) && (filters & 1) && vocab <= SP_CHUNKS * SP_CHUNK_TOKENS) {
        hipLaunchKernelGGL(sample_candidates_kernel, grid, block, 0, stream, logits, temperature, top_k, vocab, ws);
        hipLaunchKernelGGL(sample_few_kernel, dim3(rows), block, 0, stream, logits, temperature, top_k, top_p, uniform, out, vocab,
                           ws, filters, one);
        return SIA_LAUNCH_CHECK();
    }
    filters &= 7;
    const int max_threads = rows <= 16 ? SP_THREADS : 256;
    hipLaunchKernelGGL(rows <= 16 ? sample_max_kernel<SP_THREADS> : sample_max_kernel<256>, grid, dim3(max_threads), 0, stream, logits, vocab, ws,
                       (filters & 3) != 0);
    if (filters & 1)
        for (int pass = 0; pass < SP_PASSES; ++pass)
            hipLaunchKernelGGL(sample_top_k_kernel, grid, block, 0, stream, logits, temperature, top_k, vocab, ws,
                               filters, pass);
    if (filters & 2)
        for (int pass = 0; pass < SP_PASSES; ++pass)
            hipLaunchKernelGGL(sample_top_p_kernel, grid, block, 0, stream, logits, temperature, top_k, top_p, vocab,
                               ws, filters, pass, one);
    if (filters)
        hipLaunchKernelGGL(sample_kept_kernel, grid, block, 0, stream, logits, temperature, top_k, top_p, vocab, ws,
                           filters, one);
    hipLaunchKernelGGL(sample_pick_kernel, dim3(rows), dim3(SIA_WAVE), 0, stream, logits,
                       filters ? temperature : nullptr, top_k, top_p, uniform, out, vocab, ws, filters, one);
    return SIA_LAUNCH_CHECK();
}

// One token per row.  workspace: sia_sample_workspace_bytes(rows) bytes, aligned to 16, which may hold anything
// (what has to start at zero is set to zero by the first launch); calls that share a workspace must not overlap.
// filters: bit 0 set if some row may have a top-k filter, bit 1 if some row may have a top-p filter in (0, 1),
// bit 2 if some row has a temperature above 0, bit 3 only if every row with a temperature above 0 has a top_k of 1 to
// sia_sample_few_max_k(); launches for filters that no row has are skipped, and a filter
// whose bit is not set is not applied (rows decide for themselves inside the launches that run).  With
// filters == 0 the parameter pointers may be null: every row takes its argmax.
SIA_EXPORT int sia_sample(const float* logits, const float* temperature, const int* top_k, const float* top_p,
                          const float* uniform, int* out, void* workspace, int rows, int vocab, int filters,
                          hipStream_t stream) {
    if (rows <= 0) return 0;
    if (vocab <= 0 || rows > 65535 || !workspace || ((uintptr_t)workspace & 15)) return SIA_BAD_ARGUMENT;
    if (filters && (!temperature || !top_k || !top_p || !uniform)) return SIA_BAD_ARGUMENT;
    return launch_sampling(logits, temperature, top_k, top_p, uniform, out, (SampleRow*)workspace, rows, vocab, filters,
                           stream);
}

// ---- the same, for callers that cannot allocate -------------------------------------------------------------
// The workspace is a fixed array in device memory that belongs to this library: SIA_SAMPLE_STATIC_MAX_ROWS rows
// (about 4.5 MiB on every GPU the library is used on, until the process ends).  Host code never passes the
// array's name to a kernel: the name is a host-side stand-in, and each GPU holds a copy of its own, so the device
// address is asked for once per device, with that device current, and kept.
static __device__ __align__(256) unsigned char scratch[SIA_SAMPLE_STATIC_MAX_ROWS * sizeof(SampleRow)];

#define SIA_MAX_DEVICES 64
static void* scratch_on_device[SIA_MAX_DEVICES];
static std::mutex scratch_guard;

// Device address of `scratch` on the current device.
static int scratch_address(SampleRow** out) {
    int device = -1;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return (int)err;
    if (device < 0 || device >= SIA_MAX_DEVICES) return SIA_BAD_ARGUMENT;
    std::lock_guard<std::mutex> hold(scratch_guard);
    if (!scratch_on_device[device]) {
        void* ptr = nullptr;
        err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess) return (int)err;
        if (!ptr) return SIA_BAD_ARGUMENT;
        scratch_on_device[device] = ptr;
    }
    *out = (SampleRow*)scratch_on_device[device];
    return 0;
}

SIA_EXPORT int sia_sample_static_max_rows(void) { return SIA_SAMPLE_STATIC_MAX_ROWS; }

SIA_EXPORT int sia_sample_static_init(void) {
    SampleRow* ws = nullptr;
    return scratch_address(&ws);
}

SIA_EXPORT int sia_sample_static(const float* logits, const float* temperature, const int* top_k, const float* top_p,
                                 const float* uniform, int* out, int rows, int vocab, int filters,
                                 hipStream_t stream) {
    if (rows <= 0) return 0;
    if (vocab <= 0 || rows > SIA_SAMPLE_STATIC_MAX_ROWS) return SIA_BAD_ARGUMENT;
    if (filters && (!temperature || !top_k || !top_p || !uniform)) return SIA_BAD_ARGUMENT;
    SampleRow* ws = nullptr;
    const int err = scratch_address(&ws);
    if (err) return err;
    // the last call's histograms are still there: the first launch sets them to zero (with a kernel's stores, not
    // a memset, which a caller that records a graph could not rely on)
    return launch_sampling(logits, temperature, top_k, top_p, uniform, out, ws, rows, vocab, filters, stream);
}
