// One pre-norm block (attention with rotation over the paged cache, SwiGLU feed-forward, RMS norms) of a step of
// many rows, as one call: the launches that the parts' own calls would make one by one, in the same order, on the
// same buffers.  Where this package's products take a step's, the rotation with the cache write and the activation are their
// epilogues, which round first and give the bits of the kernels that they replace.  Nothing is computed here; it spares
// the host the way through the interpreter between the launches, which in a step of a few hundred tokens of a small model
// takes longer than the GPU needs for them.  The BLAS library's products and the matrix-core attention live in other
// libraries: the caller hands their entry points in.
#include "common.h"

extern "C" {
int sia_add_rmsnorm(float* residual, const void* delta, const float* weight, void* out, const int* rows, int n_out,
                    int hidden, float eps, int dtype, hipStream_t stream);
int sia_swiglu(const void* gu, void* out, int n_tokens, int inter, int dtype, hipStream_t stream);
int sia_rope_kv_write(void* qkv, int row_stride, const float* cos_table, const float* sin_table, const int* positions,
                      const int* seq_of_token, const int* block_table, int table_width, void* k_pages, void* v_pages,
                      int n_tokens, int n_heads, int n_kv, int head_dim, int rotary_dim, int page_size, int dtype,
                      hipStream_t stream);
int sia_add_rmsnorm_slices(float* residual, const float* slices, int splits, const float* weight, void* out, int n, int hidden,
                           float eps, hipStream_t stream);
int sia_gemm_tiles_takes(int M, int N, int K);
int sia_gemm_tiles_takes_swiglu(int M, int inter, int K);
int sia_gemm_tiles_splits(int M, int N, int K);
int sia_gemm_tiles(const void* X, const void* W, void* Y, float* slices, int M, int N, int K, hipStream_t stream);
int sia_gemm_tiles_swiglu(const void* X, const void* W, void* Y, int M, int inter, int K, hipStream_t stream);
int sia_sum_slices(const float* slices, void* Y, int splits, long long n, hipStream_t stream);
int sia_gemm_skinny_takes(int M, int N, int K);
int sia_gemm_skinny_takes_swiglu(int M, int inter, int K);
int sia_gemm_skinny(const void* X, const void* W, void* Y, int M, int N, int K, int out_float, hipStream_t stream);
int sia_gemm_skinny_swiglu(const void* X, const void* W, void* Y, int M, int inter, int K, const float* partials,
                           int n_partials, float eps, hipStream_t stream);
int sia_gemm_skinny_rope(const void* X, const void* W, void* Y, int M, int K, const float* cos_table, const float* sin_table,
                         const int* positions, const int* seq_of_token, const int* block_table, int table_width,
                         void* k_pages, void* v_pages, int n_heads, int n_kv, int head_dim, int page_size,
                         const float* partials, int n_partials, float eps, hipStream_t stream);
}

typedef int (*ProductFn)(const void* X, const void* W, void* Y, int M, int N, int K, int out_float, hipStream_t stream);
typedef int (*DecodeFn)(const void* q, int q_row_stride, const void* k_pages, const void* v_pages,
                        const int* block_table, int table_width, const int* cu_q, const int* kv_len, void* out,
                        float* ws_acc, float* ws_ml, int n_seqs, int n_heads, int n_kv, int page_size, float scale,
                        int window, int max_splits, hipStream_t stream);
typedef int (*PrefillFn)(const void* q, int q_row_stride, const void* k_pages, const void* v_pages,
                         const int* block_table, int table_width, const int* cu_q, const int* kv_len, void* out,
                         int seq_begin, int seq_end, int n_tiles, int n_tiles_split, int n_tiles_long, int q_bound,
                         int kv_bound, int n_heads, int n_kv, int page_size, float scale, int window,
                         hipStream_t stream);

// What a block owns: its weights (bfloat16 matrices [out, in], float gains) and its constants.
struct SiaBlockOwn {
    const float* mixer_norm_gain;
    const void* w_qkv;
    const void* w_o;
    const float* feed_forward_norm_gain;
    const void* w_gate_up;
    const void* w_down;
    const float* cos_table;  // null without rotation
    const float* sin_table;
    float mixer_norm_eps, feed_forward_norm_eps, scale;
    int hidden, n_heads, n_kv, head_dim, rotary_dim, inter, window;
};

// What a step owns, the same for every block of the same geometry: its metadata, the buffers between the launches
// (bfloat16, each used by one block after the other) and how its attention is launched.
struct SiaBlockStep {
    ProductFn product;
    DecodeFn attend_single;   // sequences that bring one token
    PrefillFn attend_runs;    // the others
    float* residual;          // [tokens, hidden]
    void* normed;             // [tokens, hidden]
    void* qkv;                // [tokens, (n_heads + 2 n_kv) head_dim]
    void* attended;           // [tokens, n_heads head_dim]
    void* mixed;              // [tokens, hidden]: the mixer's output
    void* gate_up;            // [tokens, 2 inter]
    void* activated;          // [tokens, inter]
    void* fed;                // [tokens, hidden]: the feed-forward's output, the delta of the next block
    const int* positions;
    const int* seq_of_token;
    const int* cu_q;
    const int* kv_len;
    float* ws_acc;
    float* ws_ml;
    int n_tokens, n_seqs, n_single, max_splits, n_tiles, n_tiles_split, n_tiles_long, q_bound, kv_bound;
    int own_products;         // whether products that this package's kernels take go to them, not all to `product`
    float* slices;            // room for the largest product that they leave in slices (null if none does)
    int fed_splits;           // more than 1: the block's last product stays in that many slices, for the next norm to add
};

#define SIA_STEP(call)             \
    do {                           \
        const int rc_ = (call);    \
        if (rc_ != 0) return rc_;  \
    } while (0)

// Whether this package's products may be asked: a weight that does not begin at a multiple of 16 bytes is the library's.
static bool may_own(const SiaBlockStep* S, const void* W) { return S->own_products && ((uintptr_t)W & 15) == 0; }

// Y = X W^T by whoever takes a product of this size.
static int block_product(const SiaBlockStep* S, const void* X, const void* W, void* Y, int N, int K, hipStream_t stream) {
    const int M = S->n_tokens;
    const bool own = may_own(S, W);
    if (own && sia_gemm_skinny_takes(M, N, K)) return sia_gemm_skinny(X, W, Y, M, N, K, 0, stream);
    if (own && sia_gemm_tiles_takes(M, N, K)) {
        SIA_STEP(sia_gemm_tiles(X, W, Y, S->slices, M, N, K, stream));
        const int splits = sia_gemm_tiles_splits(M, N, K);
        return splits > 1 ? sia_sum_slices(S->slices, Y, splits, (long long)M * N, stream) : 0;
    }
    return S->product(X, W, Y, M, N, K, 0, stream);
}

// residual += delta (where there is one; with delta_splits > 1 it lies in that many slices in S->slices); then the block up to
// its attention, whose results are left in S->attended, or without ``attend`` up to its projected rows, which are left in S->qkv with keys and values in the pages: what a caller that
// goes on with some rows alone needs of all of them.
// block_table [n_seqs, table_width], k_pages, v_pages: the block's cache in this step.  0, or the first launch's error.
SIA_EXPORT int sia_prenorm_mixer(const SiaBlockOwn* B, const SiaBlockStep* S, const void* delta, int delta_splits, const int* block_table,
                                 int table_width, void* k_pages, void* v_pages, int page_size, int attend, hipStream_t stream) {
    if (!B || !S || !S->product || !S->attend_runs || S->n_tokens <= 0 || S->n_tokens > 65535) return SIA_BAD_ARGUMENT;
    const int M = S->n_tokens, H = B->hidden;
    const int qkv_width = (B->n_heads + 2 * B->n_kv) * B->head_dim;
    if (delta_splits > 1)
        SIA_STEP(sia_add_rmsnorm_slices(S->residual, S->slices, delta_splits, B->mixer_norm_gain, S->normed, M, H,
                                        B->mixer_norm_eps, stream));
    else
        SIA_STEP(sia_add_rmsnorm(S->residual, delta, B->mixer_norm_gain, S->normed, nullptr, M, H, B->mixer_norm_eps,
                                 SIA_BF16, stream));
    if (may_own(S, B->w_qkv) && B->rotary_dim == B->head_dim && B->head_dim % 2 == 0 && sia_gemm_skinny_takes(M, qkv_width, H)) {
        SIA_STEP(sia_gemm_skinny_rope(S->normed, B->w_qkv, S->qkv, M, H, B->cos_table, B->sin_table, S->positions,
                                      S->seq_of_token, block_table, table_width, k_pages, v_pages, B->n_heads, B->n_kv,
                                      B->head_dim, page_size, nullptr, 0, 0.f, stream));
    } else {
        SIA_STEP(block_product(S, S->normed, B->w_qkv, S->qkv, qkv_width, H, stream));
        SIA_STEP(sia_rope_kv_write(S->qkv, qkv_width, B->cos_table, B->sin_table, S->positions, S->seq_of_token,
                                   block_table, table_width, k_pages, v_pages, M, B->n_heads, B->n_kv, B->head_dim,
                                   B->rotary_dim, page_size, SIA_BF16, stream));
    }
    if (!attend) return 0;
    if (S->n_single > 0) {
        if (!S->attend_single) return SIA_BAD_ARGUMENT;
        SIA_STEP(S->attend_single(S->qkv, qkv_width, k_pages, v_pages, block_table, table_width, S->cu_q, S->kv_len,
                                  S->attended, S->ws_acc, S->ws_ml, S->n_single, B->n_heads, B->n_kv, page_size,
                                  B->scale, B->window, S->max_splits, stream));
    }
    if (S->n_single < S->n_seqs)
        SIA_STEP(S->attend_runs(S->qkv, qkv_width, k_pages, v_pages, block_table, table_width, S->cu_q, S->kv_len,
                                S->attended, S->n_single, S->n_seqs, S->n_tiles, S->n_tiles_split, S->n_tiles_long,
                                S->q_bound, S->kv_bound, B->n_heads, B->n_kv, page_size, B->scale, B->window, stream));
    return 0;
}

// The whole block.  Leaves its last product in S->fed, not yet added (with S->fed_splits > 1, and a w_down that begins at a multiple
// of 16 bytes, in slices in S->slices).
SIA_EXPORT int sia_prenorm_block(const SiaBlockOwn* B, const SiaBlockStep* S, const void* delta, int delta_splits, const int* block_table,
                                 int table_width, void* k_pages, void* v_pages, int page_size, hipStream_t stream) {
    SIA_STEP(sia_prenorm_mixer(B, S, delta, delta_splits, block_table, table_width, k_pages, v_pages, page_size, 1, stream));
    const int M = S->n_tokens, H = B->hidden, Q = B->n_heads * B->head_dim;
    SIA_STEP(block_product(S, S->attended, B->w_o, S->mixed, H, Q, stream));
    SIA_STEP(sia_add_rmsnorm(S->residual, S->mixed, B->feed_forward_norm_gain, S->normed, nullptr, M, H,
                             B->feed_forward_norm_eps, SIA_BF16, stream));
    if (may_own(S, B->w_gate_up) && sia_gemm_skinny_takes_swiglu(M, B->inter, H)) {
        SIA_STEP(sia_gemm_skinny_swiglu(S->normed, B->w_gate_up, S->activated, M, B->inter, H, nullptr, 0, 0.f, stream));
    } else if (may_own(S, B->w_gate_up) && sia_gemm_tiles_takes_swiglu(M, B->inter, H)) {
        SIA_STEP(sia_gemm_tiles_swiglu(S->normed, B->w_gate_up, S->activated, M, B->inter, H, stream));
    } else {
        SIA_STEP(block_product(S, S->normed, B->w_gate_up, S->gate_up, 2 * B->inter, H, stream));
        SIA_STEP(sia_swiglu(S->gate_up, S->activated, M, B->inter, SIA_BF16, stream));
    }
    if (S->fed_splits > 1 && may_own(S, B->w_down))
        SIA_STEP(sia_gemm_tiles(S->activated, B->w_down, S->fed, S->slices, M, H, B->inter, stream));
    else
        SIA_STEP(block_product(S, S->activated, B->w_down, S->fed, H, B->inter, stream));
    return 0;
}
