// Launchers of the gfx950 token-loop kernels (implemented in kernels.hip).
//
// Every launcher enqueues on the given stream and returns the launch status.
// Shapes are checked by the caller (backend.cpp) before any launch: a kernel
// trusts its sizes, so a wrong size would fault instead of failing.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace plamo {

// Per-call values the kernels read from device memory, so a captured decode
// graph stays valid from one step to the next (the host rewrites this block
// before every launch).
enum { kMaxLayers = 128, kMaxVerify = 16 };
struct StepParams {
    uint32_t token;             // decode token id
    uint32_t tokens;            // prompt / candidate rows of this call
    uint32_t count[kMaxLayers]; // cache rows of each layer before this call
    uint32_t done[kMaxLayers];  // fused attention: finished KV heads (zero at launch)
    uint32_t error;             // fused attention: a wait gave up (zero at launch)
    // Bounded wait of the fused attention's O blocks: the target is the KV
    // heads plus wait_extra, polled at most wait_limit times (0: 2^22).
    // Both are zero outside tests, which raise them from the host so that a
    // wait gives up and the failure path runs with every kernel exiting.
    uint32_t wait_extra, wait_limit;
    // Nonzero tag of this decode step, new for every step of a backend: the
    // fused attention's blocks publish it in their completion flags.
    uint32_t step;
};

// Norm applied in a GEMV prologue: x = rms(src) * (bf16(w) + offset).
// With residual, the prologue first forms src' = src + rms(branch) *
// (bf16(rw) + roffset) and block 0 stores src' to state_out.
struct Prologue {
    const float *src;        // vector to normalize (or raw input when w == nullptr)
    const uint16_t *w;       // norm weights; nullptr: use src as is
    float offset;
    const float *branch;     // residual branch; nullptr: no residual
    const uint16_t *rw;
    float roffset;
    float *state_out;        // written by block 0 when branch != nullptr
    float *norm_out;         // written by block 0 when non-null (normalized x)
    // Block 0 copies *status to *status_out when non-null (the decode head
    // hands the step's error word to a pinned host word this way).
    const uint32_t *status;
    uint32_t *status_out;
};

// Rows [first_row, first_row + rows) of a rotation table: cos | sin of
// frequency times row, the product rounded to FP32 as the reference's
// (src/rope_table.s:5-30), or kept in FP64 with `exact`.
hipError_t launch_rope_table(hipStream_t, const float *freq, float scale, uint32_t half,
                             uint64_t first_row, uint64_t rows, float *table, bool exact = false);
// Row gather widened from BF16: token t reads ids[t], or params->token when
// ids is null. With `publish`, block 0 also copies *params (a pinned host
// block, read over the bus) to *publish for the later kernels of the step.
hipError_t launch_embed(hipStream_t, const uint16_t *embedding, const uint32_t *ids,
                        const StepParams *params, uint32_t tokens, uint32_t hidden, float *out,
                        StepParams *publish = nullptr);
// y[r] = W[r,:] . x (x from the prologue). swiglu_half > 0: rows r and
// r + swiglu_half are gate/up and y[r] = silu(gate) * up for r < swiglu_half.
hipError_t launch_gemv(hipStream_t, const uint16_t *w, uint64_t rows, uint64_t cols,
                       const Prologue &pro, float *y, uint64_t swiglu_half, int blocks_hint);
// Scratch of the split-BF16 GEMM: the three BF16 planes of X, split-K partial
// tiles and per-tile arrival counters (zero-initialized; every launch leaves
// them zero).
struct GemmWorkspace {
    float *partial;
    uint64_t partial_floats;
    uint32_t *counter_base;
    uint32_t counters;
    uint16_t *planes;
    uint64_t plane_elems;
    uint32_t cus;  // compute units (grid sizing)
};
struct GemmSplit {
    const float *x;
    uint64_t ldx;
    const uint16_t *w;
    uint32_t n, k, t, tp, splits;
    float *y;
    uint64_t ldy;
    float *partial;
    uint32_t *counters;
    uint16_t *planes;
    uint32_t xcd_group;  // nonzero: the M tiles of a weight tile share an XCD (see the kernel)
    // Nonzero (the intermediate size I): the rows are a gate/up pair [2I]
    // and each tile takes gate and up rows of the same intermediate columns;
    // the epilogue writes silu(gate) * up as the BF16 planes `act` (rows
    // padded to act_tp) instead of y.
    uint32_t swiglu;
    uint16_t *act;
    uint32_t act_tp;
};
constexpr uint64_t kGemmPartialFloats = 16ull << 20;  // 64 MiB
constexpr uint32_t kGemmCounters = 8192;
// BF16 elements of the planes a GEMM of `tokens` rows and `cols` columns needs.
uint64_t gemm_plane_elems(uint64_t tokens, uint64_t cols);
// C[t, r] = sum_k X[t, k] * W[r, k]. With a workspace, at most 5 tokens and
// K a multiple of 512: FP32 FMAs on the vector ALUs, weights streamed as in
// the decode GEMV. Otherwise, with a workspace, more than one token and K a
// multiple of 64: BF16 matrix cores on the exact three-term split of X; else
// FP32 MFMA with BF16 weights widened in LDS.
// planes_ready: the BF16 planes of X for the matrix-core path are already in
// ws->planes (written by a norm with SplitRows of gemm_planes_rows(tokens, cols,
// ws) rows, or by launch_gemm_swiglu), and x is not read; other paths fail.
hipError_t launch_gemm(hipStream_t, const float *x, uint64_t x_stride, const uint16_t *w,
                       uint64_t rows, uint64_t cols, uint64_t tokens, float *y,
                       uint64_t y_stride, const GemmWorkspace *ws, bool planes_ready = false);
// The padded rows of the BF16 planes launch_gemm's matrix-core path reads for
// `tokens` rows of `cols` columns, or 0 when another path takes the call.
uint32_t gemm_planes_rows(uint64_t tokens, uint64_t cols, const GemmWorkspace *ws);
// Rows of X as those planes: [cols / 32][hi, mid, lo][padded][32], exact.
struct SplitRows {
    uint16_t *planes;
    uint32_t padded;
};

// A projection's weights as scaled fp16 fragments for launch_gemm_pair, and
// each row's exponent (value = fragment * 2^-exps[row]); rows padded to 32,
// `groups` groups of 32 rows per 32-column stage of the layout.
struct PairWeight {
    uint16_t *frag;
    int32_t *exps;
    uint32_t rows, cols, groups;
};
// The rows from `first` (a multiple of 32) on.
PairWeight pair_rows_from(const PairWeight &w, uint32_t first);
// Rows of X as scaled pairs of fp16 terms: [cols / 32][hi, lo][padded][32],
// value = (hi + lo) * 2^-exps[row]. With act_exps (and act_bound,
// launch_pair_balance's) a norm also writes the exponents of the rows' SwiGLU
// activation, whose planes hold value = (hi + lo) * 2^(col_exps[column] -
// exps[row]).
constexpr uint32_t kPairK = 32;
struct PairRows {
    uint16_t *planes;
    int32_t *exps;
    uint32_t padded;
    const float *act_bound;
    int32_t *act_exps;
    const int32_t *col_exps;
};
bool pair_supported(uint64_t rows, uint64_t cols);
uint64_t pair_frag_elems(uint64_t rows, uint64_t cols);
uint64_t pair_exp_count(uint64_t rows);
// Rows of the planes for `tokens` rows (the consumer's tiles are whole).
uint32_t pair_padded(uint64_t tokens);
// FP32 rows (16-byte aligned, at most 8192 wide) into the planes, rows past
// `rows` zero.
hipError_t launch_pair_rows(hipStream_t, const float *x, uint64_t x_stride, uint64_t width,
                            uint64_t rows, const PairRows &pair);
// Fills p.frag and p.exps from p.rows x p.cols BF16 weights (16-byte aligned),
// column c times 2^col_exps[c] (optional); norms (optional): each row's 2-norm.
hipError_t launch_pair_weights(hipStream_t, const uint16_t *w, const PairWeight &p, float *norms,
                               const int32_t *col_exps);
// From the 2-norms of a gate | up projection's rows: the exponents that balance
// the columns of its SwiGLU activation, for the activation's planes and for
// down's fragments, and the bound the norms scale the activation by.
hipError_t launch_pair_balance(hipStream_t, const float *norms, uint64_t intermediate,
                               int32_t *col_exps, float *bound);
// y[t, r] = X W^T on the fp16 matrix cores, FP32 sums.
hipError_t launch_gemm_pair(hipStream_t, const PairRows &x, const PairWeight &w, uint64_t tokens,
                            float *y, uint64_t y_stride, const GemmWorkspace &ws);
// silu(gate) * up of a gate | up projection into act.planes, scaled by
// act.exps (written by the norm that formed x) and act.col_exps; w.rows / 2 a
// multiple of 32.
hipError_t launch_gemm_pair_swiglu(hipStream_t, const PairRows &x, const PairWeight &w,
                                   uint64_t tokens, const PairRows &act, const GemmWorkspace &ws);
// Multi-row RMSNorm; with branch: state += rms(branch) * (bf16(w) + offset).
// With pair, the normalized rows go there instead of y, `pair->padded` rows
// (those past `rows` zero; 16-byte-aligned rows of whole 32-column stages, at
// most 8192 wide, hipErrorInvalidValue otherwise); with split likewise, for rows
// of whole 64-column steps.
hipError_t launch_norm_rows(hipStream_t, const float *x, uint64_t x_stride, const uint16_t *w,
                            float offset, float *y, uint64_t y_stride, uint64_t width,
                            uint64_t rows, const PairRows *pair = nullptr,
                            const SplitRows *split = nullptr);
// launch_residual_rows followed by launch_norm_rows of the updated rows into
// norm, in one launch (width <= 8192; hipErrorInvalidValue otherwise), pair and
// split as launch_norm_rows.
hipError_t launch_residual_norm_rows(hipStream_t, float *state, const float *branch,
                                     const uint16_t *wr, float off_r, const uint16_t *wn,
                                     float off_n, float *norm, uint64_t norm_stride,
                                     uint64_t width, uint64_t rows,
                                     const PairRows *pair = nullptr,
                                     const SplitRows *split = nullptr);
hipError_t launch_residual_rows(hipStream_t, float *state, const float *branch,
                                const uint16_t *w, float offset, uint64_t width, uint64_t rows);
hipError_t launch_swiglu_rows(hipStream_t, const float *gate_up, float *out,
                              uint64_t intermediate, uint64_t rows);
// act[t, i] = silu(g) * u of the gate/up projection (rows i and
// intermediate + i of w): the token GEMV writes act directly; other shapes
// go through launch_gemm into gate_up ([tokens][2 * intermediate]) and
// launch_swiglu_rows. With act_planes (gemm_swiglu_planes' place, not null) the
// GEMM's epilogue writes the activation there alone, as the planes of a
// launch_gemm with planes_ready.
hipError_t launch_gemm_swiglu(hipStream_t, const float *x, uint64_t x_stride, const uint16_t *w,
                              uint64_t intermediate, uint64_t cols, uint64_t tokens, float *act,
                              float *gate_up, const GemmWorkspace *ws, bool planes_ready = false,
                              uint16_t *act_planes = nullptr);
// Where in the workspace that is, past the input's planes; null when the shape
// or the workspace (of cols + intermediate columns) does not allow it.
uint16_t *gemm_swiglu_planes(uint64_t intermediate, uint64_t cols, uint64_t tokens,
                             const GemmWorkspace *ws);

// Q/K head RMSNorm + RoPE + cache append for `tokens` rows of one layer.
struct QkvPost {
    float *qkv;              // [tokens, (qh+2kh)*dim] projection output (read)
    float *q_out;            // [tokens, qh*dim] normalized, rotated Q
    const uint16_t *qn, *kn;
    const float *table;      // RoPE rows [position][dim]: cos | sin
    const StepParams *params;
    uint32_t layer, qh, kh, dim, tokens, capacity;
    // K/V destination rows: row t goes to dst_*[(row0 + t) * width], where
    // row0 = params->count[layer] when rows_from_count, else 0.
    float *k_raw, *v, *k_rot;
    int rows_from_count;
    int rotate_k;            // 0: leave k_rot alone (sliding overflow)
    float *stage;            // optional [3][width] copy of the last row (decode mirror)
    int last_query;          // nonzero: only the last row's query heads
    uint32_t head0, token0;  // first head and row of a launch (set by the launcher)
    // Optional: Q is rotated at its virtual row (count + t, past the window's
    // capacity too) by this table instead, and the keys, rotated likewise, go
    // to k_virtual[(count + t) * width].
    const float *virtual_table;
    float *k_virtual;
};
hipError_t launch_qkv_post(hipStream_t, const QkvPost &);

// Decode attention for one token, fused with the decode form of QkvPost: each
// block normalizes and rotates the query heads of its KV head, the block that
// owns row `count` also normalizes/rotates the new key and appends K, V and
// rotated K (plus the mirror stage), and every block runs an online softmax
// over its share of rows [0, count]; the last block of a KV head merges the
// partials. Requires decode_attention_supported(dim, qh / kh), splits <= 8 and
// count < capacity (a full sliding window's rows have moved on by one). Up to 256
// rows run in one block per KV head; longer contexts use up to `splits` blocks.
struct DecodeAttention {
    const float *qkv;        // [(qh+2kh)*dim] projection output
    const uint16_t *qn, *kn;
    const float *freq;       // RoPE frequencies [dim / 2] of the layer's table
    float rope_scale;        // and its concentration (rope_cos_sin)
    float *k_raw, *v, *k_rot;  // cache rows [rows, kh*dim]
    uint32_t rows;           // allocated cache rows (every tile row is clamped below it)
    float *stage;            // optional [3][kh*dim] copy of the appended row
    float *host_k, *host_v, *host_rot;  // optional device views of the host cache rows
    float *out;              // [qh*dim]
    float *partial;          // scratch [kh][splits][qh/kh][dim + 2]
    uint32_t *counters;      // [kh] zero-initialized; reset by the kernel
    const StepParams *params;
    uint32_t layer, qh, kh, dim, splits;
};
hipError_t launch_decode_attention(hipStream_t, const DecodeAttention &);
bool decode_attention_supported(uint32_t dim, uint32_t group);
// Decode attention fused with the output projection y = W_o . attention
// (rows = hidden, cols = qh * dim). `done` must be zero at launch and counts
// the finished KV heads; x is the attention output (a.out).
struct AttentionO {
    DecodeAttention a;
    const uint16_t *w;
    const float *x;
    float *y;
    uint32_t rows, cols, heads;
    uint32_t *done;
    uint32_t *error;
    // Per attention block of this layer, the step tag of its last completed
    // partial (kAttentionFlags words, zero when allocated): up to
    // kDecodeShortRows allocated rows the O blocks wait on these instead of
    // `done`.
    uint32_t *flags;
};
constexpr uint32_t kAttentionFlags = 64;
hipError_t launch_attention_o(hipStream_t, const AttentionO &);
bool attention_o_supported(uint32_t dim, uint32_t group, uint64_t cols);
// Blocks per KV head that cover `rows` cache rows (DecodeAttention::splits
// must be at least this for the largest row count of the launch).
// Allocated rows up to which the decode attention uses its short-context
// blocks (32 rows each; 64 in the fused attention + O launch, whose O blocks
// merge the partials); a decode step whose rows all stay below it may cap
// the attention's view of the allocation here.
constexpr uint32_t kDecodeShortRows = 256;
uint32_t decode_attention_splits(uint64_t rows);

// General causal attention for `tokens` query rows, the first at virtual row
// `prefix`. Key j of query t is the virtual row j of [cache rows 0..cached) ++
// [new rows 0..). With
// window > 0 query t sees only the last `window` virtual rows ending at its
// own row; its keys are raw and rotated on the fly at their window-local
// position, or `rotated` (keys and Q at their virtual rows) where
// prompt_attention_matrix holds.
struct PromptAttention {
    const float *q;          // [tokens, qh*dim] rotated Q
    const float *k_cache, *v_cache;  // rotated (or raw when window) cache rows
    const float *k_new, *v_new;      // rotated (or raw when window) new rows
    const float *table;
    float *out;              // [tokens, qh*dim]
    uint32_t prefix, tokens, cached, qh, kh, dim, window;
    int rotated;
    // Optional scratch for key splits (prompt_attention_scratch floats): few
    // query tiles then spread their keys over several blocks and a merge.
    float *partial;
};
hipError_t launch_prompt_attention(hipStream_t, const PromptAttention &);
// Head dims and group sizes of the matrix-core form.
bool prompt_attention_matrix(uint32_t dim, uint32_t qh, uint32_t kh);
// Floats of split scratch launch_prompt_attention uses for this shape (0: none).
uint64_t prompt_attention_scratch(uint32_t prefix, uint32_t tokens, uint32_t qh, uint32_t kh,
                                  uint32_t dim, uint32_t window, int rotated);

// The same attention on the fp16 matrix cores, for prompts of more than 32
// tokens and enough query rows. scratch: pair_attention_scratch bytes (256-byte aligned). With a window
// the keys are rotated at their virtual rows.
bool pair_attention_supported(uint32_t prefix, uint32_t tokens, uint32_t qh, uint32_t kh,
                              uint32_t dim);
uint64_t pair_attention_scratch(uint32_t prefix, uint32_t tokens, uint32_t kh, uint32_t dim);
hipError_t launch_pair_attention(hipStream_t, const PromptAttention &, void *scratch);

// Rotates cache rows [0, rows) of raw K into rotated K at their row position.
hipError_t launch_rerotate(hipStream_t, const float *k_raw, float *k_rot, const float *table,
                           uint64_t rows, uint32_t kh, uint32_t dim);
// Sliding-window commit: the final `keep` rows of [cache 0..prefix) ++
// [new 0..tokens) become cache rows 0..keep, rotated at their new positions.
hipError_t launch_window_store(hipStream_t, float *k_raw, float *v, float *k_rot,
                               const float *new_k, const float *new_v, uint64_t new_stride,
                               const float *table, float *scratch, uint64_t prefix,
                               uint64_t tokens, uint64_t keep, uint32_t kh, uint32_t dim);
// Batched row copies (one launch for every layer of a commit).
struct CopyRow {
    const float *src;
    float *dst;
    uint64_t floats;
};
hipError_t launch_copy_rows(hipStream_t, const CopyRow *table, uint32_t entries);
// A copy by a kernel, for pinned host memory on either side: 16-byte-aligned
// addresses and sizes.
hipError_t launch_copy_block(hipStream_t, const void *src, void *dst, uint64_t bytes);
// Up to kCopyBlocks blocks of whole words, each of any alignment to a word, in
// one launch.
constexpr uint32_t kCopyBlocks = 6;
struct CopyBlocks {
    const void *src[kCopyBlocks];
    void *dst[kCopyBlocks];
    uint64_t words[kCopyBlocks];
    uint32_t count;
    void add(const void *from, void *to, uint64_t n) {
        src[count] = from;
        dst[count] = to;
        words[count++] = n;
    }
};
hipError_t launch_copy_blocks(hipStream_t, const CopyBlocks &blocks);
// p[0, words) = value (a kernel, so that it is also safe inside captured graphs).
hipError_t launch_fill(hipStream_t, uint32_t *p, uint64_t words, uint32_t value);
// Raises the dynamic LDS limit of the GEMV variants to hold `cols` floats.
hipError_t configure_gemv(uint64_t max_cols);
// First maximal index per row (strict >); any NaN gives 0xffffffff. scratch:
// argmax_scratch_bytes(rows) of device memory.
hipError_t launch_argmax_rows(hipStream_t, const float *x, uint64_t width, uint64_t rows,
                              uint32_t *out, void *scratch);
uint64_t argmax_scratch_bytes(uint64_t rows);

}  // namespace plamo
