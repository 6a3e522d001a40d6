/*
 * iam.h - C ABI of the MI355X (gfx950) input-adaptive sparse decode library.
 *
 * This is the boundary that replaces the reference's OpenCL runtime
 * (gpu.hpp) and the OpenCL bodies of its operator wrappers.  Every entry
 * point is extern "C", takes plain pointers and sizes, and returns an int
 * status: 0 on success, a negative IAM_E* code on failure, with a message in
 * iam_last_error() (thread-local).  The C++ headers under
 * input-adaptive-matrix-inference-optimization_amd/cpp/ keep the reference's
 * class and method surface on top of these calls and turn non-zero statuses
 * into std::runtime_error, as the reference does.
 *
 * Execution model: one HIP stream per context, in order.  Every call is
 * asynchronous except iam_write / iam_read (blocking, like the reference's
 * writeBuffer/readBuffer) and iam_sync (the reference's eval()).  A context
 * is not thread-safe.  Device pointers come from iam_alloc; "_dev" arguments
 * point to device memory.
 *
 * Citations are to files of the reference repository.
 */
#ifndef IAM_H
#define IAM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* status codes */
#define IAM_OK 0
#define IAM_E_INVALID (-1)    /* bad argument or shape */
#define IAM_E_HIP (-2)        /* HIP runtime error */
#define IAM_E_NOMEM (-3)      /* allocation failed or over the byte budget */
#define IAM_E_STATE (-4)      /* call out of order (e.g. mul before calc_dispatch) */
#define IAM_E_IO (-5)         /* file missing, truncated or malformed */

#define IAM_PROBES_COUNT 4096 /* bucketMul.cl:18, bucket_mul.hpp:101 */

typedef struct iam_ctx iam_ctx;

/* ------------------------------------------------------------------ runtime */

/* Gpu::Gpu() (gpu.hpp:109-159): one device, one in-order queue. */
int iam_ctx_create(int device, iam_ctx** out);
/* Gpu::~Gpu() (gpu.hpp:161-188); frees everything allocated through the context. */
int iam_ctx_destroy(iam_ctx* ctx);
/* Gpu::eval() (gpu.hpp:399-447): wait for the queue, fold kernel timings. */
int iam_sync(iam_ctx* ctx);
/* Gpu::checkError message (gpu.hpp:581-587), thread-local. */
const char* iam_last_error(void);
/* device name / CU count / global memory (gpu.hpp:123-135, :28-31) */
int iam_device_info(iam_ctx* ctx, char* name, size_t name_len, int* compute_units,
                    size_t* global_mem_bytes);
/* MemoryTracker (gpu.hpp:21-60): byte budget = device memory - margin.
 * allocated counts the prefill buffers the models keep (iam_model_generate);
 * an allocation that finds no room frees those first. */
int iam_mem_status(iam_ctx* ctx, size_t* allocated, size_t* usable);

/* Gpu::createBuffer (gpu.hpp:236-262) */
int iam_alloc(iam_ctx* ctx, size_t bytes, void** out_dev);
/* Gpu::releaseBuffer (gpu.hpp:264-269) */
int iam_free(iam_ctx* ctx, void* dev);
/* BufferWrapper::zero (bucket_mul.hpp:34-38): a fill kernel, safe under graph capture. */
int iam_zero(iam_ctx* ctx, void* dev, size_t offset_bytes, size_t bytes);
/* Gpu::writeBuffer (gpu.hpp:464-469), blocking. */
int iam_write(iam_ctx* ctx, void* dst_dev, size_t dst_offset, const void* src_host, size_t bytes);
/* Gpu::readBuffer (gpu.hpp:457-462), blocking (waits for prior work). */
int iam_read(iam_ctx* ctx, void* dst_host, const void* src_dev, size_t src_offset, size_t bytes);
/* Gpu::copyBuffer (gpu.hpp:449-455), asynchronous device-to-device. */
int iam_copy(iam_ctx* ctx, void* dst_dev, size_t dst_offset, const void* src_dev,
             size_t src_offset, size_t bytes);

/* Measured streaming-read bandwidth of the device (GB/s): reps timed passes
 * of 16-byte loads over a zero-filled buffer of `bytes` (allocated and freed
 * here; 2 GiB keeps it out of the 256 MB Infinity Cache).  Blocking.  No
 * counterpart in the reference: the measured peak the walk's roofline is
 * also reported against. */
int iam_read_bandwidth(iam_ctx* ctx, size_t bytes, int reps, double* gb_per_s);

/* Per-kernel profiling (gpu.hpp:104-106, :275-290, :411-432): when enabled each
 * launch is bracketed by HIP events and iam_sync folds the durations. */
int iam_profiling(iam_ctx* ctx, int enable);
/* Gpu::printKernelStats (gpu.hpp:190-234) into a text buffer. */
int iam_kernel_stats(iam_ctx* ctx, char* buf, size_t len);
int iam_kernel_stats_reset(iam_ctx* ctx);
/* total time (ms) and launch count of one kernel name since the last reset.
 * The model's walk launches are labelled by matrix group ("bucket_walk.qkv",
 * ".o", ".ffn13", ".ffn2", ".lm"); a name without a dot also sums its
 * labelled launches ("bucket_walk" = every walk); "*" sums every kernel. */
int iam_kernel_stat(iam_ctx* ctx, const char* name, double* total_ms, int* calls);

/* --------------------------------------------------------------- bucketMul */

/* One weight matrix in the reference's bucket layout
 * (preprocess_layer_fixed_gpu.py:110-242, binary_loader.hpp:30-37):
 *   buckets  fp16 [n_experts * expert_rows][bucket_cols], packed value|position
 *   stats    fp16, stats_stride values per row; selection reads
 *            stats[row * stats_stride + stats_channel]
 *            (reference files: stride 4, channel 3, bucketMul.cl:372)
 *   probes   fp16, at least (expert_no + 1) * 4096 values (bucketMul.cl:103-109)
 *   expert_rows = 16 * in_dim, bucket_cols = out_dim / 16. */
typedef struct {
    const uint16_t* buckets;
    const uint16_t* stats;
    const uint16_t* probes;
    int expert_rows;
    int bucket_cols;
    int stats_stride;
    int stats_channel;
} iam_bucket_matrix;

/* BucketMul::calcDispatch (bucket_mul.hpp:147-191): cutoff search
 * (findCutoffBinarySearch, bucketMul.cl:68-214) and row selection
 * (prepareDispatch, bucketMul.cl:351-386) for x against stats/probes in the
 * reference's 4-channel stats layout.  The dispatch is kept in the context,
 * like the BucketMul singleton's scratch (bucket_mul.hpp:125-144).
 * expert_size is the row count R of one expert; rows with r/16 >= in_size
 * are skipped, as in the reference.  x must hold at least max(4096, in_size)
 * floats, because the cutoff always reads x[0:4096] (bucketMul.cl:102-110). */
int iam_bucketmul_calc_dispatch(iam_ctx* ctx, const float* x_dev, const uint16_t* stats_dev,
                                const uint16_t* probes_dev, int expert_no, int in_size,
                                int bucket_cols, int expert_size, float effort);
/* BucketMul::mul (bucket_mul.hpp:193-252): walk the rows selected by the last
 * calc_dispatch and write y[16 * bucket_cols] (overwritten). */
int iam_bucketmul_mul(iam_ctx* ctx, const uint16_t* buckets_dev, int bucket_cols, float* y_dev);
/* BucketMul::fullMul (bucket_mul.hpp:254-267) */
int iam_bucketmul_full(iam_ctx* ctx, const float* x_dev, const uint16_t* stats_dev,
                       const uint16_t* probes_dev, const uint16_t* buckets_dev, int expert_no,
                       int in_size, int bucket_cols, int expert_size, float effort, float* y_dev);
/* Up to 3 independent matrices in one launch, like iam_bucketmul_full every
 * walk workgroup running the cutoff search of its matrix itself (the q/k/v and
 * gate/up calls of attention.hpp:160-170 and feedforward.hpp:60-68 share an
 * input).  xs[i] may repeat. */
int iam_bucketmul_multi(iam_ctx* ctx, int n, const iam_bucket_matrix* mats,
                        const float* const* xs_dev, const int* in_sizes, float* const* ys_dev,
                        int expert_no, float effort);
/* One matrix group (1..3 matrices sharing one input) in one launch, as the
 * model's decode step runs it: every walk workgroup computes the input
 * itself -- x_dev as given, or, when h_dev is not null, x = RMSNorm(h) * gain
 * (rmsNorm32fast + mul16x32, aux.cl:156-196, :434-440; written to x_dev) --
 * then the cutoff (the same bisection as calc_dispatch, in every workgroup),
 * selects and walks its input slice into fp64 (or fp32) accumulators; the
 * last workgroup to finish a column tile stores that tile of ys_dev[i].
 * Results equal calc_dispatch + mul.  A norm input of other than
 * 4096 values is normalized by a separate RMSNorm launch first.  No
 * counterpart in the reference, which runs the cutoff as a launch of its
 * own (bucket_mul.hpp:147-176). */
int iam_bucketmul_fused(iam_ctx* ctx, int n, const iam_bucket_matrix* mats, float* x_dev, int in_size,
                        float* const* ys_dev, int expert_no, float effort, const float* h_dev,
                        const uint16_t* gain_dev, float eps);
/* iam_bucketmul_fused without any device allocation at call time.  No
 * counterpart in the reference: it is for callers that cannot allocate
 * (code under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc).  The walk's scratch lives in one fixed device array per GPU
 * (about 1 MiB, held from the first call on that GPU until the process
 * ends): at most IAM_NOALLOC_MAX_OUTPUTS outputs (16 * bucket_cols summed
 * over the matrices), 256 column tiles and 1024 input slices per matrix;
 * larger groups fail with IAM_E_INVALID.  A norm input (h_dev, gain_dev)
 * must be 4096 long.  Results equal iam_bucketmul_fused's.  Every call on a
 * GPU shares that array: calls that overlap on one GPU (other streams,
 * contexts or threads) race.  The call is not recorded in the dispatch
 * slots (dispatch_info / walk_count do not see it) and launches without
 * profiling events. */
#define IAM_NOALLOC_MAX_OUTPUTS 131072
int iam_bucketmul_fused_noalloc(iam_ctx* ctx, int n, const iam_bucket_matrix* mats, float* x_dev,
                                int in_size, float* const* ys_dev, int expert_no, float effort,
                                const float* h_dev, const uint16_t* gain_dev, float eps);
/* Parity outputs of the last calc_dispatch / multi / fused call for matrix slot
 * `slot`: the cutoff (fp32, as written by findCutoffBinarySearch) and the
 * selected-row count S.  The selection is re-run by a separate list kernel
 * that recomputes the cutoff on its own; the call fails with IAM_E_STATE if
 * the two cutoffs differ.  Blocking. */
int iam_bucketmul_dispatch_info(iam_ctx* ctx, int slot, float* cutoff, uint32_t* count);
/* The selected rows (expert-local row ids, ascending) of slot `slot`; writes
 * min(S, cap) ids into rows_host.  Blocking. */
int iam_bucketmul_dispatch_rows(iam_ctx* ctx, int slot, uint32_t* rows_host, size_t cap,
                                uint32_t* count);
/* Rows the last walk (mul / multi / full) of slot `slot` selected, counted
 * inside the walk kernel.  Blocking.  No counterpart in the reference. */
int iam_bucketmul_walk_count(iam_ctx* ctx, int slot, uint32_t* count);
/* effort -> quantile exactly as bucket_mul.hpp:164 */
int iam_effort_quantile(float effort);
/* Device-side counters of the walk: the algorithmic weight bytes streamed
 * (2 * S * bucket_cols summed over every matrix walked), the selected rows
 * S and the matrices walked, since the last reset.  They are updated inside
 * the walk kernel, so graph replays count too.  Blocking. */
int iam_walk_counters(iam_ctx* ctx, uint64_t* weight_bytes, uint64_t* rows, uint64_t* matrices,
                      int reset);
/* The model's walk launches by matrix group: the counters above split by the
 * group that streamed them (IAM_WALK_GROUP_NONE: standalone calls).  Reset
 * with iam_walk_counters.  Blocking.  No counterpart in the reference. */
#define IAM_WALK_GROUP_NONE 0
#define IAM_WALK_GROUP_QKV 1
#define IAM_WALK_GROUP_O 2
#define IAM_WALK_GROUP_FFN13 3
#define IAM_WALK_GROUP_FFN2 4
#define IAM_WALK_GROUP_LM 5
int iam_walk_group_counters(iam_ctx* ctx, int group, uint64_t* weight_bytes, uint64_t* rows,
                            uint64_t* matrices);
/* Of the group's walks since the last reset: the matrices whose cutoff
 * search started from a hint (tries; see iam_set_search_hints) and those
 * whose hinted window held the cutoff's ranks (hits; the others ran the
 * full search).  Counted with the counters above (iam_set_walk_counting).
 * Blocking.  No counterpart in the reference. */
int iam_walk_group_hints(iam_ctx* ctx, int group, uint64_t* tries, uint64_t* hits);
/* Counting of the walk's selected rows (default on): the first column tile
 * of each input slice adds its row count to the counters above (three
 * 64-bit atomics per slice).  Off, the counters are not updated.  The
 * per-slice counts behind iam_bucketmul_walk_count are stored either way.
 * Changing it re-captures the model's decode graph.  Not during capture.
 * No counterpart in the reference. */
int iam_set_walk_counting(iam_ctx* ctx, int on);
/* Hints for the walk's cutoff search (default off for the calls of this
 * context; a model's decode steps always use them, one per matrix of each
 * layer).  On, each iam_bucketmul_fused call starts the search of matrix
 * slot i from the cutoff that slot found in the previous fused call: one
 * pass over the importances counts those above the window [7/8, 8/7] of the
 * hint and bins those inside it, which locates the cutoff's neighbourhood
 * (ranks t-2 .. t+2) without the coarse histogram when the input changes
 * little between calls, as from one decode step to the next; where the
 * window misses those ranks the full search runs.  The cutoff, the selected
 * rows and the outputs are the same either way.  iam_set_search_hint sets
 * slot i's hint; any value is accepted (0, a negative, a non-finite one or
 * one outside [1e-30, 1e30] means no hint).  Not during capture.  No
 * counterpart in the reference. */
int iam_set_search_hints(iam_ctx* ctx, int on);
int iam_set_search_hint(iam_ctx* ctx, int slot, float value);
/* Block-structured selection, the thesis's future work (THESIS p.42-43):
 * with block_inputs B > 1, the inputs are taken in blocks of B consecutive
 * ones, and rank k of every input of a block is selected when rank k of any
 * of them passes the cutoff (the block's largest rank-k importance >= the
 * cutoff); the cutoff itself is the reference's.  It applies to calls whose
 * effort is below below_effort (the hybrid of fine selection at moderate
 * and blocks at aggressive sparsity); B = 1 (the default) is the
 * reference's per-row selection.  B is 1, 2, 4, 8 or 16.  Changing it
 * re-captures a model's decode graph.  Not during capture.  No counterpart
 * in the reference. */
int iam_set_selection_block(iam_ctx* ctx, int block_inputs, float below_effort);
int iam_get_selection_block(iam_ctx* ctx, int* block_inputs, float* below_effort);
/* Accumulation of the bucket walk (and of attention) for this context:
 * IAM_ACC_FP64 (default) adds the exact fp64 products in fp64 and rounds each
 * output once: every output is within an fp64 rounding of the correctly
 * rounded sum, whatever the order of the additions.  IAM_ACC_FP32 forms the
 * products in fp32 as the reference's bucketMul does (bucketMul.cl:430-445)
 * and adds them in fp64; attention runs in fp32.  No counterpart in the
 * reference (its fp32 atomics are order dependent). */
#define IAM_ACC_FP32 0
#define IAM_ACC_FP64 1
int iam_set_accumulation(iam_ctx* ctx, int mode);
int iam_get_accumulation(iam_ctx* ctx, int* mode);
/* Derive a compact copy stats3[r] = stats[r*4 + 3] (device), so the
 * selection reads 2 bytes per row instead of 8.  The file layout is unchanged. */
int iam_stats_compact(iam_ctx* ctx, const uint16_t* stats_dev, size_t rows, int stride,
                      int channel, uint16_t* out_dev);

/* ------------------------------------------------------------ layer ops */

/* rmsNorm32fast (aux.cl:156-196) then the fp16 gain mul16x32 (aux.cl:434-440) /
 * mulVec32by16 (aux.cl:301-306).  n must be a multiple of 1024, at most
 * 16384; vectors 16-byte aligned, the gain 8-byte aligned. */
int iam_rmsnorm_gain(iam_ctx* ctx, const float* in_dev, const uint16_t* gain_dev, int n,
                     float eps, float* out_dev);
/* add32 (bucketMul.cl:517-520) into h, then rmsnorm_gain of the sum
 * (transformer_layer.hpp:108-112 fused).  h_dev is updated in place. */
int iam_add_rmsnorm_gain(iam_ctx* ctx, float* h_dev, const float* delta_dev,
                         const uint16_t* gain_dev, int n, float eps, float* out_dev);
/* add32 (bucketMul.cl:517-520): out = a + b */
int iam_add(iam_ctx* ctx, const float* a_dev, const float* b_dev, int n, float* out_dev);
/* silu32 (matrix.cl:27-32): out = up * gate / (1 + exp(-gate)) */
int iam_silu_mul(iam_ctx* ctx, const float* gate_dev, const float* up_dev, int n,
                 float* out_dev);
/* precompute_rope_cache (attention.hpp:207-235): host table
 * [max_pos][head_dim/2][2] of (cos, sin) in float. */
int iam_rope_table(double theta, int head_dim, int max_pos, float* table_host);
/* rope_mx (aux.cl:227-248) on n_heads heads; table row = *pos_dev. */
int iam_rope(iam_ctx* ctx, const float* in_dev, const float* table_dev, const int* pos_dev,
             int n_heads, int head_dim, float* out_dev);
/* RoPE of q (n_heads) and k (n_kv heads), then the KV append
 * (attention.hpp:172-189 and :281-309) into fp16 caches laid out
 * [max_ctx][n_kv][head_dim] at position *pos_dev (ignored unless
 * 0 <= *pos_dev < max_ctx). */
int iam_rope_kv_append(iam_ctx* ctx, const float* q_dev, const float* k_dev, const float* v_dev,
                       const float* table_dev, const int* pos_dev, int n_heads, int n_kv,
                       int head_dim, int max_ctx, float* q_out_dev, uint16_t* kcache_dev,
                       uint16_t* vcache_dev);
/* Decode attention over positions 0..*pos_dev of an fp16 GQA cache
 * (dotSetScore2 aux.cl:497-540, sum_of_exps32_mx :204-210, softmax_add32_mx
 * :219-225, sumScores32 :370-384; driver attention.hpp:311-404), split over
 * the context.  Query head h reads KV head h*n_kv/n_heads (repeat4x32). */
int iam_attention_decode(iam_ctx* ctx, const float* q_dev, const uint16_t* kcache_dev,
                         const uint16_t* vcache_dev, const int* pos_dev, int n_heads, int n_kv,
                         int head_dim, int max_ctx, float* out_dev);
/* The reference's KV cache layout and fp32 attention, the parity mode of
 * iam_rope_kv_append / iam_attention_decode: the caches hold K (after RoPE)
 * and V repeated to every query head, fp32 [max_ctx][n_heads][head_dim] per
 * layer (model.hpp:97-98).  RoPE of q and k, then K and V of KV head
 * h*n_kv/n_heads stored for every query head h at *pos_dev (repeat4x32
 * aux.cl:266-275, rope_mx :227-248, the copies of attention.hpp:281-309). */
int iam_rope_kv_append_f32(iam_ctx* ctx, const float* q_dev, const float* k_dev, const float* v_dev,
                           const float* table_dev, const int* pos_dev, int n_heads, int n_kv, int head_dim,
                           int max_ctx, float* q_out_dev, float* kcache_dev, float* vcache_dev);
/* Attention over positions 0..*pos_dev of those caches in the reference's
 * fp32 arithmetic (dotSetScore2 aux.cl:497-540 with its work-group tree,
 * sum_of_exps32_mx / softmax_add32_mx :204-225 with no maximum subtracted,
 * sumScores32 :370-384; driver attention.hpp:311-404): one IEEE operation
 * at a time, the sums of exp and of p*v in splits of 64 positions taken in
 * order (the reference's float atomics have no fixed order).  A score above
 * log(FLT_MAX) ~ 88.72 makes that head's outputs NaN, as in the reference. */
int iam_attention_decode_f32(iam_ctx* ctx, const float* q_dev, const float* kcache_dev,
                             const float* vcache_dev, const int* pos_dev, int n_heads, int head_dim,
                             int max_ctx, float* out_dev);
/* matmul16x32 (aux.cl:454-490), the reference's dense LM head (model.hpp:
 * 207-227, 256 work-items per row): out[r] = the fp16 row r of W [rows][cols]
 * times x, each row's products summed per work-item over the columns
 * l, l+256, ... in order and then by the 256-way work-group tree, in fp32
 * without contraction.  cols <= 16384. */
int iam_matmul_f16_dense(iam_ctx* ctx, const uint16_t* w_dev, const float* x_dev, int rows, int cols,
                         float* out_dev);
/* fetchRow16to32 (aux.cl:442-452): out = (float) table[*token_dev][:]; a
 * token outside [0, vocab) yields zeros. */
int iam_embed_gather(iam_ctx* ctx, const uint16_t* table_dev, int cols, int vocab,
                     const int* token_dev, float* out_dev);
/* greedy pick (test_generation.cpp:235, :276): first index of the maximum */
int iam_argmax(iam_ctx* ctx, const float* v_dev, int n, int* out_dev);

/* -------------------------------------------------------- synthetic data */

/* Counter-based generator shared with the CPU oracle: element n of tensor
 * `tensor_id` = mean + sigma * (sum of 12 uniform uint32 - 6*2^32) / 2^32,
 * rounded to float (and then to fp16 for the f16 variant). */
int iam_gen_f16(iam_ctx* ctx, uint64_t seed, uint64_t tensor_id, size_t count, double mean,
                double sigma, uint16_t* out_dev);
int iam_gen_f32(iam_ctx* ctx, uint64_t seed, uint64_t tensor_id, size_t count, double mean,
                double sigma, float* out_dev);
/* GPU bucketizer, byte-identical to bucketize_fp16_packed
 * (preprocess_layer_fixed_gpu.py:110-242): W fp16 [out_dim][in_dim] ->
 * buckets [16*in][out/16], stats [16*in][4], probes [in]. */
int iam_bucketize(iam_ctx* ctx, const uint16_t* w_dev, int out_dim, int in_dim,
                  uint16_t* buckets_dev, uint16_t* stats_dev, uint16_t* probes_dev);

/* ----------------------------------------------------------------- model */

/* Mistral-shaped decoder (model.hpp:15-30, attention.hpp:21-27): dims,
 * heads, vocabulary, KV capacity and RoPE theta are parameters. */
typedef struct {
    int n_layers;
    int dim;
    int ffn_dim;
    int n_heads;
    int n_kv_heads;
    int head_dim;
    int vocab;
    int max_ctx;
    double rope_theta;
    float norm_eps;
} iam_model_config;

typedef struct iam_model iam_model;

/* MistralModel::MistralModel (model.hpp:84-127): allocates weights (bucket
 * layout, LM head included), fp16 KV caches [n_layers][max_ctx][n_kv][hd],
 * activations and the RoPE table. */
int iam_model_create(iam_ctx* ctx, const iam_model_config* cfg, iam_model** out);
int iam_model_destroy(iam_model* m);
/* Fill every weight from the synthetic generator: matrices N(0, 0.02^2)
 * bucketized on the GPU, gains 1 + N(0, 0.01^2), embedding N(0, 0.02^2). */
int iam_model_synthesize(iam_model* m, uint64_t seed);
/* MistralModel::forward (model.hpp:152-231): one token at position pos;
 * logits (vocab floats, device) are written; the KV cache at pos is filled. */
int iam_model_forward(iam_model* m, int token, int pos, float effort, float* logits_dev);
/* Like forward, but the token and position are read from device memory
 * (token_dev, pos_dev) and the next token (first argmax) is written back to
 * token_dev and pos is advanced, so a captured step replays without host
 * involvement.  hidden_override_dev, if non-NULL, replaces the embedding. */
int iam_model_step_device(iam_model* m, float effort, const float* hidden_override_dev);
/* Greedy decode (test_generation.cpp:197-276): feeds the prompt, then
 * generates n_new tokens with first-max argmax.  With use_graph the per-token
 * step is captured once as a HIP graph and replayed.  The prompt's tokens
 * before the last go through the model in batches where that is faster (fp64
 * accumulation, from 6 to 16 tokens on by shape and effort), in buffers the
 * model keeps until an allocation needs their room (about 2 MB a token, at
 * most 512 tokens', at 4096 wide with FFN 14336; fewer where there is less
 * room).  The KV cache, the picks in "history" and the walk counters' bytes,
 * rows and matrices are as by steps; batched tokens take no search hints, so
 * they count no tries or hits of them (iam_walk_group_hints).  The last
 * token's step leaves the activations and logits.
 * out_tokens receives n_new ids. */
int iam_model_generate(iam_model* m, const int* prompt, int n_prompt, int n_new, float effort,
                       int use_graph, int* out_tokens);
/* Continue greedy decoding from the current device state (the token picked
 * by the previous step at the current position) for n_steps steps, replaying
 * the captured step when use_graph is set.  Asynchronous. */
int iam_model_decode(iam_model* m, int n_steps, float effort, int use_graph);
/* Set the device position the next step computes (0 <= pos <= max_ctx).
 * decode and step_device refuse steps past the KV capacity, counted from
 * this position (or from forward / generate / reset_caches). */
int iam_model_set_position(iam_model* m, int pos);
/* MistralModel::reset_caches (model.hpp:233-237); also rewinds the position. */
int iam_model_reset_caches(iam_model* m);
/* The LM head as the reference's dense fp16 product (matmul16x32 over
 * lm_dense_dev [vocab][dim], a caller-owned device buffer that must outlive
 * its use; model.hpp:207-227) instead of the bucket-layout one; NULL restores
 * the bucket layout.  The step then runs the final norm, the dense product
 * and the first-max pick as launches of their own. */
int iam_model_set_lm_dense(iam_model* m, const uint16_t* lm_dense_dev);
/* Per-channel fp32 factors applied to the gathered embedding before the
 * first layer (NULL restores plain fetchRow16to32).  Used for the skewed-
 * channel decode workload, which scales 1% of hidden channels. */
int iam_model_set_embed_scale(iam_model* m, const float* scale_host);
/* Device pointer and size of a named model tensor, e.g. "layer3.w1.buckets",
 * "layer0.attn_gain", "embed", "final_gain", "lm_head.stats", "kcache",
 * "vcache", "rope", "logits", "token", "pos", "hidden" (the residual stream
 * after the last layer), "hidden_norm" (its final RMSNorm, the LM head input). */
int iam_model_tensor(iam_model* m, const char* name, void** dev, size_t* bytes);
/* The bucket-matrix descriptor of "layer{L}.{wq,wk,wv,wo,w1,w3,w2}" or "lm_head". */
int iam_model_matrix(iam_model* m, const char* name, iam_bucket_matrix* out);

#ifdef __cplusplus
}
#endif
#endif
