/*
 * cbis_runtime.h -- C-ABI of the C++ host runtime (libcbis.so).
 *
 * The runtime keeps the reference's host API in C++
 * (continuous-batching-inference-server_amd/csrc/runtime/runtime.hpp):
 *   PagedKVCache        include/paged_kv_cache.hpp:17-51 (src/paged_kv_cache.cpp:5-60)
 *   ModelWeights        include/model_weights.hpp:7-25  (src/model_weights.cpp:41-75)
 *   TransformerRunner   include/transformer.hpp:15-34   (src/transformer.cpp:11-99)
 *   run_continuous      src/bench_batching.cpp:98-179
 * and reaches the GPU only through include/cbis_kernels.h.  The functions
 * below wrap those classes for callers that bind C (ctypes, cgo, JNI...).
 * C++ exceptions never cross this boundary: a failing call returns a
 * negative status (or NULL) and cbis_runtime_last_error() says why.
 */
#ifndef CBIS_RUNTIME_H
#define CBIS_RUNTIME_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct cbis_model_config {
  int vocab, d_model, n_heads, head_dim, n_layers, mlp, max_seq, page_size;
  int weight_dtype; /* CBIS_F32, CBIS_BF16 or CBIS_FP8E4M3 (linear weights) */
  int kv_dtype;     /* CBIS_F32 or CBIS_BF16 (paged K/V pools) */
} cbis_model_config;

typedef struct cbis_cache cbis_cache;
typedef struct cbis_weights cbis_weights;
typedef struct cbis_runner cbis_runner;

const char* cbis_runtime_last_error(void);

/* The reference model's dimensions (include/config.hpp:4-25), fp32. */
void cbis_default_config(cbis_model_config* cfg);

/* ---- PagedKVCache (include/paged_kv_cache.hpp:17-51) -------------------- */
/* alloc_device = 0 keeps only the bookkeeping (no HIP call at all). */
cbis_cache* cbis_cache_create(int num_layers, int max_pages, int page_size, int n_heads, int head_dim, int kv_dtype,
                              int pages_per_seq, int alloc_device);
void cbis_cache_destroy(cbis_cache* c);
int cbis_cache_allocate_sequence(cbis_cache* c);
void cbis_cache_free_sequence(cbis_cache* c, int seq_id);
/* 1: capacity ensured; 0: free list exhausted (reference returns false);
 * negative: unknown sequence (reference throws std::out_of_range). */
int cbis_cache_ensure_capacity(cbis_cache* c, int seq_id, int token_pos);
/* 0 on success; negative when the slot is not allocated (reference throws). */
int cbis_cache_resolve_slot(cbis_cache* c, int seq_id, int token_pos, int* physical_page, int* offset);
/* Writes the zero-padded pages_per_seq-entry table; returns entries written or negative. */
int cbis_cache_page_table(cbis_cache* c, int seq_id, int* out, int capacity);
/* Physical pages owned by seq_id in logical order; returns the count (may exceed capacity). */
int cbis_cache_seq_pages(cbis_cache* c, int seq_id, int* out, int capacity);
int cbis_cache_num_free_pages(cbis_cache* c);
int cbis_cache_max_pages(cbis_cache* c);
int cbis_cache_page_size(cbis_cache* c);
void* cbis_cache_k_base(cbis_cache* c, int layer);
void* cbis_cache_v_base(cbis_cache* c, int layer);
/* Fills every page of every pool with N(0, std) (cbis_fill_normal_fast). */
int cbis_cache_fill_normal(cbis_cache* c, uint64_t seed, float std);

/* ---- ModelWeights (include/model_weights.hpp:7-25) ---------------------- */
/* Seeded synthetic weights: linear / embedding weights and linear biases
 * N(0, std) from the exact counter-based generator, LayerNorm gamma 1 /
 * beta 0; linear weights stored as cfg->weight_dtype. */
cbis_weights* cbis_weights_synthetic(const cbis_model_config* cfg, uint64_t seed, float std);
/* python/export_weights.py:42-66 layout (fp32), converted to cfg's dtypes. */
cbis_weights* cbis_weights_load(const char* path, const cbis_model_config* cfg);
/* Packed checkpoint (no reference counterpart; the format the reference's
 * weights.bin reader at src/model_weights.cpp:41-75 lacks for bf16 / fp8
 * models): a versioned header with the model config and tensor table, then
 * the device image in its stored dtypes (fp8 codes with their fp32 channel
 * scales).  Saving needs the weights on the device; loading validates the
 * header, the table against the config's layout, the size and a checksum
 * before returning.  cfg_out (optional) receives the file's config. */
int cbis_weights_save_packed(const cbis_weights* w, const char* path);
cbis_weights* cbis_weights_load_packed(const char* path, cbis_model_config* cfg_out);
void cbis_weights_destroy(cbis_weights* w);
size_t cbis_weights_device_bytes(const cbis_weights* w);
/* Device pointer of a named tensor ("tok_emb", "pos_emb", "lm_head",
 * "lm_scale", "ln_f_w", "ln_f_b", or "l<i>.<name>" with name in wqkv, bqkv,
 * sqkv, wo, bo, so, w1, b1, s1, w2, b2, s2, ln1_w, ln1_b, ln2_w, ln2_b). */
void* cbis_weights_tensor(const cbis_weights* w, const char* name);

/* ---- TransformerRunner (include/transformer.hpp:15-34) ------------------ */
cbis_runner* cbis_runner_create(const cbis_weights* w, cbis_cache* c, int max_total_rows);
void cbis_runner_destroy(cbis_runner* r);
/* forward_step: row i is (token_ids[i], positions[i], seq_ids[i]); the caller
 * ran ensure_capacity for every row.  logits_out: host [n, vocab] fp32. */
int cbis_runner_forward_step(cbis_runner* r, int n, const int* token_ids, const int* positions,
                             const int* seq_ids, float* logits_out);
/* Same step with the greedy argmax of every row taken on the device, fused
 * with lm_head (cbis_gemm_argmax: the logits are not stored on the paths
 * that reduce in the GEMM epilogue); next_tokens: host [n]. */
int cbis_runner_forward_step_greedy(cbis_runner* r, int n, const int* token_ids, const int* positions,
                                    const int* seq_ids, int* next_tokens);
/* Pipelined greedy steps (no reference counterpart: they let a decode loop
 * queue step t + 1 before step t's tokens reach the host).
 * cbis_runner_enqueue_greedy queues the step of cbis_runner_forward_step_greedy
 * and returns at once with *ticket.  token_src (NULL, or n entries): row i
 * with token_src[i] >= 0 takes as its input token the greedy token of row
 * token_src[i] of the greedy step enqueued just before this one, and
 * token_ids[i] is not used.  cbis_runner_wait_greedy waits for that step and
 * writes min(capacity, rows) tokens; it returns its row count, and
 * last_margins / last_device_ms / last_host_ms then describe it.  At most two
 * steps are outstanding: enqueueing a third before the first was waited for
 * fails. */
int cbis_runner_enqueue_greedy(cbis_runner* r, int n, const int* token_ids, const int* positions, const int* seq_ids,
                               const int* token_src, int64_t* ticket);
int cbis_runner_wait_greedy(cbis_runner* r, int64_t ticket, int* next_tokens, int capacity);
/* Top-2 margins (max logit minus the runner-up) of the last greedy step's
 * rows (no reference counterpart): writes min(capacity, n); returns n, which
 * is 0 after a plain forward_step. */
int cbis_runner_last_margins(const cbis_runner* r, float* out, int capacity);
/* Device time in ms of the last step's forward (no reference counterpart: a
 * diagnostic): two events on the runner's stream around the forward's
 * kernels (the first of which also brings the step's metadata from pinned
 * host memory; a greedy step's last one stores its tokens there, a
 * forward_step's of up to 4 MiB of logits the logits). */
float cbis_runner_last_device_ms(const cbis_runner* r);
/* Host wall time in ms of the last greedy step's phases (no reference
 * counterpart: a diagnostic): out[0] host preparation of the step's
 * metadata, out[1] the forward's launch, out[2] the wait for its results. */
void cbis_runner_last_host_ms(const cbis_runner* r, double out[3]);
/* Device pointer of the last forward_step's [n, vocab] fp32 logits. */
const float* cbis_runner_logits_device(cbis_runner* r);
/* hipStream_t the runner launches on. */
void* cbis_runner_stream(cbis_runner* r);
/* Enable / disable HIP-graph replay of steps whose shape repeats. */
void cbis_runner_set_graphs(cbis_runner* r, int enable);
/* Enable (the default) / disable the fused attention + out-projection
 * launch (cbis_paged_attention_proj) that steps of at most 64 decode rows
 * with keys up to 768 use when the model's widths allow it (no reference
 * counterpart; disabled, every step runs the two launches). */
void cbis_runner_set_fused_decode(cbis_runner* r, int enable);
/* How the last step ran (no reference counterpart: a diagnostic):
 * {rows, decode rows, prefill tiles, sequences, block-table width, max_kv
 * bound, decode split_tokens (1 << 30 = one pass per row, 0 = the attention
 * library's automatic split), 1 if attention and out-projection ran as one
 * launch per layer}.  Writes min(capacity, 8) ints; returns 8. */
int cbis_runner_last_plan(const cbis_runner* r, int* out, int capacity);

/* ---- Three-tier KV block manager (include/tiered_kv_manager.hpp:21-151,
 *      include/block_storage.hpp:9-64) --------------------------------------
 * A block is one physical page's K and V slots in every layer of a cache;
 * tiers: 0 GPU (resident in a PagedKVCache page), 1 DRAM (deflated in host
 * memory), 2 NVMe (deflated in the scratch file).  Same operations, eviction
 * score and tier choice as the reference; the batch calls move all their
 * blocks with one gather / scatter launch and one host copy. */
typedef struct cbis_tiered cbis_tiered;
typedef struct cbis_eviction_params {
  double alpha_staleness, beta_restore_cost, expected_compression_ratio;
  double dram_fixed_ns, dram_ns_per_byte, nvme_fixed_ns, nvme_ns_per_byte;
} cbis_eviction_params;

/* The reference's defaults (include/tiered_kv_manager.hpp:40-48). */
void cbis_eviction_params_default(cbis_eviction_params* p);
/* params may be NULL (defaults).  kv_dtype: CBIS_F32 (the reference's pools)
 * or CBIS_BF16. */
cbis_tiered* cbis_tiered_create(int layer_count, int page_size, int n_heads, int head_dim, int kv_dtype,
                                const char* nvme_scratch_path, size_t gpu_capacity_blocks,
                                size_t dram_capacity_blocks, const cbis_eviction_params* params);
void cbis_tiered_destroy(cbis_tiered* t);
size_t cbis_tiered_raw_block_bytes(const cbis_tiered* t);
int cbis_tiered_calibrate(cbis_tiered* t);
int cbis_tiered_params(const cbis_tiered* t, cbis_eviction_params* out);
int cbis_tiered_admit_gpu_resident(cbis_tiered* t, uint64_t block_id, cbis_cache* c, int physical_page,
                                   long now_step);
/* *evicted receives the block id, or UINT64_MAX when no block is on the GPU. */
int cbis_tiered_evict_one(cbis_tiered* t, long now_step, uint64_t* evicted);
int cbis_tiered_spill(cbis_tiered* t, uint64_t block_id, int dest_tier, long now_step);
int cbis_tiered_restore(cbis_tiered* t, uint64_t block_id, cbis_cache* c, int physical_page, long now_step);
int cbis_tiered_spill_batch(cbis_tiered* t, const uint64_t* block_ids, int n, int dest_tier, long now_step);
int cbis_tiered_restore_batch(cbis_tiered* t, const uint64_t* block_ids, int n, cbis_cache* c,
                              const int* physical_pages, long now_step);
/* Tier (0, 1, 2) of a tracked block; negative for an unknown one. */
int cbis_tiered_tier_of(const cbis_tiered* t, uint64_t block_id);
int cbis_tiered_known(const cbis_tiered* t, uint64_t block_id);
int cbis_tiered_touch(cbis_tiered* t, uint64_t block_id, long now_step);
/* out[5] = GPU, DRAM, NVMe block counts, raw bytes, compressed bytes. */
int cbis_tiered_stats(const cbis_tiered* t, size_t* out);

/* Host-only block codec of the colder tiers (zlib deflate, fastest level):
 * returns the compressed length (<= cap), or negative. */
int64_t cbis_block_deflate(const void* src, size_t len, void* dst, size_t cap);
/* Inflates exactly out_len bytes; 0 or negative. */
int cbis_block_inflate(const void* src, size_t len, void* dst, size_t out_len);

/* ---- continuous batching (src/bench_batching.cpp:98-179) ---------------- */
/* All requests are present at t = 0.  prompt_tokens concatenates the
 * prompts; out_tokens receives decode_lens[i] tokens per request,
 * concatenated.  step_ms (optional, capacity max_steps) receives each
 * step's wall time; returns the number of steps run, or negative. */
int cbis_run_continuous(cbis_runner* r, cbis_cache* c, int n_requests, const int* prompt_lens,
                        const int* prompt_tokens, const int* decode_lens, int max_slots, int* out_tokens,
                        double* step_ms, int max_steps);

/* The same scheduler with chunked prefill (src/bench_tiering.cpp:78-89's
 * chunking, inside continuous batching): a slot feeds at most prefill_chunk
 * prompt rows per step (0 = its whole prompt), and one step carries at most
 * step_token_budget prompt rows (0 = no cap; decode rows are never
 * deferred).  prefill_chunk = step_token_budget = 0 is cbis_run_continuous. */
int cbis_run_continuous_chunked(cbis_runner* r, cbis_cache* c, int n_requests, const int* prompt_lens,
                                const int* prompt_tokens, const int* decode_lens, int max_slots, int prefill_chunk,
                                int step_token_budget, int* out_tokens, double* step_ms, int max_steps);

/* cbis_run_continuous_chunked with request arrival times
 * (src/bench_batching.cpp:110-121, 153-158): request i is admitted once
 * arrival_ms[i] ms have passed since the run began (nondecreasing; NULL: all
 * at 0), and a scheduler with no active request sleeps until the next
 * arrival.  finish_ms (or NULL): per request, ms since the run began when its
 * last token came back (the reference's Result::finish_ms). */
int cbis_run_continuous_timed(cbis_runner* r, cbis_cache* c, int n_requests, const int* prompt_lens,
                              const int* prompt_tokens, const int* decode_lens, const double* arrival_ms,
                              int max_slots, int prefill_chunk, int step_token_budget, int* out_tokens,
                              double* step_ms, int max_steps, double* finish_ms);

/* cbis_run_continuous_timed with one step in flight (no reference
 * counterpart): step t + 1 is built and queued before step t's tokens come
 * back, its decode rows taking their input tokens from step t on the device
 * (cbis_runner_enqueue_greedy's token_src).  Same rows, tokens and page
 * order for the same admissions; a request arriving while step t runs is
 * admitted from step t + 2 at the earliest.  step_ms[k]: host ms from the
 * later of step k's enqueue and the previous collection to its collection;
 * finish_ms: when the host collected the request's last token. */
int cbis_run_continuous_pipelined(cbis_runner* r, cbis_cache* c, int n_requests, const int* prompt_lens,
                                  const int* prompt_tokens, const int* decode_lens, const double* arrival_ms,
                                  int max_slots, int prefill_chunk, int step_token_budget, int* out_tokens,
                                  double* step_ms, int max_steps, double* finish_ms);

/* Runs the scheduler on the host only, with a stand-in step whose "greedy
 * token" of row (tok, pos, seq) is (31 tok + 7 pos + 13 seq + 1) mod vocab
 * (32-bit unsigned arithmetic), so the schedule can be checked without a
 * GPU (c may be created with alloc_device = 0).  step_rows[k] receives the
 * row count of step k (capacity max_steps); row_tok / row_pos / row_sid the
 * rows of every step, concatenated (capacity max_rows).  Returns the number
 * of steps, or negative. */
int cbis_schedule_dry_run(cbis_cache* c, int n_requests, const int* prompt_lens, const int* prompt_tokens,
                          const int* decode_lens, int max_slots, int prefill_chunk, int step_token_budget, int vocab,
                          int* out_tokens, int* step_rows, int max_steps, int* row_tok, int* row_pos, int* row_sid,
                          int max_rows);
/* The dry run with arrival times on a virtual clock: every step takes
 * step_time_ms and an idle scheduler's wait jumps the clock to the next
 * arrival; finish_ms (or NULL) as cbis_run_continuous_timed's. */
int cbis_schedule_dry_run_timed(cbis_cache* c, int n_requests, const int* prompt_lens, const int* prompt_tokens,
                                const int* decode_lens, const double* arrival_ms, double step_time_ms, int max_slots,
                                int prefill_chunk, int step_token_budget, int vocab, int* out_tokens, int* step_rows,
                                int max_steps, int* row_tok, int* row_pos, int* row_sid, int max_rows,
                                double* finish_ms);
/* The timed dry run through cbis_run_continuous_pipelined's scheduler: the
 * stand-in step resolves a row's token source against the outputs of the
 * step queued before it and runs (on the virtual clock) when it is queued,
 * so rows, tokens and admissions equal the timed dry run's; rows that take
 * their token from the device come back with row_tok -1, and finish_ms is the
 * virtual time at which the request's last token was collected. */
int cbis_schedule_dry_run_pipelined(cbis_cache* c, int n_requests, const int* prompt_lens, const int* prompt_tokens,
                                    const int* decode_lens, const double* arrival_ms, double step_time_ms,
                                    int max_slots, int prefill_chunk, int step_token_budget, int vocab,
                                    int* out_tokens, int* step_rows, int max_steps, int* row_tok, int* row_pos,
                                    int* row_sid, int max_rows, double* finish_ms);

#ifdef __cplusplus
}
#endif

#endif /* CBIS_RUNTIME_H */
