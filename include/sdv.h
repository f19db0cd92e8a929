/*
 * sdv.h -- C ABI of the MI355X (gfx950) FP8-V paged decode hot path.
 *
 * Library: libsdv.so (built by hipcc from the .hip sources in specdec-context-scaling_amd/csrc).
 * All tensor arguments are DEVICE pointers owned by the caller; the library allocates
 * nothing per call.  Every entry point validates its arguments on the host, returns
 * SDV_OK (0) or a negative status, launches asynchronously on `stream` (a hipStream_t,
 * NULL = the legacy default stream) and is re-entrant (the only process-wide state is an
 * atomic call counter that tags single-launch calls and the wait bound set by
 * sdv_attention_set_wait_limit; calls that share a workspace buffer must be ordered on one
 * stream).
 *
 * Paged cache layout (one layer; layers sit `*_layer_stride` elements apart):
 *   k_pages  [num_blocks][kv_heads][head_dim/8][16][8]  bf16: token t, dim d of a page sits at
 *                                                   ((d/8)*16 + t)*8 + d%8 (8-dim chunks, so
 *                                                   one 1 KiB load feeds a 16x32 MFMA tile)
 *   v_pages  [num_blocks][kv_heads][head_dim][16]   E4M3FN codes, dimension-major in a page
 *   v_scales [num_blocks][kv_heads][16]             fp32, one scale per (token, KV head)
 * A token's slot is block * 16 + offset; block_table[b][j] is the physical block that
 * holds tokens 16*j .. 16*j+15 of sequence b.
 *
 * Reference interfaces replaced (RichardF123/SpecDec-Context-Scaling):
 *   sdv_quant_append     <- quantize_kv_fp8 (specdec/engine/model_self.py:304-314) applied
 *                           to the current V (model_self.py:697-706) plus the v_fp8 cache
 *                           append torch.cat of payload/scale (model_self.py:795-799) and the
 *                           BF16 K write-back (model_self.py:721-722)
 *   sdv_paged_attention  <- the v_fp8 read path (dequantize_kv_fp8 + cat, model_self.py:
 *                           316-320, 715-728) and the eager GQA attention core
 *                           (model_self.py:739-776); at op level it is what
 *                           ops.attention(q, k, v, "cuda") (specdec/kernels/ops.py:67-76)
 *                           -> pybind attention (specdec/kernels/cuda/bind.cpp:16)
 *                           -> attention_cuda (specdec/kernels/cuda/attention.cu:244-288)
 *                           computes, with FP8 V dequantized inside the kernel
 *   sdv_paged_attention_append <- no counterpart: sdv_quant_append + sdv_paged_attention
 *                           in one call (the single launch writes the new tokens itself)
 *   sdv_quant_append_tiles <- no counterpart: sdv_quant_append for the engine's batched
 *                           varlen prefill (a table of 16-row tiles that follow each
 *                           sequence's start)
 *   sdv_attention_workspace_size  <- no counterpart (the reference allocates its score,
 *                           softmax and kv_repeat temporaries inside torch)
 *   sdv_fp8_encode       <- the tensor.to(torch.float8_e4m3fn) cast (model_self.py:312)
 *   sdv_status_string    <- TORCH_CHECK messages (attention.cu:245-262)
 */
#ifndef SDV_H_
#define SDV_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define SDV_BLOCK_SIZE 16
#define SDV_ABI_VERSION 1

enum sdv_status {
    SDV_OK = 0,
    SDV_ERR_NULL = -1,         /* a required pointer is NULL */
    SDV_ERR_SHAPE = -2,        /* a size argument is out of range or inconsistent */
    SDV_ERR_UNSUPPORTED = -3,  /* valid but not supported (head_dim, group size, scale mode) */
    SDV_ERR_WORKSPACE = -4,    /* workspace NULL, too small or not 256-byte aligned */
    SDV_ERR_ALIGN = -5,        /* a tensor pointer is not aligned as documented */
    SDV_ERR_HIP = -6           /* the HIP runtime reported an error at launch */
};

/* scale_mode for sdv_quant_append: how s = max|v| / 448 is evaluated.
 *  SDV_SCALE_DIV: IEEE fp32 division (torch on the CPU; the golden fixtures).
 *  SDV_SCALE_RCP: max|v| * RN_f32(1/448) (torch's CUDA/ROCm kernels for a scalar divisor). */
#define SDV_SCALE_DIV 0
#define SDV_SCALE_RCP 1

/*
 * Kernel 1: fused V quantize (+ optional BF16 K copy) and paged append.
 *
 * v_new, k_new: bf16 [num_layers][n_tokens][kv_heads][head_dim] (layers in_layer_stride
 *               elements apart; k_new may be NULL: K is then not written).
 * slot_mapping: int32 [n_tokens]; a negative slot skips the token (padding).
 * group_size must equal head_dim (the v_fp8 format: one scale per token and KV head).
 * head_dim in {64, 128}.  Alignment: v_new/k_new/k_pages/v_pages 16 B (and layer strides of
 * v_new/k_new/k_pages multiples of 8 elements), v_scales and slot_mapping 4 B.
 * Each (token, KV head) gets s = max|v| / 448 (s == 0 -> 1), payload RNE(v / s) in E4M3FN,
 * bit-exact with the reference helper evaluated per scale_mode.
 */
int sdv_quant_append(const void* v_new, const void* k_new, const int32_t* slot_mapping,
                     int32_t n_tokens, int32_t kv_heads, int32_t head_dim, int32_t group_size,
                     int32_t num_layers, int64_t in_layer_stride,
                     void* k_pages, void* v_pages, float* v_scales, int32_t num_blocks,
                     int64_t k_layer_stride, int64_t v_layer_stride, int64_t s_layer_stride,
                     int32_t scale_mode, void* stream);

/*
 * sdv_quant_append with a tile table: tile i is input rows [tile_starts[i],
 * min(tile_starts[i] + 16, tile_starts[i+1])) (n_tiles + 1 entries, non-decreasing, within
 * [0, n_tokens]; rows that no tile covers are not written).  Same results as
 * sdv_quant_append for any table that covers every row once.  No counterpart in the reference
 * (its prefill writes one 2048-token chunk of one sequence): for the batched varlen prefill of
 * the paged engine, whose sequences start anywhere in the packed input -- tiles that begin at
 * each sequence's first row let whole page blocks take the 16-byte stores instead of bytes.
 */
int sdv_quant_append_tiles(const void* v_new, const void* k_new, const int32_t* slot_mapping,
                           int32_t n_tokens, int32_t kv_heads, int32_t head_dim, int32_t group_size,
                           int32_t num_layers, int64_t in_layer_stride,
                           void* k_pages, void* v_pages, float* v_scales, int32_t num_blocks,
                           int64_t k_layer_stride, int64_t v_layer_stride, int64_t s_layer_stride,
                           int32_t scale_mode, const int32_t* tile_starts, int32_t n_tiles, void* stream);

/*
 * Slot mapping and tile table of whole prompts packed back to back, for sdv_quant_append_tiles:
 * lengths is a HOST array [batch], sequence b's rows follow those of the sequences before it, its
 * first token at position 0.  slots int32 [sum(lengths)]: the block-table slot of each row;
 * tile_starts int32 [sum(ceil(lengths/16)) + 1] or NULL: a tile per page block, the last entry the
 * row count.  Each length is at most 16 * max_blocks_per_seq and its block ids are valid (they are
 * not checked).  The lengths travel as kernel arguments: nothing is copied from the host.  No
 * counterpart in the reference.
 */
int sdv_varlen_slots(const int32_t* block_table, int32_t max_blocks_per_seq, const int32_t* lengths,
                     int32_t batch, int32_t* slots, int32_t* tile_starts, void* stream);

/* Bytes of workspace sdv_paged_attention needs for these sizes (0 on invalid sizes). */
size_t sdv_attention_workspace_size(int32_t num_layers, int32_t batch, int32_t q_heads,
                                    int32_t kv_heads, int32_t q_len, int32_t head_dim,
                                    int32_t max_seq_len);

/*
 * Zero the workspace's synchronisation area (its first SDV_SYNC_BYTES bytes) on `stream`.
 * Call it once after allocating a workspace and before its first sdv_paged_attention; every
 * call that completes normally leaves the statistics zero again (the partial slots keep the
 * last call's values, those of prefill rows among them; each item zeroes its own slot at the start
 * of the next single launch).  No counterpart in the reference (it has no workspace).
 *
 * The single-launch path exchanges (max, sum) statistics between workgroups through this
 * area as 64-bit (value, call tag) words; a reader takes a word only when it carries its own
 * call's tag, so a word an earlier call left behind is never read as current.  fp32 partials
 * travel as bits + 1 (0 = not yet written) in slots that their item zeroes, and waits for,
 * before it publishes its statistics.  Its waits are bounded (they only expire when the grid's workgroups cannot all
 * be resident at once: another process holding CUs, a CU mask): an expired wait makes the
 * outputs it could not complete NaN and counts in word 0 of the area.  A call recorded into
 * a HIP graph (its replays reuse one tag) that expires also sets word 1; while it is set,
 * every graph-recorded call writes NaN to all of its outputs and counts itself instead of
 * running, until sdv_attention_workspace_init clears the area.  Eager calls take a fresh tag
 * each and are unaffected.
 *
 * A NULL workspace names the current device's no-allocation scratch (the workspace of
 * sdv_paged_attention_noalloc; workspace_bytes is then ignored): this clears its failure
 * count and graph poison.  The first use of the scratch on a device must not be recorded into
 * a graph (SDV_ERR_UNSUPPORTED), as for sdv_paged_attention_noalloc.
 */
#define SDV_SYNC_BYTES 12583168
int sdv_attention_workspace_init(void* workspace, size_t workspace_bytes, void* stream);

/*
 * Read words 0 and 1 of a workspace's synchronisation area: `failures` = expired waits and
 * refused calls of the single-launch path since the last sdv_attention_workspace_init, and
 * `poisoned` != 0 when graph-recorded calls are refused (see above).  Synchronises `stream`
 * (a device-to-host copy); not for use while a graph is being recorded.  A NULL workspace
 * names the current device's no-allocation scratch (workspace_bytes ignored), whose words
 * count the failed and refused calls of sdv_paged_attention_noalloc.  No counterpart in the
 * reference.
 */
int sdv_attention_workspace_status(const void* workspace, size_t workspace_bytes, uint32_t* failures,
                                   uint32_t* poisoned, void* stream);

/*
 * Bound of every cross-workgroup wait of the single-launch path, in polls, for calls issued
 * after this one; 0 restores the default (2^20 polls; a poll waits for a device-scope load,
 * about a microsecond, so the default gives up after about a second).  A wait expires at its
 * `polls`-th unsuccessful poll: 1 gives up at the first entry not yet published.
 * UINT32_MAX makes every wait give up at its first check, whether or not the entries it waits
 * for are published.  For tests of the failure path: waits expire while every workgroup still
 * runs to its end.  No counterpart in the reference.
 */
int sdv_attention_set_wait_limit(uint32_t polls);

/*
 * Which path sdv_paged_attention takes for these sizes on the current device: the number of
 * workgroups of the single-launch kernel, or 0 when another path serves the call (several
 * query-row groups, or a problem the device cannot hold at once: the persistent per-group
 * kernel for 256 or more one-tile groups, the prefill kernels, else three launches).  A batch of 2..64 sequences
 * is taken to pass per-sequence lengths: its single launch uses every workgroup the device
 * holds and sizes each sequence's items from its length.  Queries the device's occupancy; no
 * launch.  No counterpart in the reference.
 */
int32_t sdv_attention_single_launch(int32_t num_layers, int32_t batch, int32_t q_heads, int32_t kv_heads,
                                    int32_t q_len, int32_t head_dim, int32_t max_seq_len);

/*
 * Kernels 2/3: paged GQA attention over BF16 K and FP8 V for q_len query rows per sequence
 * (q_len = 1: decode; q_len = k+1 = 5: speculative verify; any q_len >= 1 is accepted).
 *
 * q, out: bf16, per layer [batch][q_heads][q_len][head_dim] (q_token_major = 0, the
 *         reference op's (B,H,S,D)) or [batch][q_len][q_heads][head_dim] (q_token_major = 1,
 *         the projection layout); layers are batch*q_heads*q_len*head_dim elements apart.
 * seq_lens: int32 [batch] context length T_b including the q_len new tokens (q_len..max_seq_len;
 *           the kernels clamp T_b to [0, max_seq_len], so no value can read out of bounds), or
 *           NULL: every sequence has max_seq_len tokens (a call that a HIP graph records then
 *           needs no lengths in device memory).
 * block_table: int32 [batch][max_blocks_per_seq], max_blocks_per_seq >= ceil(max_seq_len/16);
 *           an entry outside [0, num_blocks) is never dereferenced: its tokens are masked.
 * Row i of the q_len-row block attends to keys j <= T_b - q_len + i (model_self.py:755-764).
 * Numerics follow the eager path's rounding points: BF16 q.k, BF16 (q.k)/sqrt(D), fp32
 * softmax normalised by the global max and sum, BF16 probabilities, BF16 dequantised V
 * (fp32(code) * scale rounded once), fp32 accumulation, BF16 output.
 * Alignment: q/out/k_pages/v_scales 16 B, v_pages 4 B, workspace 256 B.
 */
int sdv_paged_attention(const void* q, const void* k_pages, const void* v_pages,
                        const float* v_scales, int32_t num_blocks, int64_t k_layer_stride,
                        int64_t v_layer_stride, int64_t s_layer_stride,
                        const int32_t* block_table, int32_t max_blocks_per_seq,
                        const int32_t* seq_lens,
                        int32_t num_layers, int32_t batch, int32_t q_heads, int32_t kv_heads,
                        int32_t q_len, int32_t head_dim, int32_t max_seq_len,
                        int32_t q_token_major, void* workspace, size_t workspace_bytes,
                        void* out, void* stream);

/*
 * Profiling split of sdv_paged_attention (same arguments plus phase_mask): runs only the
 * selected launches -- SDV_PHASE_QK (scores + chunk statistics), SDV_PHASE_PV (global
 * softmax, FP8-V dequant, partial p.V), SDV_PHASE_REDUCE (sum partials, BF16 out).  Calling
 * it with SDV_PHASE_QK, then SDV_PHASE_PV, then SDV_PHASE_REDUCE on one stream with one
 * workspace computes exactly what one sdv_paged_attention call computes; a timer can record
 * events between the calls.  Batches of 1024 or more one-tile groups (layers x batch x
 * kv_heads with q_heads/kv_heads*q_len <= 16, max_seq_len <= 65536), which the persistent
 * per-group kernel serves in one launch, have no split: a mask other than SDV_PHASE_ALL
 * returns SDV_ERR_UNSUPPORTED.
 * No counterpart in the reference.
 */
#define SDV_PHASE_QK 1
#define SDV_PHASE_PV 2
#define SDV_PHASE_REDUCE 4
#define SDV_PHASE_ALL 7
int sdv_paged_attention_phases(const void* q, const void* k_pages, const void* v_pages,
                               const float* v_scales, int32_t num_blocks, int64_t k_layer_stride,
                               int64_t v_layer_stride, int64_t s_layer_stride,
                               const int32_t* block_table, int32_t max_blocks_per_seq,
                               const int32_t* seq_lens,
                               int32_t num_layers, int32_t batch, int32_t q_heads, int32_t kv_heads,
                               int32_t q_len, int32_t head_dim, int32_t max_seq_len,
                               int32_t q_token_major, void* workspace, size_t workspace_bytes,
                               void* out, void* stream, int32_t phase_mask);

/*
 * sdv_quant_append of the q_len new tokens of every sequence followed by sdv_paged_attention
 * over the context that includes them, in one call: the same bytes in the pages and the same
 * output as the two calls in that order.  k_new/v_new: bf16 [num_layers][batch*q_len][kv_heads]
 * [head_dim] (layers new_layer_stride elements apart), token b*q_len + i at position
 * seq_lens[b] - q_len + i, scale_mode as for sdv_quant_append.  slot_mapping: int32
 * [batch*q_len] (negative = skip), each the block-table slot of its position
 * (block_table[b][pos/16]*16 + pos%16: on the single launch the workgroup that streams a page
 * block writes its new tokens, so a slot elsewhere would race with another workgroup's reads),
 * or NULL: the slots are taken from the block table on the device (a call that a HIP graph
 * records then needs no host-built slot array).  On the single-launch path each workgroup writes the new tokens that
 * fall in its own page blocks before reading them, so the append costs no launch of its own;
 * otherwise the append kernel runs first on the same stream.  No counterpart in the reference:
 * its layer forward quantizes and concatenates V (model_self.py:697-706, 778-800) and then
 * attends (model_self.py:739-776) as separate steps; this is both, for the engine's per-layer
 * decode and verify calls.
 */
int sdv_paged_attention_append(const void* q, const void* k_pages, const void* v_pages,
                               const float* v_scales, int32_t num_blocks, int64_t k_layer_stride,
                               int64_t v_layer_stride, int64_t s_layer_stride,
                               const int32_t* block_table, int32_t max_blocks_per_seq,
                               const int32_t* seq_lens,
                               int32_t num_layers, int32_t batch, int32_t q_heads, int32_t kv_heads,
                               int32_t q_len, int32_t head_dim, int32_t max_seq_len,
                               int32_t q_token_major, void* workspace, size_t workspace_bytes,
                               void* out, const void* k_new, const void* v_new,
                               const int32_t* slot_mapping, int64_t new_layer_stride,
                               int32_t scale_mode, void* stream);

/*
 * sdv_paged_attention without a workspace argument and without allocating: the library's own
 * device-resident scratch array (one per GPU, SDV_NOALLOC_MAX_WORKSPACE bytes, held until the
 * process ends) serves as the workspace.  Arguments and results as sdv_paged_attention.  Calls
 * whose chosen path needs more than the array holds return SDV_ERR_WORKSPACE before launching
 * anything (the single launch -- decode and verify shapes that fit the device at once, also
 * when a multi-layer call runs it once per layer -- needs SDV_SYNC_BYTES; the per-group
 * kernel, the three-launch path and prefill rows need sdv_attention_workspace_size bytes).
 * Expired waits and graph poison are counted in the scratch: read and clear them with
 * sdv_attention_workspace_status / sdv_attention_workspace_init and a NULL workspace.  Every call on one GPU
 * shares that GPU's array: calls that overlap on one GPU (other streams, other threads) race,
 * so order them on one stream.  The first call on a device takes the array's address and
 * zeroes its synchronisation area, waiting for that to finish, so it must not be recorded
 * into a graph (SDV_ERR_UNSUPPORTED); later calls may be.  No counterpart in the reference:
 * for callers that cannot allocate (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).
 */
#define SDV_NOALLOC_MAX_WORKSPACE 33554432
int sdv_paged_attention_noalloc(const void* q, const void* k_pages, const void* v_pages,
                                const float* v_scales, int32_t num_blocks, int64_t k_layer_stride,
                                int64_t v_layer_stride, int64_t s_layer_stride,
                                const int32_t* block_table, int32_t max_blocks_per_seq,
                                const int32_t* seq_lens,
                                int32_t num_layers, int32_t batch, int32_t q_heads, int32_t kv_heads,
                                int32_t q_len, int32_t head_dim, int32_t max_seq_len,
                                int32_t q_token_major, void* out, void* stream);

/*
 * A contiguous v_fp8 cache into pages: k bf16 [batch][kv_heads][seq_len][head_dim], v_codes E4M3FN of
 * the same shape, v_scales fp32 [batch][kv_heads][seq_len].  k_pages / v_pages / page_scales hold
 * batch * ceil(seq_len/16) pages in the layout above, block b*ceil(seq_len/16) + j being tokens
 * 16j.. of sequence b, and block_table int32 [batch][ceil(seq_len/16)] receives those block ids.
 * Tokens past seq_len in a last block get K 0, code 0 and scale 1.  Alignment: k/k_pages 16 B,
 * the rest 4 B.  For callers that hold the reference's cache tensors (model_self.py:778-800) and
 * call its op over them (specdec/kernels/ops.py:67-76); no counterpart of its own.
 */
int sdv_pack_contiguous(const void* k, const void* v_codes, const float* v_scales, int32_t batch,
                        int32_t kv_heads, int32_t seq_len, int32_t head_dim, void* k_pages, void* v_pages,
                        float* page_scales, int32_t* block_table, void* stream);

/* Elementwise fp32 -> E4M3FN (RNE, NaN beyond 464 / for Inf and NaN), device buffers. */
int sdv_fp8_encode(const float* in, uint8_t* out, int64_t n, void* stream);

/* Static, thread-safe description of a status code. */
const char* sdv_status_string(int status);

/* SDV_ABI_VERSION of the built library. */
int sdv_abi_version(void);

#ifdef __cplusplus
}
#endif

#endif /* SDV_H_ */
