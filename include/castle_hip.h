/* C ABI of libcastle_hip.so: the CASTLE (causal attention with lookahead keys) hot path
 * for AMD MI355X (gfx950).  Plain pointers and sizes only; every tensor pointer is DEVICE
 * memory, every call enqueues work on the HIP stream handed in (a hipStream_t passed as
 * void*; NULL = the default stream) and returns without synchronising.
 *
 * Return value of the int entry points: 0 on success, negative on error
 * (castle_error_string() gives the text).  Inputs are never modified.
 *
 * Reference interfaces replaced (paths inside lucidrains/lookahead-keys-attention):
 *   castle_fwd          lookahead_keys_attention_triton.py:417-506  CastleAttentionFunction.forward
 *                       (= castle_attention_triton, :605, called at lookahead_keys_attention.py:122);
 *                       math of lookahead_keys_attention.py:132-164
 *   castle_bwd          lookahead_keys_attention_triton.py:508-602  CastleAttentionFunction.backward
 *   castle_decode_step  lookahead_keys_attention.py:166-203         the seq_len == 1 branch of Castle.forward
 *   castle_decode_step_device_count   the same step, row count in device memory (graph replay)
 */
#ifndef CASTLE_HIP_H_
#define CASTLE_HIP_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define CASTLE_ABI_VERSION 5

/* element types of the tensors (accumulation is always fp32) */
#define CASTLE_F32 0
#define CASTLE_BF16 1
#define CASTLE_F16 2

/* flags of castle_fwd / castle_bwd.  By default bf16 tensors are converted to fp16 when they are
 * loaded (exact for |x| < 65504) and every operand the kernels produce internally is fp16:
 * same MFMA rate, 3 more mantissa bits, which keeps the gradients of long sequences inside the
 * bf16 tolerance.  CASTLE_FLAG_BF16_OPERANDS keeps bf16 MFMA operands instead (full bf16 range).
 * castle_bwd must get the same flags as the castle_fwd call whose workspace it reads.
 * CASTLE_FLAG_ROTARY: the kernels rotate qc, kc, qu, ku, vu (not vc) by their row position
 * (rotary position embedding over interleaved pairs, base 10000: what Castle(rotary_emb=True) does
 * before its core, lookahead_keys_attention.py:106-112); castle_bwd then returns the gradients with
 * respect to the un-rotated operands; castle_decode_step rotates the new token by position t and
 * appends the rotated qu, kc rows.  The final lookahead keys U are those of the rotated operands. */
#define CASTLE_FLAG_BF16_OPERANDS 1
#define CASTLE_FLAG_ROTARY 2
/* castle_bwd / castle_bwd_workspace_bytes only: do not hand dS / dSu tiles from the first backward
 * kernel to the second (2 * B * H * Lp * Lp elements of workspace); the second kernel recomputes
 * the score chain instead.  Slower, for callers short of memory. */
#define CASTLE_FLAG_RECOMPUTE_SCORES 4
/* castle_bwd / castle_bwd_workspace_bytes only: the forward state buffer was not kept; castle_bwd
 * runs the forward scan again (from the operand copies in the forward workspace) into its own
 * workspace before anything else.  What a forward call must keep for its backward is then O(L d). */
#define CASTLE_FLAG_RECOMPUTE_STATE 8

/* castle_fwd (its U output), castle_decode_step*, castle_decode_flush; bf16 tensors only (else
 * CASTLE_ERR_DTYPE); castle_bwd ignores it.  The lookahead-key buffer U is held in a half-precision
 * cache format instead of bf16: each 2-byte element is the IEEE fp16 value of U * 2^-6, saturated at
 * +-65504 (so |U| up to 4.2e6 is held, with 11 significant bits down to |U| = 2^-8 and an absolute
 * step of 4e-6 below).  The reference's step re-rounds the whole of U to the module type at every
 * token (lookahead_keys_attention.py:183); in bf16 those roundings add up to a few per cent over some
 * hundred steps, in this format to an eighth of that, for the same bytes.  Every entry point that
 * touches one U buffer must get the same setting; a reader converts with  U = 64 * (fp16 bits). */
#define CASTLE_FLAG_U_HALF 16
/* Cached step only: the caches that are read until this one's next step exceed the last-level cache, so its rows are not
 * kept there (set by itself for a host-side row count whose cache alone is that large).  Results are the same. */
#define CASTLE_FLAG_READ_ONCE 32
/* castle_fwd: the CASTLE_AMAX_PARTIALS floats at byte 256 of the workspace hold partial maxima of |vu| and the word at its start
 * is 0; castle_bwd: the same place of the backward workspace holds partial maxima of |dout| (castle_gemm leaves them
 * there): a launch and a pass less.  Ignored for fp32. */
#define CASTLE_FLAG_AMAX_READY 64
/* castle_decode_layer_once in one launch, for tests of its waits: the jobs in reverse order and next to no patience, so that nearly all are done by
 * workgroups that had waited for them; with _GIVE_UP these leave instead, and what they were to do is NaN as described there. */
#define CASTLE_FLAG_STEP_TAKE_OVER 128
#define CASTLE_FLAG_STEP_GIVE_UP 256
/* castle_fwd: no castle_bwd follows.  What lies in the workspace behind the status word and in the state is then undefined, and short sequences (up to
 * 128 rows of 16-bit types, as long as there are few of them) take one launch, whose roundings fall in other places: out and U are as exact as without the
 * flag, not the same bits.  castle_bwd refuses it (CASTLE_ERR_ARG). */
#define CASTLE_FLAG_FORWARD_ONLY 512
#define CASTLE_AMAX_PARTIALS 256
#define CASTLE_AMAX_OFFSET 256

/* error codes */
#define CASTLE_OK 0
#define CASTLE_ERR_DTYPE (-1)      /* unknown element type */
#define CASTLE_ERR_SHAPE (-2)      /* unsupported head dim / size, or (dtype, d) does not fit the LDS */
#define CASTLE_ERR_LAUNCH (-3)     /* HIP reported a launch / configuration error */
#define CASTLE_ERR_WORKSPACE (-4)  /* workspace NULL, misaligned or too small */
#define CASTLE_ERR_ARG (-5)        /* NULL pointer, misaligned pointer or stride */
#define CASTLE_ERR_SCRATCH (-6)    /* castle_decode_step_static: partial results exceed the static scratch */

/* A (B, H, L, d) tensor view: element strides for b, h and l; the d axis has stride 1.
 * ptr must be 16-byte aligned and every stride a multiple of 16 bytes / sizeof(element). */
typedef struct castle_view4 {
  void* ptr;
  int64_t stride_b;
  int64_t stride_h;
  int64_t stride_l;
} castle_view4;

/* Deferred write-back of the lookahead keys in the cached step (optional argument of the three
 * castle_decode_step* entry points; NULL = U is written by every step, as the reference's step does,
 * lookahead_keys_attention.py:183).  With it the U rows are written on every 4th step only (the steps
 * whose row count t has (t + 1) % 4 == 0).  In between, the vu rows of the up to 3 tokens not yet
 * folded into the stored U ("pending") sit in `vu_ring`, a (B, H, 4, d) buffer in the element type
 * (token j in row j % 4, written by the step that appends j), and the gate each cached row k got from
 * pending token j in `gates`, a (B, H, capacity, 4) fp32 array ([k][j % 4]; stride_l is not used, the
 * rows are 4 floats apart).  Every step adds gate * vu of the pending tokens in fp32: a tenth less
 * HBM traffic per step and a quarter of the roundings of a 16-bit U.  `base`: every U row already
 * holds all sources below `base` (the prefill length, or the row count at the last castle_decode_flush);
 * the sources pending at row count t are max(base, t - t % 4) .. t - 1.  `base_device`, if not NULL,
 * is read by the kernels instead (graph replay).  The stored U is complete whenever nothing is
 * pending; castle_decode_flush makes it so at any other time. */
typedef struct castle_deferred {
  castle_view4 vu_ring;
  castle_view4 gates;
  int32_t base;
  const int32_t* base_device;
} castle_deferred;

int castle_abi_version(void);
const char* castle_error_string(int code);

/* Bytes of the two device buffers castle_fwd needs.  `workspace` (castle_fwd_workspace_bytes,
 * grows like L d): the forward pass leaves there what the backward pass reads again (a header with
 * the range-control scalars and a status word, operand copies in the compute type, per-block T
 * tiles, log-sum-exp); keep it alive and unmodified until castle_bwd has run.  `state`
 * (castle_fwd_state_bytes, grows like L^2 d / 128): the snapshots of the lookahead state, scratch
 * for a forward pass alone; castle_bwd reads them too, unless it is told to recompute them
 * (CASTLE_FLAG_RECOMPUTE_STATE), in which case the buffer can be dropped right after castle_fwd.
 * < 0 on error.  After the stream has finished castle_fwd, the int32 at workspace + 0 is a status
 * word: bit 0 = an input element beyond the fp16 range was clamped (bf16 tensors, fp16 operands),
 * bit 1 = an entry of T' = s qc.vu was. */
int64_t castle_fwd_workspace_bytes(int B, int H, int L, int d, int dtype);
int64_t castle_fwd_state_bytes(int B, int H, int L, int d, int dtype);

/* Parallel forward.  qc,kc,vc,qu,ku,vu: (B,H,L,d), unscaled, as handed to
 * castle_attention_triton (lookahead_keys_attention.py:122).  out: (B,H,L,d) view that is
 * written (any strides, e.g. those of a (B,L,H,d) buffer).  U: optional (NULL, or a view
 * with ptr == NULL, to skip) final lookahead keys for the decode cache
 * (lookahead_keys_attention.py:161-164).  d in {16,32,64,128}; fp32 needs d <= 64.
 * flags: any of CASTLE_FLAG_BF16_OPERANDS, CASTLE_FLAG_ROTARY, CASTLE_FLAG_U_HALF (format of U), CASTLE_FLAG_FORWARD_ONLY. */
int castle_fwd(const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
               const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
               int B, int H, int L, int d, int dtype, float scale, int flags,
               const castle_view4* out, const castle_view4* U,
               void* workspace, int64_t workspace_bytes, void* state, int64_t state_bytes, void* stream);

/* Bytes of extra device workspace castle_bwd needs: reverse state snapshots, delta, a copy of dout in
 * the compute type and, for the 16-bit element types, the dS / dSu score-gradient tiles its first
 * kernel hands to its second (2 * B * H * Lp * Lp elements, Lp = L rounded up to 128; left out, and
 * the score chain recomputed instead, under CASTLE_FLAG_RECOMPUTE_SCORES or when they would exceed
 * 40 GiB, or the byte count found in the environment variable CASTLE_MAX_SCORE_TILE_BYTES when
 * the library first needed it).  `flags`: those the castle_bwd call will get. */
int64_t castle_bwd_workspace_bytes(int B, int H, int L, int d, int dtype, int flags);

/* Parallel backward.  Same operands as castle_fwd plus the forward output `out`, the
 * upstream gradient `dout`, the forward workspace as castle_fwd left it and its state buffer
 * (NULL with CASTLE_FLAG_RECOMPUTE_STATE).  Writes the six
 * gradients (all (B,H,L,d) views; every element is written, nothing is accumulated).
 * U carries no gradient (lookahead_keys_attention_triton.py:513-515).  d in {16,32,64}, and 128 for
 * the 16-bit element types (there every kernel runs twice, each pass keeping half of the outputs). */
int castle_bwd(const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
               const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
               const castle_view4* out, const castle_view4* dout,
               int B, int H, int L, int d, int dtype, float scale, int flags,
               const castle_view4* dqc, const castle_view4* dkc, const castle_view4* dvc,
               const castle_view4* dqu, const castle_view4* dku, const castle_view4* dvu,
               const void* fwd_workspace, int64_t fwd_workspace_bytes,
               const void* fwd_state, int64_t fwd_state_bytes,
               void* bwd_workspace, int64_t bwd_workspace_bytes, void* stream);

/* Bytes of device workspace castle_decode_step needs for a cache of up to t_max rows. */
int64_t castle_decode_workspace_bytes(int B, int H, int d, int t_max);

/* One cached decode step (lookahead_keys_attention.py:166-203), in place.
 * U, qu_cache, kc_cache, vc_cache: (B,H,capacity,d) buffers holding t valid rows;
 * t >= capacity is rejected (CASTLE_ERR_SHAPE) because row t is written.  The call updates U rows 0..t-1 in place (U_k += sigmoid(s qu_k.ku) vu),
 * writes row t of all four (U_t = 0, qu, kc, vc of the new token) and writes
 * out (B,H,1,d) = softmax_k(s qc.kc_k - silu(s qc.U_k)) vc_k over k = 0..t.
 * qc..vu: the new token's (B,H,1,d) operands (stride_l unused).  After the call the cache
 * holds t+1 rows.  d in {16,32,64,128}.  flags: any of CASTLE_FLAG_ROTARY, CASTLE_FLAG_U_HALF. */
int castle_decode_step(const castle_view4* U, const castle_view4* qu_cache,
                       const castle_view4* kc_cache, const castle_view4* vc_cache, int t, int capacity,
                       const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                       const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                       int B, int H, int d, int dtype, float scale, int flags,
                       const castle_view4* out, const castle_deferred* deferred,
                       void* workspace, int64_t workspace_bytes, void* stream);

/* Folds the pending sources into the stored lookahead keys (see castle_deferred): afterwards the U
 * rows 0 .. t-1 are what a step-by-step update would have left.  POSTCONDITION the caller must
 * establish before the next step or flush on this cache: `base` (and *base_device, when the steps read
 * the base from device memory) = t.  The call does not write either; a second flush, or a step, with
 * the old base adds the same gate * vu terms again.  `gates` must hold `capacity` rows of 4 floats
 * (not checked).  flags: 0 or CASTLE_FLAG_U_HALF. */
int castle_decode_flush(const castle_view4* U, const castle_view4* qu_cache, int t, const castle_deferred* deferred,
                        int B, int H, int d, int dtype, float scale, int flags, void* stream);

/* The same step with the row count t read by the kernels from device memory (*t_device, an int32
 * the caller keeps and advances), so that the enqueued work does not depend on t: one captured HIP
 * graph of a whole model step can be replayed for every token.  `capacity` = rows of the cache
 * buffers; the work split is sized for it, and a step found at *t_device >= capacity (or < 0)
 * writes nothing.  No counterpart in the reference (its step takes t from the tensor shapes,
 * lookahead_keys_attention.py:166-203); meant for callers that replay a captured step.  The call
 * itself records only kernel launches on `stream` (no memset, no allocation, no synchronisation). */
int castle_decode_step_device_count(const castle_view4* U, const castle_view4* qu_cache,
                                    const castle_view4* kc_cache, const castle_view4* vc_cache,
                                    const int32_t* t_device, int capacity,
                                    const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                                    const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                                    int B, int H, int d, int dtype, float scale, int flags,
                                    const castle_view4* out, const castle_deferred* deferred,
                                    void* workspace, int64_t workspace_bytes, void* stream);

/* The cached step for callers that cannot allocate or bring a workspace (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  No counterpart in the
 * reference.  Same kernels and results as castle_decode_step (t_device == NULL: row count t from
 * the host) or castle_decode_step_device_count (t_device != NULL: t is ignored), but the partial
 * results of the split pass live in a 4 MiB array that is part of the library's device code, one
 * copy per GPU, held until the process ends.  The call allocates nothing and clears nothing (every
 * partial that is read was written by the same call).  B * H * splits * (d + 2) * 4 bytes must fit
 * the array (splits <= 64, about 640 / (B*H) for small batches: e.g. B*H up to 8065 heads at
 * d = 128), else CASTLE_ERR_SCRATCH.  All calls on one GPU share that GPU's array: calls that
 * overlap on one GPU (different streams, or graph replays running side by side) race.  The first
 * call on a device looks the array's address up (hipGetSymbolAddress); make that call outside
 * stream capture. */
int castle_decode_step_static(const castle_view4* U, const castle_view4* qu_cache,
                              const castle_view4* kc_cache, const castle_view4* vc_cache,
                              int t, const int32_t* t_device, int capacity,
                              const castle_view4* qc, const castle_view4* kc, const castle_view4* vc,
                              const castle_view4* qu, const castle_view4* ku, const castle_view4* vu,
                              int B, int H, int d, int dtype, float scale, int flags,
                              const castle_view4* out, const castle_deferred* deferred, void* stream);

/* A whole layer for one token per sequence: y = residual + core(norm(x) w_in^T) w_out^T, the cached step with
 * the norm and the projections around it (lookahead_keys_attention.py:95-99, 166-203, 209 with seq_len == 1) in
 * three launches behind one call.
 * x, y: B rows of `dim` elements; w_in (6 H d, dim), w_out (dim, H d), both row-major in the tensor type, `proj` a
 * B x 6 H d scratch in the tensor type (order qu, ku, vu, qc, kc, vc).  norm_weight (`dim` elements), residual
 * (B rows; may alias y) and t_device may be NULL.  dim % 8 == 0 (4 for fp32); x, w_in, w_out, proj and norm_weight
 * 16-byte aligned with leading dimensions of whole 16-byte pieces.  The other arguments, the workspace among
 * them, are those of castle_decode_step / castle_decode_step_device_count.  Meant for B up to a few dozen. */
int castle_decode_layer(const castle_view4* U, const castle_view4* qu_cache,
                        const castle_view4* kc_cache, const castle_view4* vc_cache,
                        int t, const int32_t* t_device, int capacity,
                        const void* x, int64_t ldx, int dim, const void* norm_weight, float eps,
                        const void* w_in, int64_t ldw_in, const void* w_out, int64_t ldw_out,
                        const void* residual, int64_t ldr, void* y, int64_t ldy, void* proj,
                        int B, int H, int d, int dtype, float scale, int flags, const castle_deferred* deferred,
                        void* workspace, int64_t workspace_bytes, void* stream);

/* The same in one launch where the host's work for three is what a step waits for: a few sequences, the row count from the host, up to 10 MB
 * of cached rows, caches of equal strides, and the sizes for which castle_decode_layer_once_ok says 1; otherwise in three.  `control`:
 * castle_decode_layer_control_bytes bytes, 256-byte aligned, zeroed once before the first such call and then left to these calls (NULL: three
 * launches); calls that share it must not overlap, as they must not on one cache.  Workgroups of the launch wait for each other's results for a bounded
 * time, then do themselves what no other has started: the waits end whatever else runs on the GPU.  Should results not come in some tens of seconds
 * all the same, what depends on them is NaN: in y, and in a row of vc_cache of every head whose step is not complete. */
int castle_decode_layer_once_ok(int B, int H, int d, int dtype, int t, int dim);
int64_t castle_decode_layer_control_bytes(int B, int H, int d, int dtype);
int castle_decode_layer_once(const castle_view4* U, const castle_view4* qu_cache,
                             const castle_view4* kc_cache, const castle_view4* vc_cache,
                             int t, const int32_t* t_device, int capacity,
                             const void* x, int64_t ldx, int dim, const void* norm_weight, float eps,
                             const void* w_in, int64_t ldw_in, const void* w_out, int64_t ldw_out,
                             const void* residual, int64_t ldr, void* y, int64_t ldy, void* proj,
                             int B, int H, int d, int dtype, float scale, int flags, const castle_deferred* deferred,
                             void* workspace, int64_t workspace_bytes, void* control, int64_t control_bytes, void* stream);

/* Rotary position embedding of one tensor, out of place: out[b,h,l,:] = R(first_position + l) x[b,h,l,:]
 * (the rotation CASTLE_FLAG_ROTARY applies inside the kernels; lookahead_keys_attention.py:112).  Used to
 * fill the qu / kc rows of a decode cache after a rotary prefill. */
int castle_rope(const castle_view4* x, const castle_view4* out, int B, int H, int L, int d, int dtype,
                int first_position, void* stream);

/* The first L rows of a decode cache after a parallel pass (lookahead_keys_attention.py:26, 205-214): qu, kc and vc copied
 * into its buffers, qu and kc rotated by their position under CASTLE_FLAG_ROTARY. */
int castle_cache_rows(const castle_view4* qu, const castle_view4* kc, const castle_view4* vc, const castle_view4* qu_cache,
                      const castle_view4* kc_cache, const castle_view4* vc_cache, int B, int H, int L, int d, int dtype, int flags, void* stream);

/* y[M, N] = x[M, K] w[N, K]^T, all three row-major in the 16-bit element type `dtype` (leading
 * dimensions ldx, ldw, ldy in elements; fp32 accumulation), for the few rows of a decode step: the
 * fused projection and the output projection around the cached step, which the reference runs as
 * nn.Linear on a (B, 1, dim) tensor (lookahead_keys_attention.py:99 and :209 with seq_len == 1).
 * Meant for M up to a few dozen rows (one workgroup per 16-column slice of the output, K split over its
 * waves); any M works.  K % 8 == 0, N % 2 == 0, x / w 16-byte aligned with ldx, ldw % 8 == 0. */
int castle_small_linear(const void* x, const void* w, void* y, int M, int N, int K,
                        int64_t ldx, int64_t ldw, int64_t ldy, int dtype, void* stream);

/* The same product with the per-row work of a transformer block's token step folded in (each saves a
 * launch and a pass over the activations; no counterpart in the reference, whose callers run these as
 * separate modules: train_triton.py:102-107, 161-165 around lookahead_keys_attention.py:95, 99, 209):
 *   norm_weight != NULL: RMS normalisation of the x rows in front, y = ((x / sqrt(mean(x^2) + eps)) * norm_weight) w^T
 *                        (nn.RMSNorm; K elements, 16-byte aligned);
 *   activation:          CASTLE_ACT_GELU applies the erf form of GELU to the product;
 *   residual != NULL:    a (M, N) tensor with leading dimension ldr added last (may alias y).
 * Order: normalise, multiply, activate, add. */
#define CASTLE_ACT_NONE 0
#define CASTLE_ACT_GELU 1
int castle_small_linear_fused(const void* x, const void* w, void* y, int M, int N, int K,
                              int64_t ldx, int64_t ldw, int64_t ldy, int dtype,
                              const void* norm_weight, float eps, int activation,
                              const void* residual, int64_t ldr, void* stream);

/* One token per row from its logits (train_triton.py:56-71): the k largest of `vocabulary` logits are kept (of
 * equal ones the lowest indices), and the arg-max of  logit * inv_temperature - log(-log(uniform))  over them is
 * written (both logarithms' arguments at least 1e-20); uniform: (rows, vocabulary) contiguous, or NULL for the arg-max of
 * the logits.  token: row r goes to token[r * token_ld]; token_copy: NULL, or a second copy, contiguous. */
int castle_sample(const void* logits, int64_t ld, const float* uniform, int rows, int vocabulary, int k, float inv_temperature,
                  int64_t* token, int64_t token_ld, int64_t* token_copy, int dtype, void* stream);

/* y[m] = table[index[m]], m < n: rows of `width` elements (whole 16-byte pieces), y contiguous.  An index outside
 * 0 .. table_rows - 1 gives a row of zeros.  The token embedding of a step (train_triton.py:86). */
int castle_gather_rows(const void* table, int64_t table_rows, int64_t ld, int width, const int64_t* index, int n, void* y, int dtype, void* stream);

/* The work between the products of a transformer block (train_triton.py:102-107, 150-171; lookahead_keys_attention.py:95).
 * All tensors: rows of `width` (or `classes`) elements in the type `dtype`, contiguous, a whole number of 16-byte pieces
 * (at most 512 for the norm and the embedding), 16-byte aligned.
 *
 * castle_rms_norm: h = (s / sqrt(mean(s^2) + eps)) * weight with s = x, or s = x + delta (rounded to the type and written
 * to `sum`) when delta != NULL.  rstd: NULL, or one float per row for the backward pass. */
int castle_rms_norm(const void* x, const void* delta, const void* weight, void* sum, void* h, float* rstd, int64_t rows, int width, float eps,
                    int dtype, void* stream);
/* A sum of partial results that a call has left, for castle_sums (up to CASTLE_MAX_SUMS of them, all of one type, in one launch): out[n] = sum over `parts` rows of
 * part[parts][n]; columns: rather down the columns of a few, else n is a multiple of 8.  parts = 0: there is nothing to sum.  The workspace that `part` lies in is kept until then. */
#define CASTLE_MAX_SUMS 4
typedef struct castle_sum {
  const float* part;
  int64_t n;
  void* out;
  int32_t parts, columns;
} castle_sum;
int castle_sums(const castle_sum* sums, int count, int dtype, void* stream);

/* dx = dres + d(norm)/dx dh (dres may be NULL), dweight = sum over rows; either result may be NULL.  The workspace is
 * only needed for dweight.  _parts: the sum over rows is left to castle_sums. */
int64_t castle_rms_norm_bwd_workspace_bytes(int64_t rows, int width, int dtype);
int castle_rms_norm_bwd(const void* dh, const void* x, const void* weight, const float* rstd, const void* dres, void* dx, void* dweight,
                        int64_t rows, int width, int dtype, void* workspace, int64_t workspace_bytes, void* stream);
int castle_rms_norm_bwd_parts(const void* dh, const void* x, const void* weight, const float* rstd, const void* dres, void* dx, void* dweight, castle_sum* dw_sum,
                              int64_t rows, int width, int dtype, void* workspace, int64_t workspace_bytes, void* stream);

/* c[M, N] = the product of two matrices over K, in the type `dtype` with fp32 sums: the projections of a layer and their
 * gradients over hundreds to thousands of rows (nn.Linear at lookahead_keys_attention.py:75, 80, 99, 209).  An operand
 * is contraction-contiguous (a: M rows of K, b: N rows of K) or, with its flag set, free-contiguous (K rows of M or N); a
 * free-contiguous a needs a free-contiguous b.  Rows are whole 16-byte pieces, as are leading dimensions and N.
 * epilogue: CASTLE_GEMM_GELU also writes gelu(c) (erf form) to aux, CASTLE_GEMM_GELU_SLOPE multiplies the product by the
 * derivative of gelu at aux; aux has c's shape and leading dimension.  A workspace of castle_gemm_workspace_bytes
 * (0 when the contraction is not split; then ldc may exceed N).  An operand of `rows` stored rows whose elements are further
 * than 2^31 from its start is refused (CASTLE_ERR_SHAPE): castle_gemm_operand_ok, 1 or 0.  fp32: an element goes to the 16-bit matrix instructions as three
 * bf16 numbers, which hold all of it; where sums are below 2^-90, infinite or NaN the fp32 instruction forms them. */
#define CASTLE_GEMM_PLAIN 0
#define CASTLE_GEMM_GELU 1
#define CASTLE_GEMM_GELU_SLOPE 2
int castle_gemm_operand_ok(int64_t rows, int64_t ld);
int64_t castle_gemm_workspace_bytes(int M, int N, int K, int dtype, int epilogue);
/* What castle_gemm makes of a product, for tests and measurements: rows and columns of a workgroup's tile, ranges of the contraction, groups of four waves
 * that share a tile of 64 x 64 (fp32: of 32 x 32 or 64 x 64; 1 where fewer than four waves have one). */
int castle_gemm_plan(int M, int N, int K, int dtype, int epilogue, int* rows, int* columns, int* ranges, int* groups);
/* amax != NULL: CASTLE_AMAX_PARTIALS partial maxima of |c| over `columns` columns from `column` on (whole 16-byte pieces), for
 * CASTLE_FLAG_AMAX_READY; status, if not NULL, is set to 0.  Only where castle_gemm_amax_ok says so. */
typedef struct castle_amax {
  float* partials;
  int* status;
  int32_t column, columns;
} castle_amax;
int castle_gemm_amax_ok(int M, int N, int K, int dtype, int column, int columns);
int castle_gemm(const void* a, int64_t lda, int a_free_contiguous, const void* b, int64_t ldb, int b_free_contiguous, void* c, int64_t ldc,
                int M, int N, int K, int dtype, int epilogue, void* aux, const castle_amax* amax, void* workspace, int64_t workspace_bytes, void* stream);

/* Both gradients of a projection y = x w^T in one launch: dw (N, K) = dy^T x and dx (R, K) = dy w, for dy (R, N), x (R, K) and w (N, K) with leading dimensions in
 * elements; dw and dx are contiguous.  epilogue (CASTLE_GEMM_PLAIN or CASTLE_GEMM_GELU_SLOPE), aux and amax are those of castle_gemm for dx.  Only where the workspace's
 * size is not negative: elsewhere two launches are ahead (N and K are multiples of 8).  dw_sum != NULL: a dw that is formed in ranges is left to castle_sums.  _plan: for tests and measurements, a workgroup's tile and waves and the
 * ranges of the two contractions. */
int64_t castle_projection_grads_workspace_bytes(int R, int N, int K, int dtype, int epilogue, int with_amax);
int castle_projection_grads_plan(int R, int N, int K, int dtype, int epilogue, int with_amax, int* tile, int* waves, int* dw_ranges, int* dx_ranges);
int castle_projection_grads(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, const void* w, int64_t ld_w, void* dw, void* dx, int R, int N, int K,
                            int dtype, int epilogue, const void* aux, const castle_amax* amax, castle_sum* dw_sum, void* workspace, int64_t workspace_bytes, void* stream);

/* The same of normalised rows, castle_rms_norm without a summand and castle_gemm of two contraction-contiguous operands in one launch: c
 * = (a / sqrt(mean(a^2) + eps) * weight, rounded to the type) b^T.  h (M rows of K) and rstd (M floats) keep the normalised rows and their
 * factors, or are NULL; rstd needs h.  For few rows: only where castle_gemm_norm_ok says so. */
typedef struct castle_gemm_norm {
  const void* weight;
  float eps;
  void* h;
  float* rstd;
} castle_gemm_norm;
int castle_gemm_norm_ok(int M, int N, int K, int dtype);
int castle_gemm_of_norm(const void* a, int64_t lda, const castle_gemm_norm* norm, const void* b, int64_t ldb, void* c, int64_t ldc, int M, int N, int K,
                        int dtype, const castle_amax* amax, void* stream);

/* out[i] = sum over p < parts of part[p * n + i], n % 8 == 0: partial products of a weight gradient. */
int castle_sum_parts(const float* part, int parts, int64_t n, void* out, int dtype, void* stream);

/* Mean cross entropy (train_triton.py:166-171).  Row r of the logits belongs to the class target[(r / target_n) * target_ld +
 * r % target_n]; rows of class -100 do not count, a class outside 0 .. classes - 1 makes the loss and the row's gradient NaN.  loss: one element
 * of the type; lse: one float per row and inv_count: one float, both kept for the backward pass, which multiplies by
 * the one element of `grad`. */
#define CASTLE_CROSS_ENTROPY_WORKSPACE 8192
int castle_cross_entropy(const void* logits, const int64_t* target, int64_t target_n, int64_t target_ld, int64_t rows, int classes, void* loss,
                         float* lse, float* inv_count, int dtype, void* workspace, int64_t workspace_bytes, void* stream);
int castle_cross_entropy_bwd(const void* logits, const int64_t* target, int64_t target_n, int64_t target_ld, int64_t rows, int classes,
                             const float* lse, const float* inv_count, const void* grad, void* dlogits, int dtype, void* stream);

/* dweight[v] = sum of the dy rows whose index is v (indices addressed like `target` above), summed in a fixed order.
 * For small vocabularies: rows * vocabulary at most 2^26, else castle_embedding_grad_workspace_bytes returns
 * CASTLE_ERR_SHAPE. */
int64_t castle_embedding_grad_workspace_bytes(int64_t rows, int vocabulary, int width, int dtype);
int castle_embedding_grad(const void* dy, const int64_t* index, int64_t index_n, int64_t index_ld, int64_t rows, int vocabulary, int width,
                          void* dweight, int dtype, void* workspace, int64_t workspace_bytes, void* stream);

/* Per-kernel timing (no counterpart in the reference; for benchmarks).  While enabled, every
 * kernel launched by the entry points above is bracketed by a HIP event pair on its stream.
 * castle_profile_enable(on) also discards pending records.  castle_profile_read waits for the
 * recorded kernels, writes up to max_records (slot, milliseconds) pairs in launch order, clears
 * the records and returns their number (< 0 on error).  Slots: 0 operand copies (with the pass for max|vu|), 1 forward scan (with the T' blocks),
 * 2 forward attention, 3 delta, 4 backward key-stationary, 5 backward query-stationary,
 * 6 decode stream, 7 decode finish. */
int castle_profile_enable(int on);
int castle_profile_read(int* slots, float* ms, int max_records);

#ifdef __cplusplus
}
#endif
#endif /* CASTLE_HIP_H_ */
