/* include/ntk_engine.h -- the engine-private part of libntransformer_hip.so's C ABI (round 6: split off include/ntk.h, which keeps the
 * reference's surface -- the 17 launchers of reference src/cuda/kernels.h:14-71 and the nt_cuda_* runtime of src/core/device.h:79-88).
 *
 * What is here has NO counterpart in the reference's headers: fused forms of launcher sequences (each cites the sequence it computes), the
 * engine-owned repack and the matrix-core GEMV that reads it, the prompt projections on the matrix cores, the split-KV decode attention,
 * device-side embedding / sampling, the tensor-parallel exchange, and parity / measurement instrumentation (ntk_debug_*).  Same conventions
 * as ntk.h: plain pointers and sizes, stream ordered, no allocation, NTK_OK or a negative NTK_E_* code.  Used by csrc/engine/ (nt_engine_*),
 * integration/nt_hip_repack.h, the tests and bench.py.
 */
#ifndef NTK_ENGINE_H
#define NTK_ENGINE_H

#include "ntk.h"

#if defined(__GNUC__)
#pragma GCC visibility push(default)
#endif
#ifdef __cplusplus
extern "C" {
#endif

/* launch_rope + launch_copy_to_kv_cache of a prompt as ONE launch (the two calls back to back in reference attention.cpp:164-184): q rotated in
 * place, the rotated k and v converted to F16 (RNE) into the caches at start_pos; k and v are only read.  Identical q and cache rows.  head_dim <= 256. */
int ntk_rope_kv_store(float* q, const float* k, const float* v, const int* positions, int seq_len, int n_heads, int n_kv_heads, int head_dim,
                      float theta_base, float freq_scale, int interleaved, void* k_cache, void* v_cache, int start_pos, int max_seq, void* stream);
/* ... with q, k and v as the partial sums of their projections (sums[0 .. 2]: [splits[i]][seq_len][row], ntk_gemm_partials; splits 1: the projection itself, sums[0] may be q):
 * the sums in split order, then the same; the rotated q goes to q, k and v are not stored outside the caches */
int ntk_reduce_rope_kv_store(float* q, const float* const* sums, const int* splits, const int* positions, int seq_len, int n_heads, int n_kv_heads, int head_dim, float theta_base,
                             float freq_scale, int interleaved, void* k_cache, void* v_cache, int start_pos, int max_seq, void* stream);
/* ... from pieces of query, key and value side by side: [splits][seq_len][n_heads + 2 n_kv_heads][head_dim] */
int ntk_reduce_rope_kv_store_joined(float* q, const float* sums, int splits, const int* positions, int seq_len, int n_heads, int n_kv_heads, int head_dim, float theta_base, float freq_scale,
                                    int interleaved, void* k_cache, void* v_cache, int start_pos, int max_seq, void* stream);
/* ---------------------------------------------------------------------------------------------
 * Engine-level fused operators (no reference counterpart; they compute exactly what the listed
 * sequence of reference launchers computes, in fewer launches, with device-resident positions so a
 * whole token can be replayed from a hipGraph).  Used by nt_engine_*; exported for tests/benchmarks.
 * ------------------------------------------------------------------------------------------- */
typedef struct ntk_gemv_seg {
    const void* W;      /* raw GGUF blocks [rows][in]              */
    float*      y;      /* output [rows]                            */
    int         rows;
    int         dtype;  /* one format per call, or two for the plain (no resid / SiLU) form: Q4_K with Q6_K or Q5_K */
} ntk_gemv_seg;

/* y_s = W_s . f(x) for up to 3 row segments sharing x (fused Q|K|V or gate|up):
 *   norm_w != NULL : f(x) = rmsnorm(x, norm_w, eps)           (launch_rmsnorm + launch_gemv ...)
 *   resid  != NULL : y_0[r] = resid[r] + (W_0 . f(x))[r]      (launch_gemv + launch_add_inplace); resid may == y_0
 *   silu_pair != 0 : nseg == 2, y_0[r] = silu(W_0.f(x))[r] * (W_1.f(x))[r]   (2 x launch_gemv + launch_silu_mul) */
int ntk_gemv_fused(const ntk_gemv_seg* segs, int nseg, const float* x, int in_features, const float* norm_w,
                   float eps, const float* resid, int silu_pair, void* stream);

/* Engine-owned load-time repack of a K-quant matrix and the decode GEMV on the int8 matrix cores that reads it (csrc/gemv_rp.hip; SURVEY
 * 7.1 step 7 / 8(b) "Ownership": repack buffers belong to the engine object, the 1:1 ntk_gemv above keeps taking raw GGUF).  Q4_K, Q5_K,
 * Q6_K; in_features % 256 == 0 and <= 32768; rows padded to tiles of 16 inside the buffer.  Same integers, same scales (ntk_rp_dequant gives
 * the GGUF dequantisation bit for bit), 1.028 x / 1.023 x / 1.000 x the GGUF bytes.  Arithmetic: x -> per 256-column super-block three
 * signed base-256 digit planes of rint(x 2^(22-e)) (e = exponent of the block's largest |x|: <= 2^-22 of it per term), exact integer dot
 * products per sub-block on v_mfma_i32_16x16x64_i8, the reference's factorisation (gemm.cu:190-244, 297-354, 421-459) around them.
 *   ntk_rp_bytes        size of the repacked form (0: unsupported dtype / shape)
 *   ntk_rp_pack         raw GGUF [rows][in] -> dst (16-byte aligned, ntk_rp_bytes); stream ordered
 *   ntk_rp_dequant      parity instrumentation: the weights as F32 [rows][in] from the repacked form
 *   ntk_rp_unpack       the raw GGUF bytes back (exact inverse of ntk_rp_pack)
 *   ntk_gemv_rp(_fused) = ntk_gemv / ntk_gemv_fused with segs[i].W pointing at REPACKED tensors (same epilogues; one or two formats) */
size_t ntk_rp_bytes(int dtype, int rows, int in_features);
int ntk_rp_pack(void* dst, const void* raw, int rows, int in_features, int dtype, void* stream);
int ntk_rp_dequant(float* out, const void* rp, int rows, int in_features, int dtype, void* stream);
/* the raw GGUF blocks [rows][in] back from the repacked form, byte for byte (the engine keeps ONE resident copy of a K-quant matrix and unpacks into
 * a scratch in front of the launches that read raw blocks); raw: 4-byte aligned (Q6_K: 2); stream ordered */
int ntk_rp_unpack(void* raw, const void* rp, int rows, int in_features, int dtype, void* stream);
/* y[0..rows) = W . x over a repacked matrix with F32 products and sums (in_features <= 32768; x 16-byte aligned): one row of a prompt through its head */
int ntk_gemv_rp_f32(float* y, const void* rp, const float* x, int rows, int in_features, int dtype, void* stream);
int ntk_gemv_rp(float* y, const void* rp, const float* x, int out_features, int in_features, int weight_dtype, void* stream);
int ntk_gemv_rp_fused(const ntk_gemv_seg* segs, int nseg, const float* x, int in_features, const float* norm_w, float eps,
                      const float* resid, int silu_pair, void* stream);
/* parity instrumentation of the above: the LDS image its prologue builds from x (4 in + 68 in/256 bytes: three digit planes, a zero plane,
 * 64 bytes of sub-block-sum digits and one 2^(e-22) per super-block; nsub = 8: 32-column sub-blocks (Q4_K / Q5_K), 16: Q6_K), and
 * D[16][16] = A[16][64] . B[64][16] on the matrix instruction under the lane maps the kernel assumes */
int ntk_debug_rp_prologue(uint8_t* out, const float* x, const float* norm_w, float eps, int in_features, int nsub, int nwaves, void* stream);
int ntk_debug_mfma_i8_probe(int* D, const int8_t* A, const int8_t* B, void* stream);

/* RoPE(q,k at *d_pos) + KV store + GQA decode attention over keys 0..*d_pos, one launch
 * (launch_rope + launch_copy_to_kv_cache + launch_attention_decode; attention.cpp:165-190).
 * q [nh*hd], k,v [nkv*hd] are the raw projections (left untouched); d_pos is a DEVICE int.
 * inv_freq: optional DEVICE table [hd/2] of 1/powf(theta, 2i/hd) (NULL = computed in the kernel). */
int ntk_attention_decode_fused(float* output, const float* q, const float* k, const float* v, void* k_cache,
                               void* v_cache, const int* d_pos, const float* inv_freq, int n_heads, int n_kv_heads,
                               int head_dim, int max_seq, float scale, float theta_base, float freq_scale,
                               void* stream);

/* Long-context form of ntk_attention_decode_fused: `nsplit` workgroups share a head (positions interleaved), partial
 * softmax states go through `scratch` (ntk_attention_split_scratch_bytes) and a second launch merges them.  Same
 * arguments and results (summation order aside); head_dim 64 / 128 / 256, 16-byte aligned caches.
 * head_dim 128 with nsplit >= 16 and at most 16 query heads per KV head: one workgroup per (KV head, split) on the F16
 * matrix cores, every cache row read once (q * scale and the softmax weights enter as two F16 pieces each: <= 2^-22 of
 * the operand); rows past *d_pos are loaded but take no part whatever they hold. */
size_t ntk_attention_split_scratch_bytes(int n_heads, int head_dim, int nsplit);
int ntk_attention_decode_split(float* output, const float* q, const float* k, const float* v, void* k_cache,
                               void* v_cache, const int* d_pos, const float* inv_freq, int n_heads, int n_kv_heads,
                               int head_dim, int max_seq, float scale, float theta_base, float freq_scale, int nsplit,
                               float* scratch, void* stream);
/* The same as ONE launch: the workgroup that finishes last among the nsplit (<= 64) of a head merges their states itself -- the same
 * operations in the same order as the merge launch, identical bits.  The first ntk_attention_split_scratch_bytes' n_heads u32 of
 * `scratch` are arrival counters: zero them ONCE after allocating (ntk_attention_split_scratch_init, stream ordered); every launch
 * leaves them zero.  One scratch serves one stream at a time. */
int ntk_attention_split_scratch_init(float* scratch, int n_heads, void* stream);
int ntk_attention_decode_split_merged(float* output, const float* q, const float* k, const float* v, void* k_cache,
                                      void* v_cache, const int* d_pos, const float* inv_freq, int n_heads, int n_kv_heads,
                                      int head_dim, int max_seq, float scale, float theta_base, float freq_scale, int nsplit,
                                      float* scratch, void* stream);

/* Parity instrumentation: ntk_gemv_fused with the activation form of its Q4_K / Q6_K launches chosen by the CALL.  Those launches take,
 * from 48 MiB of weights on (a constant of the library: below it the conversion costs what the decode saves), the integer-activation
 * decoders of csrc/gemv_core.hip.h (three int8 digit planes per 32-column sub-block on v_dot4).  integer_activations = 1: whenever the
 * launch is eligible, 0: never, -1: the size rule -- so that the tests reach both decoders at small sizes.  No global state. */
int ntk_debug_gemv_fused_form(const ntk_gemv_seg* segs, int nseg, const float* x, int in_features, const float* norm_w, float eps,
                              const float* resid, int silu_pair, int integer_activations, void* stream);

/* Tensor-parallel exchange (csrc/tp.hip): hidden[0..n) += sum over ranks of their partial vectors, in rank
 * order, by one kernel that reads the peers' communication buffers (mapped with ntk_ipc_open or shared in-process) -- no RCCL
 * call, no second stream, hipGraph-capturable.  A communication buffer = ntk_tp_comm_bytes(max_floats) device bytes, reset once
 * with ntk_tp_comm_reset before the peers map it.  Call k of a forward writes its partial vector to ntk_tp_slot(comm, max_floats,
 * k) (slot k & 1) with any kernel on the same stream, then runs ntk_tp_allreduce_add(..., k, n, stream); calls per forward must be
 * even in number and < 1023; ntk_tp_advance_epoch ends the forward.  All ranks must issue the same sequence.  n % 4 == 0,
 * n <= max_floats, world <= 8.  ntk_tp_error after a synchronise: 0, or non-zero if a bounded wait for a peer gave up. */
size_t   ntk_tp_comm_bytes(size_t max_floats);
void*    ntk_tp_comm_alloc(size_t bytes);   /* fine-grained device memory (peer-visible without relying on a cache write-back); nt_hip_free */
int      ntk_tp_comm_reset(void* comm, void* stream);
float*   ntk_tp_slot(void* comm, size_t max_floats, unsigned call_index);
int      ntk_tp_allreduce_add(float* hidden, void* const* peers, int rank, int world, size_t max_floats, unsigned call_index, int n, void* stream);
int      ntk_tp_advance_epoch(void* comm, void* stream);
unsigned ntk_tp_error(void* comm);
int      ntk_ipc_export(void* devptr, void* handle64);
int      ntk_ipc_open(const void* handle64, void** devptr);
int      ntk_ipc_close(void* devptr);

/* Batched prompt projection on the matrix cores (replaces the per-token launch_gemv loops of
 * attention.cpp:144-162,200-210 and ffn.cpp:96-133):  Y[t,:] = W . X[t,:] (+ resid[t,:]) for t < n_tokens.
 * X [n_tokens][in] and Y/resid [n_tokens][out] are F32, token-major; W raw GGUF blocks [out][in] (quantised dtypes
 * only); X 16-byte aligned.  W is streamed once per 16 tokens; F32 activations, F32 MFMA accumulate.  resid may == Y. */
int ntk_gemm_quant(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features,
                   int weight_dtype, const float* resid, void* stream);

/* The same projection on the FP16 matrix cores, up to 1024 tokens per pass over W (csrc/gemm_f16.hip) -- ONE entry point behind a descriptor
 * (round 6: the six ntk_gemm_quant_ws* names of round 5 were this call with different optional fields).
 * Arithmetic: the integer part of every weight is exact in FP16; every F32 activation x is scaled by a power of two s (one per token: the token's
 * largest |x| s lies in [2^14, 2^15)) and split into two FP16 pieces h1 = rn16(x s), h2 = rn16(x s - h1), so that |x s - h1 - h2| <= 2^-23 |x s|
 * -- one F32 ulp of the activation (and <= 2^-39 of the token's largest |x| for activations more than 2^17 below it: the matrix cores take FP16
 * subnormals as they are, tools/micro/mfma_f16_subnormal.hip); the FP16 x FP16 products are exact in the F32 accumulator, block scales / K-quant
 * minima are applied to the F32 block sums and 1 / s to the finished sum (exact).  Against ntk_gemv the summation order differs and the
 * activations carry that one-ulp rounding.
 * Limits: Q8_0, Q4_0, Q4_K, Q5_K and Q6_K (NTK_E_DTYPE otherwise: use ntk_gemm_quant), one format per call; in_features a multiple of 128 (Q8_0) /
 * 256 (the others), rows % 16 == 0 and rows * row_bytes < 4 GiB (NTK_E_SHAPE); W, X, Y, resid 16-byte aligned (NTK_E_ALIGN).
 * (Row pitches that are not a multiple of 4 bytes -- Q8_0 with in_features % 64 != 0, Q6_K with in_features % 512 != 0 -- run the
 * same kernel with 2-byte aligned LDS reads, several times slower; no projection of the target models has one.)
 *   segs / nseg   1..3 matrices of one format that share X (Q | K | V, gate | up): {W_i raw GGUF [rows_i][in], y = Y_i [n_tokens][rows_i], rows_i, dtype}
 *   resid         optional [n_tokens][rows_0], nseg == 1 only, may alias Y_0: Y = W . X + resid
 *   workspace     ntk_gemm_quant_workspace_bytes(in_features, sum of rows_i) device bytes, 16-byte aligned, shared by every call (the FP16 planes and
 *                 scales of up to sixteen 64-token chunks of X + the partial sums of the K splits); contents need no initialisation
 *   reuse_x       != 0: X (same pointer, n_tokens <= 1024) has not changed since the previous call with this workspace -- its planes are not rebuilt
 *   row_max       optional DEVICE [n_tokens]: the tokens' largest |X[t, :]| (NULL = computed by a pass over X): the operand pre-pass is then ONE
 *                 launch, identical results.  The kernels that usually PRODUCE X in the reference's prompt path leave it beside X: ntk_rmsnorm_rowmax
 *                 (reference src/model/norm.cpp -> launch_rmsnorm, rmsnorm.cu:60-68; same expressions and sums as ntk_rmsnorm, identical output;
 *                 zero_tokens (optional): n_tokens floats set to 0 for a later ntk_silu_mul_rowmax) and ntk_silu_mul_rowmax (reference ffn.cpp:127 ->
 *                 launch_silu_mul, gemm.cu:719-724; identical output; width % 4 == 0, 16-byte aligned pointers, output may alias gate), whose row_max
 *                 must hold zeros (or earlier maxima of the same tokens) on entry
 *   partials      optional: the split-K sums are left to the launch that CONSUMES the projection.  The same launch runs but, when it splits K, the
 *                 partial sums stay in the workspace and *partials describes them (nsplit > 1; valid until the next call with this workspace) -- or
 *                 says nsplit == 1, in which case Y was written as usual (with `resid` added by the launch's epilogue; a launch that does split K
 *                 ignores `resid`: its consumer adds the residual).  Consumers:
 *                   ntk_reduce_rmsnorm_rowmax : hidden[t] = (sum of the splits, in order) + hidden[t]  (= the residual epilogue's association; nsplit == 1:
 *                       nothing to add when the launch ran with Y = resid = hidden, else hidden += Y), x_out = rmsnorm(hidden) with row_max /
 *                       zero_tokens as ntk_rmsnorm_rowmax: Wo / down projection + residual + the next RMSNorm, one launch;
 *                   ntk_reduce_silu_mul_rowmax: output[t] = silu(gate[t]) * up[t] of a deferred two-matrix gate | up launch, row_max as ntk_silu_mul_rowmax.
 *                 Identical bits to the separate launches (same sums in the same order).
 *   weights_repacked  != 0: segs[i].W point at the engine's DECODE REPACK of the matrices (ntk_rp_pack: tiles of 16 rows x 256-column super-blocks) instead
 *                 of raw GGUF blocks -- Q4_K / Q5_K / Q6_K (NTK_E_DTYPE otherwise).  Round 6: with one resident copy of a K-quant matrix the prompt pass
 *                 needs no unpack any more.  The same integers and scale products in the same order: IDENTICAL bits to the raw form.
 * Stream ordered, no allocation, no synchronisation. */
typedef struct ntk_gemm_partials {
    const float* part[3];   /* per matrix: [nsplit][n_tokens][rows] partial sums (NULL when nsplit == 1) */
    float*       y[3];      /* per matrix: the Y passed to the launch (written when nsplit == 1)            */
    int          rows[3];
    int          nseg, n_tokens, nsplit;
} ntk_gemm_partials;
typedef struct ntk_gemm_desc {
    const ntk_gemv_seg* segs;
    int                 nseg;
    const float*        X;            /* [n_tokens][in_features] */
    int                 n_tokens, in_features;
    const float*        resid;
    void*               workspace;
    size_t              workspace_bytes;
    int                 reuse_x;
    const float*        row_max;
    ntk_gemm_partials*  partials;
    int                 weights_repacked;   /* != 0: segs[i].W are tensors of the decode repack (ntk_rp_pack; Q4_K / Q5_K / Q6_K), read as they lie */
} ntk_gemm_desc;
size_t ntk_gemm_quant_workspace_bytes(int in_features, int out_features);
int ntk_gemm_quant_f16(const ntk_gemm_desc* desc, void* stream);
int ntk_reduce_rmsnorm_rowmax(float* hidden, const ntk_gemm_partials* partials, const float* weight, float eps, float* x_out, float* row_max,
                              float* zero_tokens, void* stream);
int ntk_reduce_silu_mul_rowmax(float* output, const ntk_gemm_partials* partials, float* row_max, void* stream);
int ntk_rmsnorm_rowmax(float* output, const float* input, const float* weight, int n_tokens, int hidden_size, float eps, float* row_max,
                       float* zero_tokens, void* stream);
int ntk_silu_mul_rowmax(float* output, const float* gate, const float* up, int n_tokens, int width, float* row_max, void* stream);
/* The operand pre-pass INSIDE the launch that produces X (round 6): each of these owns a whole token per workgroup, so the workgroup that has written a
 * token's row also splits it -- planes, step sums and 1 / s go straight into `workspace` (the bits ntk_gemm_quant_f16's own pre-pass would write) and the
 * projection that follows runs with reuse_x = 1 on that workspace: no separate pre-pass launch (four to five of the fourteen launches of a prompt layer).
 *   ntk_gemm_prepare_x            X as it lies (e.g. the attention output in front of Wo): row maximum + split, one launch instead of two
 *   ntk_rmsnorm_prepare_x         ntk_rmsnorm (reference rmsnorm.cu:60-68; identical output) + the split of its output
 *   ntk_reduce_rmsnorm_prepare_x  ntk_reduce_rmsnorm_rowmax (identical hidden / x_out) + the split of x_out
 *   ntk_silu_mul_prepare_x        ntk_silu_mul (reference gemm.cu:719-724; identical output, may alias gate) + the split of its output
 *   ntk_reduce_silu_mul_prepare_x ntk_reduce_silu_mul_rowmax (identical output) + the split; `workspace` must NOT be the one the partial sums lie in
 *                                 (the launch reads those while it writes the planes: the engine alternates between two workspaces)
 * n_tokens <= 1024 (one pass), the row length a multiple of 32 (NTK_E_SHAPE), 16-byte aligned pointers (NTK_E_ALIGN).  Stream ordered, no allocation. */
int ntk_gemm_prepare_x(const float* X, int n_tokens, int in_features, void* workspace, void* stream);
int ntk_rmsnorm_prepare_x(float* output, const float* input, const float* weight, int n_tokens, int hidden_size, float eps, void* workspace, void* stream);
int ntk_reduce_rmsnorm_prepare_x(float* hidden, const ntk_gemm_partials* partials, const float* weight, float eps, float* x_out, void* workspace, void* stream);
int ntk_silu_mul_prepare_x(float* output, const float* gate, const float* up, int n_tokens, int width, void* workspace, void* stream);
int ntk_reduce_silu_mul_prepare_x(float* output, const ntk_gemm_partials* partials, void* workspace, void* stream);

/* ... and of a prompt of more than 64 tokens (up to 1024, one pass): the planes from four tokens a workgroup.  ntk_rows_prepare_takes: 1 where the three take such a prompt (norm: the second), else 0
 *   ntk_rows_prepare_x            X as it lies
 *   ntk_rows_norm_prepare_x       hidden += the deferred projection (partials; NULL: hidden as it lies), planes of its RMSNorm; x_out (may be NULL): the normalised rows themselves
 *   ntk_rows_silu_mul_prepare_x   planes of silu(gate) * up of a gate | up launch, deferred or not; output (may be NULL, may be the gate's y): the rows themselves
 * Workspace and alignments as above; results as the launches above give them, up to the order of a norm's sum. */
int ntk_rows_prepare_takes(int n_tokens, int width, int norm);
int ntk_rows_prepare_pays(int n_tokens, int width, int norm, int nsplit);   /* ... and is ahead of the launches that it replaces (nsplit: pieces to add up; 0: rows as they lie; the third has 1 at least) */
int ntk_rows_prepare_x(const float* X, int n_tokens, int width, void* workspace, void* stream);
int ntk_rows_norm_prepare_x(float* hidden, const ntk_gemm_partials* partials, const float* weight, int n_tokens, int width, float eps, float* x_out, void* workspace, void* stream);
int ntk_rows_norm_prepare_zero(float* hidden, const ntk_gemm_partials* partials, const float* weight, int n_tokens, int width, float eps, float* x_out, float* zero_tokens, void* workspace,
                               void* stream);   /* ... that clears zero_tokens (n_tokens floats, may be NULL) as ntk_rmsnorm_rowmax does */
int ntk_rows_silu_mul_prepare_x(float* output, const ntk_gemm_partials* partials, void* workspace, void* stream);

/* Prompts of at most 32 tokens, whose projections keep a K slice's planes in LDS: their producers scale X per token and 256 columns, so that they need no whole row in one workgroup.
 *   ntk_gemm_short_takes          1 where ntk_gemm_short takes matrices of these rows and format (raw or repacked) over one X of in_features, else 0
 *   ntk_short_prepare_x           planes of X as it lies
 *   ntk_short_norm_prepare_x      hidden += the deferred projection (partials; NULL: hidden as it lies), planes of hidden * weight and the rows' sums of squares: the projection that
 *                                 reads them is told `normed` and eps and divides its results by the rows' root mean squares (ntk_rmsnorm's definition)
 *   ntk_short_silu_mul_prepare_x  planes of silu(gate) * up of a deferred gate | up launch
 *   ntk_gemm_short                ntk_gemm_quant_f16 over such planes (desc->X and reuse_x are not looked at; NTK_E_SHAPE where ntk_gemm_short_takes says 0).  part_at: floats into the
 *                                 workspace's area of partial sums at which this launch's begin (a multiple of 4), so that several launches may leave theirs to one consumer
 *                                 (ntk_gemm_short_form 2: a repack's results are summed in another order than its tensor's, else they are the same bits)
 * n_tokens <= 32, rows a multiple of 32 (NTK_E_SHAPE), 16-byte aligned pointers (NTK_E_ALIGN).  `workspace` must not be the one partials lie in.  Stream ordered, no allocation. */
int ntk_gemm_short_takes(const int* rows, int nseg, int n_tokens, int in_features, int dtype);
/* how it takes them: 1 the planes in LDS, 2 in registers (K-quants, many rows, up to 16 tokens); 0 not at all */
int ntk_gemm_short_form(const int* rows, int nseg, int n_tokens, int in_features, int dtype, int repacked);
int ntk_short_prepare_x(const float* X, int n_tokens, int in_features, void* workspace, void* stream);
int ntk_short_norm_prepare_x(float* hidden, const ntk_gemm_partials* partials, const float* weight, int n_tokens, int hidden_size, void* workspace, void* stream);
int ntk_short_silu_mul_prepare_x(const ntk_gemm_partials* partials, void* workspace, void* stream);
int ntk_gemm_short(const ntk_gemm_desc* desc, int normed, float eps, size_t part_at, void* stream);
/* ntk_gemm_short of a, then of b with its partial sums behind a's: matrices of two formats over the same planes, in one launch where one of them has many rows and that is estimated to be ahead
 * (repacked K-quants, sums left) */
int ntk_gemm_short_two(const ntk_gemm_desc* a, const ntk_gemm_desc* b, int normed, float eps, size_t part_at, void* stream);
/* 1: it does these two in one launch, 0: one after the other */
int ntk_gemm_short_two_joins(const ntk_gemm_desc* a, const ntk_gemm_desc* b, size_t part_at);
/* A prompt of at most 32 tokens from position 0 on: ntk_reduce_rope_kv_store, ntk_attention_prefill and ntk_short_prepare_x of its result in one launch.  sums / splits: of q, k and v as in
 * ntk_reduce_rope_kv_store; angles: ntk_short_angles' table (ntk_short_angles_bytes, 16-byte aligned), formed once a model.  head_dim 128, an even number of heads (NTK_E_SHAPE). */
size_t ntk_short_angles_bytes(int head_dim);
int ntk_short_angles(float* table, int head_dim, float theta_base, float freq_scale, void* stream);
int ntk_short_attention(const float* const* sums, const int* splits, const float* angles, int n_tokens, int n_heads, int n_kv_heads, int head_dim, float scale, int interleaved, void* k_cache,
                        void* v_cache, int max_seq, void* workspace, void* stream);

/* Y[t][0..out) (+)= W . X[t] for the tokens of a prompt over IEEE-half weights ([out][in] row-major), one pass over W: the batched form of n_tokens ntk_gemv calls.
 * row_max: the tokens' largest |X| where their producer left it (ntk_rmsnorm_rowmax ...), NULL: taken here.  workspace (16-byte aligned): without row_max at least
 * ntk_gemm_half_workspace_bytes(n_tokens), else NULL is enough; what it holds beyond that is used for partial sums or, where that is faster (most shapes, from room for all
 * rows' halves on: 4 * in_features + 4 bytes a token), for the activations' two halves: all of it may be overwritten. */
size_t ntk_gemm_half_workspace_bytes(int n_tokens);
int ntk_gemm_half(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, int accumulate, const float* row_max, void* workspace,
                  size_t workspace_bytes, void* stream);

/* y_i (+)= W_i . x of one to three matrices of F16 or of F32 rows in one launch, each product with ntk_gemv's bits */
int ntk_gemv_dense(const ntk_gemv_seg* segs, int nseg, const float* x, int in_features, int add, void* stream);
/* Y[t] = W . X[t] of F16 or F32 rows in one launch, each product with ntk_gemv's bits.  in_features a multiple of 8, 16-byte aligned W and X (NTK_E_ALIGN: nothing was launched). */
int ntk_gemv_tokens(float* y, const void* W, const float* x, int n_tokens, int out_features, int in_features, int weight_dtype, void* stream);

/* ... for up to three such matrices over the same X (query, key and value; gate and up) in one launch, with the activations' two halves formed once per pass in the workspace
 * (ntk_gemm_half_many_bytes() of it at least, which is 16 tokens' worth; the tokens go in equal passes of what it holds, 4 * in_features + 4 bytes each, and every pass reads the weights:
 * give it room for all of them; more is used for partial sums).  Y[i] = W[i] . X; silu != 0 (n == 2, out[0] == out[1]): Y[0] = silu(W[0] . X) * (W[1] . X) alone (ntk_silu_mul).
 * accumulate only with n == 1.  NTK_E_SHAPE where in_features is no multiple
 * of 64, the workspace is too small for 16 tokens or, with silu, the two matrices lie 4 GiB apart: nothing has been launched then. */
typedef struct ntk_half_desc {
    const void* W[3]; float* Y[3]; int out[3]; int n;
    const float* X; int n_tokens, in_features, accumulate;
    const float* row_max;
    int silu;
    void* workspace; size_t workspace_bytes;
} ntk_half_desc;
size_t ntk_gemm_half_many_bytes(int n_tokens, int in_features);
int ntk_gemm_half_many(const ntk_half_desc* d, void* stream);
/* how one pass of it goes, with room floats behind the halves (silu: 0): plan = {rows, columns of a tile, tiles a CU holds at once, pieces of K} */
int ntk_gemm_half_plan(int rows, int N, int K, long long room, int* plan);
/* ... with a norm between two of them and no row in between.  ntk_gemm_half_defer: ntk_gemm_half with accumulate that may leave its pieces of K to the launch behind it (partials: as those of
 * ntk_gemm_quant_f16; they lie in the workspace).  ntk_half_norm_split: hidden += that projection (partials; NULL: hidden as it lies), and the halves of its RMSNorm into `workspace` (another one), from
 * which ntk_gemm_half_normed is ntk_gemm_half_many (X, row_max not looked at; no unit's sums are left).  ntk_half_norm_takes: 1 where the workspace holds all tokens (width a multiple of 64, up to 16384), else 0. */
int ntk_gemm_half_defer(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, const float* row_max, void* workspace, size_t workspace_bytes,
                        ntk_gemm_partials* partials, void* stream);
int ntk_half_norm_takes(int n_tokens, int width, size_t workspace_bytes);
int ntk_half_norm_split(float* hidden, const ntk_gemm_partials* partials, const float* weight, int n_tokens, int width, float eps, void* workspace, size_t workspace_bytes, void* stream);
int ntk_gemm_half_normed(const ntk_half_desc* d, ntk_gemm_partials* partials, void* stream);      /* partials (or NULL): several matrices' pieces left as those of one of all their rows */

/* Dequantise rows of a (quantised) embedding table on the device: out[t,:] = table[tokens[t],:].
 * Same arithmetic as the host loop in reference src/model/transformer.cpp:419-599; Q5_K is zero-filled
 * exactly as the reference does (:595-598).  tokens is a DEVICE int array. */
int ntk_embed_rows(float* out, const void* table, const int* tokens, int n_tokens, int hidden, int dtype,
                   void* stream);

/* Greedy sampling on the device: first index of the maximum (reference src/inference/sampler.cpp:18-28).
 * Writes the index to *d_out_token (device) -- and to *h_mirror if it is a pinned host pointer (may be NULL).
 * scratch: device buffer of >= 2*1024 floats. */
int ntk_argmax(const float* logits, int n, int* d_out_token, int* h_mirror, float* scratch, void* stream);

/* The reference's sampler on the device (reference src/inference/sampler.cpp:30-117), for temperature > 0 and
 * 0 < top_k <= 64 (NTK_E_SHAPE otherwise: the caller samples on the host): repeat penalty over d_recent[n_recent] (DEVICE
 * ints, applied in place to `logits`, once per occurrence), logits / temperature, top-k, softmax, top-p cut, and the walk of the
 * cumulative distribution against `r` -- the uniform draw the caller takes from ITS std::mt19937, one per token, so the token
 * stream equals the host sampler's for the same seed.  Result to *d_out_token and *h_mirror (pinned, may be NULL).
 * scratch: ntk_sample_scratch_bytes(n) device bytes.  Vocabularies up to 131 072. */
size_t ntk_sample_scratch_bytes(int n);
int ntk_sample_top_k(float* logits, int n, const int* d_recent, int n_recent, float repeat_penalty, float temperature,
                     int top_k, float top_p, float r, int* d_out_token, int* h_mirror, void* scratch, void* stream);
/* the repeat penalty alone (greedy decoding with a penalty = this + ntk_argmax) */
int ntk_repeat_penalty(float* logits, int n, const int* d_recent, int n_recent, float repeat_penalty, void* stream);

/* The greedy tail of a decode token in two launches instead of three: ntk_argmax, then -- in the same final launch -- the token id to the
 * pinned host ring h_ring4 (4 x 8 bytes, may be NULL): slot (*d_pos & 3) receives ONE 8-byte store {token, *d_pos + 1 in the high
 * word}, and *d_pos += 1.  The ring lets a host loop keep the NEXT token's launches queued while it polls for this one (a token that
 * runs one ahead lands in another slot), instead of synchronising the stream per token. */
int ntk_argmax_advance(const float* logits, int n, int* d_out_token, int* h_mirror, unsigned long long* h_ring4, int* d_pos,
                       float* scratch, void* stream);

/* measurement instrumentation: the shader clock right now.  d_out2 (DEVICE, 3 x 8 bytes): [0] shader cycles (s_memtime) and [1] 10 ns ticks
 * (s_memrealtime) over ~50 us of one spinning wave: MHz = 100 * [0] / [1].  bench.py records it right behind the timed region. */
int ntk_debug_sclk(unsigned long long* d_out2, void* stream);
/* ... and the AVERAGE shader clock over a span of work: _begin starts a one-wave kernel on `side_stream` (a stream other than the workload's,
 * e.g. ntk_stream(1)) that sleeps and polls until _end raises d_flag (4 DEVICE bytes) through `other_stream` (e.g. ntk_stream(2)), or 3 s
 * pass; after synchronising side_stream, d_out2 = {shader cycles, 10 ns ticks} of the span.  bench.py runs it over extra decode steps right
 * behind the timed region (never inside it). */
int ntk_debug_sclk_begin(unsigned* d_flag, unsigned long long* d_out2, void* side_stream);
int ntk_debug_sclk_end(unsigned* d_flag, void* other_stream);

/* test instrumentation: after this call nt_hip_malloc hands out at most `bytes` more device bytes and then fails like an exhausted device
 * (NULL + the reference's message), where what is freed of them counts again; bytes < 0 removes the budget.  Process-wide; tests only (the load-time repack's "does not fit" path). */
void ntk_debug_malloc_budget(long long bytes);
/* test instrumentation: how often the process has waited for a stream (ntk_stream_synchronize) */
long long ntk_debug_stream_waits(void);

/* *d_pos += 1 (one thread); keeps positions on the device across graph replays */
int ntk_advance_pos(int* d_pos, void* stream);
/* ONE token's row (as ntk_embed_rows; formats without a branch: zeros), the token and its position as arguments: they go into *d_token and *d_pos for the launches behind */
int ntk_embed_token_row(float* out, const void* table, int token, int pos, int* d_token, int* d_pos, int hidden, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#if defined(__GNUC__)
#pragma GCC visibility pop
#endif
#endif /* NTK_ENGINE_H */
