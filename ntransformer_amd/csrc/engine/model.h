// engine/model.h -- resident-weights Llama model on one MI355X.
// Replaces the resident subset of reference src/model/{transformer,attention,ffn,norm}.{h,cpp}
// (Transformer::load / load_layer / allocate_buffers / embed_tokens / forward, Attention::forward,
// FFN::forward, RMSNorm::forward).  The reference's streaming / tiered / delta / speculative paths exist
// to fit 24 GB of VRAM and are dropped: 288 GB of HBM holds every target model resident.
#pragma once
#include <chrono>
#include <cstdint>
#include <string>
#include <vector>
#include "gguf.h"
#include "host_rows.h"
#include "synth.h"

struct ihipGraphExec_t;   // hipGraphExec_t

namespace nt {

struct DevTensor {
    void* ptr = nullptr;   // device
    int dtype = 0;
    int64_t in_f = 0, out_f = 0;
    size_t nbytes = 0;
    void* rp = nullptr;    // engine-owned repack for the matrix-core decode GEMV (csrc/gemv_rp.hip); nullptr: none
    size_t rp_bytes = 0;
};

struct LayerWeights {
    DevTensor attn_norm, wq, wk, wv, wo, ffn_norm, w_gate, w_up, w_down;
};

class Model {
public:
    Model() = default;
    ~Model();
    Model(const Model&) = delete;
    Model& operator=(const Model&) = delete;

    // reference Transformer::load (transformer.cpp:59-126): parse, cap context, weights -> HBM, buffers
    int load(const std::string& gguf_path, int max_context);
    // same model object built from the seeded generator, tensor by tensor, without a file
    int load_synthetic(const SynthSpec& spec, int max_context, int nthreads);
    // A SECOND SEQUENCE over the weights `src` holds resident (round 6; SURVEY 8(e): the path shards across requests -- independent sequences share
    // nothing but the read-only weights): this object gets src's tensor table (the same device pointers, raw and repacked; it owns none of them), its
    // own KV caches, activation buffers, device scalars, captured graphs and its own non-blocking stream, so two host threads can decode two requests
    // on one GPU at once.  `src` must outlive this object and must not be re-loaded or switch its repack level meanwhile; a source with one resident
    // copy of its K-quant weights gives this sequence an unpack scratch of its own; tensor-parallel slices are refused (NTK_E_SHAPE).
    int share_weights(const Model& src, int max_context);

    // reference Transformer::forward (transformer.cpp:604-669): the reference's launcher sequence, 1:1,
    // any seq_len (prefill = per-token GEMV loops like the reference).  Returns device logits [vocab].
    float* forward(const int* tokens, int seq_len, int start_pos);

    // Fused single-token step: 5 launches per layer, position and token id stay on the device so the whole
    // token is one hipGraph replay.  Token comes from d_token_ (set_device_token / previous argmax).
    // If greedy: also runs the device argmax and advances the position.
    int decode_step_fused(bool greedy, bool use_graph);
    int decode_token(int token, int pos, bool use_graph, float* host);   // a given token's logits: set_device_step, a step and copy_logits with two launches less
    int set_device_token(int token);
    int set_device_pos(int pos);
    int set_device_step(int pos, int token);   // both for ONE step, as arguments of a launch: in the stream's order, nothing waited for
    // attention regime by context length (each regime is its own captured graph: the grid of the attention launch is fixed in it).
    // 0: the single-pass kernel, one workgroup per query head, walks the head's cache serially (4.2 us per layer at 16 positions, 7.5 at
    //    512, 30.7 at 4095).  Beyond 544 positions: ntk_attention_decode_split = partial states of `splits` workgroups + a combine launch:
    // 1: 8 splits -- the per-query-head walk (8.7 us per layer at 1023 positions, 10.1 at 2047, 13.5 at 4095);
    // 2: head_dim 128, from 3072 positions: 32 splits -- the matrix-core form, one workgroup per (KV head, split), every cache row read
    //    once, one 32-row chunk per wave up to 4096 positions (12.75 us at 4095; 70B geometry 13.5 vs 16.5; decode behind a 3900-token
    //    prompt 467 -> 482 tokens/s; with 16 splits the two forms tie between 2300 and 3300 positions:
    //    profiles/r04_attention_kvhead_form.txt); other head sizes: the walk with 16 splits from 16384 positions.
    //    Contexts beyond 4096 (round 5; the reference's -c / --ctx-size, main.cpp:74-75): 32 splits STAY the best count however long the context --
    //    8B geometry, us per layer incl. the combine launch, caches past the Infinity Cache (tools/attn_bench.py --max-seq,
    //    profiles/r05_attention_long_context.txt): 8191 positions 17.2 / 14.6 / 19.1 / 27.2 with 16 / 32 / 64 / 128 splits; 32767: 30.1 /
    //    35.8 / 42.8 / 59.4 with 32 / 64 / 128 / 256 (4.45 TB/s of cache bytes at 32); 131071: 103 / 108 / 118 with 64 / 128 / 256 (5.2
    //    TB/s): one workgroup per CU (8 KV heads x 32), the chunks of 32 rows go round ALL waves of the launch, and every further split
    //    costs a redundant RoPE prologue and a longer serial walk in the combine launch.
    static constexpr int kAttnRegimes = 3;
    static int attention_regime(int pos, int head_dim) {
        if (pos < 544) return 0;
        return pos < (head_dim == 128 ? 3072 : 16384) ? 1 : 2;
    }
    static int attention_splits(int regime, int head_dim) { return regime <= 1 ? 8 : head_dim == 128 ? 32 : 16; }
    static constexpr int kMaxAttnSplits = 32;
    void pick_attention_regime();
    int sync();
    int host_token() const;                 // token written by the last device argmax (after sync)
    // token of the greedy fused step that decoded position `pos`, polled from the pinned ring without a stream synchronisation (the
    // caller may already have queued the next step)
    int wait_token(int pos, int* token);
    float* logits_ptr() { return logits_; }
    int copy_logits(float* host);           // D2H of [vocab] floats (blocking)
    // Sample the next token from the device logits with the reference's sampler (ntk_sample_top_k / penalty + ntk_argmax when
    // temperature <= 0): result in d_token_ and, after sync(), host_token().  recent: the last tokens (host), r: the host's draw.
    int sample_on_device(const int* recent, int n_recent, float repeat_penalty, float temperature, int top_k, float top_p, float r);
    static bool device_sampler_supports(float temperature, int top_k, int vocab) {
        return temperature <= 0.0f || (top_k > 0 && top_k <= 64 && top_k < vocab && vocab <= 131072);
    }

    const ModelConfig& config() const { return cfg_; }
    const GgufVocab& vocab() const { return vocab_; }
    const std::string& error() const { return err_; }
    uint64_t weight_bytes() const { return weight_bytes_; }
    // algorithmic bytes one decode token must move at position `pos`
    uint64_t bytes_per_token(int pos) const;
    // Prompts (seq_len > 1) project all tokens of a chunk with one pass over each weight matrix (ntk_gemm_quant) instead
    // of the reference's per-token GEMV loops; off = the reference's exact launch sequence.
    void set_batched_prefill(bool on) { batched_prefill_ = on; }
    // One decode token as ONE persistent launch (csrc/decode_persistent.hip) instead of 5 launches per layer.  On by default
    // when the model qualifies (quantised matrices, head_dim 64 / 128); short contexts only (single-pass attention regime),
    // longer ones keep the launch path.  Turned off for good if the kernel ever reports a bounded wait that gave up.
    void set_persistent(int level);   // 0 off, 1 decode_persistent.hip, 2 layer_engine.hip (round 5); EXPERIMENTS=1 builds only, otherwise stays off
    int persistent_kind() const { return persistent_plan_ ? persistent_kind_ : 0; }
    void set_fuse_attention(bool on) { fuse_attention_ = on; }
    void set_prefill_row_max(bool on) { prefill_row_max_ = on; }
    void set_prefill_fused_split(bool on) { prefill_fused_split_ = on; }
    // Split-KV decode attention as ONE launch (the last workgroup of a head merges the partial states: attention_merge.hip.h) or -- the default --
    // with the separate combine launch of rounds 3-5; same bits either way, the one-launch form measured 0.1-0.6 us (walk) / 1.5-4 us (matrix-core
    // form) per layer slower (profiles/NEGATIVE_RESULTS.md 8).  Captured graphs are dropped when the setting changes.
    int set_attention_merge(bool on);
    // Decode GEMVs of the K-quant matrices from the load-time repack (ntk_gemv_rp_fused) instead of the raw GGUF blocks (ntk_gemv_fused).
    // level 0: no repack (raw path).  1: repack AND the uploaded GGUF bytes stay resident (K-quant weights x 2 in HBM; round 4's form).
    // 2: ONE resident copy (round 5) -- the GGUF bytes of every repacked matrix are freed after the repack; the launches that read raw blocks
    // (prompt GEMM, the 1:1 ntk_gemv sequence, fallbacks) get the tensor unpacked into a scratch right in front of them (ntk_rp_unpack:
    // byte-exact inverse; + 2 x the model's bytes of HBM traffic per PROMPT PASS whatever its length: 8B Q4_K_M +4 ms = -30 % on a 64-token
    // prompt, -6 % on 1024 tokens; 70B -7 %; decode unchanged).  3 (default): round 5: 2 only when memory was short; ROUND 6: always 2 -- the FP16 prompt
    // GEMM reads the repack itself (ntk_gemm_desc.weights_repacked: identical bits, no unpack), so the batched prompt path and the fused decode path need
    // no GGUF bytes of a repacked matrix; what still unpacks into the scratch: the 1:1 launcher sequence (--no-fuse / tests) and the prompt's LM-head GEMV.
    // The repack is made at load unless the option was switched off BEFORE the load; switching after the load works in every direction
    // (2 -> 0 / 1 re-materialises the GGUF bytes from the repack).  Returns a status (NTK_E_NOMEM: the model keeps running on what it has).
    int set_repack(int level);
    bool repack() const { return repack_ != 0; }
    int repack_level() const { return repack_; }
    uint64_t repack_bytes() const { return repack_bytes_; }
    uint64_t resident_weight_bytes() const { return weight_bytes_ - raw_freed_bytes_ + repack_bytes_ + raw_scratch_bytes_; }
    void set_bf16_prefill(bool on) { bf16_prefill_ = on; }   // batched prompt: FP16-MFMA (gemm_f16.hip; the option keeps its round-2 name) or the F32-MFMA form (16)
    bool persistent_available() const { return persistent_plan_ != nullptr; }
    void* persistent_plan() const { return persistent_plan_; }
    // which form decode_step_fused(…) emits at the current position: "persistent" / "fused launches"
    const char* decode_path() const;
    int check_persistent();   // after a sync: NTK_OK, or NTK_E_LAUNCH if an in-kernel bounded wait gave up (TP exchange, experiments)
    int check_tp();           // the tensor-parallel part of it: error word of the exchange kernel, surfaced and cleared
    // parity instrumentation (tests): layers [first, first+count) on caller-supplied hidden states; KV cache rows in / out
    int debug_run_layers(const float* hidden_in, int T, int start_pos, int first, int count, int mode, float* hidden_out);
    int debug_kv(int layer, int pos0, int n, uint16_t* k, uint16_t* v, bool write);
    // One fused token launched eagerly and timed with HIP events on the compute stream.
    // ms[c] / calls[c] per class c: 0 quant GEMV, 1 attention, 2 everything else (embed, argmax, pos); calls[3] = timed
    // intervals.  fine (coarse = false): an event pair around every launch.  coarse: one event per change of class, so
    // a run of GEMV launches is timed as a whole (kernels + the boundaries between them) and the event cost is per run.
    int profile_token(float ms[4], int calls[4], bool coarse);
    void* stream() const { return stream_; }

    // ---- tensor parallelism (csrc/tp.hip) -------------------------------------------------------------
    // Call before load(): this model object holds slice `rank` of `world` -- rows [rank/world) of Wq, Wk, Wv, gate, up (whole
    // heads), columns of Wo and down -- so config() reports the LOCAL head / FFN counts.  After load(): exchange comm()
    // addresses (tp_export: a hipIpc handle and the raw pointer) and tp_connect() them on every rank before the first forward.
    int tp_configure(int rank, int world);
    int tp_rank() const { return tp_rank_; }
    int tp_world() const { return tp_world_; }
    int tp_export(void* handle64, void** raw);
    int tp_connect(const void* handles, void* const* raws);   // world x 64-byte handles (other processes) or raw pointers (same process)
    unsigned tp_error();                                      // after sync(): 0, or the call that gave up waiting for a peer
    // the host-side column slice of a GGUF matrix: columns [rank * in/world, (rank+1) * in/world) of every row, re-packed
    static int slice_columns(void* dst, const void* src, int dtype, int64_t out_f, int64_t in_f, int rank, int world);

private:
    int load_impl(const std::string& gguf_path, int max_context);
    int finish_load(int max_context);
    int alloc_buffers();
    int upload(DevTensor& dst, const void* host, int dtype, int64_t in_f, int64_t out_f, size_t nbytes);
    enum Shard { WHOLE, ROWS, COLS };
    // upload this rank's part of a full host tensor [out_f][in_f]: everything, rows [rank * out/world ...), or the column slice
    int upload_shard(DevTensor& dst, const void* host_full, int dtype, int64_t in_f, int64_t out_f, size_t nbytes_full, Shard how);
    int repack_all();                 // the repacked form of every K-quant projection (after the upload)
    int repack_one(DevTensor& t);
    int drop_raw_all();               // level 2: free the GGUF bytes of every repacked matrix, size the unpack scratch
    int restore_raw_all();            // ... and back: the GGUF bytes re-materialised from the repack
    // the raw GGUF blocks of a projection for a launch that reads them: the resident bytes, or the tensor unpacked into the scratch (stream
    // ordered; raw_begin() starts a new group of tensors that must be valid together: Q | K | V, gate | up)
    void raw_begin() { raw_cursor_ = 0; }
    const void* raw_of(const DevTensor& t);
    int tp_check_shapes();            // the head / FFN / block divisibility the slices need
    int tp_allreduce(float* hidden, int n);   // hidden += sum over ranks of the partial vectors in the current slot
    float* tp_slot() const;           // where the next partial vector goes
    void free_all();
    enum TokenKind { kSampled = 0, kGreedy = 1, kBare = 2 };    // bare: the embedded row is there, and the caller's launch behind the logits advances the position
    int enqueue_token(TokenKind kind);   // the fused launch sequence for one token
    int run_token(TokenKind kind, bool use_graph);
    int enqueue_layers(int first, int last);            // its layer loop
    int layers_1to1(int T, int start_pos, int first, int last, bool keys_last = false, float* queries = nullptr);   // the layer loop of forward()
    bool short_prompt(int T) const;
    bool short_matrices(int T) const;
    mutable int short_known_[2] = {-1, -1};   // short_matrices of up to 16 and up to 32 tokens: not asked yet, no, yes
    int layers_short(int T, int start_pos, int first, int last_layer);
    void prof_mark(int cls, bool begin);
    bool use_persistent_now() const;
    int build_persistent_plan(int kind);   // the same operator sequence as a table for ntk_persistent_launch / ntk_layer_engine_launch (nullptr plan if unsupported)

    ModelConfig cfg_;
    GgufVocab vocab_;
    std::string err_;
    std::vector<LayerWeights> layers_;
    DevTensor token_embd_, output_norm_, output_;
    bool output_tied_ = false;
    uint64_t weight_bytes_ = 0;
    std::vector<void*> allocs_;
    bool shares_weights_ = false;    // the tensor table points into ANOTHER Model's allocations (share_weights): nothing of it is freed here

    // buffers (reference transformer.cpp:330-391)
    uint16_t* k_cache_ = nullptr;   // [L][max_seq][nkv][hd] half
    uint16_t* v_cache_ = nullptr;
    float* hidden_ = nullptr;       // [max_seq][H]
    float* residual_ = nullptr;     // [max_seq][H]
    float* workspace_ = nullptr;    // max(attention, ffn) floats, shared by all layers
    size_t workspace_floats_ = 0;
    float* logits_ = nullptr;       // [V]
    int* positions_ = nullptr;      // [max_seq]
    int* tokens_dev_ = nullptr;     // [max_seq]
    int* d_pos_ = nullptr;          // device scalar: position of the token being decoded
    int* d_token_ = nullptr;        // device scalar: id of the token being decoded
    int* h_token_ = nullptr;        // pinned mirror of the argmax result
    unsigned long long* h_ring_ = nullptr;   // pinned ring of 4 x {token, position + 1}: ntk_argmax_advance / wait_token
    HostRows out_row_;                // the logits on their way to the caller
    std::chrono::steady_clock::time_point wait_t0_;
    float* argmax_scratch_ = nullptr;
    void* sample_scratch_ = nullptr;
    int* d_recent_ = nullptr;       // device copy of the repeat-penalty window
    int* h_recent_ = nullptr;       // pinned staging of it
    static constexpr int kRecentCap = 4096;
    float* rope_inv_freq_ = nullptr; // [hd/2] 1/powf(theta, 2i/hd), computed once on the host (rotary.cu:47)
    float* rope_angles_ = nullptr;     // ntk_short_angles of the first 32 positions
    void* stream_ = nullptr;
    bool batched_prefill_ = true;
    struct Timed { int cls; void* a; void* b; int n; bool shared_a; };   // n launches between events a and b
    bool prof_coarse_ = false;
    std::vector<Timed>* prof_ = nullptr;   // non-null while profile_token() runs
    // one captured token per (greedy?, attention regime)
    static constexpr int kPersistentSlot = kAttnRegimes;   // the persistent forms of regime 0 have their own slot
    ihipGraphExec_t* graphs_[3][kAttnRegimes + 1] = {};   // [sampled, greedy, layers and head alone][attention regime 0..2, 3 = persistent]
    int host_pos_ = 0;               // host mirror of *d_pos_ (set_device_pos + one per fused step): picks the regime
    int attn_regime_ = 0;            // regime enqueue_token() emits
    float* attn_scratch_ = nullptr;  // partial softmax states of the split-KV attention
    bool prefill_row_max_ = true;    // RMSNorm / SiLU launches of the prompt pass leave the tokens' largest |x| for the FP16 GEMM's pre-pass (A/B switch)
    float* row_max_ = nullptr;       // [2][max_seq]: the prompt tokens' largest |x| beside the RMSNorm / SiLU outputs (FP16 GEMM pre-pass)
    void* gemm_ws_ = nullptr;        // workspace of ntk_gemm_quant_ws (FP16 prompt projections), sized for max(H, I) columns
    void* gemm_ws2_ = nullptr;       // a second one: the launch that produces a projection's input writes that projection's planes (ntk_*_prepare_x) while it may
                                     // still read the previous projection's partial sums out of the other workspace
    bool prefill_fused_split_ = true;   // (A/B switch of that: 0 = the FP16 GEMM's own pre-pass launches)
    size_t gemm_ws_bytes_ = 0;
    bool bf16_prefill_ = true;
    unsigned* attn_sync_ = nullptr;  // 3 words for ntk_attention_gemv_fused (attention producers inside the Wo launch)
    int repack_ = 3;                 // EFFECTIVE level: 0 raw path, 1 repack + raw resident, 2 repack only (one resident copy); 3 only before a load
    int repack_wanted_ = 3;          // the level as ASKED (3 = "2 if memory is short else 1"): re-evaluated by every load
    bool repack_done_ = false;       // repack_all() ran on the loaded tensors
    uint64_t repack_bytes_ = 0;
    uint64_t raw_freed_bytes_ = 0;   // GGUF bytes released after the repack (level 2)
    void* raw_scratch_ = nullptr;    // where raw_of() unpacks to
    size_t raw_scratch_bytes_ = 0, raw_cursor_ = 0;
    int raw_err_ = 0;                // first failure inside raw_of() (it returns a pointer): ok() folds it into the forward's status
    bool attn_merge_ = false;        // split-KV attention without the combine launch (round 5; identical bits, measured 0-2 us per layer SLOWER: opt-in)
    bool fuse_attention_ = false;    // attention + Wo projection as one launch: measured SLOWER than two launches (profiles/r02_*): opt-in
    int tp_rank_ = 0, tp_world_ = 1;
    void* tp_comm_ = nullptr;        // this rank's communication buffer (flags + two slots of max_seq x H floats)
    size_t tp_max_floats_ = 0;
    void* tp_peers_[8] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    bool tp_peer_opened_[8] = {false, false, false, false, false, false, false, false};   // mapped through hipIpc (to be closed)
    bool tp_connected_ = false;
    unsigned tp_call_ = 0;           // all-reduce calls of the forward being enqueued (call k uses slot k & 1)
    bool own_stream_ = false;        // tensor-parallel ranks that share a process need private streams
    ModelConfig cfg_full_;           // the unsliced configuration (cfg_ holds the local head / FFN counts)
    void* persistent_plan_ = nullptr;
    bool persistent_on_ = false;   // opt-in until it beats the launch path on the bench (set_persistent / "persistent" option)
    int persistent_wanted_ = 0;    // the option as last set (re-applied after a load)
    int persistent_kind_ = 1;      // which kernel persistent_plan_ belongs to
};

}  // namespace nt
