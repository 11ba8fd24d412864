// engine/model.cpp -- see model.h
#include "model.h"
#include "../../../include/ntk_engine.h"
#include "../../../include/ntk_layers.h"
#ifdef NTK_EXPERIMENTS
#include "ntk_experiments.h"
#endif

#include <hip/hip_runtime.h>
#include <initializer_list>
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <chrono>
#include <thread>

namespace nt {

#define NT_TRY(expr)                       \
    do {                                   \
        const int st__ = (expr);           \
        if (st__ != NTK_OK) return st__;   \
    } while (0)

static bool is_quant(int dt) {
    return dt == NTK_DT_Q8_0 || dt == NTK_DT_Q4_0 || dt == NTK_DT_Q4_K || dt == NTK_DT_Q5_K || dt == NTK_DT_Q6_K;
}

Model::~Model() { free_all(); }

void Model::free_all() {
    for (auto& row : graphs_)
        for (auto& gx : row) {
            if (gx) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(gx));
            gx = nullptr;
        }
#ifdef NTK_EXPERIMENTS
    if (persistent_plan_) { if (persistent_kind_ == 2) ntk_layer_engine_plan_destroy(persistent_plan_); else ntk_persistent_plan_destroy(persistent_plan_); }
#endif
    persistent_plan_ = nullptr;
    persistent_on_ = false;
    for (int r = 0; r < 8; ++r) {   // peers' communication buffers mapped through hipIpc
        if (tp_peer_opened_[r] && tp_peers_[r]) (void)ntk_ipc_close(tp_peers_[r]);
        tp_peers_[r] = nullptr;
        tp_peer_opened_[r] = false;
    }
    tp_connected_ = false;
    tp_comm_ = nullptr;
    tp_call_ = 0;
    if (own_stream_ && stream_) (void)hipStreamDestroy(static_cast<hipStream_t>(stream_));
    own_stream_ = false;
    stream_ = nullptr;
    for (void* p : allocs_) nt_hip_free(p);
    allocs_.clear();
    if (h_token_) nt_hip_free_host(h_token_);
    h_token_ = nullptr;
    if (h_ring_) nt_hip_free_host(h_ring_);
    h_ring_ = nullptr;
    if (h_recent_) nt_hip_free_host(h_recent_);
    h_recent_ = nullptr;
    out_row_.clear();
    sample_scratch_ = nullptr;
    d_recent_ = nullptr;
    attn_sync_ = nullptr;
    gemm_ws_ = gemm_ws2_ = nullptr;
    shares_weights_ = false;   // (allocs_ held only this object's own buffers: the tensors belong to the model they were shared from)
    layers_.clear();
    // a second load() on the same object starts from a clean slate
    token_embd_ = output_norm_ = output_ = DevTensor();
    weight_bytes_ = 0;
    repack_bytes_ = 0;
    raw_freed_bytes_ = 0;
    raw_scratch_ = nullptr; raw_scratch_bytes_ = raw_cursor_ = 0; raw_err_ = 0;
    repack_done_ = false;
    output_tied_ = false;
    host_pos_ = 0;
    attn_regime_ = 0;
    k_cache_ = v_cache_ = nullptr;
    hidden_ = residual_ = workspace_ = logits_ = argmax_scratch_ = rope_inv_freq_ = rope_angles_ = attn_scratch_ = row_max_ = nullptr;
    positions_ = tokens_dev_ = d_pos_ = d_token_ = nullptr;
}

int Model::upload(DevTensor& dst, const void* host, int dtype, int64_t in_f, int64_t out_f, size_t nbytes) {
    void* d = nt_hip_malloc((nbytes + 255) / 256 * 256 + 256);   // tail padding: kernels may read the last 16-byte chunk whole
    if (!d) { err_ = "out of device memory"; return NTK_E_NOMEM; }
    allocs_.push_back(d);
    if (host && nbytes) {   // a failed upload must not leave silently garbage weights behind
        if (hipMemcpy(d, host, nbytes, hipMemcpyHostToDevice) != hipSuccess) { err_ = "weight upload (H2D copy) failed"; return NTK_E_LAUNCH; }
    }
    dst.ptr = d; dst.dtype = dtype; dst.in_f = in_f; dst.out_f = out_f; dst.nbytes = nbytes;
    weight_bytes_ += nbytes;
    return NTK_OK;
}

// ---- tensor parallelism: slices ---------------------------------------------------------------------------------------------
int Model::tp_configure(int rank, int world) {
    if (world < 1 || world > 8 || rank < 0 || rank >= world) { err_ = "bad tensor-parallel rank / world"; return NTK_E_SHAPE; }
    if (!layers_.empty()) { err_ = "tp_configure must precede load"; return NTK_E_SHAPE; }
    tp_rank_ = rank;
    tp_world_ = world;
    return NTK_OK;
}

int Model::slice_columns(void* dst, const void* src, int dtype, int64_t out_f, int64_t in_f, int rank, int world) {
    if (!dst || !src) return NTK_E_NULL;
    if (world < 1 || rank < 0 || rank >= world || in_f % world != 0) return NTK_E_SHAPE;
    const int64_t in_l = in_f / world;
    const size_t rb_full = ntk_row_bytes(dtype, in_f), rb_loc = ntk_row_bytes(dtype, in_l);
    if (!rb_full || !rb_loc || rb_loc * (size_t)world != rb_full) return NTK_E_SHAPE;   // the slice must be whole blocks
    const uint8_t* s8 = static_cast<const uint8_t*>(src);
    uint8_t* d8 = static_cast<uint8_t*>(dst);
    for (int64_t r = 0; r < out_f; ++r) memcpy(d8 + (size_t)r * rb_loc, s8 + (size_t)r * rb_full + (size_t)rank * rb_loc, rb_loc);
    return NTK_OK;
}

int Model::upload_shard(DevTensor& dst, const void* host_full, int dtype, int64_t in_f, int64_t out_f, size_t nbytes_full, Shard how) {
    if (tp_world_ == 1 || how == WHOLE) return upload(dst, host_full, dtype, in_f, out_f, nbytes_full);
    if (how == ROWS) {   // rows are contiguous: a byte range
        const int64_t rows = out_f / tp_world_;
        const size_t rb = ntk_row_bytes(dtype, in_f);
        if (out_f % tp_world_ != 0 || !rb) { err_ = "tensor rows do not divide over the tensor-parallel ranks"; return NTK_E_SHAPE; }
        return upload(dst, static_cast<const uint8_t*>(host_full) + (size_t)tp_rank_ * rows * rb, dtype, in_f, rows, (size_t)rows * rb);
    }
    const int64_t in_l = in_f / tp_world_;
    const size_t rb_loc = ntk_row_bytes(dtype, in_l);
    std::vector<uint8_t> tmp((size_t)out_f * rb_loc);
    const int st = slice_columns(tmp.data(), host_full, dtype, out_f, in_f, tp_rank_, tp_world_);
    if (st != NTK_OK) { err_ = "tensor columns do not divide into whole blocks over the tensor-parallel ranks"; return st; }
    return upload(dst, tmp.data(), dtype, in_l, out_f, tmp.size());
}

int Model::tp_check_shapes() {
    if (tp_world_ == 1) return NTK_OK;
    if (cfg_.n_heads % tp_world_ || cfg_.n_kv_heads % tp_world_ || cfg_.intermediate_size % tp_world_) {
        err_ = "heads / KV heads / FFN width do not divide over the tensor-parallel ranks";
        return NTK_E_SHAPE;
    }
    return NTK_OK;
}

int Model::tp_export(void* handle64, void** raw) {
    if (!tp_comm_) return NTK_E_NULL;
    if (raw) *raw = tp_comm_;
    if (handle64) return ntk_ipc_export(tp_comm_, handle64);
    return NTK_OK;
}

int Model::tp_connect(const void* handles, void* const* raws) {
    if (tp_world_ == 1) { tp_connected_ = true; return NTK_OK; }
    if (!tp_comm_ || (!handles && !raws)) return NTK_E_NULL;
    for (int r = 0; r < tp_world_; ++r) {
        if (r == tp_rank_) { tp_peers_[r] = tp_comm_; continue; }
        if (raws) { tp_peers_[r] = raws[r]; continue; }
        void* p = nullptr;
        const int st = ntk_ipc_open(static_cast<const uint8_t*>(handles) + 64 * r, &p);
        if (st != NTK_OK) { err_ = "mapping a peer's communication buffer failed (hipIpcOpenMemHandle)"; return st; }
        tp_peers_[r] = p;
        tp_peer_opened_[r] = true;
    }
    for (int r = 0; r < tp_world_; ++r)
        if (!tp_peers_[r]) return NTK_E_NULL;
    tp_connected_ = true;
    return NTK_OK;
}

unsigned Model::tp_error() {
    if (!tp_comm_) return 0u;
    unsigned v = 0;   // read on the model's own stream (no legacy-stream traffic next to another rank's capture)
    if (ntk_memcpy_d2h_async(&v, static_cast<uint8_t*>(tp_comm_) + 128, 4, stream_) != NTK_OK || ntk_stream_synchronize(stream_) != NTK_OK) return ~0u;
    return v;
}
float* Model::tp_slot() const { return ntk_tp_slot(tp_comm_, tp_max_floats_, tp_call_); }
int Model::tp_allreduce(float* hidden, int n) {
    if (!tp_connected_) { err_ = "tensor-parallel ranks are not connected (tp_connect)"; return NTK_E_NULL; }
    const int st = ntk_tp_allreduce_add(hidden, tp_peers_, tp_rank_, tp_world_, tp_max_floats_, tp_call_, n, stream_);
    ++tp_call_;
    return st;
}

int Model::load(const std::string& path, int max_context) {
    const int st = load_impl(path, max_context);
    if (st != NTK_OK) free_all();   // nothing stays resident after a failed load
    return st;
}

int Model::load_impl(const std::string& path, int max_context) {
    free_all();
    fprintf(stderr, "Loading model: %s\n", path.c_str());
    GgufFile f;
    int st = f.open(path);
    if (st != NTK_OK) { err_ = f.error(); fprintf(stderr, "%s\n", err_.c_str()); return st; }
    cfg_ = f.config();
    vocab_ = f.vocab();
    if (cfg_.max_seq_len > max_context) {   // transformer.cpp:70-74
        fprintf(stderr, "Note: Capping context from %d to %d tokens (use --ctx-size to change)\n", cfg_.max_seq_len, max_context);
        cfg_.max_seq_len = max_context;
    }
    cfg_.print();
    f.print_info();
    int dev = 0;
    if (const char* e = getenv("NTK_DEVICE")) dev = atoi(e);
    st = ntk_device_init(dev);
    if (st != NTK_OK) { err_ = "no usable GPU (HIP device init failed)"; fprintf(stderr, "%s\n", err_.c_str()); return st; }

    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim;
    const int64_t qd = (int64_t)cfg_.n_heads * hd, kvd = (int64_t)cfg_.n_kv_heads * hd;
    NT_TRY(tp_check_shapes());
    auto take = [&](const std::string& name, DevTensor& dst, int64_t in_f, int64_t out_f, bool vec, Shard how = WHOLE) -> int {
        const GgufTensor* t = f.find(name);
        if (!t) { err_ = "Tensor not found: " + name; return NTK_E_FORMAT; }
        if (t->numel() != in_f * out_f || (!vec && (t->dims.size() != 2 || t->dims[0] != in_f))) {
            err_ = "Unexpected shape for " + name;
            return NTK_E_SHAPE;
        }
        if (vec && t->dtype != NTK_DT_F32) { err_ = name + " must be F32"; return NTK_E_DTYPE; }
        if (t->nbytes == 0 || !t->known_type) { err_ = "Unsupported tensor type for " + name; return NTK_E_DTYPE; }
        return upload_shard(dst, f.data(*t), t->dtype, in_f, out_f, t->nbytes, how);
    };
    NT_TRY(take("token_embd.weight", token_embd_, H, cfg_.vocab_size, false));
    if (f.find("output.weight")) {   // transformer.cpp:92-99
        NT_TRY(take("output.weight", output_, H, cfg_.vocab_size, false));
    } else {
        output_ = token_embd_;
        output_tied_ = true;
    }
    NT_TRY(take("output_norm.weight", output_norm_, H, 1, true));
    layers_.resize(cfg_.n_layers);
    for (int i = 0; i < cfg_.n_layers; ++i) {   // transformer.cpp:286-328
        const std::string p = "blk." + std::to_string(i) + ".";
        LayerWeights& L = layers_[i];
        NT_TRY(take(p + "attn_norm.weight", L.attn_norm, H, 1, true));
        NT_TRY(take(p + "attn_q.weight", L.wq, H, qd, false, ROWS));      // whole heads per rank
        NT_TRY(take(p + "attn_k.weight", L.wk, H, kvd, false, ROWS));
        NT_TRY(take(p + "attn_v.weight", L.wv, H, kvd, false, ROWS));
        NT_TRY(take(p + "attn_output.weight", L.wo, qd, H, false, COLS));  // the columns of this rank's heads
        NT_TRY(take(p + "ffn_norm.weight", L.ffn_norm, H, 1, true));
        NT_TRY(take(p + "ffn_gate.weight", L.w_gate, H, I, false, ROWS));
        NT_TRY(take(p + "ffn_up.weight", L.w_up, H, I, false, ROWS));
        NT_TRY(take(p + "ffn_down.weight", L.w_down, I, H, false, COLS));
    }
    return finish_load(max_context);
}

int Model::load_synthetic(const SynthSpec& spec, int max_context, int nthreads) {
    free_all();
    std::vector<SynthTensor> plan;
    if (!synth_plan(spec, plan)) { err_ = "bad synthetic spec"; return NTK_E_SHAPE; }
    cfg_ = ModelConfig();
    cfg_.model_name = "synthetic-" + spec.mix;
    cfg_.vocab_size = spec.vocab; cfg_.hidden_size = spec.hidden; cfg_.intermediate_size = spec.inter;
    cfg_.n_layers = spec.layers; cfg_.n_heads = spec.heads; cfg_.n_kv_heads = spec.kv_heads;
    cfg_.head_dim = spec.hidden / spec.heads;
    cfg_.norm_eps = spec.eps; cfg_.rope_theta = spec.theta;
    cfg_.max_seq_len = std::min(spec.ctx, max_context);
    cfg_.bos_token_id = spec.bos; cfg_.eos_token_id = spec.eos;
    synth_vocab(spec, vocab_.tokens, vocab_.token_types);
    int dev = 0;
    if (const char* e = getenv("NTK_DEVICE")) dev = atoi(e);
    const int st = ntk_device_init(dev);
    if (st != NTK_OK) { err_ = "no usable GPU (HIP device init failed)"; return st; }
    { const int ts = tp_check_shapes(); if (ts != NTK_OK) return ts; }

    size_t biggest = 0;
    for (const auto& t : plan) biggest = std::max(biggest, t.nbytes);
    void* stage = nt_hip_malloc_host(biggest);
    if (!stage) { err_ = "pinned staging allocation failed"; return NTK_E_NOMEM; }
    layers_.resize(cfg_.n_layers);
    int rc = NTK_OK;
    for (const auto& t : plan) {
        synth_fill(stage, t, spec.seed, nthreads);
        DevTensor* dst = nullptr;
        if (t.name == "token_embd.weight") dst = &token_embd_;
        else if (t.name == "output.weight") dst = &output_;
        else if (t.name == "output_norm.weight") dst = &output_norm_;
        else {
            int li = 0;
            char what[64] = {0};
            if (sscanf(t.name.c_str(), "blk.%d.%63s", &li, what) != 2) { rc = NTK_E_FORMAT; break; }
            LayerWeights& L = layers_[li];
            const std::string w = what;
            dst = w == "attn_norm.weight" ? &L.attn_norm : w == "attn_q.weight" ? &L.wq : w == "attn_k.weight" ? &L.wk
                : w == "attn_v.weight" ? &L.wv : w == "attn_output.weight" ? &L.wo : w == "ffn_norm.weight" ? &L.ffn_norm
                : w == "ffn_gate.weight" ? &L.w_gate : w == "ffn_up.weight" ? &L.w_up : &L.w_down;
        }
        Shard how = WHOLE;
        if (t.name.find("attn_q.") != std::string::npos || t.name.find("attn_k.") != std::string::npos || t.name.find("attn_v.") != std::string::npos ||
            t.name.find("ffn_gate.") != std::string::npos || t.name.find("ffn_up.") != std::string::npos) how = ROWS;
        else if (t.name.find("attn_output.") != std::string::npos || t.name.find("ffn_down.") != std::string::npos) how = COLS;
        rc = upload_shard(*dst, stage, ggml_type_to_dtype((uint32_t)t.ggml_type), t.in_f, t.out_f, t.nbytes, how);
        if (rc != NTK_OK) break;
    }
    nt_hip_free_host(stage);
    if (rc == NTK_OK) rc = finish_load(max_context);
    if (rc != NTK_OK) free_all();
    return rc;
}

int Model::share_weights(const Model& src, int max_context) {
    if (&src == this) { err_ = "share_weights: a model cannot share its own weights"; return NTK_E_NULL; }
    free_all();
    if (src.layers_.empty()) { err_ = "share_weights: the source model is not loaded"; return NTK_E_NULL; }
    if (src.tp_world_ != 1 || src.shares_weights_) {
        err_ = "share_weights: the source must hold whole tensors of its own (no tensor parallelism, not itself a sharing sequence)";
        return NTK_E_SHAPE;
    }
    cfg_ = src.cfg_;
    cfg_full_ = src.cfg_;
    if (max_context > 0) cfg_.max_seq_len = max_context;
    vocab_ = src.vocab_;
    layers_ = src.layers_;               // the same device pointers (raw GGUF bytes and the decode repack): read-only for every launch
    token_embd_ = src.token_embd_; output_norm_ = src.output_norm_; output_ = src.output_;
    output_tied_ = src.output_tied_;
    weight_bytes_ = src.weight_bytes_;   // (bytes_per_token: the bytes a token of THIS sequence streams)
    repack_ = src.repack_; repack_wanted_ = src.repack_; repack_done_ = true;
    repack_bytes_ = 0;                   // none of it is this object's
    shares_weights_ = true;
    if (src.raw_freed_bytes_ > 0 && src.raw_scratch_bytes_ > 0) {   // one resident copy: what still reads raw blocks (the 1:1 sequence, the prompt's LM head) unpacks
        void* d = nt_hip_malloc(src.raw_scratch_bytes_);         // into a scratch of THIS sequence (stream ordered on this sequence's stream)
        if (!d) { err_ = "share_weights: no device memory for the unpack scratch"; free_all(); return NTK_E_NOMEM; }
        allocs_.push_back(d);
        raw_scratch_ = d; raw_scratch_bytes_ = src.raw_scratch_bytes_;
        raw_freed_bytes_ = src.raw_freed_bytes_;
    }
    hipStream_t own = nullptr;
    if (hipStreamCreateWithFlags(&own, hipStreamNonBlocking) != hipSuccess) { err_ = "stream creation failed"; free_all(); return NTK_E_LAUNCH; }
    stream_ = own;
    own_stream_ = true;
    const int rc = alloc_buffers();
    if (rc != NTK_OK) free_all();
    return rc;
}

int Model::finish_load(int /*max_context*/) {
    cfg_full_ = cfg_;
    if (tp_world_ > 1) {   // from here on this object IS a model with 1/W of the heads and of the FFN width (hidden size unchanged)
        cfg_.n_heads /= tp_world_;
        cfg_.n_kv_heads /= tp_world_;
        cfg_.intermediate_size /= tp_world_;
        hipStream_t own = nullptr;   // ranks that share a process (tests) must not queue behind each other's waiting kernels
        if (hipStreamCreateWithFlags(&own, hipStreamNonBlocking) != hipSuccess) { err_ = "stream creation failed"; return NTK_E_LAUNCH; }
        stream_ = own;
        own_stream_ = true;
    } else {
        stream_ = ntk_stream(0);
    }
    if (!stream_) { err_ = "no compute stream"; return NTK_E_NODEVICE; }
    NT_TRY(alloc_buffers());
    repack_ = repack_wanted_;   // every load decides anew (a level-3 request that ended as 1 or 2 on the previous model must not stick)
    if (repack_) {
        // ADVICE (round 4): a repack that does not fit must not fail the load -- the raw path decodes every tensor that has no repacked form
        const int st = repack_all();
        if (st == NTK_E_NOMEM) {
            int kept = 0;
            for (auto& L : layers_) for (DevTensor* t : {&L.wq, &L.wk, &L.wv, &L.wo, &L.w_gate, &L.w_up, &L.w_down}) kept += t->rp ? 0 : 1;
            fprintf(stderr, "warning: not enough device memory for the decode repack of every matrix: %d projection tensors stay on the raw-GGUF path\n", kept);
            err_.clear();
        } else if (st != NTK_OK) {
            return st;
        }
        if (repack_ == 3) repack_ = 2;   // round 6: the prompt GEMM reads the repack itself, so the second copy buys the batched paths nothing
        if (repack_ == 2) NT_TRY(drop_raw_all());
    }
    if (persistent_wanted_) set_persistent(persistent_wanted_);
    size_t fr = 0, tot = 0;
    ntk_device_mem_info(&fr, &tot);
    fprintf(stderr, "Model loaded successfully! (resident on MI355X: %.2f GB of weights%s)\nFree VRAM: %.1f GB\n",
            (weight_bytes_ - raw_freed_bytes_) / 1073741824.0, repack_bytes_ ? (" + " + std::to_string(repack_bytes_ / 1073741824.0).substr(0, 5) + " GB repacked for decode").c_str() : "",
            fr / 1073741824.0);
    return NTK_OK;
}

// ---- engine-owned repack of the K-quant projections (csrc/gemv_rp.hip): made once, on the device, from the uploaded GGUF bytes, which
//      stay resident for the 1:1 launchers and the prompt GEMM ----
int Model::repack_one(DevTensor& t) {
    if (t.rp || !t.ptr) return NTK_OK;
    if (t.out_f <= 0 || t.out_f > 0x7FFFFFFF || t.in_f <= 0 || t.in_f > 32768) return NTK_OK;
    const size_t n = ntk_rp_bytes(t.dtype, (int)t.out_f, (int)t.in_f);
    if (n == 0 || n > 0xFFFFFFF0ull) return NTK_OK;   // formats / shapes the matrix-core GEMV does not take keep the raw path
    void* d = nt_hip_malloc(n + 256);
    if (!d) return NTK_E_NOMEM;   // (the caller keeps the tensors that did fit and lets the raw path take the rest)
    allocs_.push_back(d);
    const int st = ntk_rp_pack(d, t.ptr, (int)t.out_f, (int)t.in_f, t.dtype, stream_);
    if (st != NTK_OK) { err_ = std::string("decode repack failed: ") + ntk_status_string(st); return st; }
    t.rp = d;
    t.rp_bytes = n;
    repack_bytes_ += n;
    return NTK_OK;
}

int Model::repack_all() {
    int rc = NTK_OK;
    auto one = [&](DevTensor& t) { const int st = repack_one(t); if (st != NTK_OK && rc == NTK_OK) rc = st; return st; };
    for (auto& L : layers_) {
        if (one(L.wq) == NTK_E_NOMEM) break;
        one(L.wk); one(L.wv); one(L.wo); one(L.w_gate); one(L.w_up); one(L.w_down);
        if (rc == NTK_E_NOMEM) break;
    }
    if (rc != NTK_E_NOMEM) one(output_);
    repack_done_ = true;
    const int sy = ntk_stream_synchronize(stream_);
    return rc != NTK_OK ? rc : sy;
}

// ---- one resident copy (level 2): the uploaded GGUF bytes of every repacked matrix go; raw_of() unpacks on demand ----
int Model::drop_raw_all() {
    size_t need = 0;
    auto grp = [&](std::initializer_list<DevTensor*> ts) {
        size_t g = 0;
        for (DevTensor* t : ts) if (t->rp && !(output_tied_ && t->ptr == token_embd_.ptr)) g += (t->nbytes + 255) / 256 * 256 + 256;
        need = std::max(need, g);
    };
    for (auto& L : layers_) { grp({&L.wq, &L.wk, &L.wv}); grp({&L.wo}); grp({&L.w_gate, &L.w_up}); grp({&L.w_down}); }
    grp({&output_});
    if (need == 0) return NTK_OK;
    if (!raw_scratch_ || raw_scratch_bytes_ < need) {
        void* d = nt_hip_malloc(need);
        if (!d) { fprintf(stderr, "warning: no device memory for the unpack scratch: the GGUF bytes stay resident beside the repack\n"); repack_ = 1; return NTK_OK; }
        allocs_.push_back(d);
        raw_scratch_ = d; raw_scratch_bytes_ = need;
    }
    auto drop = [&](DevTensor& t) {
        if (!t.rp || !t.ptr || (output_tied_ && t.ptr == token_embd_.ptr)) return;
        auto it = std::find(allocs_.begin(), allocs_.end(), t.ptr);
        if (it != allocs_.end()) allocs_.erase(it);
        nt_hip_free(t.ptr);
        t.ptr = nullptr;
        raw_freed_bytes_ += t.nbytes;
    };
    NT_TRY(ntk_stream_synchronize(stream_));
    for (auto& L : layers_) { drop(L.wq); drop(L.wk); drop(L.wv); drop(L.wo); drop(L.w_gate); drop(L.w_up); drop(L.w_down); }
    drop(output_);
    return NTK_OK;
}

int Model::restore_raw_all() {
    int rc = NTK_OK;
    auto back = [&](DevTensor& t) {
        if (t.ptr || !t.rp || rc != NTK_OK) return;
        void* d = nt_hip_malloc((t.nbytes + 255) / 256 * 256 + 256);
        if (!d) { rc = NTK_E_NOMEM; return; }
        const int st = ntk_rp_unpack(d, t.rp, (int)t.out_f, (int)t.in_f, t.dtype, stream_);
        if (st != NTK_OK) { nt_hip_free(d); rc = st; return; }
        allocs_.push_back(d);
        t.ptr = d;
        raw_freed_bytes_ -= t.nbytes;
    };
    for (auto& L : layers_) { back(L.wq); back(L.wk); back(L.wv); back(L.wo); back(L.w_gate); back(L.w_up); back(L.w_down); }
    back(output_);
    const int sy = ntk_stream_synchronize(stream_);
    return rc != NTK_OK ? rc : sy;
}

const void* Model::raw_of(const DevTensor& t) {
    if (t.ptr) return t.ptr;
    if (!t.rp || !raw_scratch_) { raw_err_ = NTK_E_NULL; return nullptr; }
    const size_t n = (t.nbytes + 255) / 256 * 256 + 256;
    if (raw_cursor_ + n > raw_scratch_bytes_) {   // a group never exceeds the scratch (sized for the largest in drop_raw_all): wrapping would overwrite a tensor the same launch still reads
        if (!raw_err_) raw_err_ = NTK_E_NOMEM;
        return nullptr;
    }
    void* d = static_cast<uint8_t*>(raw_scratch_) + raw_cursor_;
    raw_cursor_ += n;
    const int st = ntk_rp_unpack(d, t.rp, (int)t.out_f, (int)t.in_f, t.dtype, stream_);
    if (st != NTK_OK) { raw_err_ = st; return nullptr; }
    return d;
}

int Model::set_attention_merge(bool on) {
    if (on == attn_merge_) return NTK_OK;
    if (!layers_.empty()) {
        NT_TRY(sync());
        for (auto& row : graphs_) for (auto& gx : row) { if (gx) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(gx)); gx = nullptr; }
    }
    attn_merge_ = on;
    return NTK_OK;
}

int Model::set_repack(int level) {
    level = level < 0 ? 0 : level > 3 ? 3 : level;
    if (shares_weights_) { err_ = "set_repack: this sequence shares another model's tensors"; return NTK_E_SHAPE; }
    repack_wanted_ = level;
    if (layers_.empty()) { repack_ = level; return NTK_OK; }   // before the load: finish_load() decides
    if (level == 3) level = 2;   // (round 6: one resident copy; what is gone stays gone)
    if (level == repack_) return NTK_OK;
    NT_TRY(sync());
    for (auto& row : graphs_) for (auto& gx : row) { if (gx) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(gx)); gx = nullptr; }
    int rc = NTK_OK;
    if (level < 2 && raw_freed_bytes_ > 0) rc = restore_raw_all();           // the GGUF bytes come back first (levels 0 and 1 read them)
    if (rc == NTK_OK && level > 0 && !repack_done_) {
        rc = repack_all();
        if (rc == NTK_E_NOMEM) { fprintf(stderr, "warning: decode repack incomplete (device memory): the rest stays on the raw path\n"); rc = NTK_OK; err_.clear(); }
    }
    if (rc != NTK_OK) { err_ = std::string("set_repack: ") + ntk_status_string(rc); return rc; }
    repack_ = level;
    if (level == 2) {
#ifdef NTK_EXPERIMENTS
        // the persistent kernels stream the uploaded GGUF bytes through the pointers their plan recorded: a plan must not outlive them
        if (persistent_plan_) {
            for (auto& row : graphs_) { if (row[kPersistentSlot]) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(row[kPersistentSlot])); row[kPersistentSlot] = nullptr; }
            if (persistent_kind_ == 2) ntk_layer_engine_plan_destroy(persistent_plan_); else ntk_persistent_plan_destroy(persistent_plan_);
            persistent_plan_ = nullptr;
        }
#endif
        persistent_on_ = false;
        rc = drop_raw_all();
    }
    return rc;
}

int Model::alloc_buffers() {   // transformer.cpp:330-391
    const size_t S = (size_t)cfg_.max_seq_len, H = (size_t)cfg_.hidden_size, L = (size_t)cfg_.n_layers;
    const size_t per = (size_t)cfg_.n_kv_heads * cfg_.head_dim;
    auto dev = [&](size_t bytes, bool zero) -> void* {
        void* p = nt_hip_malloc(bytes + 256);
        if (p) { allocs_.push_back(p); if (zero) nt_hip_memset(p, 0, bytes); }
        return p;
    };
    // the attention kernels address a layer's cache rows with 32-bit byte offsets (attention.hip): a context whose per-layer cache reaches
    // 3.75 GiB is refused here, at load, rather than as NTK_E_SHAPE from the first decode step (8 KV heads of 128: 1.9 M positions)
    if (S * per * sizeof(uint16_t) >= 0xF0000000ull) { err_ = "context too long: one layer's K cache must stay below 3.75 GiB (32-bit row offsets)"; return NTK_E_SHAPE; }
    const size_t kvb = L * S * per * sizeof(uint16_t);
    k_cache_ = (uint16_t*)dev(kvb, true);
    v_cache_ = (uint16_t*)dev(kvb, true);
    hidden_ = (float*)dev(std::max<size_t>(S, 2) * H * 4, false);
    residual_ = (float*)dev(std::max<size_t>(S, 2) * H * 4, false);
    logits_ = (float*)dev((size_t)cfg_.vocab_size * 4, false);
    const size_t attn_ws = S * (size_t)(2 * cfg_.n_heads + 2 * cfg_.n_kv_heads) * cfg_.head_dim;
    const size_t ffn_ws = 2 * S * (size_t)cfg_.intermediate_size;
    workspace_floats_ = std::max(attn_ws, ffn_ws);
    workspace_ = (float*)dev(workspace_floats_ * 4, false);
    positions_ = (int*)dev(S * 4, false);
    tokens_dev_ = (int*)dev(S * 4, false);
    d_pos_ = (int*)dev(64, true);
    d_token_ = (int*)dev(64, true);
    argmax_scratch_ = (float*)dev(2 * 1024 * 4, false);
    rope_inv_freq_ = (float*)dev((size_t)cfg_.head_dim / 2 * 4 + 64, false);
    rope_angles_ = (float*)dev(ntk_short_angles_bytes(cfg_.head_dim) + 64, false);
    row_max_ = (float*)dev((size_t)S * 2 * 4, true);
    attn_scratch_ = (float*)dev(ntk_attention_split_scratch_bytes(cfg_.n_heads, cfg_.head_dim, kMaxAttnSplits), true);   // (zeroed: the arrival counters in front)
    h_token_ = (int*)nt_hip_malloc_host(64);
    h_ring_ = (unsigned long long*)nt_hip_malloc_host(64);
    out_row_.alloc((size_t)cfg_.vocab_size);   // (none: a copy of the runtime's)
    if (h_ring_) memset(h_ring_, 0, 64);
    sample_scratch_ = dev(ntk_sample_scratch_bytes(cfg_.vocab_size), false);
    attn_sync_ = (unsigned*)dev(4096, true);
    {   // one workspace for every projection: the largest need over the launches the prompt pass makes (Q|K|V and gate|up go out as one)
        const int H = cfg_.hidden_size, I = cfg_.intermediate_size, qkv = (cfg_.n_heads + 2 * cfg_.n_kv_heads) * cfg_.head_dim;
        const int shapes[][2] = {{H, qkv}, {H, cfg_.n_heads * cfg_.head_dim}, {H, cfg_.n_kv_heads * cfg_.head_dim}, {cfg_.n_heads * cfg_.head_dim, H},
                                 {H, 2 * I}, {H, I}, {I, H}};
        gemm_ws_bytes_ = 0;
        for (const auto& sh : shapes) gemm_ws_bytes_ = std::max(gemm_ws_bytes_, ntk_gemm_quant_workspace_bytes(sh[0], sh[1]));
    }
    short_known_[0] = short_known_[1] = -1;
    gemm_ws_ = dev(gemm_ws_bytes_, false);
    gemm_ws2_ = dev(gemm_ws_bytes_, false);
    if (tp_world_ > 1) {   // communication buffer: flags + two slots of one prompt's worth of hidden vectors
        tp_max_floats_ = S * H;
        tp_comm_ = ntk_tp_comm_alloc(ntk_tp_comm_bytes(tp_max_floats_));   // fine-grained: csrc/tp.hip
        if (tp_comm_) allocs_.push_back(tp_comm_);
        if (!tp_comm_ || ntk_tp_comm_reset(tp_comm_, nullptr) != NTK_OK || ntk_device_synchronize() != NTK_OK) { err_ = "communication buffer allocation failed"; return NTK_E_NOMEM; }
    }
    d_recent_ = (int*)dev(kRecentCap * 4, false);
    h_recent_ = (int*)nt_hip_malloc_host(kRecentCap * 4);
    if (!k_cache_ || !v_cache_ || !hidden_ || !residual_ || !logits_ || !workspace_ || !positions_ || !tokens_dev_ ||
        !d_pos_ || !d_token_ || !argmax_scratch_ || !h_token_ || !h_ring_) {
        err_ = "buffer allocation failed";
        return NTK_E_NOMEM;
    }
    *h_token_ = 0;
    if (rope_inv_freq_) {
        std::vector<float> f((size_t)cfg_.head_dim / 2);
        for (int i = 0; i < cfg_.head_dim / 2; ++i) f[i] = 1.0f / powf(cfg_.rope_theta, (2.0f * i) / cfg_.head_dim);
        nt_hip_memcpy_h2d(rope_inv_freq_, f.data(), f.size() * 4);
    }
    if (rope_angles_) {   // (none: short prompts rotate in a launch of their own)
        if (ntk_short_angles(rope_angles_, cfg_.head_dim, cfg_.rope_theta, cfg_.rope_freq_scale, stream_) != NTK_OK || ntk_stream_synchronize(stream_) != NTK_OK) return NTK_E_LAUNCH;
    }
    return NTK_OK;
}

uint64_t Model::bytes_per_token(int pos) const {
    uint64_t b = 0;
    for (const auto& L : layers_)
        b += L.wq.nbytes + L.wk.nbytes + L.wv.nbytes + L.wo.nbytes + L.w_gate.nbytes + L.w_up.nbytes + L.w_down.nbytes;
    b += output_.nbytes;
    b += (uint64_t)(2 * cfg_.n_layers + 1) * cfg_.hidden_size * 4;
    const uint64_t kv_row = (uint64_t)cfg_.n_kv_heads * cfg_.head_dim * 2;
    b += 2ull * cfg_.n_layers * kv_row * (uint64_t)(pos + 1) + 2ull * cfg_.n_layers * kv_row;
    b += ntk_row_bytes(token_embd_.dtype, cfg_.hidden_size);
    return b;
}

// ---------------------------------------------------------------------------------------------------
// 1:1 path: the reference's own launcher sequence (transformer.cpp:604-669, attention.cpp:120-211,
// ffn.cpp:85-134), through the same C ABI an external caller would use
// ---------------------------------------------------------------------------------------------------
float* Model::forward(const int* tokens, int T, int start_pos) {
    if (T <= 0 || start_pos < 0 || start_pos + T > cfg_.max_seq_len) { err_ = "forward: sequence exceeds context"; return nullptr; }
    for (int i = 0; i < T; ++i)   // the embedding gather indexes the table with these on the device
        if (tokens[i] < 0 || tokens[i] >= cfg_.vocab_size) { err_ = "forward: token id out of range"; return nullptr; }
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim, nh = cfg_.n_heads, nkv = cfg_.n_kv_heads;
    const int qd = nh * hd, kvd = nkv * hd;
    void* s = stream_;
    tp_call_ = 0;
    // embedding rows are dequantised on the device (the reference does it on the host and uploads, :419-599)
    std::vector<int> pos(T);
    for (int i = 0; i < T; ++i) pos[i] = start_pos + i;
    const bool words = T <= 16;   // (tokens and positions as arguments of one launch)
    if (words) {
        std::vector<int> both(tokens, tokens + T);
        both.insert(both.end(), pos.begin(), pos.end());
        if (ntk_store_words(tokens_dev_, T, positions_, T, both.data(), s) != NTK_OK) return nullptr;
    } else if (ntk_memcpy_h2d_async(tokens_dev_, tokens, (size_t)T * 4, s) != NTK_OK) return nullptr;
    const int est = ntk_embed_rows(hidden_, token_embd_.ptr, tokens_dev_, T, H, token_embd_.dtype, s);
    if (est == NTK_E_DTYPE) fprintf(stderr, "Error: Unsupported embedding dtype: %s\n", dtype_name(token_embd_.dtype));
    else if (est != NTK_OK) return nullptr;
    if (!words && ntk_memcpy_h2d_async(positions_, pos.data(), (size_t)T * 4, s) != NTK_OK) return nullptr;
    if (!words && ntk_stream_synchronize(s) != NTK_OK) return nullptr;   // `pos` / `tokens` are host temporaries

    // The last layer's results are read at the last token only: of the others it needs their cache rows, and from its attention on the pass goes on with the last few tokens -- from a row on 16 bytes,
    // two at least, by a prompt's own launches.  (As a decoded token the last one would have a K-quant's inputs rounded to 22 bits of their block's largest: 3.1e-7 of a product of normal
    // values, 1.6e-6 beside outliers, 1.6e-7 here in both; and those launches take fewer head sizes, contexts and widths.)  us, whole / so: four layers of the 8B shape in Q8_0, 33 tokens
    // 764 / 723, 1000 4643 / 3803; in Q4_K_M, 17 tokens 623 / 587; in F16, 33 tokens 661 / 642; two of the 70B shape in Q6_K, 17 tokens 1085 / 881.  Prompts of up to 16 tokens, and those of up to
    // 32 that layers_short takes or that are half-precision, spend a layer on its weights, not on its tokens.
    const bool tail = batched_prefill_ && tp_world_ == 1 && cfg_.n_layers > 0 && (T > 32 || (T > 16 && is_quant(layers_.back().w_down.dtype) && !short_prompt(T)));
    int rc = layers_1to1(T, start_pos, 0, cfg_.n_layers, tail);
    if (rc == NTK_OK && tail) {
        float* const rows = hidden_;
        const int few = 4 + T % 4;
        hidden_ += (size_t)(T - few) * H;
        rc = layers_1to1(few, start_pos + T - few, cfg_.n_layers - 1, cfg_.n_layers, false, workspace_ + (size_t)(T - few) * qd);
        hidden_ = rows;
    }
    auto ok = [&](int st) { if (st != NTK_OK && rc == NTK_OK) rc = st; };
    float* last = hidden_ + (size_t)(T - 1) * H;
    ok(ntk_rmsnorm(last, last, (const float*)output_norm_.ptr, 1, H, cfg_.norm_eps, s));   // in place, :658-659
    // (a repacked head is read as it lies, whether its GGUF blocks are resident or not: the same bits either way.  us, the GEMV over resident blocks / unpacking and that GEMV / so, Q4_K:
    // 32000 x 2048 17.6 / 41.9 / 14.5, 32000 x 4096 18.4 / 60.8 / 25.5, 128256 x 4096 55.6 / 262.8 / 67.0, 128256 x 8192 105.9 / 508.4 / 125.4: with the blocks resident, which has to be
    // asked for, up to 20 us of a pass are given for results that do not depend on it)
    int head = NTK_E_DTYPE;
    if (output_.rp) head = ntk_gemv_rp_f32(logits_, output_.rp, last, (int)output_.out_f, (int)output_.in_f, output_.dtype, s);
    if (head != NTK_E_DTYPE && head != NTK_E_SHAPE && head != NTK_E_ALIGN) ok(head);
    else {
        raw_begin();
        const int st = ntk_gemv(logits_, raw_of(output_), last, (int)output_.out_f, (int)output_.in_f, output_.dtype, s);
        if (st == NTK_E_DTYPE) fprintf(stderr, "Unsupported dtype for GEMV: %s\n", dtype_name(output_.dtype));   // gemm.cu:801-803
        else ok(st);
    }
    if (tp_world_ > 1) ok(ntk_tp_advance_epoch(tp_comm_, s));
    ok(ntk_stream_synchronize(s));
    if (raw_err_ != NTK_OK) { rc = raw_err_; raw_err_ = NTK_OK; }
    if (rc == NTK_OK) rc = check_tp();
    if (rc != NTK_OK) { if (err_.empty() || rc != NTK_E_LAUNCH) err_ = std::string("forward failed: ") + ntk_status_string(rc); return nullptr; }
    return logits_;
}

// a prompt of T <= 32 tokens whose matrices all take the form that keeps a K slice's planes in LDS (ntk_gemm_short): layers_short
bool Model::short_prompt(int T) const {
    if (T < 2 || T > 32 || !batched_prefill_ || !bf16_prefill_ || !gemm_ws_ || !gemm_ws2_ || tp_world_ > 1 || !row_max_ || !prefill_row_max_ || !prefill_fused_split_) return false;
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, qd = cfg_.n_heads * cfg_.head_dim;
    if (H % 32 || I % 32 || qd % 32) return false;
    // (the plans depend on the matrices and on how many blocks of 16 tokens there are)
    int& known = short_known_[T <= 16 ? 0 : 1];
    if (known < 0) known = short_matrices(T) ? 1 : 0;
    return known == 1;
}
bool Model::short_matrices(int T) const {
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, qd = cfg_.n_heads * cfg_.head_dim;
    auto takes = [&](const DevTensor& w, int in) {
        const int rows = (int)w.out_f;
        return is_quant(w.dtype) && (w.ptr || w.rp) && (int)w.in_f == in && ntk_gemm_short_takes(&rows, 1, T, in, w.dtype);
    };
    for (const LayerWeights& L : layers_) {
        if (!takes(L.wq, H) || !takes(L.wk, H) || !takes(L.wv, H) || !takes(L.wo, qd) || !takes(L.w_gate, H) || !takes(L.w_up, H) || !takes(L.w_down, I)) return false;
        if (L.w_gate.dtype != L.w_up.dtype || L.w_gate.out_f != L.w_up.out_f || (int)L.w_gate.out_f != I || (int)L.wo.out_f != H || (int)L.w_down.out_f != H) return false;
        // (matrices of one format go out together: their plan is the launch's, not each one's)
        const DevTensor* qkv[3] = {&L.wq, &L.wk, &L.wv};
        for (int a = 0; a < 3; ++a) {
            int rows[3], n = 0;
            for (int b = 0; b < 3; ++b)
                if (qkv[b]->dtype == qkv[a]->dtype) rows[n++] = (int)qkv[b]->out_f;
            if (!ntk_gemm_short_takes(rows, n, T, H, qkv[a]->dtype)) return false;
        }
        const int gu[2] = {I, I};
        if (!ntk_gemm_short_takes(gu, 2, T, H, L.w_gate.dtype)) return false;
    }
    return true;
}

// layers_1to1 for such a prompt: every producer of a projection's input leaves its planes in the workspace that the projection before it does not use (no whole row in one workgroup:
// gemm_f16.hip), every projection leaves its partial sums to the launch behind it.
int Model::layers_short(int T, int start_pos, int first, int last_layer) {
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim, nh = cfg_.n_heads, nkv = cfg_.n_kv_heads;
    const int qd = nh * hd, kvd = nkv * hd;
    void* s = stream_;
    const size_t kv_layer = (size_t)cfg_.max_seq_len * kvd;
    const float scale = 1.0f / sqrtf((float)hd);
    float* q_buf = workspace_;
    float* k_buf = q_buf + (size_t)T * qd;
    float* v_buf = k_buf + (size_t)T * kvd;
    float* attn_out = v_buf + (size_t)T * kvd;
    float* gate_buf = workspace_;
    float* up_buf = gate_buf + (size_t)T * I;
    void* ws = gemm_ws_;
    auto other = [&]() { ws = ws == gemm_ws_ ? gemm_ws2_ : gemm_ws_; return ws; };
    // (the repack wherever it is there, the file's blocks beside it or not: up to 16 tokens of many rows are multiplied in another order from it, and a prompt's bits are to be the same either way.
    // us, both copies resident, 16 tokens, sixteen 8B layers in Q4_K_M 1542 / 1329, eight in Q6_K 953 / 800)
    auto repacked = [&](const DevTensor* const* Ws, int n) {
        bool rp = true;
        for (int i = 0; i < n; ++i) rp = rp && Ws[i]->rp && Ws[i]->dtype != NTK_DT_Q8_0 && Ws[i]->dtype != NTK_DT_Q4_0;
        return rp;
    };
    auto describe = [&](const DevTensor* const* Ws, float* const* Ys, int n, const float* resid, ntk_gemm_partials* pt, bool rp, ntk_gemv_seg (&segs)[3]) {
        for (int i = 0; i < n; ++i) segs[i] = {rp ? Ws[i]->rp : raw_of(*Ws[i]), Ys[i], (int)Ws[i]->out_f, Ws[i]->dtype};
        ntk_gemm_desc d{};
        d.segs = segs; d.nseg = n; d.n_tokens = T; d.in_features = (int)Ws[0]->in_f; d.resid = resid;
        d.workspace = ws; d.workspace_bytes = gemm_ws_bytes_; d.partials = pt; d.weights_repacked = rp ? 1 : 0;
        return d;
    };
    auto gemm = [&](const DevTensor* const* Ws, float* const* Ys, int n, const float* resid, bool normed, size_t part_at, ntk_gemm_partials* pt) {
        const bool rp = repacked(Ws, n);
        if (!rp) raw_begin();
        ntk_gemv_seg segs[3];
        const ntk_gemm_desc d = describe(Ws, Ys, n, resid, pt, rp, segs);
        return ntk_gemm_short(&d, normed ? 1 : 0, cfg_.norm_eps, part_at, s);
    };
    NT_TRY(ntk_short_norm_prepare_x(hidden_, nullptr, (const float*)layers_[first].attn_norm.ptr, T, H, ws, s));
    for (int i = first; i < last_layer; ++i) {
        const LayerWeights& L = layers_[i];
        uint16_t* kc = k_cache_ + (size_t)i * kv_layer;
        uint16_t* vc = v_cache_ + (size_t)i * kv_layer;
        const DevTensor* const qkv[3] = {&L.wq, &L.wk, &L.wv};
        float* const ys[3] = {q_buf, k_buf, v_buf};
        const float* sums[3] = {q_buf, k_buf, v_buf};
        int splits[3] = {1, 1, 1};
        bool done[3] = {false, false, false};
        size_t at = 0;
        // from the prompt's first token on: everything between the projections in one launch
        const bool whole = start_pos == 0 && hd == 128 && nh % 2 == 0 && rope_angles_ != nullptr;
        const bool defer = whole || (T >= 4 && hd <= 256);   // (the prompt form of the rotation: ntk_rope takes it from 4 tokens on, too; wider heads are turned in place)
        // (one launch a format; two formats together)
        struct Of { const DevTensor* w[3]; float* y[3]; int idx[3], n = 0; ntk_gemm_partials pt; } of[3];
        int kinds = 0;
        for (int a = 0; a < 3; ++a) {
            if (done[a]) continue;
            Of& o = of[kinds++];
            for (int b = a; b < 3; ++b)
                if (qkv[b]->dtype == qkv[a]->dtype) { o.w[o.n] = qkv[b]; o.y[o.n] = ys[b]; o.idx[o.n++] = b; done[b] = true; }
        }
        auto leaves = [&](const Of& o) {
            if (!defer || o.pt.nsplit <= 1) return;
            for (int k = 0; k < o.n; ++k) {
                sums[o.idx[k]] = o.pt.part[k];
                splits[o.idx[k]] = o.pt.nsplit;
                at += (size_t)o.pt.nsplit * T * o.w[k]->out_f;
            }
        };
        if (kinds == 2 && defer && repacked(of[0].w, of[0].n) && repacked(of[1].w, of[1].n)) {
            ntk_gemv_seg sa[3], sb[3];
            const ntk_gemm_desc da = describe(of[0].w, of[0].y, of[0].n, nullptr, &of[0].pt, true, sa), db = describe(of[1].w, of[1].y, of[1].n, nullptr, &of[1].pt, true, sb);
            NT_TRY(ntk_gemm_short_two(&da, &db, 1, cfg_.norm_eps, 0, s));
            leaves(of[0]);
            leaves(of[1]);
        } else
            for (int a = 0; a < kinds; ++a) {
                NT_TRY(gemm(of[a].w, of[a].y, of[a].n, nullptr, true, at, defer ? &of[a].pt : nullptr));
                leaves(of[a]);
            }
        if (whole) {
            NT_TRY(ntk_short_attention(sums, splits, rope_angles_, T, nh, nkv, hd, scale, cfg_.rope_interleaved, kc, vc, cfg_.max_seq_len, other(), s));
        } else if (defer) {
            NT_TRY(ntk_reduce_rope_kv_store(q_buf, sums, splits, positions_, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, kc, vc, start_pos, cfg_.max_seq_len, s));
        } else {
            NT_TRY(ntk_rope(q_buf, k_buf, positions_, 1, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, s));
            NT_TRY(ntk_copy_to_kv_cache(kc, vc, k_buf, v_buf, T, nkv, hd, start_pos, cfg_.max_seq_len, s));
        }
        if (!whole) {
            NT_TRY(ntk_attention_prefill(attn_out, q_buf, kc, vc, T, start_pos, nh, nkv, hd, cfg_.max_seq_len, scale, s));
            NT_TRY(ntk_short_prepare_x(attn_out, T, qd, other(), s));
        }
        ntk_gemm_partials pt;
        const DevTensor* w[2] = {&L.wo, nullptr};
        float* y[2] = {hidden_, nullptr};
        NT_TRY(gemm(w, y, 1, hidden_, false, 0, &pt));
        NT_TRY(ntk_short_norm_prepare_x(hidden_, &pt, (const float*)L.ffn_norm.ptr, T, H, other(), s));
        w[0] = &L.w_gate; w[1] = &L.w_up;
        y[0] = gate_buf; y[1] = up_buf;
        NT_TRY(gemm(w, y, 2, nullptr, true, 0, &pt));
        NT_TRY(ntk_short_silu_mul_prepare_x(&pt, other(), s));
        w[0] = &L.w_down;
        y[0] = hidden_;
        const bool more = i + 1 < last_layer;
        NT_TRY(gemm(w, y, 1, hidden_, false, 0, more ? &pt : nullptr));
        if (more) NT_TRY(ntk_short_norm_prepare_x(hidden_, &pt, (const float*)layers_[i + 1].attn_norm.ptr, T, H, other(), s));
    }
    int rc = NTK_OK;
    if (raw_err_ != NTK_OK) { rc = raw_err_; raw_err_ = NTK_OK; }
    return rc;
}

// layers [first, last) of the 1:1 path on hidden_[T][H] at positions start_pos.. (positions_ already on the device).  keys_last: of the last one only the cache rows, the rotated queries left at the
// front of workspace_; queries: those of the first one's T tokens, whose cache rows are written, with room for as many behind them
int Model::layers_1to1(int T, int start_pos, int first, int last_layer, bool keys_last, float* queries) {
    if (!queries && short_prompt(T) && first < last_layer) return layers_short(T, start_pos, first, last_layer);
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim, nh = cfg_.n_heads, nkv = cfg_.n_kv_heads;
    const int qd = nh * hd, kvd = nkv * hd;
    void* s = stream_;
    const size_t kv_layer = (size_t)cfg_.max_seq_len * kvd;
    const float scale = 1.0f / sqrtf((float)hd);
    float* q_buf = workspace_;
    float* k_buf = q_buf + (size_t)T * qd;
    float* v_buf = k_buf + (size_t)T * kvd;
    float* attn_out = queries ? queries + (size_t)T * qd : v_buf + (size_t)T * kvd;
    float* gate_buf = workspace_;
    float* up_buf = gate_buf + (size_t)T * I;
    int rc = NTK_OK;
    auto ok = [&](int st) { if (st != NTK_OK && rc == NTK_OK) rc = st; };
    // (wp: the tensor's raw GGUF blocks -- resident, or unpacked from the repack by raw_of() once per projection, not per token)
    auto gemv = [&](float* y, const DevTensor& w, const void* wp, const float* x) {
        const int st = ntk_gemv(y, wp, x, (int)w.out_f, (int)w.in_f, w.dtype, s);
        if (st == NTK_E_DTYPE) fprintf(stderr, "Unsupported dtype for GEMV: %s\n", dtype_name(w.dtype));   // gemm.cu:801-803
        else ok(st);
    };
    // Y[t] = W . X[t] for the T tokens: one pass over W per 16 tokens on the matrix cores, or the reference's loop
    const bool batched = batched_prefill_ && T > 1;
    // (rounds 2-5: a prompt of <= 16 tokens was one pass of the F32-MFMA GEMM -- 2 217 tok/s against 1 727 through the 64-token form of the FP16 GEMM; round 6:
    // prompts of <= 32 tokens take the FP16 GEMM's weight-streaming form, gemm_quant_f16_small_kernel)
    const bool bf16_now = bf16_prefill_ && gemm_ws_ && T > 1;
    // ... but a matrix that exists ONLY as its decode repack goes through the FP16 GEMM (which reads the repack) from 2 tokens on: the F32-MFMA form would
    // need the GGUF bytes unpacked first (a 16-token pass of the 8B Q4_K_M model: 9 ms this way, 11 ms with the unpack)
    const bool bf16_rp = bf16_prefill_ && gemm_ws_ && T > 1;
    const float* planes_of = nullptr;   // the x whose FP16 planes sit in the current workspace (Q, K, V and gate, up share one x)
    // Two workspaces, used alternately: the launch that PRODUCES a projection's input also splits it into that projection's planes (ntk_*_prepare_x,
    // round 6) -- into the workspace the previous projection did NOT use, whose partial sums it may still be reading.
    void* cur_ws = gemm_ws_;
    auto flip_ws = [&]() { cur_ws = cur_ws == gemm_ws_ ? gemm_ws2_ : gemm_ws_; return cur_ws; };
    const float* planes_ready = nullptr;   // written by such a producer: becomes planes_of where the old contents are declared stale
    // rm: the tokens' largest |X| when the kernel that produced X left them (ntk_rmsnorm_rowmax / ntk_silu_mul_rowmax): the FP16 GEMM's operand
    // pre-pass then needs no pass of its own over X for the token scales
    // the FP16 GEMM behind its descriptor (ntk_engine.h): matrices of one format sharing X
    auto gemm_f16 = [&](const ntk_gemv_seg* segs, int nseg, const float* X, int in_f, const float* resid, int reuse_x, const float* rm, ntk_gemm_partials* pt,
                        bool repacked) {
        ntk_gemm_desc d{};
        d.segs = segs; d.nseg = nseg; d.X = X; d.n_tokens = T; d.in_features = in_f; d.resid = resid;
        d.workspace = cur_ws; d.workspace_bytes = gemm_ws_bytes_; d.reuse_x = reuse_x; d.row_max = rm; d.partials = pt;
        d.weights_repacked = repacked ? 1 : 0;
        return ntk_gemm_quant_f16(&d, s);
    };
    // RMSNorm / SiLU x up in front of an FP16-GEMM projection also leave the tokens' largest |x| (row_max_: [2][max_seq]; the second array is
    // zeroed by the layer's first RMSNorm launch for the SiLU launch's atomic maxima)
    const bool with_max = batched && bf16_now && row_max_ != nullptr && prefill_row_max_;
    float* rm_a = with_max ? row_max_ : nullptr;
    float* rm_b = with_max ? row_max_ + cfg_.max_seq_len : nullptr;
    // what a projection may take from them: NULL unless the launch that wrote ITS input wrote (rm_b: and an earlier one of this layer cleared) the array -- a launch that
    // splits its rows itself (below) does neither, and a matrix of another format that shares the input would scale by another pass's maxima
    const float* max_a = nullptr;
    const float* max_b = nullptr;
    bool b_clear = false;
    // (round 6) ... or split X themselves: the projection then needs no pre-pass launch at all
    // (up to 64 tokens: a producer that owns a whole token per workgroup writes its planes in 16-byte pieces a kilobyte apart -- at 1024 tokens the pass
    // measured 5 % SLOWER than with the GEMM's own pre-pass, 8B Q8_0 28 010 -> 26 460 tok/s; at 16 - 64 tokens it is 2 - 5 % faster)
    const bool fuse_split = with_max && prefill_fused_split_ && gemm_ws2_ != nullptr && T <= 64;
    // (... beyond: four tokens a workgroup, rows_split_kernel, where its registers hold the row and few pieces are added up; other rows leave their maxima)
    const bool rows_split = with_max && prefill_fused_split_ && gemm_ws2_ != nullptr && T > 64;
    auto splits_rows = [&](size_t width, bool norm, int nsplit) { return fuse_split || (rows_split && ntk_rows_prepare_pays(T, (int)width, norm ? 1 : 0, nsplit)); };
    auto f16_ok = [&](const DevTensor& w) {   // the formats and shapes ntk_gemm_quant_f16 takes
        const bool kq = w.dtype == NTK_DT_Q4_0 || w.dtype == NTK_DT_Q4_K || w.dtype == NTK_DT_Q5_K || w.dtype == NTK_DT_Q6_K;
        return (w.dtype == NTK_DT_Q8_0 || kq) && w.in_f % (kq ? 256 : 128) == 0 && w.out_f % 16 == 0 && (w.ptr || w.rp);
    };
    // nothing but planes is read of X where every matrix that reads it goes through that GEMM, whatever it would refuse looked at ahead: such rows are not written at all
    auto planes_only = [&](std::initializer_list<const DevTensor*> ws, size_t width) {
        if (!rows_split) return false;
        for (const DevTensor* w : ws)
            if (!f16_ok(*w) || (size_t)w->in_f != width || w->nbytes > 0xE0000000u || (reinterpret_cast<uintptr_t>(w->ptr ? w->ptr : w->rp) & 15)) return false;
        return true;
    };
    auto prepare_x = [&](const float* X, const DevTensor& w) {   // X as it lies (the attention output): row maximum + split in one launch
        if (!splits_rows(w.in_f, false, 0) || !f16_ok(w) || X == planes_of) return;
        void* ws = flip_ws();
        if ((fuse_split ? ntk_gemm_prepare_x(X, T, (int)w.in_f, ws, s) : ntk_rows_prepare_x(X, T, (int)w.in_f, ws, s)) == NTK_OK) planes_of = X;
        else planes_of = nullptr;
    };
    // One resident copy (round 6): a K-quant matrix whose GGUF bytes were freed after the load-time repack is read by the FP16 GEMM FROM THE REPACK
    // (ntk_gemm_desc.weights_repacked: identical bits) -- no unpack in front of the prompt launches any more.  rp_only(w): that is the tensor's state.
    auto rp_only = [&](const DevTensor& w) {
        return !w.ptr && w.rp && (w.dtype == NTK_DT_Q4_K || w.dtype == NTK_DT_Q5_K || w.dtype == NTK_DT_Q6_K) && w.out_f % 16 == 0;
    };
    // half-precision weights: one pass over them for all tokens, too (false: not such a matrix, nothing was launched).  From 3072 inputs on: there the tiles' results are no further
    // from 64 bits than the one-token products' (gemm_tile.hip.h: 1.30e-7 against 1.42e-7 of the result at 3072, with channels that tower over the others 1.43 and 1.42; 2.14 and
    // 2.78 at 14336), at 2560 they are with such channels (1.37 and 1.32), at 1024 in every case (1.07 and 0.99).  Time would draw the line lower: 40 tokens through 2048 x 2048 take 10 us, 130 one by one
    auto project_half = [&](float* Y, const DevTensor& w, const float* X, size_t ystride, size_t xstride, bool accumulate, const float* rm) -> bool {
        if (!bf16_now || !w.ptr || w.dtype != NTK_DT_F16 || w.in_f < 3072 || ystride != (size_t)w.out_f || xstride != (size_t)w.in_f) return false;
        void* ws = cur_ws == gemm_ws_ ? gemm_ws2_ : gemm_ws_;   // (not the one that holds the planes of a quantised matrix's input)
        if (!ws) { ws = cur_ws; planes_of = nullptr; }
        ok(ntk_gemm_half(Y, w.ptr, X, T, (int)w.out_f, (int)w.in_f, accumulate ? 1 : 0, rm, ws, gemm_ws_bytes_, s));
        return true;
    };
    // halves_of: the input whose halves ntk_half_norm_split has left in cur_ws (no rows are written: half_only of what reads it)
    const float* halves_of = nullptr;
    auto half_only = [&](std::initializer_list<const DevTensor*> ws) {
        if (!with_max || !prefill_fused_split_ || tp_world_ > 1 || !gemm_ws2_ || !ntk_half_norm_takes(T, H, gemm_ws_bytes_)) return false;
        for (const DevTensor* w : ws)
            if (!w->ptr || w->dtype != NTK_DT_F16 || w->in_f < 3072 || (int)w->in_f != H || (reinterpret_cast<uintptr_t>(w->ptr) & 15)) return false;
        return true;
    };
    // several of them over one X in one launch (silu: gate and up, Y[0] = silu(gate) * up); false: not such matrices, nothing was launched
    auto project_half_many = [&](float* const* Ys, const DevTensor* const* Ws, int n, const float* X, const float* rm, bool silu, ntk_gemm_partials* joined = nullptr) -> bool {     // joined: the pieces of a product over ready halves may be left there
        ntk_half_desc d{};
        for (int i = 0; i < n; ++i) {
            if (!batched || !bf16_now || !Ws[i]->ptr || Ws[i]->dtype != NTK_DT_F16 || Ws[i]->in_f < 3072 || Ws[i]->in_f != Ws[0]->in_f) return false;
            d.W[i] = Ws[i]->ptr; d.Y[i] = Ys[i]; d.out[i] = (int)Ws[i]->out_f;
        }
        const bool ready = X == halves_of;
        void* ws = ready ? cur_ws : cur_ws == gemm_ws_ ? gemm_ws2_ : gemm_ws_;   // (as above)
        const bool own = ws != nullptr;
        d.n = n; d.X = X; d.n_tokens = T; d.in_features = (int)Ws[0]->in_f; d.row_max = rm; d.silu = silu ? 1 : 0;
        d.workspace = own ? ws : cur_ws; d.workspace_bytes = gemm_ws_bytes_;
        const int st = ready ? ntk_gemm_half_normed(&d, joined, s) : ntk_gemm_half_many(&d, s);
        if (st == NTK_E_SHAPE || st == NTK_E_ALIGN) return false;
        if (!own) planes_of = nullptr;
        ok(st);
        return true;
    };
    auto project = [&](float* Y, const DevTensor& w, const float* X, size_t ystride, size_t xstride, const float* rm) {
        if (batched && project_half(Y, w, X, ystride, xstride, false, rm)) return;
        if (batched && bf16_rp && rp_only(w) && ystride == (size_t)w.out_f && xstride == (size_t)w.in_f) {   // straight from the repack
            const ntk_gemv_seg sg{w.rp, Y, (int)w.out_f, w.dtype};
            const int st = gemm_f16(&sg, 1, X, (int)w.in_f, nullptr, X == planes_of ? 1 : 0, rm, nullptr, true);
            if (st == NTK_OK) { planes_of = X; return; }
            if (st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) { ok(st); return; }
        }
        raw_begin();
        const void* wp = raw_of(w);
        if (batched && is_quant(w.dtype) && ystride == (size_t)w.out_f && xstride == (size_t)w.in_f) {
            int st = NTK_E_DTYPE;
            if (bf16_now) {   // FP16 matrix cores, up to 1024 tokens per pass (Q8_0 / Q4_K / Q5_K / Q6_K)
                const ntk_gemv_seg sg{wp, Y, (int)w.out_f, w.dtype};
                st = gemm_f16(&sg, 1, X, (int)w.in_f, nullptr, X == planes_of ? 1 : 0, rm, nullptr, false);
            }
            if (st == NTK_OK) planes_of = X;
            if (st == NTK_E_DTYPE || st == NTK_E_SHAPE || st == NTK_E_ALIGN)
                st = ntk_gemm_quant(Y, wp, X, T, (int)w.out_f, (int)w.in_f, w.dtype, nullptr, s);
            if (st != NTK_E_ALIGN && st != NTK_E_SHAPE) { ok(st); return; }   // those two: shapes only the per-token loop takes
        }
        if (batched && wp && (w.dtype == NTK_DT_F16 || w.dtype == NTK_DT_F32) && ystride == (size_t)w.out_f && xstride == (size_t)w.in_f) {
            const int st = ntk_gemv_tokens(Y, wp, X, T, (int)w.out_f, (int)w.in_f, w.dtype, s);
            if (st != NTK_E_ALIGN && st != NTK_E_SHAPE) { ok(st); return; }
        }
        for (int t = 0; t < T; ++t) gemv(Y + (size_t)t * ystride, w, wp, X + (size_t)t * xstride);
    };
    // matrices that share X (Q | K | V, gate | up): those of one format go out as ONE launch of the FP16 GEMM, the rest one by one, ahead of them.  sums / splits: the LAST launch may
    // leave the partial sums of its K splits to the consumer (its matrices' places in the two are then set; a launch behind it would overwrite them)
    auto project_many = [&](float* const* Ys, const DevTensor* const* Ws, int n, const float* X, const float* rm, const float** sums = nullptr, int* splits = nullptr, ntk_gemm_partials* joined = nullptr) {
        bool done[3] = {false, false, false};
        if (project_half_many(Ys, Ws, n, X, rm, false, joined)) return;
        struct Group { int idx[3], m; } groups[3];
        int n_groups = 0;
        if (batched && bf16_now)
            for (int a = 0; a < n; ++a) {
                if (done[a]) continue;
                Group& g = groups[n_groups];
                g.m = 0;
                for (int b = a; b < n; ++b)
                    if (!done[b] && Ws[b]->dtype == Ws[a]->dtype && Ws[b]->in_f == Ws[a]->in_f) g.idx[g.m++] = b;
                if (g.m < 2) continue;
                for (int k = 0; k < g.m; ++k) done[g.idx[k]] = true;
                ++n_groups;
            }
        for (int a = 0; a < n; ++a)
            if (!done[a]) project(Ys[a], *Ws[a], X, (size_t)Ws[a]->out_f, (size_t)Ws[a]->in_f, rm);
        for (int gi = 0; gi < n_groups; ++gi) {
            const Group& g = groups[gi];
            ntk_gemv_seg segs[3];
            ntk_gemm_partials pt;
            const bool defer = sums && gi + 1 == n_groups;
            bool all_rp = true;
            for (int k = 0; k < g.m; ++k) all_rp = all_rp && rp_only(*Ws[g.idx[k]]);
            if (!all_rp) raw_begin();   // (the group's tensors side by side in the unpack scratch when their GGUF bytes are not resident)
            for (int k = 0; k < g.m; ++k) segs[k] = {all_rp ? Ws[g.idx[k]]->rp : raw_of(*Ws[g.idx[k]]), Ys[g.idx[k]], (int)Ws[g.idx[k]]->out_f, Ws[g.idx[k]]->dtype};
            const int st = gemm_f16(segs, g.m, X, (int)Ws[g.idx[0]]->in_f, nullptr, X == planes_of ? 1 : 0, rm, defer ? &pt : nullptr, all_rp);
            if (st == NTK_OK) {
                planes_of = X;
                if (defer && pt.nsplit > 1)
                    for (int k = 0; k < g.m; ++k)
                        if (pt.part[k]) { sums[g.idx[k]] = pt.part[k]; splits[g.idx[k]] = pt.nsplit; }
            } else if (st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) { ok(st); return; }
            else
                for (int k = 0; k < g.m; ++k) project(Ys[g.idx[k]], *Ws[g.idx[k]], X, (size_t)Ws[g.idx[k]]->out_f, (size_t)Ws[g.idx[k]]->in_f, rm);
        }
    };
    // hidden += W . X (attention.cpp:207 + transformer.cpp:645, ffn.cpp:130 + transformer.cpp:652): the batched
    // projection adds the residual in its epilogue, the reference sequence goes through residual_ and launch_add_inplace
    auto project_add = [&](const DevTensor& w, const float* X, size_t xstride, const float* rm) {
        if (tp_world_ > 1) {   // this rank's columns give a PARTIAL sum: into the exchange slot, then hidden += sum over ranks
            project(tp_slot(), w, X, H, xstride, rm);
            planes_of = nullptr;
            ok(tp_allreduce(hidden_, T * H));
            return;
        }
        if (batched && (size_t)w.out_f == (size_t)H && project_half(hidden_, w, X, H, xstride, true, rm)) return;
        if (batched && bf16_now && (size_t)w.out_f == (size_t)H && xstride == (size_t)w.in_f) prepare_x(X, w);
        if (batched && bf16_rp && rp_only(w) && (size_t)w.out_f == (size_t)H && xstride == (size_t)w.in_f) {   // straight from the repack
            const ntk_gemv_seg sg{w.rp, hidden_, (int)w.out_f, w.dtype};
            const int st = gemm_f16(&sg, 1, X, (int)w.in_f, hidden_, X == planes_of ? 1 : 0, rm, nullptr, true);
            if (st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) { planes_of = nullptr; ok(st); return; }
        }
        if (batched && is_quant(w.dtype) && (size_t)w.out_f == (size_t)H && xstride == (size_t)w.in_f) {
            int st = NTK_E_DTYPE;
            raw_begin();
            const void* wp = raw_of(w);
            if (bf16_now) {
                const ntk_gemv_seg sg{wp, hidden_, (int)w.out_f, w.dtype};
                st = gemm_f16(&sg, 1, X, (int)w.in_f, hidden_, X == planes_of ? 1 : 0, rm, nullptr, false);
            }
            planes_of = nullptr;   // (this projection rewrites hidden_, and the next group has a new x)
            if (st == NTK_E_DTYPE || st == NTK_E_SHAPE || st == NTK_E_ALIGN)
                st = ntk_gemm_quant(hidden_, wp, X, T, (int)w.out_f, (int)w.in_f, w.dtype, hidden_, s);
            if (st != NTK_E_ALIGN && st != NTK_E_SHAPE) { ok(st); return; }
        }
        project(residual_, w, X, H, xstride, rm);
        ok(ntk_add_inplace(hidden_, residual_, T * H, s));
    };
    auto left_max = [&](bool written, bool zero_b, bool cleared = false) {   // a norm has written residual_ (zero_b: the layer's first, which clears rm_b if it leaves maxima at all, or cleared)
        max_a = written ? rm_a : nullptr;
        if (zero_b) b_clear = (written || cleared) && rm_b;
    };
    auto norm = [&](const DevTensor& nw, bool zero_b, const DevTensor& next_w, bool only, bool half) {     // only, half: planes_only, half_only of the matrices that read it
        halves_of = nullptr;
        if (half) {
            planes_of = planes_ready = nullptr;
            ok(ntk_half_norm_split(hidden_, nullptr, (const float*)nw.ptr, T, H, cfg_.norm_eps, cur_ws, gemm_ws_bytes_, s));
            halves_of = residual_;
            left_max(false, zero_b);
            return;
        }
        if (splits_rows(H, true, 0) && f16_ok(next_w) && (int)next_w.in_f == H) {
            void* ws = flip_ws();
            ok(fuse_split ? ntk_rmsnorm_prepare_x(residual_, hidden_, (const float*)nw.ptr, T, H, cfg_.norm_eps, ws, s)
                          : ntk_rows_norm_prepare_zero(hidden_, nullptr, (const float*)nw.ptr, T, H, cfg_.norm_eps, only ? nullptr : residual_, zero_b ? rm_b : nullptr, ws, s));
            planes_ready = residual_;
            left_max(false, zero_b, !fuse_split);
            return;
        }
        left_max(with_max, zero_b);
        if (with_max) ok(ntk_rmsnorm_rowmax(residual_, hidden_, (const float*)nw.ptr, T, H, cfg_.norm_eps, rm_a, zero_b ? rm_b : nullptr, s));
        else ok(ntk_rmsnorm(residual_, hidden_, (const float*)nw.ptr, T, H, cfg_.norm_eps, s));
    };
    // hidden += W . X followed by the NEXT RMSNorm (nw; into residual_, with the token maxima) as one consumer launch of the projection's K splits
    // (ntk_gemm_quant_f16 with `partials` + ntk_reduce_rmsnorm_rowmax); false = not this shape / format: the caller runs project_add + norm
    auto project_add_norm = [&](const DevTensor& w, const float* X, const float* rm, const DevTensor& nw, bool zero_b, const DevTensor& next_w, bool only, bool half) -> bool {
        if (half && w.ptr && w.dtype == NTK_DT_F16 && w.in_f >= 3072 && (size_t)w.out_f == (size_t)H) {   // (the pieces lie in the other workspace: the halves go to this one)
            ntk_gemm_partials pt;
            void* ws = cur_ws == gemm_ws_ ? gemm_ws2_ : gemm_ws_;
            int st = ntk_gemm_half_defer(hidden_, w.ptr, X, T, H, (int)w.in_f, rm, ws, gemm_ws_bytes_, &pt, s);
            planes_of = planes_ready = nullptr;
            if (st == NTK_OK) st = ntk_half_norm_split(hidden_, &pt, (const float*)nw.ptr, T, H, cfg_.norm_eps, cur_ws, gemm_ws_bytes_, s);
            halves_of = residual_;
            left_max(false, zero_b);
            ok(st);
            return true;
        }
        if (!with_max || tp_world_ > 1 || !is_quant(w.dtype) || (size_t)w.out_f != (size_t)H) return false;
        ntk_gemm_partials pt;
        int st = NTK_E_DTYPE;
        if (fuse_split || !rm) prepare_x(X, w);   // (where its maxima are there, the GEMM's own split is the faster)
        if (rp_only(w)) {   // straight from the repack
            const ntk_gemv_seg sg{w.rp, hidden_, (int)w.out_f, w.dtype};
            st = gemm_f16(&sg, 1, X, (int)w.in_f, hidden_, X == planes_of ? 1 : 0, rm, &pt, true);
        }
        if (st == NTK_E_DTYPE || st == NTK_E_SHAPE || st == NTK_E_ALIGN) {
            raw_begin();
            const void* wp = raw_of(w);
            // (a launch that does not split K adds the residual in its own epilogue, in place, as project_add does: nothing is deferred then)
            const ntk_gemv_seg sg{wp, hidden_, (int)w.out_f, w.dtype};
            st = gemm_f16(&sg, 1, X, (int)w.in_f, hidden_, X == planes_of ? 1 : 0, rm, &pt, false);
        }
        if (st == NTK_E_DTYPE || st == NTK_E_SHAPE || st == NTK_E_ALIGN) return false;   // (nothing was launched)
        if (half) {   // (an unquantised group behind a quantised projection)
            if (st == NTK_OK) st = ntk_half_norm_split(hidden_, &pt, (const float*)nw.ptr, T, H, cfg_.norm_eps, flip_ws(), gemm_ws_bytes_, s);
            planes_of = planes_ready = nullptr;
            halves_of = residual_;
            left_max(false, zero_b);
            ok(st);
            return true;
        }
        halves_of = nullptr;
        planes_of = nullptr;
        const int pieces = pt.nsplit > 1 ? pt.nsplit : pt.y[0] != hidden_ ? 1 : 0;
        if (st == NTK_OK && splits_rows(H, true, pieces) && f16_ok(next_w) && (int)next_w.in_f == H) {   // (the partial sums lie in cur_ws: the planes go to the other one)
            void* ws = flip_ws();
            st = fuse_split ? ntk_reduce_rmsnorm_prepare_x(hidden_, &pt, (const float*)nw.ptr, cfg_.norm_eps, residual_, ws, s)
                            : ntk_rows_norm_prepare_zero(hidden_, &pt, (const float*)nw.ptr, T, H, cfg_.norm_eps, only ? nullptr : residual_, zero_b ? rm_b : nullptr, ws, s);
            planes_ready = residual_;
            left_max(false, zero_b, !fuse_split);
        } else
        if (st == NTK_OK) left_max(true, zero_b), st = ntk_reduce_rmsnorm_rowmax(hidden_, &pt, (const float*)nw.ptr, cfg_.norm_eps, residual_, rm_a, zero_b ? rm_b : nullptr, s);
        ok(st);
        return true;
    };
    bool normed_ahead = false;   // residual_ / rm_a already hold this layer's normalised input (written with the previous layer's down projection)
    for (int i = first; i < last_layer; ++i) {
        const LayerWeights& L = layers_[i];
        uint16_t* kc = k_cache_ + (size_t)i * kv_layer;
        uint16_t* vc = v_cache_ + (size_t)i * kv_layer;
        auto only_qkv = [&](const LayerWeights& l) { return planes_only({&l.wq, &l.wk, &l.wv}, H); };
        auto half_qkv = [&](const LayerWeights& l) { return half_only({&l.wq, &l.wk, &l.wv}); };
        const bool given = queries && i == first;
        if (!given) {
            if (!normed_ahead) norm(L.attn_norm, true, L.wq, only_qkv(L), half_qkv(L));
            normed_ahead = false;
            planes_of = planes_ready;   // residual_ has new contents (split already by the launch that wrote them, or not)
            planes_ready = nullptr;
            const bool one_launch = with_max && T >= 4 && hd <= 256;
            const float* sums[3] = {q_buf, k_buf, v_buf};     // what the rotation reads: the projections, or the partial sums of the last launch's
            int splits[3] = {1, 1, 1};
            ntk_gemm_partials joined{};                       // (or of all three side by side)
            {
                float* const ys[3] = {q_buf, k_buf, v_buf};
                const DevTensor* const ws[3] = {&L.wq, &L.wk, &L.wv};
                project_many(ys, ws, 3, residual_, max_a, one_launch ? sums : nullptr, splits, one_launch ? &joined : nullptr);
            }
            if (one_launch) {                            // (the prompt form of the rotation: ntk_rope takes it from 4 tokens on, too)
                if (joined.part[0])
                    ok(ntk_reduce_rope_kv_store_joined(q_buf, joined.part[0], joined.nsplit, positions_, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, kc, vc, start_pos,
                                                       cfg_.max_seq_len, s));
                else if (splits[0] + splits[1] + splits[2] > 3)
                    ok(ntk_reduce_rope_kv_store(q_buf, sums, splits, positions_, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, kc, vc, start_pos, cfg_.max_seq_len, s));
                else
                    ok(ntk_rope_kv_store(q_buf, k_buf, v_buf, positions_, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, kc, vc,
                                         start_pos, cfg_.max_seq_len, s));
            } else {
                ok(ntk_rope(q_buf, k_buf, positions_, 1, T, nh, nkv, hd, cfg_.rope_theta, cfg_.rope_freq_scale, cfg_.rope_interleaved, s));
                ok(ntk_copy_to_kv_cache(kc, vc, k_buf, v_buf, T, nkv, hd, start_pos, cfg_.max_seq_len, s));
            }
        }
        if (keys_last && i + 1 == last_layer) break;
        if (T == 1) ok(ntk_attention_decode(attn_out, q_buf, kc, vc, start_pos + T, nh, nkv, hd, cfg_.max_seq_len, scale, s));
        else ok(ntk_attention_prefill(attn_out, given ? queries : q_buf, kc, vc, T, start_pos, nh, nkv, hd, cfg_.max_seq_len, scale, s));
        const bool only_unit = planes_only({&L.w_gate, &L.w_up}, H);
        const intptr_t apart = (intptr_t)L.w_gate.ptr - (intptr_t)L.w_up.ptr;
        const bool half_unit = half_only({&L.w_gate, &L.w_up}) && std::abs(apart) < (1LL << 32) - (intptr_t)L.w_gate.out_f * H * 2;   // (what ntk_gemm_half_many takes as a gated pair)
        if (!project_add_norm(L.wo, attn_out, nullptr, L.ffn_norm, false, L.w_gate, only_unit, half_unit)) {
            project_add(L.wo, attn_out, qd, nullptr);
            norm(L.ffn_norm, false, L.w_gate, only_unit, half_unit);
        }
        planes_of = planes_ready;
        planes_ready = nullptr;
        // gate | up and SiLU x up (per token in the reference, ffn.cpp:127: the same elementwise op): with the token maxima, the gate | up launch's K
        // splits are summed by the SiLU launch itself (ntk_gemm_quant_f16 with `partials` + ntk_reduce_silu_mul_rowmax)
        bool ffn_done = false;
        max_b = nullptr;
        if (with_max && rm_b && tp_world_ == 1 && L.w_gate.dtype == L.w_up.dtype && is_quant(L.w_gate.dtype) && L.w_gate.in_f == L.w_up.in_f &&
            (size_t)L.w_gate.out_f == (size_t)I && (size_t)L.w_up.out_f == (size_t)I && I % 4 == 0) {
            const bool both_rp = rp_only(L.w_gate) && rp_only(L.w_up);
            if (!both_rp) raw_begin();
            ntk_gemv_seg segs[2] = {{both_rp ? L.w_gate.rp : raw_of(L.w_gate), gate_buf, (int)I, L.w_gate.dtype},
                                    {both_rp ? L.w_up.rp : raw_of(L.w_up), up_buf, (int)I, L.w_up.dtype}};
            ntk_gemm_partials pt;
            int st = gemm_f16(segs, 2, residual_, (int)L.w_gate.in_f, nullptr, residual_ == planes_of ? 1 : 0, max_a, &pt, both_rp);
            if (st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) {   // (those three: nothing was launched)
                if (st == NTK_OK && splits_rows(I, false, pt.nsplit) && f16_ok(L.w_down) && (size_t)L.w_down.in_f == (size_t)I) {
                    void* ws = flip_ws();
                    st = fuse_split ? ntk_reduce_silu_mul_prepare_x(gate_buf, &pt, ws, s) : ntk_rows_silu_mul_prepare_x(planes_only({&L.w_down}, I) ? nullptr : gate_buf, &pt, ws, s);
                    planes_ready = gate_buf;
                } else
                if (st == NTK_OK) st = ntk_reduce_silu_mul_rowmax(gate_buf, &pt, rm_b, s), max_b = b_clear ? rm_b : nullptr;
                ok(st);
                ffn_done = true;
            }
        }
        if (!ffn_done && tp_world_ == 1 && (size_t)L.w_gate.out_f == (size_t)I && (size_t)L.w_up.out_f == (size_t)I) {      // half-precision gate and up meet in their product's launch
            float* const ys[2] = {gate_buf, nullptr};
            const DevTensor* const ws[2] = {&L.w_gate, &L.w_up};
            ffn_done = project_half_many(ys, ws, 2, residual_, max_a, true);
        }
        if (!ffn_done) {
            float* const ys[2] = {gate_buf, up_buf};
            const DevTensor* const ws[2] = {&L.w_gate, &L.w_up};
            project_many(ys, ws, 2, residual_, max_a);
            int st_silu = NTK_E_SHAPE;   // (in place: exactly one of these launches runs)
            if (splits_rows(I, false, 1) && f16_ok(L.w_down) && (size_t)L.w_down.in_f == (size_t)I && tp_world_ == 1) {
                ntk_gemm_partials pt{};
                pt.nseg = 2; pt.n_tokens = T; pt.nsplit = 1; pt.y[0] = gate_buf; pt.y[1] = up_buf; pt.rows[0] = pt.rows[1] = I;
                void* ws = flip_ws();
                st_silu = fuse_split ? ntk_silu_mul_prepare_x(gate_buf, gate_buf, up_buf, T, I, ws, s) : ntk_rows_silu_mul_prepare_x(planes_only({&L.w_down}, I) ? nullptr : gate_buf, &pt, ws, s);
                if (st_silu == NTK_OK) planes_ready = gate_buf;
            } else if (with_max && rm_b) {
                st_silu = ntk_silu_mul_rowmax(gate_buf, gate_buf, up_buf, T, I, rm_b, s);
                if (st_silu == NTK_OK && b_clear) max_b = rm_b;
            }
            if (st_silu == NTK_E_SHAPE || st_silu == NTK_E_ALIGN) { st_silu = ntk_silu_mul(gate_buf, gate_buf, up_buf, T * I, s); rm_b = nullptr; }   // (then for the rest of the pass)
            ok(st_silu);
        }
        planes_of = planes_ready;
        planes_ready = nullptr;
        // down projection + residual, and the NEXT layer's first RMSNorm in the same consumer launch when there is a next layer in this pass
        if (i + 1 < last_layer && project_add_norm(L.w_down, gate_buf, max_b, layers_[i + 1].attn_norm, true, layers_[i + 1].wq, only_qkv(layers_[i + 1]), half_qkv(layers_[i + 1]))) normed_ahead = true;
        else project_add(L.w_down, gate_buf, I, max_b);
        if (rc != NTK_OK) break;
    }
    if (raw_err_ != NTK_OK) { rc = raw_err_; raw_err_ = NTK_OK; }   // what raw_of() could not report through its pointer (it precedes the consumer's NTK_E_NULL)
    return rc;
}

// ---------------------------------------------------------------------------------------------------
// fused single-token path
// ---------------------------------------------------------------------------------------------------
int Model::set_device_token(int token) {
    if (token < 0 || token >= cfg_.vocab_size) { err_ = "token id out of range"; return NTK_E_SHAPE; }
    *h_token_ = token;
    return ntk_memcpy_h2d_async(d_token_, h_token_, 4, stream_);
}
int Model::set_device_pos(int pos) {
    host_pos_ = pos;
    // small copy, once per generation -- on the model's own stream: a blocking copy on the legacy stream would collide with a
    // hipGraph capture in progress on another thread's stream (tensor-parallel ranks sharing a process)
    NT_TRY(ntk_memcpy_h2d_async(d_pos_, &pos, 4, stream_));
    NT_TRY(ntk_stream_synchronize(stream_));
    // nothing is in flight: forget the tokens of earlier positions (a re-based position could otherwise match a stale {token, position} tag)
    if (h_ring_) memset(h_ring_, 0, 64);
    return NTK_OK;
}
int Model::sync() { return ntk_stream_synchronize(stream_); }
int Model::host_token() const { return *h_token_; }
int Model::set_device_step(int pos, int token) {
    if (token < 0 || token >= cfg_.vocab_size) { err_ = "token id out of range"; return NTK_E_SHAPE; }
    *h_token_ = token;
    host_pos_ = pos;
    const int words[2] = {token, pos};
    return ntk_store_words(d_token_, 1, d_pos_, 1, words, stream_);
}
int Model::copy_logits(float* host) {
    if (out_row_) return out_row_.fetch(host, logits_, nullptr, stream_);
    NT_TRY(ntk_memcpy_d2h_async(host, logits_, (size_t)cfg_.vocab_size * 4, stream_));
    return ntk_stream_synchronize(stream_);
}

int Model::sample_on_device(const int* recent, int n_recent, float repeat_penalty, float temperature, int top_k, float top_p, float r) {
    if (!sample_scratch_ || !d_recent_ || !h_recent_) return NTK_E_NOMEM;
    if (n_recent > kRecentCap) { recent += n_recent - kRecentCap; n_recent = kRecentCap; }
    void* s = stream_;
    if (repeat_penalty > 1.0f && n_recent > 0) {
        // the previous token's copy of the window has completed (the host synchronised to read that token)
        memcpy(h_recent_, recent, (size_t)n_recent * 4);
        NT_TRY(ntk_memcpy_h2d_async(d_recent_, h_recent_, (size_t)n_recent * 4, s));
    } else {
        n_recent = 0;
    }
    if (temperature <= 0.0f) {   // greedy with a repeat penalty: Sampler::sample returns argmax of the penalised logits
        NT_TRY(ntk_repeat_penalty(logits_, cfg_.vocab_size, d_recent_, n_recent, repeat_penalty, s));
        return ntk_argmax(logits_, cfg_.vocab_size, d_token_, h_token_, argmax_scratch_, s);
    }
    return ntk_sample_top_k(logits_, cfg_.vocab_size, d_recent_, n_recent, repeat_penalty, temperature, top_k, top_p, r, d_token_,
                            h_token_, sample_scratch_, s);
}

// profiling hook (only inside profile_token(), never while capturing).  Fine mode: an event pair around every
// launch.  Coarse mode: ONE event where the launch class changes -- a run of same-class launches is timed as a
// whole (its kernels and the boundaries between them), so the cost of the events is paid once per run.
void Model::prof_mark(int cls, bool begin) {
    if (!prof_) return;
    void* s = stream_;
    if (prof_coarse_) {
        if (!begin) return;
        if (!prof_->empty() && prof_->back().cls == cls) { ++prof_->back().n; return; }
        void* e = ntk_event_create();
        ntk_event_record(e, s);
        const bool shared = !prof_->empty();
        if (shared) prof_->back().b = e;
        prof_->push_back({cls, e, nullptr, 1, shared});
        return;
    }
    void* e = ntk_event_create();
    ntk_event_record(e, s);
    if (begin) prof_->push_back({cls, e, nullptr, 1, false}); else prof_->back().b = e;
}

// which launch kinds read the repacked tensors: 1 Q|K|V, 2 Wo, 4 gate|up, 8 down, 16 LM head (tuning builds: NTK_RP_MASK)
static int rp_mask() {
#ifdef NTK_TUNE
    static const int m = [] { const char* e = getenv("NTK_RP_MASK"); return e ? atoi(e) : 31; }();
    return m;
#else
    return 31;
#endif
}

int Model::enqueue_token(TokenKind kind) {
    const int H = cfg_.hidden_size;
    const bool greedy = kind == kGreedy;
    void* s = stream_;
    tp_call_ = 0;
    if (kind != kBare) {
        prof_mark(2, true);
        const int est = ntk_embed_rows(hidden_, token_embd_.ptr, d_token_, 1, H, token_embd_.dtype, s);
        prof_mark(2, false);
        if (est != NTK_OK && est != NTK_E_DTYPE) return est;
    }
#ifdef NTK_EXPERIMENTS
    if (use_persistent_now()) {   // every layer and the LM head in one launch
        NT_TRY(persistent_kind_ == 2 ? ntk_layer_engine_launch(persistent_plan_, d_pos_, s) : ntk_persistent_launch(persistent_plan_, d_pos_, s));
        if (greedy) NT_TRY(ntk_argmax_advance(logits_, cfg_.vocab_size, d_token_, h_token_, h_ring_, d_pos_, argmax_scratch_, s));
        else NT_TRY(ntk_advance_pos(d_pos_, s));
        return NTK_OK;
    }
#endif
    NT_TRY(enqueue_layers(0, cfg_.n_layers));
    // final RMSNorm + LM head (one launch for a quantised output matrix), then the token's tail
    {
        const DevTensor& w = output_;
        if (is_quant(w.dtype)) {
            prof_mark(0, true);
            int st = NTK_E_DTYPE;
            if (repack_ && w.rp && (rp_mask() & 16)) {
                ntk_gemv_seg rs = {w.rp, logits_, (int)w.out_f, w.dtype};
                st = ntk_gemv_rp_fused(&rs, 1, hidden_, (int)w.in_f, (const float*)output_norm_.ptr, cfg_.norm_eps, nullptr, 0, s);
                if (st != NTK_OK && st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) return st;
            }
            if (st != NTK_OK) {
                raw_begin();
                ntk_gemv_seg seg = {raw_of(w), logits_, (int)w.out_f, w.dtype};
                NT_TRY(ntk_gemv_fused(&seg, 1, hidden_, (int)w.in_f, (const float*)output_norm_.ptr, cfg_.norm_eps, nullptr, 0, s));
            }
            prof_mark(0, false);
        } else {
            NT_TRY(ntk_rmsnorm(residual_ + H, hidden_, (const float*)output_norm_.ptr, 1, (int)w.in_f, cfg_.norm_eps, s));
            NT_TRY(ntk_gemv(logits_, w.ptr, residual_ + H, (int)w.out_f, (int)w.in_f, w.dtype, s));
        }
    }
    if (kind == kBare) return NTK_OK;
    prof_mark(2, true);
    // greedy: arg-max, token -> device word + pinned ring, position + 1 in ONE tail (ntk_argmax_advance); otherwise only the position
    if (greedy) NT_TRY(ntk_argmax_advance(logits_, cfg_.vocab_size, d_token_, h_token_, h_ring_, d_pos_, argmax_scratch_, s));
    else NT_TRY(ntk_advance_pos(d_pos_, s));
    if (tp_world_ > 1) NT_TRY(ntk_tp_advance_epoch(tp_comm_, s));
    prof_mark(2, false);
    return NTK_OK;
}

// The token decoded at position `pos` by a greedy fused step, without synchronising the stream: the final launch of the step stores
// {token, pos + 1} into slot (pos & 3) of the pinned ring; the host polls that word.  Meanwhile the NEXT step may already be queued (its
// token lands in another slot), so the GPU never waits for the host between tokens (Engine::run / decode_greedy_steps keep one step
// ahead).  A poll that sees nothing for 2 s falls back to a stream synchronisation and reports what that returns.
int Model::wait_token(int pos, int* token) {
    volatile unsigned long long* slot = h_ring_ + (pos & 3);
    const unsigned want = (unsigned)(pos + 1);
    for (unsigned spins = 0;; ++spins) {
        const unsigned long long v = *slot;
        if ((unsigned)(v >> 32) == want) { *token = (int)(unsigned)v; return NTK_OK; }
#if defined(__x86_64__) || defined(__i386__)
        __builtin_ia32_pause();
#else
        std::this_thread::yield();
#endif
        if ((spins & 0xFFFFu) == 0xFFFFu) {
            const auto now = std::chrono::steady_clock::now();
            if (spins == 0xFFFFu) wait_t0_ = now;
            else if (std::chrono::duration<double>(now - wait_t0_).count() > 2.0) break;
        }
    }
    static bool warned = false;
    if (!warned) { warned = true; fprintf(stderr, "warning: the pinned token ring was not seen updating for 2 s (host memory not coherent with a running kernel?); falling back to a stream synchronisation per token\n"); }
    NT_TRY(ntk_stream_synchronize(stream_));
    const unsigned long long v = *slot;
    if ((unsigned)(v >> 32) != want) { err_ = "decode step finished without publishing its token"; return NTK_E_LAUNCH; }
    *token = (int)(unsigned)v;
    return NTK_OK;
}

// layers [first, last) of the fused single-token path on hidden_[H] (position in *d_pos_)
int Model::enqueue_layers(int first, int last_layer) {
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim, nh = cfg_.n_heads, nkv = cfg_.n_kv_heads;
    const int qd = nh * hd, kvd = nkv * hd;
    void* s = stream_;
    auto mark = [&](int cls, bool begin) { prof_mark(cls, begin); };
    const float scale = 1.0f / sqrtf((float)hd);
    const size_t kv_layer = (size_t)cfg_.max_seq_len * kvd;
    float* q_buf = workspace_;
    float* k_buf = q_buf + qd;
    float* v_buf = k_buf + kvd;
    float* attn_out = v_buf + kvd;
    float* gate_buf = workspace_;
    float* up_buf = gate_buf + I;

    // y_k = W_k . f(x) for n <= 3 matrices sharing x.  Matrices with one quantised dtype go out as one fused
    // launch (RMSNorm prologue when `norm`, residual epilogue when `resid`, n == 1); dense F16/F32 tensors take
    // the 1:1 launchers.  Scratch: residual_[0,H) = dense output before the residual add, residual_[H,2H) = norm(x).
    auto project = [&](const DevTensor* const* ws, float* const* ys, int n, const float* x, const DevTensor* norm,
                       const float* resid, int kind) -> int {
        const float* nw = norm ? (const float*)norm->ptr : nullptr;
        bool done[3] = {false, false, false};
        if (repack_ && (rp_mask() & kind)) {   // every matrix has its repacked form: one launch of the matrix-core GEMV, whatever the mix of K-quant formats
            bool all = true;
            for (int a = 0; a < n; ++a) all = all && ws[a]->rp != nullptr && ws[a]->in_f == ws[0]->in_f;
            if (all) {
                ntk_gemv_seg segs[3];
                for (int a = 0; a < n; ++a) segs[a] = {ws[a]->rp, ys[a], (int)ws[a]->out_f, ws[a]->dtype};
                mark(0, true);
                const int st = ntk_gemv_rp_fused(segs, n, x, (int)ws[0]->in_f, nw, cfg_.norm_eps, resid, 0, s);
                mark(0, false);
                if (st == NTK_OK) return NTK_OK;
                if (st != NTK_E_DTYPE && st != NTK_E_ALIGN && st != NTK_E_SHAPE) return st;   // (those: the raw-GGUF launches below take over)
            }
        }
        if (n > 1 && !resid) {   // matrices in two K-quant formats (Q4_K_M's attn_v): still one launch when the library has the pair
            bool all_quant = true, mixed = false;
            for (int a = 0; a < n; ++a) { all_quant = all_quant && is_quant(ws[a]->dtype); mixed = mixed || ws[a]->dtype != ws[0]->dtype; }
            if (all_quant && mixed) {
                ntk_gemv_seg segs[3];
                raw_begin();
                for (int a = 0; a < n; ++a) segs[a] = {raw_of(*ws[a]), ys[a], (int)ws[a]->out_f, ws[a]->dtype};
                mark(0, true);
                const int st = ntk_gemv_fused(segs, n, x, (int)ws[0]->in_f, nw, cfg_.norm_eps, nullptr, 0, s);
                mark(0, false);
                if (st == NTK_OK) return NTK_OK;
                // formats / alignment / workgroup split / LDS size the optional one-launch form does not take: the per-format
                // launches below do (the pair kernel is an optimisation, never the only way)
                if (st != NTK_E_DTYPE && st != NTK_E_ALIGN && st != NTK_E_SHAPE) return st;
            }
        }
        const float* normed = nullptr;   // norm(x) for the matrices that do not form it themselves
        for (int a = 0; a < n; ++a) {
            if (done[a]) continue;
            const DevTensor& w = *ws[a];
            if (!is_quant(w.dtype)) {
                const float* xin = x;
                if (nw) {
                    if (!normed) NT_TRY(ntk_rmsnorm(residual_ + H, x, nw, 1, (int)w.in_f, cfg_.norm_eps, s));
                    xin = normed = residual_ + H;
                }
                if ((w.dtype == NTK_DT_F16 || w.dtype == NTK_DT_F32) && w.ptr && (!resid || resid == ys[a])) {   // those of its type in one launch, a residual added where it lies
                    ntk_gemv_seg segs[3];
                    int m = 0;
                    for (int b = a; b < n; ++b) {
                        if (done[b] || ws[b]->dtype != w.dtype || ws[b]->in_f != w.in_f || !ws[b]->ptr || (resid && b != a)) continue;
                        segs[m++] = {ws[b]->ptr, ys[b], (int)ws[b]->out_f, w.dtype};
                        done[b] = true;
                    }
                    NT_TRY(ntk_gemv_dense(segs, m, xin, (int)w.in_f, resid ? 1 : 0, s));
                    continue;
                }
                float* y = resid ? residual_ : ys[a];
                raw_begin();
                NT_TRY(ntk_gemv(y, raw_of(w), xin, (int)w.out_f, (int)w.in_f, w.dtype, s));
                if (resid) NT_TRY(ntk_add(ys[a], resid, residual_, (int)w.out_f, s));
                done[a] = true;
                continue;
            }
            ntk_gemv_seg segs[3];
            int m = 0;
            raw_begin();
            for (int b = a; b < n; ++b) {
                if (done[b] || ws[b]->dtype != w.dtype) continue;
                segs[m++] = {raw_of(*ws[b]), ys[b], (int)ws[b]->out_f, ws[b]->dtype};
                done[b] = true;
            }
            mark(0, true);
            NT_TRY(ntk_gemv_fused(segs, m, x, (int)w.in_f, nw, cfg_.norm_eps, resid, 0, s));
            mark(0, false);
        }
        return NTK_OK;
    };
    auto project1 = [&](const DevTensor& w, float* y, const float* x, const DevTensor* norm, const float* resid, int kind) -> int {
        const DevTensor* ws[1] = {&w};
        float* ys[1] = {y};
        return project(ws, ys, 1, x, norm, resid, kind);
    };

    for (int i = first; i < last_layer; ++i) {
        const LayerWeights& L = layers_[i];
        uint16_t* kc = k_cache_ + (size_t)i * kv_layer;
        uint16_t* vc = v_cache_ + (size_t)i * kv_layer;
        {
            const DevTensor* ws[3] = {&L.wq, &L.wk, &L.wv};
            float* ys[3] = {q_buf, k_buf, v_buf};
            NT_TRY(project(ws, ys, 3, hidden_, &L.attn_norm, nullptr, 1));
        }
#ifdef NTK_EXPERIMENTS
        if (attn_regime_ == 0 && fuse_attention_ && attn_sync_ && is_quant(L.wo.dtype) && tp_world_ == 1) {
            // attention producers inside the Wo launch: one launch, one boundary and one first-byte latency less per layer
            raw_begin();
            ntk_gemv_seg wo = {raw_of(L.wo), hidden_, (int)L.wo.out_f, L.wo.dtype};
            mark(0, true);
            const int st = ntk_attention_gemv_fused(attn_out, q_buf, k_buf, v_buf, kc, vc, d_pos_, rope_inv_freq_, nh, nkv, hd,
                                                    cfg_.max_seq_len, scale, cfg_.rope_theta, cfg_.rope_freq_scale, &wo, hidden_,
                                                    attn_sync_, s);
            mark(0, false);
            if (st == NTK_OK) goto ffn;
            if (st != NTK_E_ALIGN && st != NTK_E_SHAPE && st != NTK_E_DTYPE) return st;   // those: shapes only the two launches take
        }
#endif
        mark(1, true);
        if (attn_regime_ == 0)
            NT_TRY(ntk_attention_decode_fused(attn_out, q_buf, k_buf, v_buf, kc, vc, d_pos_, rope_inv_freq_, nh, nkv, hd,
                                              cfg_.max_seq_len, scale, cfg_.rope_theta, cfg_.rope_freq_scale, s));
        else
            NT_TRY((attn_merge_ ? ntk_attention_decode_split_merged : ntk_attention_decode_split)(
                attn_out, q_buf, k_buf, v_buf, kc, vc, d_pos_, rope_inv_freq_, nh, nkv, hd, cfg_.max_seq_len, scale, cfg_.rope_theta,
                cfg_.rope_freq_scale, attention_splits(attn_regime_, hd), attn_scratch_, s));
        mark(1, false);
        if (tp_world_ > 1) {   // partial sum over this rank's heads -> exchange slot -> hidden += sum over ranks
            NT_TRY(project1(L.wo, tp_slot(), attn_out, nullptr, nullptr, 2));
            NT_TRY(tp_allreduce(hidden_, H));
        } else {
            NT_TRY(project1(L.wo, hidden_, attn_out, nullptr, hidden_, 2));
        }
#ifdef NTK_EXPERIMENTS
    ffn:
#endif
        if (is_quant(L.w_gate.dtype) && L.w_gate.dtype == L.w_up.dtype) {
            mark(0, true);
            int st = NTK_E_DTYPE;
            if (repack_ && L.w_gate.rp && L.w_up.rp && (rp_mask() & 4)) {
                ntk_gemv_seg rs[2] = {{L.w_gate.rp, gate_buf, I, L.w_gate.dtype}, {L.w_up.rp, up_buf, I, L.w_up.dtype}};
                st = ntk_gemv_rp_fused(rs, 2, hidden_, H, (const float*)L.ffn_norm.ptr, cfg_.norm_eps, nullptr, 1, s);
                if (st != NTK_OK && st != NTK_E_DTYPE && st != NTK_E_SHAPE && st != NTK_E_ALIGN) return st;
            }
            if (st != NTK_OK) {
                raw_begin();
                ntk_gemv_seg segs[2] = {{raw_of(L.w_gate), gate_buf, I, L.w_gate.dtype}, {raw_of(L.w_up), up_buf, I, L.w_up.dtype}};
                NT_TRY(ntk_gemv_fused(segs, 2, hidden_, H, (const float*)L.ffn_norm.ptr, cfg_.norm_eps, nullptr, 1, s));
            }
            mark(0, false);
        } else {
            const DevTensor* ws[2] = {&L.w_gate, &L.w_up};
            float* ys[2] = {gate_buf, up_buf};
            NT_TRY(project(ws, ys, 2, hidden_, &L.ffn_norm, nullptr, 4));
            NT_TRY(ntk_silu_mul(gate_buf, gate_buf, up_buf, I, s));
        }
        if (tp_world_ > 1) {
            NT_TRY(project1(L.w_down, tp_slot(), gate_buf, nullptr, nullptr, 8));
            NT_TRY(tp_allreduce(hidden_, H));
        } else {
            NT_TRY(project1(L.w_down, hidden_, gate_buf, nullptr, hidden_, 8));
        }
    }
    return NTK_OK;
}

// ---- parity instrumentation (tests; reached through nt_engine_debug_*, never from the generate loop) --------------------------
// Layers [first, first + count) on caller-supplied hidden states: hidden_in [T][H] (host) -> hidden_out [T][H] (host), tokens at
// positions start_pos...  mode 0: the 1:1 launcher sequence (prompt projections batched or per token as set_batched_prefill says);
// mode 1: the fused single-token launches (T == 1); mode 2: the same replayed from a freshly captured hipGraph.  The KV cache
// rows of the T positions are written by the layers as in a normal forward; rows of earlier positions are whatever the cache
// holds (debug_kv_write puts a checker's rows there: layer-wise teacher forcing).
int Model::debug_run_layers(const float* hidden_in, int T, int start_pos, int first, int count, int mode, float* hidden_out) {
    if (!hidden_in || !hidden_out) return NTK_E_NULL;
    if (T <= 0 || start_pos < 0 || start_pos + T > cfg_.max_seq_len || first < 0 || count < 0 || first + count > cfg_.n_layers) return NTK_E_SHAPE;
    if (mode != 0 && T != 1) return NTK_E_SHAPE;
    if (tp_world_ > 1) return NTK_E_SHAPE;
    const size_t bytes = (size_t)T * cfg_.hidden_size * 4;
    void* s = stream_;
    NT_TRY(ntk_memcpy_h2d_async(hidden_, hidden_in, bytes, s));
    int rc;
    if (mode == 0) {
        std::vector<int> pos(T);
        for (int i = 0; i < T; ++i) pos[i] = start_pos + i;
        NT_TRY(ntk_memcpy_h2d_async(positions_, pos.data(), (size_t)T * 4, s));
        NT_TRY(ntk_stream_synchronize(s));
        rc = layers_1to1(T, start_pos, first, first + count);
    } else {
        NT_TRY(set_device_pos(start_pos));
        pick_attention_regime();
        if (mode == 1) {
            rc = enqueue_layers(first, first + count);
        } else {
            hipStream_t st = static_cast<hipStream_t>(s);
            hipGraph_t g = nullptr;
            if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess) return NTK_E_LAUNCH;
            rc = enqueue_layers(first, first + count);
            const hipError_t e = hipStreamEndCapture(st, &g);
            if (rc == NTK_OK && (e != hipSuccess || !g)) rc = NTK_E_LAUNCH;
            hipGraphExec_t ex = nullptr;
            if (rc == NTK_OK && hipGraphInstantiate(&ex, g, nullptr, nullptr, 0) != hipSuccess) rc = NTK_E_LAUNCH;
            if (g) (void)hipGraphDestroy(g);
            if (rc == NTK_OK && hipGraphLaunch(ex, st) != hipSuccess) rc = NTK_E_LAUNCH;
            if (rc == NTK_OK) rc = ntk_stream_synchronize(s);
            if (ex) (void)hipGraphExecDestroy(ex);
        }
    }
    if (rc != NTK_OK) return rc;
    NT_TRY(ntk_memcpy_d2h_async(hidden_out, hidden_, bytes, s));
    return ntk_stream_synchronize(s);
}

// cache rows [pos0, pos0 + n) of one layer, [n][n_kv_heads * head_dim] halves each (reference layout, transformer.cpp:340-346)
int Model::debug_kv(int layer, int pos0, int n, uint16_t* k, uint16_t* v, bool write) {
    if (!k || !v) return NTK_E_NULL;
    if (layer < 0 || layer >= cfg_.n_layers || pos0 < 0 || n < 0 || pos0 + n > cfg_.max_seq_len) return NTK_E_SHAPE;
    const size_t per = (size_t)cfg_.n_kv_heads * cfg_.head_dim;
    const size_t off = ((size_t)layer * cfg_.max_seq_len + pos0) * per, bytes = (size_t)n * per * 2;
    void* s = stream_;
    if (write) {
        NT_TRY(ntk_memcpy_h2d_async(k_cache_ + off, k, bytes, s));
        NT_TRY(ntk_memcpy_h2d_async(v_cache_ + off, v, bytes, s));
    } else {
        NT_TRY(ntk_memcpy_d2h_async(k, k_cache_ + off, bytes, s));
        NT_TRY(ntk_memcpy_d2h_async(v, v_cache_ + off, bytes, s));
    }
    return ntk_stream_synchronize(s);
}

// A tensor-parallel exchange whose bounded wait for a peer gave up has added garbage: surface it (and clear the sticky word)
int Model::check_tp() {
    if (tp_world_ <= 1 || !tp_comm_) return NTK_OK;
    const unsigned e = tp_error();
    if (e == 0u) return NTK_OK;
    const unsigned zero = 0u;
    (void)ntk_memcpy_h2d_async(static_cast<uint8_t*>(tp_comm_) + 128, &zero, 4, stream_);
    (void)ntk_stream_synchronize(stream_);
    err_ = "tensor-parallel exchange: a peer rank did not arrive (call tag " + std::to_string(e) + "); the token's results are invalid";
    fprintf(stderr, "%s\n", err_.c_str());
    return NTK_E_LAUNCH;
}

bool Model::use_persistent_now() const {
    return persistent_plan_ && persistent_on_ && attn_regime_ == 0 && !prof_;
}

void Model::set_persistent(int level) {   // 0 off, 1 the round-2 token kernel (decode_persistent.hip), 2 the loader / consumer engine (layer_engine.hip)
    const bool on = level != 0;
    persistent_on_ = false;
    persistent_wanted_ = level;   // (asked before the load: finish_load() applies it)
#ifndef NTK_EXPERIMENTS
    if (on) fprintf(stderr, "note: the persistent token kernels are built by experiments/Makefile only (experiments/libntransformer_hip_exp.so); this library decodes with fused launches\n");
#else
    if (persistent_plan_ && persistent_kind_ != (level == 2 ? 2 : 1)) {   // the other kernel's plan: drop it and its captured graphs
        (void)sync();
        for (auto& row : graphs_) { if (row[kPersistentSlot]) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(row[kPersistentSlot])); row[kPersistentSlot] = nullptr; }
        if (persistent_kind_ == 2) ntk_layer_engine_plan_destroy(persistent_plan_); else ntk_persistent_plan_destroy(persistent_plan_);
        persistent_plan_ = nullptr;
    }
#endif
    if (!on || tp_world_ != 1 || layers_.empty()) return;
    if (raw_freed_bytes_ > 0) (void)set_repack(1);   // the persistent kernels stream the GGUF bytes themselves: those must be resident
    if (!persistent_plan_) (void)build_persistent_plan(level == 2 ? 2 : 1);   // built on first use (EXPERIMENTS=1 builds only): it allocates device memory
    persistent_on_ = persistent_plan_ != nullptr;
}

// what decode_step_fused() emits at the CURRENT position (the persistent form covers the single-pass attention regime only)
const char* Model::decode_path() const {
    if (persistent_plan_ && persistent_on_ && persistent_kind_ == 2)
        return attn_regime_ == 0 ? "persistent layer engine (1 launch per token: loader / consumer waves, granule hand-offs; fused launches beyond the single-pass attention regime)"
                                 : "fused (5 launches/layer; persistent layer engine below the split-attention regime)";
    if (persistent_plan_ && persistent_on_)
        return attn_regime_ == 0 ? "persistent (1 launch per token in the single-pass attention regime, fused launches beyond)"
                                 : "fused (5 launches/layer; persistent below the split-attention regime)";
    return "fused (5 launches/layer)";
}

// after a sync: NTK_OK, or NTK_E_LAUNCH when an in-kernel bounded wait gave up (tensor-parallel exchange; with
// EXPERIMENTS=1 also the persistent token kernel and the attention-in-Wo launch, which are then disabled)
int Model::check_persistent() {
    NT_TRY(check_tp());
#ifdef NTK_EXPERIMENTS
    if (attn_sync_ && fuse_attention_) {   // ntk_attention_gemv_fused: a bounded in-kernel wait that gave up
        unsigned w[3] = {0, 0, 0};
        if (ntk_memcpy_d2h_async(w, attn_sync_, sizeof w, stream_) != NTK_OK || ntk_stream_synchronize(stream_) != NTK_OK) return NTK_E_LAUNCH;
        if (w[2] != 0) {
            fuse_attention_ = false;
            nt_hip_memset(attn_sync_, 0, 4096);
            for (auto& row : graphs_) for (auto& gx : row) { if (gx) (void)hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(gx)); gx = nullptr; }
            err_ = "attention + Wo fused launch: the wait for the attention workgroups gave up; falling back to separate launches";
            fprintf(stderr, "%s\n", err_.c_str());
            return NTK_E_LAUNCH;
        }
    }
    if (!persistent_plan_ || !persistent_on_) return NTK_OK;
    int op = -1;
    int st;
    if (persistent_kind_ == 2) {
        unsigned code = 0;
        st = ntk_layer_engine_error(persistent_plan_, &code);
        op = code ? (int)((code - 1u) & 4095u) : -1;
        if (st != NTK_OK) fprintf(stderr, "layer engine: error word %u (operator %d, wait kind %u, CU %u)\n", code, op, ((code - 1u) >> 12) & 15u, (code - 1u) >> 16);
    } else {
        st = ntk_persistent_error(persistent_plan_, &op);
    }
    if (st != NTK_OK) {
        persistent_on_ = false;
        err_ = "persistent decode kernel: a bounded grid wait gave up at operator " + std::to_string(op) + "; falling back to launches";
        fprintf(stderr, "%s\n", err_.c_str());
    }
    return st;
#else
    return NTK_OK;
#endif
}

#ifdef NTK_EXPERIMENTS
// The token's operator table for the persistent kernel: exactly the sequence enqueue_token() launches.
int Model::build_persistent_plan(int kind) {
    const int H = cfg_.hidden_size, I = cfg_.intermediate_size, hd = cfg_.head_dim, nh = cfg_.n_heads, nkv = cfg_.n_kv_heads;
    const int qd = nh * hd, kvd = nkv * hd;
    if (hd != 64 && hd != 128) return NTK_E_SHAPE;
    if (const char* e = getenv("NTK_NO_PERSISTENT")) { if (atoi(e)) return NTK_E_SHAPE; }
    const float scale = 1.0f / sqrtf((float)hd);
    const size_t kv_layer = (size_t)cfg_.max_seq_len * kvd;
    float* q_buf = workspace_;
    float* k_buf = q_buf + qd;
    float* v_buf = k_buf + kvd;
    float* attn_out = v_buf + kvd;
    float* gate_buf = workspace_;
    float* up_buf = gate_buf + I;
    std::vector<ntk_pop> ops;
    bool ok = true;
    // n matrices sharing x: one operator per dtype group (Q4_K_M: attn_v is Q6_K / Q5_K next to Q4_K q, k); only the first
    // waits for x, only the last signals
    auto gemv_group = [&](const DevTensor* const* ws, float* const* ys, int n, const float* x, const DevTensor* norm, const float* resid,
                          bool wait, bool arrive, bool plain) {
        bool done[3] = {false, false, false};
        std::vector<ntk_pop> grp;
        for (int a = 0; a < n; ++a) {
            if (done[a]) continue;
            if (!is_quant(ws[a]->dtype)) { ok = false; return; }
            ntk_pop o;
            memset(&o, 0, sizeof o);
            o.kind = NTK_POP_GEMV;
            for (int b = a; b < n; ++b) {
                if (done[b] || ws[b]->dtype != ws[a]->dtype) continue;
                o.segs[o.nseg++] = {ws[b]->ptr, ys[b], (int)ws[b]->out_f, ws[b]->dtype};
                done[b] = true;
            }
            o.in_features = (int)ws[a]->in_f;
            o.eps = cfg_.norm_eps;
            o.x = x;
            o.norm_w = norm ? (const float*)norm->ptr : nullptr;
            o.resid = resid;
            o.plain_store = plain ? 1 : 0;
            grp.push_back(o);
        }
        for (size_t i = 0; i < grp.size(); ++i) {
            grp[i].wait = (wait && i == 0) ? 1 : 0;
            grp[i].arrive = (arrive && i + 1 == grp.size()) ? 1 : 0;
            ops.push_back(grp[i]);
        }
    };
    for (int i = 0; i < cfg_.n_layers && ok; ++i) {
        const LayerWeights& L = layers_[i];
        {
            const DevTensor* ws[3] = {&L.wq, &L.wk, &L.wv};
            float* ys[3] = {q_buf, k_buf, v_buf};
            gemv_group(ws, ys, 3, hidden_, &L.attn_norm, nullptr, i > 0, true, false);   // layer 0 reads the embedding kernel's output
        }
        ntk_pop a;
        memset(&a, 0, sizeof a);
        a.kind = NTK_POP_ATTENTION; a.wait = 1; a.arrive = 1;
        a.out = attn_out; a.q = q_buf; a.k = k_buf; a.v = v_buf;
        a.k_cache = k_cache_ + (size_t)i * kv_layer; a.v_cache = v_cache_ + (size_t)i * kv_layer;
        a.inv_freq = rope_inv_freq_;
        a.n_heads = nh; a.n_kv_heads = nkv; a.head_dim = hd; a.max_seq = cfg_.max_seq_len;
        a.scale = scale; a.theta_base = cfg_.rope_theta; a.freq_scale = cfg_.rope_freq_scale;
        ops.push_back(a);
        {
            const DevTensor* ws[1] = {&L.wo};
            float* ys[1] = {hidden_};
            gemv_group(ws, ys, 1, attn_out, nullptr, hidden_, true, true, false);
        }
        if (!(is_quant(L.w_gate.dtype) && L.w_gate.dtype == L.w_up.dtype)) { ok = false; break; }
        {
            ntk_pop o;
            memset(&o, 0, sizeof o);
            o.kind = NTK_POP_GEMV; o.wait = 1; o.arrive = 1;
            o.segs[0] = {L.w_gate.ptr, gate_buf, I, L.w_gate.dtype};
            o.segs[1] = {L.w_up.ptr, up_buf, I, L.w_up.dtype};
            o.nseg = 2; o.in_features = H; o.silu_pair = 1; o.eps = cfg_.norm_eps;
            o.x = hidden_; o.norm_w = (const float*)L.ffn_norm.ptr;
            ops.push_back(o);
        }
        {
            const DevTensor* ws[1] = {&L.w_down};
            float* ys[1] = {hidden_};
            gemv_group(ws, ys, 1, gate_buf, nullptr, hidden_, true, true, false);
        }
    }
    if (ok) {
        const DevTensor* ws[1] = {&output_};
        float* ys[1] = {logits_};
        gemv_group(ws, ys, 1, hidden_, &output_norm_, nullptr, true, false, true);
    }
    if (!ok) return NTK_E_DTYPE;
    persistent_kind_ = kind;
    if (kind == 2) return ntk_layer_engine_plan_create(ops.data(), (int)ops.size(), &persistent_plan_);
    return ntk_persistent_plan_create(ops.data(), (int)ops.size(), &persistent_plan_);
}
#else
int Model::build_persistent_plan(int) { return NTK_E_SHAPE; }
#endif

void Model::pick_attention_regime() {
    attn_regime_ = (attn_scratch_ && (cfg_.head_dim == 64 || cfg_.head_dim == 128 || cfg_.head_dim == 256))
                       ? attention_regime(host_pos_, cfg_.head_dim) : 0;
    ++host_pos_;   // every fused token ends with ntk_advance_pos on the device; set_device_pos() re-bases both
}

int Model::decode_step_fused(bool greedy, bool use_graph) { return run_token(greedy ? kGreedy : kSampled, use_graph); }

// A given token at a given position: its words go with the launch of its embedding row, in front of the captured layers, and the launch that takes the logits out advances the position -- a token is
// two launches shorter than set_device_step, decode_step_fused and copy_logits one after the other.
int Model::decode_token(int token, int pos, bool use_graph, float* host) {
    if (tp_world_ > 1 || !out_row_ || use_persistent_now()) {
        NT_TRY(set_device_step(pos, token));
        NT_TRY(decode_step_fused(false, use_graph));
        return copy_logits(host);
    }
    if (token < 0 || token >= cfg_.vocab_size) { err_ = "token id out of range"; return NTK_E_SHAPE; }
    *h_token_ = token;
    host_pos_ = pos;
    NT_TRY(ntk_embed_token_row(hidden_, token_embd_.ptr, token, pos, d_token_, d_pos_, cfg_.hidden_size, token_embd_.dtype, stream_));
    NT_TRY(run_token(kBare, use_graph));
    return out_row_.fetch(host, logits_, d_pos_, stream_);
}

int Model::run_token(TokenKind kind, bool use_graph) {
    pick_attention_regime();
    if (!use_graph) return enqueue_token(kind);
    ihipGraphExec_t*& slot = graphs_[kind][use_persistent_now() ? kPersistentSlot : attn_regime_];
    hipStream_t st = static_cast<hipStream_t>(stream_);
    if (!slot) {   // capture once: every per-token quantity (token id, position) lives in device memory
        hipGraph_t g = nullptr;
        // (relaxed under tensor parallelism: ranks sharing a process run their own runtime calls on other threads meanwhile)
        if (hipStreamBeginCapture(st, tp_world_ > 1 ? hipStreamCaptureModeRelaxed : hipStreamCaptureModeThreadLocal) != hipSuccess) return NTK_E_LAUNCH;
        const int rc = enqueue_token(kind);
        const hipError_t e = hipStreamEndCapture(st, &g);
        if (rc != NTK_OK || e != hipSuccess || !g) { if (g) (void)hipGraphDestroy(g); return rc != NTK_OK ? rc : NTK_E_LAUNCH; }
        hipGraphExec_t ex = nullptr;
        const hipError_t ie = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ie != hipSuccess) return NTK_E_LAUNCH;
        slot = reinterpret_cast<ihipGraphExec_t*>(ex);
    }
    return hipGraphLaunch(reinterpret_cast<hipGraphExec_t>(slot), st) == hipSuccess ? NTK_OK : NTK_E_LAUNCH;
}

int Model::profile_token(float ms[4], int calls[4], bool coarse) {
    std::vector<Timed> rec;
    rec.reserve(1024);
    prof_ = &rec;
    prof_coarse_ = coarse;
    pick_attention_regime();
    int rc = enqueue_token(kGreedy);
    if (coarse && !rec.empty()) {   // close the last run
        void* e = ntk_event_create();
        ntk_event_record(e, stream_);
        rec.back().b = e;
    }
    prof_ = nullptr;
    prof_coarse_ = false;
    if (rc == NTK_OK) rc = ntk_stream_synchronize(stream_);
    for (int c = 0; c < 4; ++c) { ms[c] = 0.0f; calls[c] = 0; }
    for (auto& t : rec) {
        float m = 0.0f;
        if (t.a && t.b && ntk_event_elapsed_ms(t.a, t.b, &m) == NTK_OK) { ms[t.cls] += m; calls[t.cls] += t.n; }
        ++calls[3];   // timed intervals
    }
    for (auto& t : rec) {   // coarse: record i's `b` is record i+1's `a` -- destroy every event once
        if (t.a && !t.shared_a) ntk_event_destroy(t.a);
        if (t.b) ntk_event_destroy(t.b);
    }
    return rc;
}

}  // namespace nt
