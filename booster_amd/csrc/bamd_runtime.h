// bamd_runtime.h — what the model families of the library share: the model / context objects behind include/bamd.h, error handling, device allocation,
// and the interface a family implements.  bamd_engine.cpp holds the GGUF Llama pipeline and the C entry points; a family registered in bamd_arch.cpp that is not
// that pipeline hangs a bamd_arch_runtime on its model, and the entry points hand over to it.
#pragma once
#include "../../include/bamd.h"
#include "bamd_formats.h"
#include "bamd_gguf.h"
#include "bamd_kernels.h"
#include "bamd_aql.h"

#include <hip/hip_runtime.h>
#include <memory>
#include <string>
#include <vector>

int bamd_fail(const std::string & m);                 // sets bamd_last_error of this thread, returns 1
#define HIPC(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return bamd_fail(std::string(#x) + ": " + hipGetErrorString(e_)); } while (0)

struct bamd_arch_runtime {
    virtual ~bamd_arch_runtime() {}
    virtual int context_init(bamd_context * c) = 0;                  // c->m, n_ctx, n_seq, stream, logits, logits_host, co_err are set
    virtual void context_free(bamd_context * c) = 0;
    virtual void clear(bamd_context * c) = 0;                        // every sequence forgotten
    virtual int seq_len(bamd_context * c, int seq) = 0;
    virtual int seq_free(bamd_context * c, int seq) = 0;
    // one batch: the entries' tokens run behind what their sequences hold; logits of the wanted places in order to `logits` (host, may be null).  Rows stay in
    // c->logits while they fit BAMD_LOGIT_ROWS.  wait = false: everything enqueued on the context's stream, nothing copied
    virtual int decode_batch(bamd_context * c, const bamd_batch_entry * e, int n, float * logits, bool wait) = 0;
    // greedy steps on the device; first: token fed to each sequence's first step (null: one sequence, the arg-max of row 0 of c->logits); out [n_seqs][n_steps + 1]
    virtual int generate(bamd_context * c, const int32_t * seqs, int n_seqs, int n_steps, const int32_t * first, int32_t * out, float * ms) = 0;
    // layer-split stage: n tokens of sequence 0; token_dev: device int32 instead of `tokens` (n = 1)
    virtual int stage(bamd_context * c, const int32_t * tokens, const void * token_dev, int n, int n_past, const void * hidden_in, void * hidden_out, bool want_logits, hipStream_t s) = 0;
    virtual int argmax_to(bamd_context * c, int32_t * token_dev, hipStream_t s) = 0;
    virtual int profile_kinds(bamd_context * c, int pos, int * launches, double * ms, double * bytes) = 0;
    virtual const char * vocab_path() = 0;                            // GGUF with the tokenizer, "" = none
};
#define BAMD_LOGIT_ROWS 64

// -------------------------------------------------------------------------------------------------------
struct DevMat {                      // one quantised matrix resident in HBM
    void * stream = nullptr;         // wave-stream records (matmul operand)
    void * raw = nullptr;            // GGUF layout (kept only for token_embd: row gather)
    int type = 0, nrows = 0, K = 0;  // nrows = rows in the GGUF
    int nrows_pad = 0;               // rows of the stream (next multiple of 8; missing rows are zero records)
    size_t bytes = 0;
};
struct DevLayer {
    float * attn_norm = nullptr, * ffn_norm = nullptr;
    DevMat wq, wk, wv, wo, wg, wu, wd;
    // prefill side tables (bamd_prefill2.hip), built at the first batched evaluation: one per QKV segment as enqueue_prefill_batch merges them, wo, gate, up, down
    void * aux_qkv[3] = { nullptr, nullptr, nullptr }, * aux_o = nullptr, * aux_g = nullptr, * aux_u = nullptr, * aux_d = nullptr;
};

struct bamd_model {
    const char * arch = "llama";
    std::unique_ptr<bamd_arch_runtime> rt;      // null: the GGUF Llama pipeline of bamd_engine.cpp
    int device = 0;
    int E = 0, H = 0, Hkv = 0, hd = 0, L = 0, F = 0, V = 0, n_ctx_train = 0, n_rot = 0;
    float eps = 1e-5f, rope_theta = 10000.f, rope_freq_scale = 1.f, rope_ext_factor = 0.f, rope_attn_factor = 1.f;
    int rope_n_ctx_orig = 0;
    int layer_first = 0, layer_last = 0;
    bool with_embd = true, with_output = true;
    std::vector<float> rope_freqs;   // host copy (optional)
    std::vector<DevLayer> layers;    // [layer_last - layer_first]
    DevMat tok_embd, output;
    float * out_norm = nullptr;
    int64_t weight_bytes = 0;
    int n_cu = 256;
    std::unique_ptr<GgufFile> file;  // stays mapped (bamd_model_tensor_raw)
    std::vector<void *> allocs;
    bool aux_ok = false; int64_t aux_bytes = 0; std::string aux_why;      // prefill side tables: all matrices or none (build_prefill_aux)
};

struct bamd_context {
    bamd_model * m = nullptr;
    int n_ctx = 0;
    int n_seq = 1;                   // sequences the context holds (more than one: families with a bamd_arch_runtime)
    void * arch_state = nullptr;     // of that family
    std::vector<unsigned short *> kc, vc;
    float * rope = nullptr, * rope_cur = nullptr;   // rope_cur [hd]: the cos / sin row of the current step's position (step_begin_kernel -> attn_qk_kernel)
    float * x = nullptr, * x2 = nullptr, * q = nullptr, * k = nullptr, * v = nullptr, * att = nullptr, * h = nullptr, * scores = nullptr, * probs = nullptr;
    int n_ctx_pad = 0;              // KV row stride: n_ctx rounded up to 64 (V^T rows are stored in 64-position blocks)
    float * logits = nullptr;        // device
    float * logits_host = nullptr;   // pinned
    bool logits_readback = true, logits_host_valid = false;
    bool status_pending = false;     // a bamd_decode without read-back returned before its stream was waited for: the next synchronising call checks the give-up words
    // sampler prefilter (bamd_logits_shortlist): per-vocabulary tables, penalty list and result (device + pinned mirrors)
    uint8_t * samp_cls = nullptr; float * samp_cut = nullptr;
    bamd_logit_penalty * samp_pen = nullptr, * samp_pen_host = nullptr;
    unsigned char * samp_out = nullptr, * samp_out_host = nullptr;
    bamd_step_state * st = nullptr;
    int32_t * forced = nullptr; int forced_cap = 0;
    int32_t * out_tokens = nullptr; int out_cap = 0;
    hipStream_t stream = nullptr;
    hipGraphExec_t graph = nullptr; int graph_fused = -1;
    bamd_aql_graph * aql = nullptr; int aql_key = -1; bool aql_failed = false; int aql_runs = 0;    // the same step as AQL packets for the own queue (bamd_aql.h)
    bamd_aql_graph * aql_step[4] = {}; int aql_steps = 0, aql_recorded = 0;                        // stage_step's single-token steps on the own queue: fused attention x logits to the host
    bamd_step_state * inbox = nullptr;           // pinned host memory: the state of that step, read by step_begin_kernel itself (no copy in front of the step)
    unsigned long long * co_gran = nullptr;   // co-launch granules [H * hd] {value, tag} + give-up counter behind them (bamd_colaunch.hip), zero-initialised
    uint32_t * co_err = nullptr;
    int32_t * slots = nullptr; int slots_cap = 0;   // device-side greedy loop after a context shift: {cell, padded KV length} of every step (bamd_generate_greedy)
    int host_serial = 0;             // host calls that set the device state so far (bamd_step_state.serial)
    // KV cell metadata (llama_kv_cache cells: pos / delta / head / used, llama.cpp:2700-2760) — inactive (cell i holds position i, nothing to
    // track) until the first bamd_kv_seq_rm / bamd_kv_seq_add
    struct Cells { bool active = false, has_shift = false; std::vector<int32_t> pos, delta; int head = 0, used = 0; } cells;
    int n_cached = 0;               // positions evaluated so far (highest n_past + n_tokens seen): what the cells hold when tracking starts
    int32_t * cellpos = nullptr;    // device copy of cells.pos (attention mask of the shifted path)
    int32_t * shift_idx = nullptr; float * shift_tab = nullptr; int shift_tab_cap = 0;
    // stage-step graphs (bamd_stage_step): one per (want_logits, prefill_mode), valid for the pointers it was captured with
    struct StageGraph { hipGraphExec_t exec = nullptr; const void * token_src = nullptr, * hin = nullptr; void * hout = nullptr; int fused = -1; };
    StageGraph sgraph[2][2];
    // batched prefill buffers, [bcap] tokens each (allocated at the first multi-token decode)
    // phase-stamp blocks (bamd_timeline_step, BAMD_TIMING builds): one block of BAMD_TL_SLOT_WORDS u64 per launch
    unsigned long long * tl_base = nullptr; int tl_slot = 0, tl_cap = 0;
    int bcap = 0; bool bwide_failed = false;
    float * attn_bscr = nullptr; size_t attn_bscr_bytes = 0, attn_bscr_failed = 0;   // score rows of the matrix-core prefill attention beyond BAMD_AM_MAXPOS = 896 positions (grow-only; absent = the VALU kernel runs)
    float * bx = nullptr, * bx2 = nullptr, * bqkv = nullptr, * batt = nullptr, * bh = nullptr; bamd_step_state * bst = nullptr;
    void * blay[3] = {}; int blay_tokens[3] = {};                   // activations quantised: rows of bytes, f16 records, f16 fragments (each allocated when a product first reads it)
    std::vector<void *> allocs;
};

// fresh memory is given its pages here (a fault per 4 KiB: 130 us for sixteen rows of 32 000 logits), in time that the host would wait for the device
static inline void bamd_touch(float * p, size_t n) { for (size_t i = 0; i < n; i += 1024) ((volatile float *) p)[i] = 0.f; if (n) ((volatile float *) p)[n - 1] = 0.f; }
static inline int dev_alloc(std::vector<void *> & keep, void ** p, size_t bytes) {
    HIPC(hipMalloc(p, bytes + 4096));           // + 4 KiB: the sixteen-wave prefill kernel's nibble loads of the two super-blocks behind the end of K run past
                                                // the last record group (bamd_prefill2.hip)
    keep.push_back(*p);
    return 0;
}
