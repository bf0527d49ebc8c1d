// engine.h -- host-side state shared by the libpgmi engines: the context, its weight slab and captured
// graphs, error reporting, and the helpers the C ABI files use (internal, not the C ABI).
//
//   engine_core.hip     family-independent ABI: weights, loading, sampling, stop tokens, replicas
//   engine.hip          the PaliGemma family
//   engine_decoder.hip  the layered-decoder family (a list of layers, each a mixer and a feed-forward)
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "../../include/pgmi.h"
#include "common.h"
#include "launch.h"

using namespace pgmi;

struct DecoderState;  // engine_decoder.hip

int pgmi_fail(int code, const std::string& msg);  // sets pgmi_last_error() of the calling thread, returns code
static inline int fail(int code, const std::string& msg) { return pgmi_fail(code, msg); }

#define HIPCHK(expr)                                                                       \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess) return fail(PGMI_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define LAUNCHCHK()                                                                        \
    do {                                                                                   \
        hipError_t e_ = hipGetLastError();                                                 \
        if (e_ != hipSuccess) return fail(PGMI_E_HIP, std::string("kernel launch: ") + hipGetErrorString(e_)); \
    } while (0)

struct Slot {
    std::string name;
    int64_t off;
    int64_t shape[4];
    int ndim;
    int64_t numel;
};

struct GraphKey {
    int B;
    void* kv;
    int kv_batch, kv_max;
    float* logits;
    int64_t* next;
    const int64_t* ids;  // the ids that the graph reads: those it feeds back in place (null: the launch in front of it reads them)
    bool emb;            // the step's input is the staged embedding rows (pgmi_decode_embeds), not ids
    int masked;          // 0: no mask (a zero word), 1: staged bf16 mask (sum rounded), 2: staged fp32 mask
    int n_steps;         // decode steps captured back to back (pgmi_decode_steps; 1 otherwise)
    int64_t* tokens;     // their per-step token record ([n_steps][B], may be null)
    bool operator<(const GraphKey& o) const {
        return std::tie(B, kv, kv_batch, kv_max, logits, next, ids, emb, masked, n_steps, tokens) <
               std::tie(o.B, o.kv, o.kv_batch, o.kv_max, o.logits, o.next, o.ids, o.emb, o.masked, o.n_steps,
                        o.tokens);
    }
};

// a decode step, its first launch (the only one that reads its token ids), or all but that
enum StepPart { STEP_ALL, STEP_HEAD, STEP_REST };

struct GraphEntry {
    int seen = 0;
    hipGraphExec_t exec = nullptr;
};

// Which engine a context belongs to, and what the family-independent ABI asks of it
enum Family : int { FAMILY_PALIGEMMA = 0, FAMILY_DECODER = 1 };

struct pgmi_ctx {
    Family family = FAMILY_PALIGEMMA;
    int (*prepare)(pgmi_ctx*) = nullptr;                          // pgmi_prepare
    int64_t (*kv_bytes)(const pgmi_ctx*, int, int) = nullptr;     // pgmi_kv_bytes
    void (*release)(pgmi_ctx*) = nullptr;                         // family part of pgmi_destroy (may be null)
    DecoderState* dec = nullptr;                                  // FAMILY_DECODER
    pgmi_config c;                                                // FAMILY_PALIGEMMA
    int device;
    std::vector<Slot> slots;
    std::unordered_map<std::string, int> index;
    int64_t slab_bytes = 0;
    uint8_t* slab = nullptr;
    std::vector<float> inv_freq;
    std::vector<uint16_t> host_cos, host_sin;  // optional exact table
    bool prepared = false;
    std::vector<void*> allocs;
    // derived
    uint16_t* patch_w = nullptr;  // [v_hidden][kpad]
    int kpad = 0;
    int ipad = 0;  // v_intermediate rounded up to 64: the row pitch of vH
    uint16_t* cosT = nullptr;
    uint16_t* sinT = nullptr;
    // text prefill workspace (rows = max_batch*max_seq)
    uint16_t *Hs, *Tn, *QKV, *Qr, *AO, *ACT, *lastrows;
    long tn_rows = 0;  // rows of Tn holding the final RMSNorm of the last pgmi_lm_forward (pgmi_lm_final_hidden)
    int64_t* dpos;
    int64_t* dids_tmp;
    // vision workspace (rows = max_batch*N)
    uint16_t *vX, *vT, *vQKV, *vAO, *vH, *vP;
    float* ws;
    size_t ws_bytes;
    // decode workspace
    uint16_t *dH, *dQ, *dAO, *dACT;
    uint16_t* dHn;  // batched decode (B >= 3): the RMSNorm'd rows the unstaged MFMA projections read
    float* dSS;     // batched decode: o_proj's 16-column partial sums of squares of h, [B][H / 16]
    // batched decode (max_batch >= 3): fragment-major images of every layer's gate|up, q|k|v (in the GEMV's row
    // order), o_proj and down weights (mf_swizzle), [layer][gate|up 2 I x H | q|k|v QKVN x H | o_proj | down H x I]
    uint16_t* mfw = nullptr;
    size_t mfw_layer = 0;
    bool mfw_dirty = false;  // the fragment-major images are (re)built by the next batched decode step
    float *opart, *pmax, *dlogits, *amax_v;
    int *pidx, *amax_i;
    int max_chunks;
    StepState* step;
    StepState* pstep;  // the generate-loop prefill's last-row attention (flash-decoding over the prompt's keys)
    uint16_t* d_emb;             // staged input rows of pgmi_decode_embeds ([max_batch][hidden] bf16)
    float* d_mask;               // staged additive decode mask ([max_batch][max_kv] fp32, pgmi_decode_embeds_dev)
    float* d_zero;               // one zero word: the "no mask" mask of the decode attention
    int64_t* d_next;             // argmax target when the caller passes none
    unsigned* lm_done;           // lm_head arrival counter (argmax folded into its last workgroup)
    hipStream_t cap_stream = nullptr;
    std::map<GraphKey, GraphEntry> graphs;
    // prefill graphs (vision tower, language-model forward): replayed for repeated calls with
    // identical pointer/shape arguments (a replay is the eager call: kernels read the same
    // addresses at run time), captured on the second such call
    bool prefill_graph = true;
    int mf_staged = -1;  // batched decode RMSNorm form (mf_staged()); -1 = default (unstaged)
    // device step state as the last enqueued per-phase decode step leaves it (advanced in-graph)
    bool step_known = false;
    int step_kv = 0, step_pos = 0;
    std::map<std::vector<intptr_t>, GraphEntry> pgraphs;
    // in-situ timing probe of the prefill MLP GEMMs (pgmi_prefill_probe): events around layer i's gate|up
    // GEMM (ev[4i], ev[4i+1]) and down GEMM (ev[4i+2], ev[4i+3]) of eager forwards
    std::vector<hipEvent_t> probe_ev;
    bool probe_on = false;
    bool graph_before_probe = true;  // prefill_graph as the caller left it before the probe turned it off
};

inline void clear_pgraphs(pgmi_ctx* x) {
    for (auto& kv : x->pgraphs)
        if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    x->pgraphs.clear();
}

// the captured decode steps
inline void clear_dgraphs(pgmi_ctx* x) {
    for (auto& kv : x->graphs)
        if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    x->graphs.clear();
}

inline void add_slot(pgmi_ctx* x, const std::string& name, std::initializer_list<int64_t> shape) {
    Slot s;
    s.name = name;
    s.ndim = (int)shape.size();
    s.numel = 1;
    int i = 0;
    for (int64_t d : shape) { s.shape[i++] = d; s.numel *= d; }
    for (; i < 4; ++i) s.shape[i] = 1;
    s.off = x->slab_bytes;
    x->slab_bytes += (s.numel * 2 + 255) / 256 * 256;
    x->index[name] = (int)x->slots.size();
    x->slots.push_back(s);
}

inline uint16_t* W(pgmi_ctx* x, const std::string& name) {
    auto it = x->index.find(name);
    if (it == x->index.end()) return nullptr;
    return reinterpret_cast<uint16_t*>(x->slab + x->slots[it->second].off);
}

inline uint16_t host_f2bf(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

inline float bf16_round_host(float f) {
    uint32_t u = (uint32_t)host_f2bf(f) << 16;
    float r;
    std::memcpy(&r, &u, 4);
    return r;
}

inline uint64_t fnv1a(const char* s) {
    uint64_t h = 0xCBF29CE484222325ULL;
    for (const unsigned char* p = (const unsigned char*)s; *p; ++p) { h ^= *p; h *= 0x100000001B3ULL; }
    return h;
}

inline uint64_t splitmix64_h(uint64_t x) {
    x += 0x9E3779B97F4A7C15ULL;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ULL;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBULL;
    return x ^ (x >> 31);
}

inline int dalloc(pgmi_ctx* x, void** p, size_t bytes) {
    if (bytes == 0) bytes = 256;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) return fail(PGMI_E_NOMEM, std::string("hipMalloc ") + std::to_string(bytes) + ": " + hipGetErrorString(e));
    x->allocs.push_back(*p);
    return 0;
}

template <typename T>
int dalloc_t(pgmi_ctx* x, T** p, size_t count) {
    return dalloc(x, reinterpret_cast<void**>(p), count * sizeof(T));
}


inline int ensure_prepared(pgmi_ctx* x, Family family = FAMILY_PALIGEMMA) {
    if (!x) return fail(PGMI_E_ARG, "null context");
    if (x->family != family) return fail(PGMI_E_STATE, "this call belongs to another model family");
    if (!x->prepared) return fail(PGMI_E_STATE, "pgmi_prepare() has not been called");
    if (!x->slab) return fail(PGMI_E_STATE, "weights are not bound (pgmi_bind_weights)");
    return 0;
}

// Run body(stream) eagerly, or replay its captured hipGraph: the first call with a given key
// runs eagerly (kernel attributes are set on first launch), the second captures, later ones
// replay.  The key holds every pointer and size the body reads, so a replay is that call.
template <class F>
static int run_graphed(pgmi_ctx* x, hipStream_t s, const std::vector<intptr_t>& key, F body) {
    if (!x->prefill_graph) return body(s);
    GraphEntry& ge = x->pgraphs[key];
    if (!ge.exec) {
        if (ge.seen++ == 0) return body(s);
        if (x->pgraphs.size() > 64) {  // bound the cache (e.g. fresh buffers every call)
            clear_pgraphs(x);
            return body(s);
        }
        hipGraph_t g;
        HIPCHK(hipStreamBeginCapture(x->cap_stream, hipStreamCaptureModeThreadLocal));
        const int rc = body(x->cap_stream);
        HIPCHK(hipStreamEndCapture(x->cap_stream, &g));
        if (rc) {
            (void)hipGraphDestroy(g);
            return rc;
        }
        GraphEntry& ge2 = x->pgraphs[key];
        HIPCHK(hipGraphInstantiate(&ge2.exec, g, nullptr, nullptr, 0));
        (void)hipGraphDestroy(g);
        HIPCHK(hipGraphLaunch(ge2.exec, s));
        return 0;
    }
    HIPCHK(hipGraphLaunch(ge.exec, s));
    return 0;
}
