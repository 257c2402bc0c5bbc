// qwen_runtime_api.cpp -- C ABI of the decode runtime (include/qwen_kernels.h):
// the reference's rmsnorm ... rmsnorm_gated on host pointers, and its compiled
// forward loop (forward_linear_layer, forward_mlp, forward_token_c) run on
// the GPU with weights, parameters and activations resident in HBM.  All
// arithmetic is in the HIP kernels (runtime_ftz.hip, bfp8_ftz.hip,
// bf16_head.hip); nothing here computes results on the CPU.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "host_internal.h"
#include "runtime_internal.h"

namespace qhost {
namespace {

// ---- host-pointer calls: one arena in, kernels, the same arena out --------------------
// Arguments are packed at 256-byte offsets into a pinned buffer, copied to the
// device in one transfer, and copied back in one transfer after the kernels.
struct HostCall {
    struct Arg {
        void* host;
        size_t bytes, off;
        bool out;
    };
    std::vector<Arg> args;
    size_t total = 0;
    // Registers an argument; returns its offset in the arena.
    size_t add(const void* p, size_t bytes, bool out) {
        const size_t off = total;
        args.push_back(Arg{const_cast<void*>(p), bytes, off, out});
        total += (bytes + 255) & ~(size_t)255;
        return off;
    }
    int upload() {
        int rc;
        if ((rc = g.rt_pin.reserve(total)) || (rc = g.rt_dev.reserve(total))) return rc;
        char* pin = static_cast<char*>(g.rt_pin.p);
        for (const Arg& a : args)
            if (a.bytes) memcpy(pin + a.off, a.host, a.bytes);
        HIP_OK(hipMemcpyAsync(g.rt_dev.p, pin, total, hipMemcpyHostToDevice, g.stream));
        return BFP8_OK;
    }
    template <class T>
    T* dev(size_t off) const {
        return reinterpret_cast<T*>(static_cast<char*>(g.rt_dev.p) + off);
    }
    int download() {
        HIP_OK(hipMemcpyAsync(g.rt_pin.p, g.rt_dev.p, total, hipMemcpyDeviceToHost, g.stream));
        HIP_OK(hipStreamSynchronize(g.stream));
        const char* pin = static_cast<const char*>(g.rt_pin.p);
        for (const Arg& a : args)
            if (a.out && a.bytes) memcpy(a.host, pin + a.off, a.bytes);
        return BFP8_OK;
    }
};

#define RT_CHECK(where, expr)                                                            \
    do {                                                                                 \
        int rc_ = (expr);                                                                \
        if (rc_ != BFP8_OK) fatal(where);                                                \
    } while (0)

#define RT_LAUNCH(expr)                                                                  \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess) {                                                          \
            set_error("%s: %s", #expr, hipGetErrorString(e_));                           \
            return BFP8_EHIP;                                                            \
        }                                                                                \
    } while (0)

// ---- the forward -----------------------------------------------------------------------
constexpr int kHidden = RT_HIDDEN, kConv = RT_CONV_CH, kHD = RT_HEADS * RT_HEAD_DIM, kMlp = 3584;
constexpr int kVocab = 65536, kLayers = 24;
constexpr size_t kTapsLen = (size_t)3 * kConv, kStateLen = (size_t)RT_HEADS * RT_HEAD_DIM * RT_HEAD_DIM;

// Device copies of parameters the forward reads (float vectors, bf16 tables,
// writable BFP8 planes), keyed by host address and size, kept until
// bfp8_cache_clear().
struct ParamKey {
    const void* p;
    size_t bytes;
    bool operator<(const ParamKey& o) const { return p != o.p ? p < o.p : bytes < o.bytes; }
};

struct DevState {
    // [3][6144] taps and [16][128*128] blocked state, the current ones conv[cur]
    // and rec[rcur] (the separate launches update rec in place; rec[1] is there
    // where the device has room for it: the layer can run in a chain)
    DevBuf buf;                              // conv[0], conv[1], rec[0]
    float *conv[2], *rec[2] = {nullptr, nullptr};
    int cur = 0, rcur = 0;
    float* host_conv;     // the caller's buffers
    float* host_rec;
    bool resident_used = false;  // advanced on the device while resident
    bool dirty = false;          // device copy newer than the caller's buffers
};

// One layer (linear-attention layer or MLP of a full-attention layer).
struct FwdLayer {
    bool linear;
    LinearLayerPlan lp;  // the plan it was built from
    MlpPlan mp;
    // parameters (device)
    const float *in_ln_w = nullptr, *conv_w = nullptr, *wa = nullptr, *wb = nullptr, *nea = nullptr,
                *dt = nullptr, *norm_w = nullptr, *post_ln_w = nullptr;
    DevState* st = nullptr;
    // GPU planes: linear = qkv, z, o, gate, up, down; MLP = gate, up, down
    DevWeights w[6];
    int slot = -1;  // in the chain's layer table (-1: runs as separate launches)
};

// Runs of layers in one launch (forward_chain.hip).
// A run takes under 0.5 ms once its workgroups are all there.  Other work on the
// GPU may hold some of them back: longer than kChainWait (2 ms of the 100 MHz
// clock) and the run gives up and is done again by separate launches, as are
// the rest of the token and the next calls.  Two processes that both run the
// forward hold back each other's workgroups now and then (one run in about 500),
// and a process whose separate launches go in between the other's runs is the
// slower one, so the rest is short; it doubles when the next run gives up too (and
// shortens by a call with each run that ends), so that work which never lets go of
// a CU costs 2 ms once in 65,536 calls.  Two such processes, four tokens: 3.75 ms
// each (1.94 alone; 3.2 if both only ever took separate launches), at most 10;
// with a wait of 0.25 s and a rest of 256, 6.1 and 506.
constexpr uint64_t kChainWait = 200000;
constexpr int kChainRest = 4, kChainRestMax = 65536;
constexpr int kSeconds = 6;  // second state buffers in one allocation (one each costs a cold token 2 ms of 48)
struct Chain {
    std::vector<RtChainLayer> host;  // the layer table
    DevBuf layers;                   // ... its device copy, the first `uploaded` entries
    size_t uploaded = 0;
    std::vector<DevBuf> seconds;     // the states' rec[1], kSeconds each
    int second_left = 0;             // free places of the last one
    DevBuf xch;                      // two sets of exchange words; each launch takes the other one and clears its predecessor's
    int set = 0;                     // the clean set
    int used[2] = {0, 0};            // words of each that are not clean
    PinnedBuf io;                    // ChainIo
    uint64_t wait_ticks = kChainWait;
    int rest = 0;                // calls still to go as separate launches, after a run gave up
    int next_rest = kChainRest;  // ... when the next one does
    long long done = 0, gave_up = 0;  // runs
    bool in_flight = false;
    bool off = false;  // its memory was given back: separate launches until the caches are cleared
};
// Host memory that the launches read and write.
struct ChainIo {
    float h_in[RT_HIDDEN], h_out[RT_HIDDEN];
    int lm[4];        // [ids 1, scores 1, count, argmax]
    uint32_t status;  // 1: the launch gave up
};

struct Workspace {
    DevBuf buf;
    float *h, *h2;  // the hidden state ping-pongs between these (see RtRowsArgs::h_out)
    float *normed, *qkv, *z, *zsilu, *attn, *o, *gate, *up, *down;
    int* lm;        // [ids 1, scores 1, count, argmax]; directly after h2
    bool start_h2;  // a token's embedding goes to h2 (see result_out)
};

struct Forward {
    std::map<ParamKey, DevBuf> params;
    std::map<ParamKey, CachedWeights> planes;           // writable BFP8 planes
    std::map<std::vector<char>, std::unique_ptr<FwdLayer>> layers;
    std::map<std::pair<const float*, const float*>, std::unique_ptr<DevState>> states;  // by the caller's buffers
    Workspace ws{};
    bool ws_ready = false;
    int resident = 0;
    Chain chain;
};

Forward F;

int fwd_param(const void* p, size_t bytes, const void** out) {
    const ParamKey key{p, bytes};
    auto it = F.params.find(key);
    if (it == F.params.end()) {
        DevBuf d;
        int rc;
        if ((rc = d.reserve(bytes))) return rc;
        HIP_OK(hipMemcpy(d.p, p, bytes, hipMemcpyHostToDevice));
        it = F.params.emplace(key, d).first;
    }
    *out = it->second.p;
    return BFP8_OK;
}

template <class T>
int fwd_vec(const T* p, size_t n, const T** out) {
    const void* d;
    int rc = fwd_param(p, n * sizeof(T), &d);
    *out = static_cast<const T*>(d);
    return rc;
}

// GPU-layout planes: the shared read-only cache, else a forward-owned copy.
int fwd_planes(const int8_t* mant, const uint8_t* exps, int M, int K, DevWeights* out) {
    const size_t mb = (size_t)M * K, eb = (size_t)M * bfp8_nblocks(K);
    if (range_readonly_cached(mant, mb) && range_readonly_cached(exps, eb)) return weights_for(mant, exps, M, K, out);
    const ParamKey key{mant, mb};
    auto it = F.planes.find(key);
    if (it == F.planes.end()) {
        int rc;
        if ((rc = g.soa_m.reserve(mb)) || (rc = g.soa_e.reserve(eb))) return rc;
        HIP_OK(hipMemcpyAsync(g.soa_m.p, mant, mb, hipMemcpyHostToDevice, g.stream));
        HIP_OK(hipMemcpyAsync(g.soa_e.p, exps, eb, hipMemcpyHostToDevice, g.stream));
        CachedWeights cw;
        if ((rc = cw.mant.reserve(bfp8_gpu_mant_bytes(M, K))) || (rc = cw.exps.reserve(bfp8_gpu_exps_bytes(M, K))))
            return rc;
        HIP_OK(bfp8_launch_pack(cw.mant.as<uint8_t>(), cw.exps.as<uint8_t>(), g.soa_m.as<int8_t>(),
                                g.soa_e.as<uint8_t>(), M, K, g.stream));
        HIP_OK(hipStreamSynchronize(g.stream));
        it = F.planes.emplace(key, cw).first;
    }
    out->mant = it->second.mant.as<uint8_t>();
    out->exps = it->second.exps.as<uint8_t>();
    return BFP8_OK;
}

int ensure_workspace() {
    if (F.ws_ready) return BFP8_OK;
    Workspace& w = F.ws;
    const int nf[] = {kHidden, kHidden, kHidden, kConv, kHD, kHD, kHD, kHidden, kMlp, kMlp, kHidden};
    size_t total = 256;
    for (int n : nf) total += ((size_t)n * 4 + 255) & ~(size_t)255;
    int rc;
    if ((rc = w.buf.reserve(total))) return rc;
    char* p = w.buf.as<char>();
    auto take = [&](size_t bytes) {
        char* r = p;
        p += (bytes + 255) & ~(size_t)255;
        return r;
    };
    float** fl[] = {&w.h, &w.h2, &w.normed, &w.qkv, &w.z, &w.zsilu, &w.attn, &w.o, &w.gate, &w.up, &w.down};
    for (int i = 0; i < 11; ++i) {
        *fl[i] = reinterpret_cast<float*>(take((size_t)nf[i] * 4));
        if (i == 1) w.lm = reinterpret_cast<int*>(take(16));  // h2 is a multiple of 256 B
    }
    F.ws_ready = true;
    return BFP8_OK;
}

bool linear_shapes_ok(const LinearLayerPlan& p) {
    return p.M_qkv == kConv && p.K_qkv == kHidden && p.M_z == kHD && p.K_z == kHidden && p.M_o == kHidden &&
           p.K_o == kHD && p.M_gate == kMlp && p.K_gate == kHidden && p.M_up == kMlp && p.K_up == kHidden &&
           p.M_down == kHidden && p.K_down == kMlp;
}

bool mlp_shapes_ok(const MlpPlan& p) {
    return p.M_gate == kMlp && p.K_gate == kHidden && p.M_up == kMlp && p.K_up == kHidden && p.M_down == kHidden &&
           p.K_down == kMlp;
}

// A second state buffer, or null (no chain here, no room).
float* second_state() {
    Chain& c = F.chain;
    if (!rt_chain_fits() || c.off) return nullptr;
    if (c.second_left == 0) {
        DevBuf b;
        if (b.reserve(kSeconds * kStateLen * 4, true)) return nullptr;
        c.seconds.push_back(b);
        c.second_left = kSeconds;
    }
    return c.seconds.back().as<float>() + kStateLen * (kSeconds - c.second_left--);
}

// Device state of a layer, keyed by the caller's conv-state buffer.  A new
// one starts from the caller's buffers.
int fwd_state(float* conv_s, float* state, DevState** out) {
    const std::pair<const float*, const float*> key{conv_s, state};
    auto it = F.states.find(key);
    if (it != F.states.end()) {
        *out = it->second.get();
        return BFP8_OK;
    }
    std::unique_ptr<DevState> st(new DevState());
    if (int rc = st->buf.reserve((2 * kTapsLen + kStateLen) * 4)) return rc;
    float* p = st->buf.as<float>();
    st->rec[0] = p;
    st->conv[0] = p + kStateLen;
    st->conv[1] = p + kStateLen + kTapsLen;
    st->rec[1] = second_state();
    st->host_conv = conv_s;
    st->host_rec = state;
    HIP_OK(hipMemcpy(st->conv[0], conv_s, kTapsLen * 4, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(st->rec[0], state, kStateLen * 4, hipMemcpyHostToDevice));
    *out = st.get();
    F.states[key] = std::move(st);
    return BFP8_OK;
}

int state_in(DevState* st) {
    HIP_OK(hipMemcpyAsync(st->conv[st->cur], st->host_conv, (size_t)3 * kConv * 4, hipMemcpyHostToDevice, g.stream));
    HIP_OK(hipMemcpyAsync(st->rec[st->rcur], st->host_rec, (size_t)RT_HEADS * RT_HEAD_DIM * RT_HEAD_DIM * 4,
                          hipMemcpyHostToDevice, g.stream));
    return BFP8_OK;
}

int state_out(DevState* st) {
    HIP_OK(hipMemcpyAsync(st->host_conv, st->conv[st->cur], (size_t)3 * kConv * 4, hipMemcpyDeviceToHost, g.stream));
    HIP_OK(hipMemcpyAsync(st->host_rec, st->rec[st->rcur], (size_t)RT_HEADS * RT_HEAD_DIM * RT_HEAD_DIM * 4,
                          hipMemcpyDeviceToHost, g.stream));
    return BFP8_OK;
}

std::vector<char> key_of(const void* p, size_t n, char tag) {
    std::vector<char> k(n + 1);
    k[0] = tag;
    memcpy(k.data() + 1, p, n);
    return k;
}

// Enters a layer into the chain's table, where it fits (else slot stays -1).
void chain_add(FwdLayer* L) {
    Chain& c = F.chain;
    if (!rt_chain_fits() || c.off || c.host.size() >= 0xffff) return;
    RtChainLayer y{};
    for (int i = 0; i < (L->linear ? 6 : 3); ++i) {
        y.mant[L->linear ? i : 3 + i] = L->w[i].mant;
        y.exps[L->linear ? i : 3 + i] = L->w[i].exps;
    }
    y.post_ln_w = L->post_ln_w;
    if (L->linear) {
        DevState* st = L->st;
        if (!st->rec[1]) return;  // (no room: separate launches)
        y.in_ln_w = L->in_ln_w;
        y.conv_w = L->conv_w;
        y.wa = L->wa;
        y.wb = L->wb;
        y.nea = L->nea;
        y.dt = L->dt;
        y.norm_w = L->norm_w;
        for (int i = 0; i < 2; ++i) {
            y.conv[i] = st->conv[i];
            y.rec[i] = st->rec[i];
        }
        y.linear = 1;
    }
    constexpr size_t kSet = (size_t)RT_CHAIN_SET_WORDS * 8;
    if (!c.xch.p) {
        if (c.xch.reserve(2 * kSet, true) || hipMemsetAsync(c.xch.p, 0xff, 2 * kSet, g.stream) != hipSuccess) {
            c.xch.release();
            return;
        }
        c.used[0] = c.used[1] = 0;
    }
    if (c.io.reserve(sizeof(ChainIo))) return;
    c.host.push_back(y);
    L->slot = (int)c.host.size() - 1;
}

// The table's new entries to the device (no launch of this library is in
// flight: its forward calls wait for theirs).  Where there is no room for a
// larger table the old one stays, with the entries that it has.
int chain_upload() {
    Chain& c = F.chain;
    const size_t n = c.host.size(), bytes = n * sizeof(RtChainLayer);
    if (c.uploaded == n) return BFP8_OK;
    if (bytes > c.layers.n) {
        DevBuf larger;
        if (int rc = larger.reserve(std::max<size_t>(2 * bytes, 64 * sizeof(RtChainLayer)), true)) return rc;
        c.layers.release();
        c.layers = larger;
        c.uploaded = 0;
    }
    HIP_OK(hipMemcpy(c.layers.as<RtChainLayer>() + c.uploaded, c.host.data() + c.uploaded,
                     (n - c.uploaded) * sizeof(RtChainLayer), hipMemcpyHostToDevice));
    c.uploaded = n;
    return BFP8_OK;
}

int fwd_linear_layer(const LinearLayerPlan* p, FwdLayer** out) {
    if (!linear_shapes_ok(*p)) {
        set_error("linear-layer plan shapes differ from the model's (qkv %dx%d, z %dx%d, o %dx%d, gate %dx%d, "
                  "up %dx%d, down %dx%d)", p->M_qkv, p->K_qkv, p->M_z, p->K_z, p->M_o, p->K_o, p->M_gate,
                  p->K_gate, p->M_up, p->K_up, p->M_down, p->K_down);
        return BFP8_EINVAL;
    }
    const std::vector<char> key = key_of(p, sizeof *p, 'L');
    auto it = F.layers.find(key);
    if (it != F.layers.end()) {
        *out = it->second.get();
        return BFP8_OK;
    }
    std::unique_ptr<FwdLayer> L(new FwdLayer());
    L->linear = true;
    L->lp = *p;
    int rc;
    const int8_t* m[6] = {p->mant_qkv, p->mant_z, p->mant_o, p->mant_gate, p->mant_up, p->mant_down};
    const uint8_t* e[6] = {p->exp_qkv, p->exp_z, p->exp_o, p->exp_gate, p->exp_up, p->exp_down};
    const int Ms[6] = {p->M_qkv, p->M_z, p->M_o, p->M_gate, p->M_up, p->M_down};
    const int Ks[6] = {p->K_qkv, p->K_z, p->K_o, p->K_gate, p->K_up, p->K_down};
    for (int i = 0; i < 6; ++i)
        if ((rc = fwd_planes(m[i], e[i], Ms[i], Ks[i], &L->w[i]))) return rc;
    if ((rc = fwd_vec(p->in_ln_w, kHidden, &L->in_ln_w)) || (rc = fwd_vec(p->conv_w, (size_t)kConv * 4, &L->conv_w)) ||
        (rc = fwd_vec(p->wa, (size_t)RT_HEADS * kHidden, &L->wa)) ||
        (rc = fwd_vec(p->wb, (size_t)RT_HEADS * kHidden, &L->wb)) || (rc = fwd_vec(p->nea, RT_HEADS, &L->nea)) ||
        (rc = fwd_vec(p->dt, RT_HEADS, &L->dt)) || (rc = fwd_vec(p->norm_w, RT_HEAD_DIM, &L->norm_w)) ||
        (rc = fwd_vec(p->post_ln_w, kHidden, &L->post_ln_w)) || (rc = fwd_state(p->conv_s, p->state, &L->st)))
        return rc;
    chain_add(L.get());
    *out = L.get();
    F.layers.emplace(key, std::move(L));
    return BFP8_OK;
}

int fwd_mlp_layer(const MlpPlan* p, FwdLayer** out) {
    if (!mlp_shapes_ok(*p)) {
        set_error("MLP plan shapes differ from the model's (gate %dx%d, up %dx%d, down %dx%d)", p->M_gate, p->K_gate,
                  p->M_up, p->K_up, p->M_down, p->K_down);
        return BFP8_EINVAL;
    }
    const std::vector<char> key = key_of(p, sizeof *p, 'M');
    auto it = F.layers.find(key);
    if (it != F.layers.end()) {
        *out = it->second.get();
        return BFP8_OK;
    }
    std::unique_ptr<FwdLayer> L(new FwdLayer());
    L->linear = false;
    L->mp = *p;
    int rc;
    const int8_t* m[3] = {p->mant_gate, p->mant_up, p->mant_down};
    const uint8_t* e[3] = {p->exp_gate, p->exp_up, p->exp_down};
    const int Ms[3] = {p->M_gate, p->M_up, p->M_down};
    const int Ks[3] = {p->K_gate, p->K_up, p->K_down};
    for (int i = 0; i < 3; ++i)
        if ((rc = fwd_planes(m[i], e[i], Ms[i], Ks[i], &L->w[i]))) return rc;
    if ((rc = fwd_vec(p->post_ln_w, kHidden, &L->post_ln_w))) return rc;
    chain_add(L.get());
    *out = L.get();
    F.layers.emplace(key, std::move(L));
    return BFP8_OK;
}

// Profiled step: while profiling, each step is synchronised and its wall time
// booked to its slot.
struct Step {
    int slot;
    double t0;
    explicit Step(int s) : slot(s), t0(g_prof_on ? now_ms() : 0.0) {}
    int done() {
        if (!g_prof_on) return BFP8_OK;
        HIP_OK(hipStreamSynchronize(g.stream));
        g_prof_ms[slot] += now_ms() - t0;
        return BFP8_OK;
    }
};

RtRowsGemv rows_gemv(const DevWeights& w, float* y, int M) {
    RtRowsGemv r{};
    r.mant = w.mant;
    r.exps = w.exps;
    r.y = y;
    r.M = M;
    r.pair_rows = M & ~1;
    return r;
}

int rows_step(const RtRowsArgs& a) {
    Step s(QP_GEMV);
    RT_LAUNCH(rt_launch_rows(a, g.stream));
    return s.done();
}

// The other buffer of the hidden state's ping-pong.
float* other_h(const float* h) { return h == F.ws.h ? F.ws.h2 : F.ws.h; }

// rmsnorm of *h (after adding res, if any) into y, in place (the final norm).
int norm_step(float* h, const float* res, const float* w, float* y) {
    Step s(QP_RMSNORM);
    RtNormArgs a{};
    a.h = h;
    a.res = res;
    a.w = w;
    a.y = y;
    a.n = kHidden;
    a.eps = 1e-6f;
    RT_LAUNCH(rt_launch_rmsnorm(a, g.stream));
    return s.done();
}

// The MLP half shared by both layer kinds (planes gud = gate, up, down):
// rmsnorm(h + res) -> gate, up in one launch; swiglu -> down in another.
// *h moves to the other buffer when a residual is added.  Leaves the down
// projection in ws.down, not yet added.
int mlp_steps(const FwdLayer& L, const DevWeights* gud, float** h, const float* res) {
    Workspace& w = F.ws;
    RtRowsArgs a{};
    a.g[0] = rows_gemv(gud[0], w.gate, kMlp);
    a.g[1] = rows_gemv(gud[1], w.up, kMlp);
    a.ngemv = 2;
    a.split = kMlp / 16;
    a.K = kHidden;
    a.mode = RT_ROWS_NORM;
    a.h = *h;
    a.res = res;
    a.w = L.post_ln_w;
    a.eps = 1e-6f;
    a.h_out = res ? other_h(*h) : nullptr;
    int rc;
    if ((rc = rows_step(a))) return rc;
    if (res) *h = a.h_out;
    RtRowsArgs d{};
    d.g[0] = rows_gemv(gud[2], w.down, kHidden);
    d.ngemv = 1;
    d.split = kHidden / 16;
    d.K = kMlp;
    d.mode = RT_ROWS_SWIGLU;
    d.gate = w.gate;
    d.up = w.up;
    return rows_step(d);
}

// forward_linear_layer on the device: *h the hidden state, res a pending
// residual to add first (null for none).  Leaves the MLP's down projection in
// ws.down.
int linear_steps(const FwdLayer& L, float** h, const float* res) {
    Workspace& w = F.ws;
    RtRowsArgs a{};
    a.g[0] = rows_gemv(L.w[0], w.qkv, kConv);
    a.g[1] = rows_gemv(L.w[1], w.z, kHD);
    a.ngemv = 2;
    a.split = kConv / 16;
    a.K = kHidden;
    a.mode = RT_ROWS_NORM;
    a.h = *h;
    a.res = res;
    a.w = L.in_ln_w;
    a.eps = 1e-6f;
    a.y_norm = w.normed;
    a.h_out = res ? other_h(*h) : nullptr;
    int rc;
    if ((rc = rows_step(a))) return rc;
    if (res) *h = a.h_out;
    {
        Step s(QP_GDN);
        DevState* st = L.st;
        RtLinearAttnArgs la{};
        la.qkv = w.qkv;
        la.normed = w.normed;
        la.conv_in = st->conv[st->cur];
        la.conv_out = st->conv[st->cur ^ 1];
        la.conv_w = L.conv_w;
        la.wa = L.wa;
        la.wb = L.wb;
        la.nea = L.nea;
        la.dt = L.dt;
        la.state = st->rec[st->rcur];
        la.attn = w.attn;
        la.z = w.z;
        la.zsilu = w.zsilu;
        RT_LAUNCH(rt_launch_linear_attn(la, g.stream));
        st->cur ^= 1;
        if ((rc = s.done())) return rc;
    }
    // the gated RMSNorm runs in the o GEMV's prologue
    RtRowsArgs o{};
    o.g[0] = rows_gemv(L.w[2], w.o, kHidden);
    o.ngemv = 1;
    o.split = kHidden / 16;
    o.K = kHD;
    o.mode = RT_ROWS_GATED;
    o.attn = w.attn;
    o.zsilu = w.zsilu;
    o.w = L.norm_w;
    o.eps = 1e-6f;
    if ((rc = rows_step(o))) return rc;
    return mlp_steps(L, &L.w[3], h, w.o);
}

int layer_steps(const FwdLayer& L, float** h, const float* res) {
    return L.linear ? linear_steps(L, h, res) : mlp_steps(L, &L.w[0], h, res);
}

int add_pending(float* h, const float* res) {
    if (!res) return BFP8_OK;
    Step s(QP_RESID);
    RT_LAUNCH(rt_launch_add_residual(h, res, kHidden, g.stream));
    return s.done();
}

int h_in(float* dev, const float* h) {
    HIP_OK(hipMemcpyAsync(dev, h, (size_t)kHidden * 4, hipMemcpyHostToDevice, g.stream));
    return BFP8_OK;
}

int h_out(float* h, const float* dev) {
    HIP_OK(hipMemcpyAsync(h, dev, (size_t)kHidden * 4, hipMemcpyDeviceToHost, g.stream));
    HIP_OK(hipStreamSynchronize(g.stream));
    return BFP8_OK;
}

// A token's hidden state hd and lm_head result back to the host.  When hd is
// h2 the two are adjacent and come back in one copy through pinned memory;
// otherwise in two, and the next token starts in the other buffer: the layer
// sequence fixes how often the state moves between h and h2, so it then ends
// in h2.
int result_out(float* h, const float* hd, int* out) {
    Workspace& w = F.ws;
    const size_t hb = (size_t)kHidden * 4;
    if (hd == w.h2) {
        if (int rc = g.rt_pin.reserve(hb + 16)) return rc;
        HIP_OK(hipMemcpyAsync(g.rt_pin.p, w.h2, hb + 16, hipMemcpyDeviceToHost, g.stream));
        HIP_OK(hipStreamSynchronize(g.stream));
        memcpy(h, g.rt_pin.p, hb);
        memcpy(out, static_cast<const char*>(g.rt_pin.p) + hb, 16);
        return BFP8_OK;
    }
    w.start_h2 = !w.start_h2;
    HIP_OK(hipMemcpyAsync(out, w.lm, 16, hipMemcpyDeviceToHost, g.stream));
    return h_out(h, hd);
}

// Copies back the device states that resident calls left newer than the
// caller's buffers.
int sync_states_out() {
    for (auto& kv : F.states) {
        DevState* st = kv.second.get();
        if (!st->dirty) continue;
        if (int rc = state_out(st)) return rc;
        st->dirty = false;
    }
    HIP_OK(hipStreamSynchronize(g.stream));
    return BFP8_OK;
}

// A layer's states before a forward call: refreshed from the caller's
// buffers unless resident.
int states_in(const std::vector<FwdLayer*>& layers) {
    for (FwdLayer* L : layers) {
        if (!L->linear) continue;
        if (F.resident) {
            L->st->resident_used = true;
            L->st->dirty = true;
        } else if (int rc = state_in(L->st)) {
            return rc;
        }
    }
    return BFP8_OK;
}

int states_out(const std::vector<FwdLayer*>& layers) {
    if (F.resident) return BFP8_OK;
    for (FwdLayer* L : layers)
        if (L->linear)
            if (int rc = state_out(L->st)) return rc;
    return BFP8_OK;
}

// ---- runs of layers in one launch -------------------------------------------------------
ChainIo& chain_io() { return *static_cast<ChainIo*>(F.chain.io.p); }

// Every layer of [l, e) in the device's table (a layer seen while the device was
// full is not).
bool chain_has(const std::vector<FwdLayer*>& layers, int l, int e) {
    int top = -1;
    for (int i = l; i < e; ++i) {
        if (layers[i]->slot < 0) return false;
        top = std::max(top, layers[i]->slot);
    }
    return (size_t)top < F.chain.uploaded || chain_upload() == BFP8_OK;
}

// Every layer in the table, and no per-step profile asked for.
bool chain_ok(const std::vector<FwdLayer*>& layers) {
    if (F.chain.rest > 0) {
        --F.chain.rest;
        return false;
    }
    return !g_prof_on && chain_has(layers, 0, (int)layers.size());
}

// Whether a run can hand h on as it is: no pair of its words is all ones, the
// pattern of a pair that is not there yet (NaNs whose bits would be lost).
bool chain_takes(const float* h) {
    uint64_t found = 0;
    for (int i = 0; i < kHidden; i += 2) {
        uint64_t v;
        memcpy(&v, h + i, 8);
        found |= v == ~0ull;
    }
    return !found;
}

// Layers [l, e), no two with one state, in one launch, from row `row` of the
// table (table != null) or from io.h_in, the hidden state to io.h_out; with fnorm
// also its final norm to ws.normed.  chain_done says whether it ran to its end.
int chain_launch(const std::vector<FwdLayer*>& layers, int l, int e, const uint16_t* table, int ntiles, int row,
                 const float* fnorm) {
    Chain& c = F.chain;
    ChainIo& io = chain_io();
    RtChainArgs a{};
    a.layers = c.layers.as<RtChainLayer>();
    a.n = e - l;
    for (int i = l; i < e; ++i) {
        const FwdLayer* L = layers[i];
        a.idx[i - l] = (uint16_t)L->slot;
        if (L->linear) {
            a.cur |= (uint32_t)L->st->cur << (i - l);
            a.rcur |= (uint32_t)L->st->rcur << (i - l);
        }
    }
    a.table = table;
    a.ntiles = ntiles;
    a.row = row;
    a.h_in = io.h_in;
    a.h_out = io.h_out;
    a.final_w = fnorm;
    a.y_norm = fnorm ? F.ws.normed : nullptr;
    a.eps = 1e-6f;
    uint64_t* sets = c.xch.as<uint64_t>();
    a.xch = sets + (size_t)c.set * RT_CHAIN_SET_WORDS;
    a.xch_clear = sets + (size_t)(c.set ^ 1) * RT_CHAIN_SET_WORDS;
    a.clear_words = c.used[c.set ^ 1];
    a.wait_ticks = c.wait_ticks;
    a.status = &io.status;
    io.status = 0;
    RT_LAUNCH(rt_launch_chain(a, g.stream));
    c.in_flight = true;
    c.used[c.set] = a.n * RT_CHAIN_LAYER_WORDS + RT_HIDDEN / 2;
    c.used[c.set ^ 1] = 0;
    c.set ^= 1;
    return BFP8_OK;
}

// After the stream is synchronized: the run's states become the current ones
// (*ok), or it gave up or was not to be made (!*ok on entry), and nothing of it
// counts (!*ok).
int chain_done(const std::vector<FwdLayer*>& layers, int l, int e, bool* ok) {
    Chain& c = F.chain;
    c.in_flight = false;
    const bool gave_up = __atomic_load_n(&chain_io().status, __ATOMIC_ACQUIRE) != 0;
    *ok = *ok && !gave_up;
    if (*ok) {
        ++c.done;
        c.next_rest = std::max(c.next_rest - 1, kChainRest);
        for (int i = l; i < e; ++i) {
            if (!layers[i]->linear) continue;
            layers[i]->st->cur ^= 1;
            layers[i]->st->rcur ^= 1;
        }
        return BFP8_OK;
    }
    if (!gave_up) return BFP8_OK;
    ++c.gave_up;
    HIP_OK(hipMemsetAsync(c.xch.p, 0xff, 2 * (size_t)RT_CHAIN_SET_WORDS * 8, g.stream));
    c.used[0] = c.used[1] = 0;
    c.rest = c.next_rest;
    c.next_rest = std::min(2 * c.next_rest, kChainRestMax);
    return BFP8_OK;
}

int layer_call(const FwdLayer& L, float* h, int slot) {
    const double t0 = g_prof_on ? now_ms() : 0.0;
    int rc;
    const std::vector<FwdLayer*> one{const_cast<FwdLayer*>(&L)};
    if (chain_ok(one)) {
        if ((rc = states_in(one))) return rc;
        memcpy(chain_io().h_in, h, (size_t)kHidden * 4);
        if ((rc = chain_launch(one, 0, 1, nullptr, 0, 0, nullptr))) return rc;
        bool ok = chain_takes(h);  // (while the run is under way)
        HIP_OK(hipStreamSynchronize(g.stream));
        if ((rc = chain_done(one, 0, 1, &ok))) return rc;
        if (ok) {
            if ((rc = states_out(one))) return rc;
            if (L.linear && !F.resident) HIP_OK(hipStreamSynchronize(g.stream));
            memcpy(h, chain_io().h_out, (size_t)kHidden * 4);
            return BFP8_OK;
        }
    }
    float* hd = F.ws.h;
    if ((rc = h_in(hd, h)) || (rc = states_in(one))) return rc;
    if ((rc = layer_steps(L, &hd, nullptr)) || (rc = add_pending(hd, F.ws.down))) return rc;
    if ((rc = states_out(one))) return rc;
    if ((rc = h_out(h, hd))) return rc;
    if (g_prof_on) g_prof_ms[slot] += now_ms() - t0;
    return BFP8_OK;
}

// Layers [l, e) as separate launches from the hidden state in F.ws.h, which
// ends, the last residual added, at *hd.
int separate_steps(const std::vector<FwdLayer*>& layers, int l, int e, float** hd) {
    const float* pending = nullptr;
    int rc;
    *hd = F.ws.h;
    for (int i = l; i < e; ++i, pending = F.ws.down)
        if ((rc = layer_steps(*layers[i], hd, pending))) return rc;
    return add_pending(*hd, pending);
}

// Whether a layer of [l, e) advances the state that layer e does.  A run takes a
// state's current buffer as its input and writes the other one, so it advances
// each state once; plans may name the same buffers for several layers.
bool state_in_run(const std::vector<FwdLayer*>& layers, int l, int e) {
    for (int i = l; i < e; ++i)
        if (layers[e]->st && layers[i]->st == layers[e]->st) return true;
    return false;
}

// forward_token_c's layers and head, the layers in runs of one launch: up to
// the next full-attention layer whose callback edits the hidden state on the
// host, the next layer whose state the run advances already, or the end.  A run
// that gives up is done again by separate launches.
int token_chain(std::unique_lock<std::mutex>& lk, const std::vector<FwdLayer*>& layers, const int* layer_is_full,
                FullAttnCallback cb, void* py_context, const uint16_t* table, int tiled, int row, const float* fnorm, float* h,
                int* id) {
    Workspace& w = F.ws;
    const size_t hb = (size_t)kHidden * 4;
    const int ntiles = tiled ? bfp8_ntiles(kVocab) : 0;
    int rc;
    if ((rc = states_in(layers))) return rc;
    bool embed = true;  // the hidden state is still the table's row, else it is in h
    for (int l = 0, e; l < kLayers; l = e) {
        if (layer_is_full[l] && cb) {
            if (embed) {
                RT_LAUNCH(rt_launch_embed(w.h, table, ntiles, row, kHidden, g.stream));
                if ((rc = h_out(h, w.h))) return rc;
                embed = false;
            }
            lk.unlock();
            cb(l, h, py_context);
            lk.lock();
        }
        for (e = l + 1; e < kLayers && !(layer_is_full[e] && cb) && !state_in_run(layers, l, e); ++e) {}
        const bool last = e == kLayers;
        ChainIo& io = chain_io();
        auto head = [&] {
            return bf16_lm_head_dev(io.lm, reinterpret_cast<float*>(io.lm + 1), io.lm + 2, io.lm + 3, nullptr, w.normed, table,
                                    tiled, kVocab, kHidden, 1, 0, g.stream);
        };
        // (an earlier run of the token may have given up, a callback's calls may have changed the table)
        bool ok = F.chain.rest == 0 && chain_has(layers, l, e);
        if (ok) {
            if (!embed) memcpy(io.h_in, h, hb);
            if ((rc = chain_launch(layers, l, e, embed ? table : nullptr, ntiles, row, last ? fnorm : nullptr))) return rc;
            if (last && (rc = head())) return rc;
            ok = embed || chain_takes(h);  // (while the run is under way)
            HIP_OK(hipStreamSynchronize(g.stream));
            if ((rc = chain_done(layers, l, e, &ok))) return rc;
        }
        if (ok) {
            memcpy(h, io.h_out, hb);
        } else {
            float* hd;
            if (embed)
                RT_LAUNCH(rt_launch_embed(w.h, table, ntiles, row, kHidden, g.stream));
            else if ((rc = h_in(w.h, h)))
                return rc;
            if ((rc = separate_steps(layers, l, e, &hd))) return rc;
            if (last && ((rc = norm_step(hd, nullptr, fnorm, w.normed)) || (rc = head()))) return rc;
            if ((rc = h_out(h, hd))) return rc;
        }
        embed = false;
    }
    *id = chain_io().lm[3];
    if ((rc = states_out(layers))) return rc;
    if (!F.resident) HIP_OK(hipStreamSynchronize(g.stream));
    return BFP8_OK;
}

void drop_chain() {
    F.chain.host.clear();
    F.chain.uploaded = 0;
    F.chain.layers.release();
    F.chain.xch.release();
    for (DevBuf& b : F.chain.seconds) b.release();
    F.chain.seconds.clear();
    F.chain.second_left = 0;
}

void drop_forward() {
    F.layers.clear();
    for (auto& kv : F.params) kv.second.release();
    F.params.clear();
    for (auto& kv : F.planes) {
        kv.second.mant.release();
        kv.second.exps.release();
    }
    F.planes.clear();
    for (auto& kv : F.states) {
        kv.second->buf.release();
    }
    F.states.clear();
    drop_chain();
    F.chain.off = false;
}

}  // namespace

// The chain's memory: the states' second buffers (1 MiB a layer) and the exchange
// words (3.9 MB), without which the layers run as separate launches.
bool release_spare(size_t bytes) {
    Chain& c = F.chain;
    size_t held = c.xch.n + c.layers.n;
    for (const DevBuf& b : c.seconds) held += b.n;
    if (!held || c.in_flight) return false;
    size_t room = 0, total = 0;
    if (g_dev_limit)
        room = g_dev_limit > g_dev_bytes ? g_dev_limit - g_dev_bytes : 0;
    else if (hipMemGetInfo(&room, &total) != hipSuccess)
        return false;
    if (room + held < bytes) return false;
    for (auto& kv : F.states) {  // a state in its second buffer moves to the first
        DevState* st = kv.second.get();
        if (st->rcur && hipMemcpyAsync(st->rec[0], st->rec[1], kStateLen * 4, hipMemcpyDeviceToDevice, g.stream) != hipSuccess)
            return false;
    }
    if (hipStreamSynchronize(g.stream) != hipSuccess) return false;
    for (auto& kv : F.states) {
        DevState* st = kv.second.get();
        st->rcur = 0;
        st->rec[1] = nullptr;
    }
    for (auto& kv : F.layers) kv.second->slot = -1;
    drop_chain();
    c.off = true;
    return true;
}

// Called by bfp8_cache_clear (lock held).
void forward_cache_clear() { drop_forward(); }

int forward_preload_param(const void* p, size_t bytes) {
    const void* d;
    return fwd_param(p, bytes, &d);
}

}  // namespace qhost

using namespace qhost;

extern "C" {

// ---- reference runtime symbols, host pointers ---------------------------------------------
void rmsnorm(float* y, const float* x, const float* w, int n, float eps) {
    if (n <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("rmsnorm", ensure_init_locked());
    HostCall c;
    const size_t oy = c.add(y, (size_t)n * 4, true), ox = c.add(x, (size_t)n * 4, false),
                 ow = c.add(w, (size_t)n * 4, false);
    RT_CHECK("rmsnorm", c.upload());
    RtNormArgs a{};
    a.h = c.dev<float>(ox);
    a.w = c.dev<float>(ow);
    a.y = c.dev<float>(oy);
    a.n = n;
    a.eps = eps;
    if (rt_launch_rmsnorm(a, g.stream) != hipSuccess) {
        set_error("rmsnorm launch failed");
        fatal("rmsnorm");
    }
    RT_CHECK("rmsnorm", c.download());
}

void swiglu(float* y, const float* gate, const float* up, int n) {
    if (n <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("swiglu", ensure_init_locked());
    HostCall c;
    const size_t oy = c.add(y, (size_t)n * 4, true), og = c.add(gate, (size_t)n * 4, false),
                 ou = c.add(up, (size_t)n * 4, false);
    RT_CHECK("swiglu", c.upload());
    RtSwigluArgs a{};
    a.y = c.dev<float>(oy);
    a.gate = c.dev<float>(og);
    a.up = c.dev<float>(ou);
    a.n = n;
    if (rt_launch_swiglu(a, g.stream) != hipSuccess) {
        set_error("swiglu launch failed");
        fatal("swiglu");
    }
    RT_CHECK("swiglu", c.download());
}

void add_residual(float* x, const float* res, int n) {
    if (n <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("add_residual", ensure_init_locked());
    HostCall c;
    const size_t ox = c.add(x, (size_t)n * 4, true), orr = c.add(res, (size_t)n * 4, false);
    RT_CHECK("add_residual", c.upload());
    if (rt_launch_add_residual(c.dev<float>(ox), c.dev<float>(orr), n, g.stream) != hipSuccess) {
        set_error("add_residual launch failed");
        fatal("add_residual");
    }
    RT_CHECK("add_residual", c.download());
}

void causal_conv1d_update_silu(float* y, const float* x, float* conv_state, const float* weight, int channels) {
    if (channels <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("causal_conv1d_update_silu", ensure_init_locked());
    HostCall c;
    const size_t C = (size_t)channels;
    const size_t oy = c.add(y, C * 4, true), ox = c.add(x, C * 4, false), os = c.add(conv_state, 3 * C * 4, true),
                 ow = c.add(weight, 4 * C * 4, false);
    RT_CHECK("causal_conv1d_update_silu", c.upload());
    RtConvArgs a{};
    a.y = c.dev<float>(oy);
    a.x = c.dev<float>(ox);
    a.state = c.dev<float>(os);
    a.w = c.dev<float>(ow);
    a.channels = channels;
    if (rt_launch_conv1d(a, g.stream) != hipSuccess) {
        set_error("conv1d launch failed");
        fatal("causal_conv1d_update_silu");
    }
    RT_CHECK("causal_conv1d_update_silu", c.download());
}

void qk_l2norm(float* q, float* k, int num_heads, int head_dim) {
    if (num_heads <= 0 || head_dim <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("qk_l2norm", ensure_init_locked());
    HostCall c;
    const size_t n = (size_t)num_heads * head_dim * 4;
    const size_t oq = c.add(q, n, true), ok = c.add(k, n, true);
    RT_CHECK("qk_l2norm", c.upload());
    if (rt_launch_qk_l2norm(c.dev<float>(oq), c.dev<float>(ok), num_heads, head_dim, g.stream) != hipSuccess) {
        set_error("qk_l2norm launch failed");
        fatal("qk_l2norm");
    }
    RT_CHECK("qk_l2norm", c.download());
}

void gdn_gates(float* alpha, float* beta, const float* x, const float* wa, const float* wb, const float* neg_exp_alog,
               const float* dt, int H, int K) {
    if (H <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("gdn_gates", ensure_init_locked());
    HostCall c;
    const size_t kk = (size_t)(K > 0 ? K : 0);
    const size_t oa = c.add(alpha, (size_t)H * 4, true), ob = c.add(beta, (size_t)H * 4, true),
                 ox = c.add(x, kk * 4, false), owa = c.add(wa, (size_t)H * kk * 4, false),
                 owb = c.add(wb, (size_t)H * kk * 4, false), on = c.add(neg_exp_alog, (size_t)H * 4, false),
                 od = c.add(dt, (size_t)H * 4, false);
    RT_CHECK("gdn_gates", c.upload());
    RtGatesArgs a{};
    a.alpha = c.dev<float>(oa);
    a.beta = c.dev<float>(ob);
    a.x = c.dev<float>(ox);
    a.wa = c.dev<float>(owa);
    a.wb = c.dev<float>(owb);
    a.nea = c.dev<float>(on);
    a.dt = c.dev<float>(od);
    a.H = H;
    a.K = (int)kk;
    if (rt_launch_gates(a, g.stream) != hipSuccess) {
        set_error("gdn_gates launch failed");
        fatal("gdn_gates");
    }
    RT_CHECK("gdn_gates", c.download());
}

void gdn_recurrent_step(float* attn_out, float* state, const float* q, const float* k, const float* v,
                        const float* alpha, const float* beta, int num_heads, int head_dim) {
    if (num_heads <= 0 || head_dim <= 0) return;
    if ((head_dim & 3) || head_dim > RT_MAX_HEAD_DIM) {
        set_error("gdn_recurrent_step: head_dim %d is not a multiple of 4 up to %d", head_dim, RT_MAX_HEAD_DIM);
        fatal("gdn_recurrent_step");
    }
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("gdn_recurrent_step", ensure_init_locked());
    HostCall c;
    const size_t H = (size_t)num_heads, D = (size_t)head_dim;
    const size_t oo = c.add(attn_out, H * D * 4, true), os = c.add(state, H * D * D * 4, true),
                 oq = c.add(q, H * D * 4, false), ok = c.add(k, H * D * 4, false), ov = c.add(v, H * D * 4, false),
                 oa = c.add(alpha, H * 4, false), ob = c.add(beta, H * 4, false);
    RT_CHECK("gdn_recurrent_step", c.upload());
    RtGdnArgs a{};
    a.out = c.dev<float>(oo);
    a.state = c.dev<float>(os);
    a.q = c.dev<float>(oq);
    a.k = c.dev<float>(ok);
    a.v = c.dev<float>(ov);
    a.alpha = c.dev<float>(oa);
    a.beta = c.dev<float>(ob);
    a.H = num_heads;
    a.D = head_dim;
    if (rt_launch_gdn_step(a, g.stream) != hipSuccess) {
        set_error("gdn_recurrent_step launch failed");
        fatal("gdn_recurrent_step");
    }
    RT_CHECK("gdn_recurrent_step", c.download());
}

void rmsnorm_gated(float* y, const float* x, const float* z, const float* norm_w, int num_heads, int head_dim,
                   float eps) {
    if (num_heads <= 0 || head_dim <= 0) return;
    std::lock_guard<std::mutex> lk(g.mu);
    RT_CHECK("rmsnorm_gated", ensure_init_locked());
    HostCall c;
    const size_t n = (size_t)num_heads * head_dim * 4;
    const size_t oy = c.add(y, n, true), ox = c.add(x, n, false), oz = c.add(z, n, false),
                 ow = c.add(norm_w, (size_t)head_dim * 4, false);
    RT_CHECK("rmsnorm_gated", c.upload());
    RtGatedArgs a{};
    a.y = c.dev<float>(oy);
    a.x = c.dev<float>(ox);
    a.z = c.dev<float>(oz);
    a.w = c.dev<float>(ow);
    a.H = num_heads;
    a.D = head_dim;
    a.eps = eps;
    if (rt_launch_gated(a, g.stream) != hipSuccess) {
        set_error("rmsnorm_gated launch failed");
        fatal("rmsnorm_gated");
    }
    RT_CHECK("rmsnorm_gated", c.download());
}

// ---- the forward loop ------------------------------------------------------------------------
void forward_linear_layer(const LinearLayerPlan* p, float* h) {
    if (!p || !h) return;
    std::lock_guard<std::mutex> lk(g.mu);
    FwdLayer* L = nullptr;
    RT_CHECK("forward_linear_layer", ensure_init_locked());
    RT_CHECK("forward_linear_layer", ensure_workspace());
    RT_CHECK("forward_linear_layer", fwd_linear_layer(p, &L));
    RT_CHECK("forward_linear_layer", layer_call(*L, h, QP_LINEAR));
}

void forward_mlp(const MlpPlan* p, float* h) {
    if (!p || !h) return;
    std::lock_guard<std::mutex> lk(g.mu);
    FwdLayer* L = nullptr;
    RT_CHECK("forward_mlp", ensure_init_locked());
    RT_CHECK("forward_mlp", ensure_workspace());
    RT_CHECK("forward_mlp", fwd_mlp_layer(p, &L));
    RT_CHECK("forward_mlp", layer_call(*L, h, QP_MLP));
}

int forward_token_c(int token_id, float* h, const LinearLayerPlan* linear_plans, const MlpPlan* mlp_plans,
                    const int* layer_is_full, const float* final_norm_w, const uint16_t* embed_table,
                    FullAttnCallback full_attn_cb, void* py_context) {
    if (!h || !linear_plans || !mlp_plans || !layer_is_full || !final_norm_w || !embed_table) {
        set_error("forward_token_c: null argument");
        fatal("forward_token_c");
    }
    std::unique_lock<std::mutex> lk(g.mu);
    const double t_total = g_prof_on ? now_ms() : 0.0;
    RT_CHECK("forward_token_c", ensure_init_locked());
    RT_CHECK("forward_token_c", ensure_workspace());
    // layers, the table and the final norm (built on first use)
    std::vector<FwdLayer*> layers(kLayers);
    int li = 0;
    for (int l = 0; l < kLayers; ++l) {
        if (layer_is_full[l])
            RT_CHECK("forward_token_c", fwd_mlp_layer(&mlp_plans[l], &layers[l]));
        else
            RT_CHECK("forward_token_c", fwd_linear_layer(&linear_plans[li++], &layers[l]));
    }
    const float* fnorm = nullptr;
    const uint16_t* table = nullptr;
    const size_t tbytes = (size_t)kVocab * kHidden * 2;
    RT_CHECK("forward_token_c", fwd_vec(final_norm_w, kHidden, &fnorm));
    int tiled = 0;  // the cached table's layout
    if (bf16_table_lookup(embed_table, kVocab, kHidden, &table, &tiled)) {
        // cached on an earlier token: no /proc/self/maps scan
    } else if (range_readonly_cached(embed_table, tbytes)) {
        RT_CHECK("forward_token_c", bf16_table_for(embed_table, kVocab, kHidden, &table, &tiled));
    } else {
        RT_CHECK("forward_token_c", fwd_vec(embed_table, (size_t)kVocab * kHidden, &table));
    }
    // the lm_head's lists, before a run of layers is in flight (nothing is given back then)
    RT_CHECK("forward_token_c", scratch_for(g.stream).partials.reserve((size_t)bfp8_ntiles(kVocab) * 8));
    int row = token_id % kVocab;
    if (row < 0) row += kVocab;
    if (chain_ok(layers)) {
        int id = 0;
        RT_CHECK("forward_token_c", token_chain(lk, layers, layer_is_full, full_attn_cb, py_context, table, tiled, row, fnorm,
                                                h, &id));
        return id;
    }
    Workspace& w = F.ws;
    float* hd = w.start_h2 ? w.h2 : w.h;  // the hidden state on the device
    RT_CHECK("forward_token_c", states_in(layers));
    {
        Step s(QP_EMBED);
        if (rt_launch_embed(hd, table, tiled ? bfp8_ntiles(kVocab) : 0, row, kHidden, g.stream) != hipSuccess) {
            set_error("embedding launch failed");
            fatal("forward_token_c");
        }
        RT_CHECK("forward_token_c", s.done());
    }
    const float* pending = nullptr;  // down projection not yet added to h
    for (int l = 0; l < kLayers; ++l) {
        FwdLayer& L = *layers[l];
        const double t_layer = g_prof_on ? now_ms() : 0.0;
        if (layer_is_full[l]) {
            if (full_attn_cb) {
                RT_CHECK("forward_token_c", add_pending(hd, pending));
                pending = nullptr;
                RT_CHECK("forward_token_c", h_out(h, hd));
                const double t_cb = g_prof_on ? now_ms() : 0.0;
                lk.unlock();
                full_attn_cb(l, h, py_context);
                lk.lock();
                if (g_prof_on) g_prof_ms[QP_PYCALLBACK] += now_ms() - t_cb;
                RT_CHECK("forward_token_c", h_in(hd, h));
            }
            RT_CHECK("forward_token_c", layer_steps(L, &hd, pending));
            if (g_prof_on) g_prof_ms[QP_MLP] += now_ms() - t_layer;
        } else {
            RT_CHECK("forward_token_c", layer_steps(L, &hd, pending));
            if (g_prof_on) g_prof_ms[QP_LINEAR] += now_ms() - t_layer;
        }
        pending = w.down;
    }
    RT_CHECK("forward_token_c", norm_step(hd, pending, fnorm, w.normed));
    {
        Step s(QP_LMHEAD);
        RT_CHECK("forward_token_c", bf16_lm_head_dev(w.lm, reinterpret_cast<float*>(w.lm + 1), w.lm + 2, w.lm + 3,
                                                     nullptr, w.normed, table, tiled, kVocab, kHidden, 1, 0,
                                                     g.stream));
        RT_CHECK("forward_token_c", s.done());
    }
    int out[4] = {0, 0, 0, 0};
    RT_CHECK("forward_token_c", states_out(layers));
    RT_CHECK("forward_token_c", result_out(h, hd, out));
    if (g_prof_on) g_prof_ms[QP_TOTAL] += now_ms() - t_total;
    return out[3];
}

void qwen_debug_chain_wait(long long ticks) {
    std::lock_guard<std::mutex> lk(g.mu);
    F.chain.wait_ticks = ticks < 0 ? kChainWait : (uint64_t)ticks;
    F.chain.rest = 0;
    F.chain.next_rest = kChainRest;
}

int qwen_debug_chain_rest(int calls) {
    std::lock_guard<std::mutex> lk(g.mu);
    const int prev = F.chain.rest;
    if (calls >= 0) F.chain.rest = calls;
    return prev;
}

void qwen_debug_chain_runs(long long* done, long long* gave_up) {
    std::lock_guard<std::mutex> lk(g.mu);
    if (done) *done = F.chain.done;
    if (gave_up) *gave_up = F.chain.gave_up;
}

int qwen_forward_state_resident(int on) {
    std::lock_guard<std::mutex> lk(g.mu);
    const int prev = F.resident;
    if (prev && !on && g.ready && sync_states_out() != BFP8_OK) fatal("qwen_forward_state_resident");
    F.resident = on ? 1 : 0;
    return prev;
}

void qwen_forward_reset_state(void) {
    std::lock_guard<std::mutex> lk(g.mu);
    if (!g.ready) return;
    for (auto& kv : F.states) {
        DevState* st = kv.second.get();
        // hipMemsetAsync is fine here: this call is never captured in a graph
        if (hipMemsetAsync(st->conv[st->cur], 0, (size_t)3 * kConv * 4, g.stream) != hipSuccess ||
            hipMemsetAsync(st->rec[st->rcur], 0, (size_t)RT_HEADS * RT_HEAD_DIM * RT_HEAD_DIM * 4, g.stream) != hipSuccess) {
            set_error("state reset failed");
            fatal("qwen_forward_reset_state");
        }
        st->dirty = st->resident_used;
    }
    if (hipStreamSynchronize(g.stream) != hipSuccess) fatal("qwen_forward_reset_state");
}

void qwen_forward_sync_state(void) {
    std::lock_guard<std::mutex> lk(g.mu);
    if (g.ready && sync_states_out() != BFP8_OK) fatal("qwen_forward_sync_state");
}

}  // extern "C"
