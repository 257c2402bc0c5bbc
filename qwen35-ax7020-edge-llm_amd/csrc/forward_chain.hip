// forward_chain.hip -- a run of decode layers in one launch.
//
// A decode token is a chain of small dependent steps: per linear-attention
// layer the qkv / z GEMVs, the attention step, o, gate / up and down
// (04/qwen_kernels_opt.c:920-1010).  Run as one launch per step (fused_gemv.hip,
// runtime_ftz.hip) each costs 5 to 7.5 us, of which 2.3 us are the launch
// itself and about 1 us the step's inputs' way back from memory, while its
// weights would stream in a fraction of a microsecond.  Here 256 workgroups, one
// per CU, stay for the whole run and hand the vectors on among themselves:
//
//   * a produced vector goes out as 64-bit words of two floats, one agent-scope
//     atomic store each, and a consumer re-reads the words that it needs until
//     none is the "not yet" pattern (all ones: a NaN that no operation gives;
//     a float pair that happens to carry it is stored as the canonical NaN).
//     Data and flag are one word, so no fence and no second round trip.  Every
//     (layer, vector) has words of its own, and a launch that follows uses the
//     other of two sets, which this one leaves cleared;
//   * every workgroup keeps the hidden state in registers and computes each
//     norm and activation itself, as the separate launches do;
//   * weights and parameters are loaded into registers a step or more ahead,
//     right after the inputs of the current step have arrived (a wavefront's
//     loads complete in order: issued earlier they would hold up the inputs).
//
// Every operation and its order are those of the separate kernels (the GEMV
// terms and block-order sums of fused_gemv.hip, the attention step of
// runtime_ftz.hip), so results are the same bit for bit.
//
// All 256 workgroups have to run at once: the host launches this only where
// they fit (one per CU).  Work of other streams may hold back some of them for
// a while; the waits are bounded by the clock, a workgroup that gives up says so
// in `status` and leaves, and so do the others.  The launch writes the layers'
// states to their second buffers, so the host can then run the separate
// launches from the unchanged ones.
//
// Compiled with f32 flush-to-zero and -ffp-contract=off.
#include <hip/hip_runtime.h>

#include "bfp8_internal.h"
#include "gemv_dev.h"
#include "quant_block.h"
#include "runtime_dev.h"
#include "runtime_internal.h"

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kMlpRows = 3584;
constexpr int kHD = RT_HEADS * RT_HEAD_DIM;
constexpr int kMaxNb = kMlpRows / 64;
constexpr uint64_t kNotYet = ~0ull;
// words of one layer's vectors
constexpr int kWDown = 0, kWO = kWDown + RT_HIDDEN / 2, kWQkv = kWO + RT_HIDDEN / 2, kWZ = kWQkv + RT_CONV_CH / 2,
              kWAttn = kWZ + kHD / 2, kWZs = kWAttn + kHD / 2, kWGate = kWZs + kHD / 2, kWUp = kWGate + kMlpRows / 2,
              kWEnd = kWUp + kMlpRows / 2;
static_assert(kWEnd == RT_CHAIN_LAYER_WORDS, "exchange words of a layer");
// the attention step's columns of a workgroup: 16 workgroups per head
constexpr int kParts = RT_CHAIN_WGS / RT_HEADS, kCols = RT_HEAD_DIM / kParts;
static_assert(kCols == 8 && kCols * RT_HEAD_DIM == 2 * kThreads, "two state elements per thread");
constexpr int kBigRows = 32;                  // rows per workgroup of the K = 1024 GEMVs
constexpr int kBigPitch = 16 + 4, kSmallPitch = kMaxNb + 4;  // floats per chain of terms (16-byte rows)

struct ChainLds {
    __attribute__((aligned(16))) uint32_t xs[kMaxNb * 32];  // split activation records
    float xsc[kMaxNb];
    __attribute__((aligned(16))) float terms[4 * kBigRows * kBigPitch];
    __attribute__((aligned(16))) float sq[4][kChunk / 4 + 4];      // rmsnorm's squares, a row per residue
    __attribute__((aligned(16))) float pg[2][4][kChunk / 4 + 4];   // the gates' products
    __attribute__((aligned(16))) float normed[RT_HIDDEN];
    __attribute__((aligned(16))) float kq[2][RT_HEAD_DIM];         // k, q
    float vv[RT_HEAD_DIM];
    __attribute__((aligned(16))) float lq[2][4][36];               // k and q squares; q * k
    __attribute__((aligned(16))) float sp[2][kCols][RT_HEAD_DIM + 4];  // S * k, S * q per column
    __attribute__((aligned(16))) float gp[RT_HEADS][4][36];        // the gated norm's squares
    float gr[RT_HEADS];
    float dcol[kCols];
    float sc[5];  // alpha, beta, k scale, q scale, q.k
    float scale;
    int fail;
};
static_assert(sizeof(float) * 16 * kSmallPitch <= sizeof(ChainLds::terms), "the small GEMVs' terms fit");

// The layers' descriptions do not change during a launch: scalar loads.
typedef const __attribute__((address_space(4))) RtChainLayer ChainLayer;

__device__ __forceinline__ void lds_barrier() {  // LDS only: loads stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ float word_lo(uint64_t v) { return __uint_as_float((uint32_t)v); }
__device__ __forceinline__ float word_hi(uint64_t v) { return __uint_as_float((uint32_t)(v >> 32)); }

__device__ __forceinline__ void publish(uint64_t* p, float lo, float hi) {
    uint64_t v = ((uint64_t)__float_as_uint(hi) << 32) | __float_as_uint(lo);
    if (v == kNotYet) v = 0x7fc000007fc00000ull;
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// v[i] = *p[i], re-read until each has been written (lanes without `mine` read
// nothing); false when the launch's time is up.
template <int N>
__device__ __forceinline__ bool await(uint64_t (&v)[N], const uint64_t* const (&p)[N], bool mine, uint64_t deadline) {
    for (int i = 0; i < N; ++i) v[i] = 0;
    for (uint32_t spin = 1;; ++spin) {
        bool ok = true;
        if (mine) {
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] = __hip_atomic_load(p[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int i = 0; i < N; ++i) ok &= v[i] != kNotYet;
        }
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) return true;
        if (((spin & 15) == 0 || deadline == 0) && wall_clock64() > deadline) return false;
    }
}

// Weights of 32 rows (half s of tile t) of a K = 1024 GEMV: wavefront w blocks
// 2w and 2w + 1; lane = row (lane & 31), residue 2p + lane / 32 of load p.
struct BigW {
    u32x4 w[2][2];
    uint32_t e;  // the row's exponents of blocks 4(w / 2) ..
};
__device__ __forceinline__ void load_big(BigW& r, const uint8_t* mant, const uint8_t* exps, int half, int w, int lane) {
    const int t = half >> 1, row = (half & 1) * 32 + (lane & 31);
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mant + (size_t)t * 16 * 4096u, 16 * 4096u);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)t * 4 * 256u, 4 * 256u);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
            r.w[i][p] = load_w(wrs, (2 * w + i) * 4096 + (2 * p + (lane >> 5)) * 1024 + row * 16, 0);
    r.e = load_e(ers, (w >> 1) * 256 + row * 4, 0);
}

// Weights of 4 rows (sub-tile sub) of a GEMV of kNb blocks: lane = row (lane &
// 3), residue (lane >> 2) & 3, block 4(w + 8i) + lane / 16 of load i.
template <int kNb>
struct SmallW {
    static constexpr int kLd = (kNb / 4 + kWaves - 1) / kWaves;
    u32x4 w[kLd];
    uint32_t e[kLd];
};
template <int kNb>
__device__ __forceinline__ void load_small(SmallW<kNb>& r, const uint8_t* mant, const uint8_t* exps, int sub, int w,
                                           int lane) {
    const int t = sub >> 4, row = (sub & 15) * 4 + (lane & 3), q = (lane >> 2) & 3;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mant + (size_t)t * kNb * 4096u, kNb * 4096u);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)t * (kNb / 4) * 256u, (kNb / 4) * 256u);
#pragma unroll
    for (int i = 0; i < SmallW<kNb>::kLd; ++i) {  // (past the tile: zeros, no memory touched)
        r.w[i] = load_w(wrs, ((w + kWaves * i) * 4 + (lane >> 4)) * 4096 + q * 1024 + row * 16, 0);
        r.e[i] = load_e(ers, (w + kWaves * i) * 256 + row * 4, 0);
    }
}

// The block's term (float(S) * 2^(e-134)) * xscale of one residue chunk.
__device__ __forceinline__ float chunk_term(const ChainLds& L, const u32x4& wq, int b, int q, uint32_t e) {
    const uint4 xh = *reinterpret_cast<const uint4*>(&L.xs[(b * 4 + q) * 8]);
    const uint4 xl = *reinterpret_cast<const uint4*>(&L.xs[(b * 4 + q) * 8 + 4]);
    int S = __builtin_amdgcn_sdot4((int)wq.x, (int)xh.x, 0, false);
    S = __builtin_amdgcn_sdot4((int)wq.y, (int)xh.y, S, false);
    S = __builtin_amdgcn_sdot4((int)wq.z, (int)xh.z, S, false);
    S = __builtin_amdgcn_sdot4((int)wq.w, (int)xh.w, S, false);
    S = (int)((uint32_t)S << 8);
    S = __builtin_amdgcn_sdot4((int)wq.x, (int)xl.x, S, false);
    S = __builtin_amdgcn_sdot4((int)wq.y, (int)xl.y, S, false);
    S = __builtin_amdgcn_sdot4((int)wq.z, (int)xl.z, S, false);
    S = __builtin_amdgcn_sdot4((int)wq.w, (int)xl.w, S, false);
    const float t1 = (float)S * exp_scale_ftz(e);
    return t1 * L.xsc[b];
}

// p[0] + ... + p[n - 1] from +0 in this order (LDS, 16-byte aligned); the
// reads run kAhead ahead of the adds (spread as in chain_add256).
template <int kN>
__device__ __forceinline__ float chain_n(const float* p) {
    constexpr int kV = kN / 4, kAhead = kV < 8 ? kV : 8;
    const float4* p4 = reinterpret_cast<const float4*>(p);
    float4 v[kV];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) v[i] = p4[i];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < kV; ++i) {
        if (i + kAhead < kV) v[i + kAhead] = p4[i + kAhead];
        s = s + v[i].x;
        s = s + v[i].y;
        s = s + v[i].z;
        s = s + v[i].w;
        asm volatile("" : "+v"(s)::"memory");
    }
    return s;
}

// Four swiglu elements (swiglu_elem's vector part): the float instructions
// where everything is normal, else the exact helpers, in one place.
__device__ __forceinline__ void swiglu4(float (&y)[4], const float (&gt)[4], const float (&up)[4]) {
    uint32_t ok = 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float d = 1.0f + exp_neon(-gt[j]), r = __fdiv_rn(gt[j], d);
        ok &= normal_u(gt[j]) & normal_u(d) & normal_u(r);
        y[j] = r * up[j];
    }
    if (!ok) {
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            const float gj = j == 0 ? gt[0] : j == 1 ? gt[1] : j == 2 ? gt[2] : gt[3];
            const float uj = j == 0 ? up[0] : j == 1 ? up[1] : j == 2 ? up[2] : up[3];
            const float v = swiglu_elem(gj, uj, true);
            y[0] = j == 0 ? v : y[0];
            y[1] = j == 1 ? v : y[1];
            y[2] = j == 2 ? v : y[2];
            y[3] = j == 3 ? v : y[3];
        }
    }
}

// Four gated-norm elements (gated_mul), likewise.
__device__ __forceinline__ void gated4(float (&y)[4], const float (&x)[4], float r, const float4& w4, const float (&z)[4]) {
    const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
    uint32_t ok = normal_u(r);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float a = x[j] * r, b = a * wv[j], c = b * z[j];
        ok &= normal_u(x[j]) & normal_u(a) & normal_u(wv[j]) & normal_u(b) & normal_u(z[j]) & normal_u(c);
        y[j] = c;
    }
    if (!ok) {
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            const float xj = j == 0 ? x[0] : j == 1 ? x[1] : j == 2 ? x[2] : x[3];
            const float wj = j == 0 ? w4.x : j == 1 ? w4.y : j == 2 ? w4.z : w4.w;
            const float zj = j == 0 ? z[0] : j == 1 ? z[1] : j == 2 ? z[2] : z[3];
            const float v = gated_mul(xj, r, wj, zj);
            y[0] = j == 0 ? v : y[0];
            y[1] = j == 1 ? v : y[1];
            y[2] = j == 2 ? v : y[2];
            y[3] = j == 3 ? v : y[3];
        }
    }
}

__device__ __forceinline__ void big_terms(ChainLds& L, const BigW& W, int w, int lane) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int b = 2 * w + i;
        const uint32_t e = (W.e >> (8 * (b & 3))) & 0xffu;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int q = 2 * p + (lane >> 5);
            L.terms[(q * kBigRows + (lane & 31)) * kBigPitch + b] = chunk_term(L, W.w[i][p], b, q, e);
        }
    }
}
// Wavefronts 0 and 1: rows 16w .. 16w + 15, lane = residue * 16 + row; the
// rows' words 8w .. 8w + 7 of `out`.
__device__ __forceinline__ void big_sums(const ChainLds& L, uint64_t* out, int w, int lane) {
    const int q = lane >> 4, r = lane & 15;
    const float fs = chain_n<16>(&L.terms[(q * kBigRows + 16 * w + r) * kBigPitch]);
    const float f0 = __shfl(fs, r, 64), f1 = __shfl(fs, 16 + r, 64), f2 = __shfl(fs, 32 + r, 64), f3 = __shfl(fs, 48 + r, 64);
    const float y = (f0 + f2) + (f1 + f3);
    const float lo = __shfl(y, 2 * (lane & 7), 64), hi = __shfl(y, 2 * (lane & 7) + 1, 64);
    if (lane < 8) publish(out + 8 * w + lane, lo, hi);
}

template <int kNb>
__device__ __forceinline__ void small_terms(ChainLds& L, const SmallW<kNb>& W, int w, int lane) {
    const int r = lane & 3, q = (lane >> 2) & 3, blk = lane >> 4;
#pragma unroll
    for (int i = 0; i < SmallW<kNb>::kLd; ++i) {
        const int b = (w + kWaves * i) * 4 + blk;
        if (b < kNb) L.terms[(q * 4 + r) * kSmallPitch + b] = chunk_term(L, W.w[i], b, q, (W.e[i] >> (8 * blk)) & 0xffu);
    }
}
// Wavefront 0: 16 chains, lane = residue * 4 + row; the four rows' two words.
template <int kNb>
__device__ __forceinline__ void small_sums(const ChainLds& L, uint64_t* out, int lane) {
    const float fs = chain_n<kNb>(&L.terms[(lane & 15) * kSmallPitch]);
    const int r = lane & 3;
    const float f0 = __shfl(fs, r, 64), f1 = __shfl(fs, 4 + r, 64), f2 = __shfl(fs, 8 + r, 64), f3 = __shfl(fs, 12 + r, 64);
    const float y = (f0 + f2) + (f1 + f3);
    const float lo = __shfl(y, 2 * (lane & 1), 64), hi = __shfl(y, 2 * (lane & 1) + 1, 64);
    if (lane < 2) publish(out + lane, lo, hi);
}

// rmsnorm of x (threads below 256, elements 4 tid + j) times (1 + nw): into
// L.normed, and quantized into the LDS activation.  false: give up.
__device__ __forceinline__ bool norm_step(ChainLds& L, const float (&x)[4], const float4& nw, float eps, int tid, int lane,
                                          int w) {
    if (tid < 256) {
#pragma unroll
        for (int j = 0; j < 4; ++j) L.sq[j][tid] = x[j] * x[j];
    }
    lds_barrier();
    if (L.fail) return false;
    if (w == 0) {
        float s = 0.0f;
        if (lane < 4) s = chain_add256(0.0f, &L.sq[lane][0]);
        const float r = (readlane_f(s, 0) + readlane_f(s, 2)) + (readlane_f(s, 1) + readlane_f(s, 3));
        if (lane == 0) L.scale = rms_scale(r, RT_HIDDEN, eps);
    }
    lds_barrier();
    const float r = L.scale;
    if (tid < 256) {
        const float y[4] = {x[0] * (r * (1.0f + nw.x)), x[1] * (r * (1.0f + nw.y)), x[2] * (r * (1.0f + nw.z)),
                            x[3] * (r * (1.0f + nw.w))};
        *reinterpret_cast<float4*>(&L.normed[4 * tid]) = make_float4(y[0], y[1], y[2], y[3]);
        bfp8_quant4_store_lds(y, tid & 15, &L.xsc[tid >> 4], &L.xs[(tid >> 4) * 32], true);
    }
    lds_barrier();
    return true;
}

}  // namespace

extern "C" __global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void rt_chain_kernel(
    RtChainArgs a) {
    __shared__ ChainLds L;
    const int tid = threadIdx.x, lane = tid & 63, g = blockIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t deadline = a.wait_ticks ? wall_clock64() + a.wait_ticks : 0;  // 0: no waiting at all
    // sub-tile of four rows: the two that share 128-byte lines go to one XCD
    // (workgroups are dealt to the 8 XCDs in turn)
    const int sub = 2 * ((g >> 4) * 8 + (g & 7)) + ((g >> 3) & 1);
    const int head = g / kParts, part = g % kParts;
    if (tid == 0) L.fail = 0;
    ChainLayer* const layers = (ChainLayer*)a.layers;
    auto give_up = [&] {
        L.fail = 1;
        __hip_atomic_store(a.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    };

    BigW bw;
    SmallW<32> sc;
    SmallW<56> se;
    float4 nw;  // norm weights of elements 4 tid + j (tid < 256)
    const int t4 = 4 * (tid & 255);
    // a layer's first step: qkv / z, or gate / up
    auto load_first = [&](ChainLayer& y) {
        if (y.linear) {
            load_big(bw, g < 192 ? y.mant[0] : y.mant[1], g < 192 ? y.exps[0] : y.exps[1], g < 192 ? g : g - 192, w, lane);
            nw = *reinterpret_cast<const float4*>(y.in_ln_w + t4);
        } else {
            if (g < 224)
                load_big(bw, g < 112 ? y.mant[3] : y.mant[4], g < 112 ? y.exps[3] : y.exps[4], g < 112 ? g : g - 112, w, lane);
            nw = *reinterpret_cast<const float4*>(y.post_ln_w + t4);
        }
    };

    // the hidden state, elements 4 tid + j of threads below 256
    float h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    lds_barrier();  // L.fail
    if (a.table) {
        if (tid < 256) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = 4 * tid + j;
                size_t at = (size_t)a.row * RT_HIDDEN + e;
                if (a.ntiles) {  // the lm_head's tile layout (see rt_embed_kernel)
                    const int c = e >> 3, q = c >> 2;
                    const size_t slot =
                        (((size_t)(q >> 1) * (size_t)(4 * a.ntiles) + (size_t)(a.row >> 4)) * 2 + (q & 1)) * 64 +
                        4 * (a.row & 15) + (e & 3);
                    at = slot * 8 + 2 * (c & 3) + ((e >> 2) & 1);
                }
                h[j] = __uint_as_float((uint32_t)a.table[at] << 16);
            }
        }
        load_first(layers[a.idx[0]]);
    } else {
        // one workgroup reads the host's copy and hands it on
        uint64_t* in = a.xch + (size_t)a.n * kWEnd;
        if (g == 0 && tid < 256) {
            const float4 v = *reinterpret_cast<const float4*>(a.h_in + 4 * tid);
            publish(in + 2 * tid, v.x, v.y);
            publish(in + 2 * tid + 1, v.z, v.w);
        }
        uint64_t v[2];
        if (!await(v, {in + 2 * (tid & 255), in + 2 * (tid & 255) + 1}, tid < 256, deadline)) give_up();
        load_first(layers[a.idx[0]]);
        h[0] = word_lo(v[0]);
        h[1] = word_hi(v[0]);
        h[2] = word_lo(v[1]);
        h[3] = word_hi(v[1]);
    }

    // h += the vector at `words` (add_residual)
    auto add_words = [&](const uint64_t* words) {
        uint64_t v[2];
        if (!await(v, {words + 2 * (tid & 255), words + 2 * (tid & 255) + 1}, tid < 256, deadline)) give_up();
        h[0] = h[0] + word_lo(v[0]);
        h[1] = h[1] + word_hi(v[0]);
        h[2] = h[2] + word_lo(v[1]);
        h[3] = h[3] + word_hi(v[1]);
    };

    for (int l = 0; l < a.n; ++l) {
        ChainLayer& y = layers[a.idx[l]];
        uint64_t* const X = a.xch + (size_t)l * kWEnd;
        const uint32_t cur = (a.cur >> l) & 1u, rcur = (a.rcur >> l) & 1u;
        if (l > 0) add_words(a.xch + (size_t)(l - 1) * kWEnd + kWDown);
        if (y.linear) {
            // ---- rmsnorm, then qkv and z (04/qwen_kernels_opt.c:925-941) ----
            // loads for the gates, the attention step and o
            const float4 gwt = *reinterpret_cast<const float4*>((tid < 256 ? y.wa : y.wb) + (size_t)head * RT_HIDDEN + t4);
            const float nea = y.nea[head], dt = y.dt[head];
            const int sect = min(tid >> 6, 2), ch = sect * kHD + head * RT_HEAD_DIM + 2 * lane;  // two channels (tid < 192)
            const float* ci = y.conv[cur];
            const float2 c0 = *reinterpret_cast<const float2*>(ci + ch);
            const float2 c1 = *reinterpret_cast<const float2*>(ci + RT_CONV_CH + ch);
            const float2 c2 = *reinterpret_cast<const float2*>(ci + 2 * RT_CONV_CH + ch);
            const float4 cw0 = *reinterpret_cast<const float4*>(y.conv_w + (size_t)ch * 4);
            const float4 cw1 = *reinterpret_cast<const float4*>(y.conv_w + (size_t)ch * 4 + 4);
            // two elements of this workgroup's eight state columns (blocked layout, contiguous)
            const size_t so = (size_t)head * RT_HEAD_DIM * RT_HEAD_DIM + (size_t)part * kCols * RT_HEAD_DIM + 2 * tid;
            const float2 S = *reinterpret_cast<const float2*>(y.rec[rcur] + so);
            const int si = 4 * ((tid >> 3) & 31) + 2 * (tid & 1);        // their row i (and i + 1)
            const int sj = 4 * (tid >> 8) + ((tid >> 1) & 3);            // and column of the eight
            load_small<32>(sc, y.mant[2], y.exps[2], sub, w, lane);
            const float4 gnw = *reinterpret_cast<const float4*>(y.norm_w + ((4 * tid) & (RT_HEAD_DIM - 1)));
            if (!norm_step(L, h, nw, a.eps, tid, lane, w)) return;
            {
                const float4 n4 = *reinterpret_cast<const float4*>(&L.normed[t4]);
                float(*pg)[kChunk / 4 + 4] = L.pg[tid >> 8];
                pg[0][tid & 255] = gwt.x * n4.x;
                pg[1][tid & 255] = gwt.y * n4.y;
                pg[2][tid & 255] = gwt.z * n4.z;
                pg[3][tid & 255] = gwt.w * n4.w;
            }
            big_terms(L, bw, w, lane);
            lds_barrier();
            if (w < 2) {
                big_sums(L, X + (g < 192 ? kWQkv + g * 16 : kWZ + (g - 192) * 16), w, lane);
            } else if (w == 4) {  // the gates (read after the attention step's barriers; waves 0 - 3 have the conv)
                float s = 0.0f;
                if (lane < 8) s = chain_add256(0.0f, &L.pg[lane >> 2][lane & 3][0]);
                const float r = lanes4_combine(s);
                const float bv = readlane_f(r, 4);
                if (lane == 0) gates_scalar(r, bv, nea, dt, &L.sc[0], &L.sc[1]);
            }
            // ---- conv1d + SiLU, q/k L2 norm, recurrent step (:943-967) ----
            {
                const bool conv = tid < 192, zcol = tid >= 192 && tid < 192 + kCols / 2;
                uint64_t v[1];
                const int zi = (head * RT_HEAD_DIM + part * kCols) / 2 + (tid - 192);
                if (!await(v, {X + (conv ? kWQkv + (sect * kHD + head * RT_HEAD_DIM) / 2 + lane : zcol ? kWZ + zi : kWQkv)},
                           conv || zcol, deadline))
                    give_up();
                // the next step's weights, behind the inputs
                if (g < 224)
                    load_big(bw, g < 112 ? y.mant[3] : y.mant[4], g < 112 ? y.exps[3] : y.exps[4], g < 112 ? g : g - 112, w,
                             lane);
                nw = *reinterpret_cast<const float4*>(y.post_ln_w + t4);
                const float x0 = word_lo(v[0]), x1 = word_hi(v[0]);
                if (conv) {
                    float d0 = cw0.x * c0.x, d1 = cw1.x * c0.y;
                    d0 = d0 + cw0.y * c1.x;
                    d1 = d1 + cw1.y * c1.y;
                    d0 = d0 + cw0.z * c2.x;
                    d1 = d1 + cw1.z * c2.y;
                    d0 = d0 + cw0.w * x0;
                    d1 = d1 + cw1.w * x1;
                    const float y0 = ieee_div(d0, 1.0f + exp_neon(-d0)), y1 = ieee_div(d1, 1.0f + exp_neon(-d1));
                    const int e = 2 * lane;
                    if (sect == 2) {
                        L.vv[e] = y0;
                        L.vv[e + 1] = y1;
                    } else {  // sect 0: q (row 1), 1: k (row 0)
                        L.kq[1 - sect][e] = y0;
                        L.kq[1 - sect][e + 1] = y1;
                        L.lq[1 - sect][e & 3][e >> 2] = y0 * y0;
                        L.lq[1 - sect][(e & 3) + 1][e >> 2] = y1 * y1;
                    }
                    if (part == 0) {  // one writer for the shifted taps
                        float* co = y.conv[cur ^ 1];
                        *reinterpret_cast<float2*>(co + ch) = c1;
                        *reinterpret_cast<float2*>(co + RT_CONV_CH + ch) = c2;
                        *reinterpret_cast<float2*>(co + 2 * RT_CONV_CH + ch) = make_float2(x0, x1);
                    }
                } else if (zcol) {
                    publish(X + kWZs + zi, silu_scalar(x0), silu_scalar(x1));
                }
            }
            lds_barrier();
            if (L.fail) return;
            if (w == 0) {
                float s = 0.0f;
                if (lane < 8) s = chain_n<RT_HEAD_DIM / 4>(&L.lq[lane >> 2][lane & 3][0]);
                const float r = lanes4_combine(s);
                const float q_sq = readlane_f(r, 4);
                if (lane == 0) {
                    // 1 / sqrtf(D): both steps of normal constants, so the instructions are exact
                    const float q_scale = __fdiv_rn(1.0f, (float)__builtin_sqrt((double)RT_HEAD_DIM));
                    L.sc[2] = div_sqrt_add(1.0f, r, 1e-6f);
                    L.sc[3] = div_sqrt_add(q_scale, q_sq, 1e-6f);
                }
            }
            lds_barrier();
            if (tid < RT_HEAD_DIM) {
                const float k = L.kq[0][tid] * L.sc[2], q = L.kq[1][tid] * L.sc[3];
                L.kq[0][tid] = k;
                L.kq[1][tid] = q;
                L.lq[0][tid & 3][tid >> 2] = q * k;
            }
            lds_barrier();
            const float2 k2 = *reinterpret_cast<const float2*>(&L.kq[0][si]);
            {
                const float2 q2 = *reinterpret_cast<const float2*>(&L.kq[1][si]);
                *reinterpret_cast<float2*>(&L.sp[0][sj][si]) = make_float2(S.x * k2.x, S.y * k2.y);
                *reinterpret_cast<float2*>(&L.sp[1][sj][si]) = make_float2(S.x * q2.x, S.y * q2.y);
            }
            if (w == 1) {
                float s = 0.0f;
                if (lane < 4) s = chain_n<RT_HEAD_DIM / 4>(&L.lq[0][lane][0]);
                const float r = lanes4_combine(s);
                if (lane == 0) L.sc[4] = r;
            }
            lds_barrier();
            const float alpha = L.sc[0], beta = L.sc[1];
            if (w == 0) {  // lane = role * 8 + column: sum_i k[i] S[i][j], sum_i q[i] S[i][j]
                const float acc = chain_n<RT_HEAD_DIM>(&L.sp[(lane >> 3) & 1][lane & 7][0]);
                const int c = lane & 7;
                const float kvs = __shfl(acc, c, 64), qss = __shfl(acc, 8 + c, 64);
                const float d = (L.vv[part * kCols + c] - kvs * alpha) * beta;
                const float o = qss * alpha + L.sc[4] * d;
                if (lane < kCols) L.dcol[lane] = d;
                const float lo = __shfl(o, 2 * (lane & 3), 64), hi = __shfl(o, 2 * (lane & 3) + 1, 64);
                if (lane < kCols / 2) publish(X + kWAttn + (head * RT_HEAD_DIM + part * kCols) / 2 + lane, lo, hi);
            }
            lds_barrier();
            {
                const float d = L.dcol[sj];
                *reinterpret_cast<float2*>(y.rec[rcur ^ 1] + so) = make_float2(S.x * alpha + d * k2.x, S.y * alpha + d * k2.y);
            }
            // ---- gated RMSNorm, then o (:968-985) ----
            float at[4], zs[4];
            {
                uint64_t v[4];
                const uint64_t* pa = X + kWAttn + 2 * tid;
                const uint64_t* pz = X + kWZs + 2 * tid;
                if (!await(v, {pa, pa + 1, pz, pz + 1}, true, deadline)) give_up();
                at[0] = word_lo(v[0]);
                at[1] = word_hi(v[0]);
                at[2] = word_lo(v[1]);
                at[3] = word_hi(v[1]);
                zs[0] = word_lo(v[2]);
                zs[1] = word_hi(v[2]);
                zs[2] = word_lo(v[3]);
                zs[3] = word_hi(v[3]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) L.gp[tid >> 5][j][tid & 31] = at[j] * at[j];
            lds_barrier();
            if (L.fail) return;
            if (w == 0) {
                const float r = lanes4_combine(chain_n<RT_HEAD_DIM / 4>(&L.gp[lane >> 2][lane & 3][0]));
                if ((lane & 3) == 0) L.gr[lane >> 2] = rms_scale(r, RT_HEAD_DIM, a.eps);
            }
            lds_barrier();
            {
                const float gr = L.gr[tid >> 5];
                float v[4];
                gated4(v, at, gr, gnw, zs);
                bfp8_quant4_store_lds(v, tid & 15, &L.xsc[tid >> 4], &L.xs[(tid >> 4) * 32], true);
            }
            lds_barrier();
            small_terms<32>(L, sc, w, lane);
            lds_barrier();
            if (w == 0) small_sums<32>(L, X + kWO + 2 * sub, lane);
            add_words(X + kWO);
        }
        // ---- rmsnorm, gate and up (:987-997) ----
        load_small<56>(se, y.mant[5], y.exps[5], sub, w, lane);
        if (!norm_step(L, h, nw, a.eps, tid, lane, w)) return;
        if (g < 224) big_terms(L, bw, w, lane);
        lds_barrier();
        if (g < 224 && w < 2) big_sums(L, X + (g < 112 ? kWGate + g * 16 : kWUp + (g - 112) * 16), w, lane);
        // ---- swiglu, down (:998-1004) ----
        {
            uint64_t v[4], u[4];
            const uint64_t* pg = X + kWGate + 2 * tid;
            const uint64_t* pu = X + kWUp + 2 * tid;
            bool ok = await(v, {pg, pg + 1, pu, pu + 1}, true, deadline);
            // (the last 1536 elements: threads below 384)
            const int m = tid < 384 ? 1024 : 0;
            ok = await(u, {pg + m, pg + m + 1, pu + m, pu + m + 1}, tid < 384, deadline) && ok;
            if (!ok) give_up();
            if (l + 1 < a.n) load_first(layers[a.idx[l + 1]]);
            // (one body for both halves: the code stays short)
#pragma unroll 1
            for (int half = 0; half < 2; ++half) {
                if (half && w >= 6) break;
                const uint64_t g0 = half ? u[0] : v[0], g1 = half ? u[1] : v[1], u0 = half ? u[2] : v[2], u1 = half ? u[3] : v[3];
                const float gt[4] = {word_lo(g0), word_hi(g0), word_lo(g1), word_hi(g1)};
                const float up[4] = {word_lo(u0), word_hi(u0), word_lo(u1), word_hi(u1)};
                float s[4];
                swiglu4(s, gt, up);
                const int b = 32 * half + (tid >> 4);
                bfp8_quant4_store_lds(s, tid & 15, &L.xsc[b], &L.xs[b * 32], true);
            }
        }
        lds_barrier();
        if (L.fail) return;
        small_terms<56>(L, se, w, lane);
        lds_barrier();
        if (w == 0) small_sums<56>(L, X + kWDown + 2 * sub, lane);
    }

    // the other set's words, for the launch after this one
    for (int i = g * kThreads + tid; i < a.clear_words; i += RT_CHAIN_WGS * kThreads) a.xch_clear[i] = kNotYet;
    // one workgroup finishes the hidden state (and the final norm)
    if (g != 0) return;
    add_words(a.xch + (size_t)(a.n - 1) * kWEnd + kWDown);
    if (tid < 256) *reinterpret_cast<float4*>(a.h_out + 4 * tid) = make_float4(h[0], h[1], h[2], h[3]);
    if (a.y_norm) {
        nw = *reinterpret_cast<const float4*>(a.final_w + t4);
        if (!norm_step(L, h, nw, a.eps, tid, lane, w)) return;
        if (tid < 256) *reinterpret_cast<float4*>(a.y_norm + 4 * tid) = *reinterpret_cast<const float4*>(&L.normed[4 * tid]);
    }
}

// Whether the device runs the chain's workgroups all at once.
bool rt_chain_fits() {
    static const bool fits = [] {
        int occ = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(rt_chain_kernel), kThreads, 0) !=
            hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return occ >= 1 && bfp8_cu_count() >= RT_CHAIN_WGS;
    }();
    return fits;
}

hipError_t rt_launch_chain(const RtChainArgs& a, hipStream_t s) {
    if (a.n < 1 || a.n > RT_CHAIN_MAX_LAYERS || (!a.table && !a.h_in) || !a.h_out || !a.status || !a.xch ||
        a.xch == a.xch_clear || (a.y_norm && !a.final_w))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(rt_chain_kernel, dim3(RT_CHAIN_WGS), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}
