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
//     none is the "not yet" pattern (all ones: a NaN that no operation gives, but
//     passes on; a float pair that carries it is stored as the canonical NaN,
//     which makes no difference but in the hidden state handed in, and the host
//     takes separate launches for one with such a pair).
//     Data and flag are one word, so no fence and no second round trip.  Every
//     (layer, vector) has words of its own, and a launch that follows uses the
//     other of two sets, which this one leaves cleared;
//   * every workgroup keeps the hidden state in registers and computes each
//     norm and activation itself, as the separate launches do;
//   * a ninth wavefront loads the weights a step or more ahead, into LDS.  In the
//     others' registers they held up the exchange (a wavefront's loads complete
//     in order), and so do any loads of the CU in flight: they go out where the
//     workgroup computes (see loader);
//   * the workgroup that has 16 rows of gate has those of up too and hands on
//     their swiglu: half the words, and no workgroup computes all 3584.
//
// Bound by latency: a linear-attention layer is 20.5 us, of them 8 in five
// exchanges, of which one between all workgroups takes 1.3 to 2.2 us (store,
// memory-side cache, the last of 256 readers' polls) and one between a head's
// 0.8; 2.9 in 824 dependent float adds, 8 cycles each, that the results' order
// fixes; its 21.5 MB of weights would stream in 4.  Weights in the wavefronts'
// registers, gate and up from different workgroups, 16-bit layer indices (read
// by vector loads): 24.0 us, a token's launch 517; with the loader, 438; with
// the attention step on four wavefronts without barriers and stores of 32
// bytes, 422.
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

constexpr int kThreads = 512, kWaves = kThreads / 64;  // and one more wavefront, the loader
constexpr int kMlpRows = 3584;
constexpr int kHD = RT_HEADS * RT_HEAD_DIM;
constexpr int kMaxNb = kMlpRows / 64;
constexpr uint64_t kNotYet = ~0ull;
// words of one layer's vectors
constexpr int kRowWords = RT_CHAIN_ROW_WORDS;
constexpr int kWDown = 0, kWO = kWDown + RT_CHAIN_WGS * kRowWords, kWQkv = kWO + RT_CHAIN_WGS * kRowWords, kWZ = kWQkv + RT_CONV_CH / 2,
              kWAttn = kWZ + kHD / 2, kWZs = kWAttn + kHD / 2, kWMlp = kWZs + kHD / 2, kWEnd = kWMlp + kMlpRows / 2;
static_assert(kWEnd == RT_CHAIN_LAYER_WORDS, "exchange words of a layer");
// the attention step's columns of a workgroup: 16 workgroups per head
constexpr int kParts = RT_CHAIN_WGS / RT_HEADS, kCols = RT_HEAD_DIM / kParts;
static_assert(kCols == 8 && kCols / 2 * 256 == kCols * RT_HEAD_DIM, "four state elements per thread of four wavefronts");
constexpr int kWaitLoads = 0x0F70;             // s_waitcnt vmcnt(0)
constexpr int kBigRows = 32;                  // rows per workgroup of the K = 1024 GEMVs
constexpr int kBigPitch = 16 + 4, kSmallPitch = kMaxNb + 4;  // floats per chain of terms (16-byte rows)

// Weights of 2 x 16 rows of K = 1024 (16 blocks) and the norm weights of their
// activation.  Block b of half m: one load, lane = residue * 16 + row.
struct BigLds {
    u32x4 w[16][2][64];
    uint32_t e[2][4][16];  // exponents of blocks 4i .. 4i + 3 of a row
    float4 nw[RT_HIDDEN / 4];
};
// Weights of 4 rows of up to kMaxNb blocks.  Blocks 4j .. 4j + 3: one load, lane =
// block * 16 + residue * 4 + row.
struct SmallLds {
    u32x4 w[kMaxNb / 4][64];
    uint32_t e[16][4];
};

struct ChainLds {
    BigLds big[2];  // a step's, the next one's
    SmallLds small[2];
    __attribute__((aligned(16))) uint32_t xs[kMaxNb * 32];  // split activation records
    float xsc[kMaxNb];
    __attribute__((aligned(16))) float terms[4 * kBigRows * kBigPitch];
    __attribute__((aligned(16))) float sq[4][kChunk / 4 + 4];      // rmsnorm's squares, a row per residue
    __attribute__((aligned(16))) float pg[2][4][kChunk / 4 + 4];   // the gates' products
    __attribute__((aligned(16))) float normed[RT_HIDDEN];
    __attribute__((aligned(16))) float kq[2][RT_HEAD_DIM];         // k, q
    __attribute__((aligned(16))) float vv[RT_HEAD_DIM];
    __attribute__((aligned(16))) float lq[2][4][36];               // k and q squares
    __attribute__((aligned(16))) float qk[kCols / 2][4][36];       // a wavefront's q * k
    __attribute__((aligned(16))) float sp[2][kCols][RT_HEAD_DIM + 4];  // S * k, S * q per column
    __attribute__((aligned(16))) float gp[RT_HEADS][4][36];        // the gated norm's squares
    float sc[2];  // alpha, beta
    __attribute__((aligned(8))) float ocol[kCols];
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

// Orders a wavefront's own LDS writes before its reads of other lanes' ones.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float word_lo(uint64_t v) { return __uint_as_float((uint32_t)v); }
__device__ __forceinline__ float word_hi(uint64_t v) { return __uint_as_float((uint32_t)(v >> 32)); }

__device__ __forceinline__ void publish(uint64_t* p, float lo, float hi) {
    uint64_t v = ((uint64_t)__float_as_uint(hi) << 32) | __float_as_uint(lo);
    if (v == kNotYet) v = 0x7fc000007fc00000ull;
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// v[i] = *p[i], re-read until each has been written (lanes without `mine` read
// nothing, lanes that have all of theirs no more: every workgroup reads every
// word past its L2, so re-reads get in the way of the stores they wait for);
// false when the launch's time is up.
template <int N>
__device__ __forceinline__ bool await(uint64_t (&v)[N], const uint64_t* const (&p)[N], bool mine, uint64_t deadline) {
    for (int i = 0; i < N; ++i) v[i] = 0;
    bool ok = !mine;
    for (uint32_t spin = 1;; ++spin) {
        if (!ok) {
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] = __hip_atomic_load(p[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ok = true;
#pragma unroll
            for (int i = 0; i < N; ++i) ok &= v[i] != kNotYet;
        }
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) return true;
        if (((spin & 15) == 0 || deadline == 0) && wall_clock64() > deadline) return false;
    }
}

// The loader's side of BigLds and SmallLds: loads straight into LDS (lane i's
// piece goes to base + i * its size).
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t rs, void* lds, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, kNonTemporal);
}
__device__ __forceinline__ void lds_load4(__amdgpu_buffer_rsrc_t rs, void* lds, int voff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 4, voff, 0, 0, 0);
}
// Rows 16 r0 .. and 16 r1 .. of two (or one) matrices of 1024 columns, with the
// norm weights (only these without `rows`).
__device__ __forceinline__ void load_big(BigLds& L, const uint8_t* m0, const uint8_t* e0, int r0, const uint8_t* m1,
                                         const uint8_t* e1, int r1, const float* nw, bool rows, int lane) {
    const int at[2] = {(r0 & 3) * 16 + (lane & 15), (r1 & 3) * 16 + (lane & 15)};
    const __amdgpu_buffer_rsrc_t nr = make_rsrc(nw, RT_HIDDEN * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_load16(nr, &L.nw[64 * i], lane * 16, i * 1024);
    if (!rows) return;
    const __amdgpu_buffer_rsrc_t er[2] = {make_rsrc(e0 + (size_t)(r0 >> 2) * 4 * 256u, 4 * 256u),
                                          make_rsrc(e1 + (size_t)(r1 >> 2) * 4 * 256u, 4 * 256u)};
    const __amdgpu_buffer_rsrc_t wr[2] = {make_rsrc(m0 + (size_t)(r0 >> 2) * 16 * 4096u, 16 * 4096u),
                                          make_rsrc(m1 + (size_t)(r1 >> 2) * 16 * 4096u, 16 * 4096u)};
#pragma unroll
    for (int m = 0; m < 2; ++m) lds_load4(er[m], &L.e[m][0][0], (lane >> 4) * 256 + at[m] * 4);
#pragma unroll 1
    for (int b = 0; b < 16; ++b)
#pragma unroll
        for (int m = 0; m < 2; ++m) lds_load16(wr[m], &L.w[b][m][0], (lane >> 4) * 1024 + at[m] * 16, b * 4096);
}
// Rows 4 sub .. of a matrix of nb blocks.
__device__ __forceinline__ void load_small(SmallLds& L, const uint8_t* mant, const uint8_t* exps, int nb, int sub, int lane) {
    const int t = sub >> 4, row = (sub & 15) * 4 + (lane & 3), q = (lane >> 2) & 3;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mant + (size_t)t * nb * 4096u, nb * 4096u);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)t * (nb / 4) * 256u, (nb / 4) * 256u);
    lds_load4(ers, &L.e[0][0], (lane >> 2) * 256 + row * 4);  // (past the tile: zeros, no memory touched)
#pragma unroll 1
    for (int j = 0; j < nb / 4; ++j) lds_load16(wrs, &L.w[j][0], (lane >> 4) * 4096 + q * 1024 + row * 16, j * 4 * 4096);
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

// s + p[0] + ... + p[n - 1] in this order (LDS, 16-byte aligned); the
// reads run kAhead ahead of the adds (spread as in chain_add256).
template <int kN>
__device__ __forceinline__ float chain_n(const float* p, float s = 0.0f) {
    constexpr int kV = kN / 4, kAhead = kV < 8 ? kV : 8;
    const float4* p4 = reinterpret_cast<const float4*>(p);
    float4 v[kV];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) v[i] = p4[i];
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

// swiglu_elem's vector part: the float instructions where everything is
// normal, else the exact helpers.
__device__ __forceinline__ float swiglu1(float gt, float up) {
    const float d = 1.0f + exp_neon(-gt), r = __fdiv_rn(gt, d);
    if (normal_u(gt) & normal_u(d) & normal_u(r)) return r * up;
    return swiglu_elem(gt, up, true);
}

// One block of 64 elements quantized by 8 lanes, eight consecutive elements
// per lane (bfp8_quant4_store_lds with a lane's elements 4 ii and 4 ii + 4 as one
// 16-bit store).  ii: the lane's place among the eight.
__device__ __forceinline__ void quant8_store_lds(const float (&x)[8], int ii, float* xscale_b, uint32_t* xsplit_b) {
    float v = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float aj = fabsf(x[j]);
        v = fmaxf(v, (aj > 0.0f) ? aj : 0.0f);  // a NaN never wins `v > amax`
    }
    int m = __float_as_int(v);
    m = max(m, __builtin_amdgcn_mov_dpp(m, 0xB1, 0xF, 0xF, false));
    m = max(m, __builtin_amdgcn_mov_dpp(m, 0x4E, 0xF, 0xF, false));
    m = max(m, __builtin_amdgcn_mov_dpp(m, 0x141, 0xF, 0xF, false));
    const float amax = __int_as_float(m);
    const bool live = amax > 1e-20f;
    const float q = __fdiv_rn(16384.0f, live ? amax : 1.0f);
    typedef __attribute__((address_space(3))) uint16_t lds_u16;
    typedef __attribute__((address_space(3))) float lds_f32;
    lds_u16* rb = (lds_u16*)xsplit_b;
    if (ii == 0) *(lds_f32*)xscale_b = live ? amax * 0x1p-14f : 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t hi = 0, lo = 0;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const float p = __fmul_rn(x[j + 4 * t], q);
            const int xq = (int)__builtin_rintf((live && p == p) ? p : 0.0f);
            const int xl = (int)(int8_t)(xq & 0xff);
            lo |= (uint32_t)(xl & 0xff) << (8 * t);
            hi |= (uint32_t)(((xq - xl) >> 8) & 0xff) << (8 * t);
        }
        rb[j * 16 + ii] = (uint16_t)hi;
        rb[j * 16 + 8 + ii] = (uint16_t)lo;
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

__device__ __forceinline__ void big_terms(ChainLds& L, const BigLds& W, int w, int lane) {
    const int row = lane & 15, q = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int b = 2 * w + i;
#pragma unroll
        for (int m = 0; m < 2; ++m)
            L.terms[(q * kBigRows + 16 * m + row) * kBigPitch + b] =
                chunk_term(L, W.w[b][m][lane], b, q, (W.e[m][b >> 2][row] >> (8 * (b & 3))) & 0xffu);
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

// Wavefront 0, the halves being 16 rows of gate and up: swiglu of the 16 rows.
__device__ __forceinline__ void mlp_sums(const ChainLds& L, uint64_t* out, int lane) {
    const int q = lane >> 4, r = lane & 15;
    float y[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const float fs = chain_n<16>(&L.terms[(q * kBigRows + 16 * m + r) * kBigPitch]);
        const float f0 = __shfl(fs, r, 64), f1 = __shfl(fs, 16 + r, 64), f2 = __shfl(fs, 32 + r, 64), f3 = __shfl(fs, 48 + r, 64);
        y[m] = (f0 + f2) + (f1 + f3);
    }
    const float v = swiglu1(y[0], y[1]);
    const float lo = __shfl(v, 2 * (lane & 7), 64), hi = __shfl(v, 2 * (lane & 7) + 1, 64);
    if (lane < 8) publish(out + lane, lo, hi);
}

template <int kNb>
__device__ __forceinline__ void small_terms(ChainLds& L, const SmallLds& W, int w, int lane) {
    const int r = lane & 3, q = (lane >> 2) & 3, blk = lane >> 4;
#pragma unroll
    for (int i = 0; i < (kNb / 4 + kWaves - 1) / kWaves; ++i) {
        const int j = w + kWaves * i;
        if (j < kNb / 4)
            L.terms[(q * 4 + r) * kSmallPitch + 4 * j + blk] =
                chunk_term(L, W.w[j][lane], 4 * j + blk, q, (W.e[j][r] >> (8 * blk)) & 0xffu);
    }
}
// Wavefront 0: 16 chains, lane = residue * 4 + row; the four rows' two words,
// twice (a store of less than 32 bytes arrives later: 429 us for a token's
// launch with the 16 bytes alone, 422 with 32).
template <int kNb>
__device__ __forceinline__ void small_sums(const ChainLds& L, uint64_t* out, int lane) {
    const float fs = chain_n<kNb>(&L.terms[(lane & 15) * kSmallPitch]);
    const int r = lane & 3;
    const float f0 = __shfl(fs, r, 64), f1 = __shfl(fs, 4 + r, 64), f2 = __shfl(fs, 8 + r, 64), f3 = __shfl(fs, 12 + r, 64);
    const float y = (f0 + f2) + (f1 + f3);
    const float lo = __shfl(y, 2 * (lane & 1), 64), hi = __shfl(y, 2 * (lane & 1) + 1, 64);
    if (lane < kRowWords) publish(out + lane, lo, hi);
}

// rmsnorm of x (threads below 256, elements 4 tid + j) times (1 + nws): into
// L.normed, and quantized into the LDS activation.  false: give up.
__device__ __forceinline__ bool norm_step(ChainLds& L, const float (&x)[4], const float4* nws, float eps, int tid,
                                          int lane, int w) {
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
        const float4 nw = nws[tid];
        const float y[4] = {x[0] * (r * (1.0f + nw.x)), x[1] * (r * (1.0f + nw.y)), x[2] * (r * (1.0f + nw.z)),
                            x[3] * (r * (1.0f + nw.w))};
        *reinterpret_cast<float4*>(&L.normed[4 * tid]) = make_float4(y[0], y[1], y[2], y[3]);
        bfp8_quant4_store_lds(y, tid & 15, &L.xsc[tid >> 4], &L.xs[(tid >> 4) * 32], true);
    }
    lds_barrier();
    return true;
}

// The loader: the wavefront that does every load of weights, into LDS.  A step
// is a norm, its GEMVs (the first buffer), and the GEMV behind them that the
// hidden state waits for (the second): norm .. o of a linear-attention layer, or
// norm .. down.  The next steps' loads go out right behind the barriers that tell
// that an exchange is over, and that leave the longest way to the next: a CU's
// loads return in order, so a read of the exchange words waits for every load
// before it (a buffer's loads as soon as it is free: 530 us for a token's launch
// where this took 438).  The loader passes every barrier of the steps with the
// others; its loads are waited for by a step's first one.  It waits for nothing
// else, and runs on alone where the others gave up.
__device__ __forceinline__ void loader(ChainLds& L, const RtChainArgs& a, ChainLayer* layers, int sub, int lane, int g) {
    auto load_first = [&](int l, bool attn, int t) {  // step t, of layer l
        if (l >= a.n) return;
        ChainLayer& y = layers[a.idx[l]];
        BigLds& B = L.big[t & 1];
        if (attn) {
            const uint8_t *m = g < 192 ? y.mant[0] : y.mant[1], *e = g < 192 ? y.exps[0] : y.exps[1];
            const int r = 2 * (g < 192 ? g : g - 192);
            load_big(B, m, e, r, m, e, r + 1, y.in_ln_w, true, lane);
        } else {  // (the last workgroups use only the norm weights)
            load_big(B, y.mant[3], y.exps[3], g, y.mant[4], y.exps[4], g, y.post_ln_w, g < kMlpRows / 16, lane);
        }
    };
    auto load_second = [&](int l, bool attn, int t) {
        if (l >= a.n) return;
        ChainLayer& y = layers[a.idx[l]];
        const int i = attn ? 2 : 5;
        load_small(L.small[t & 1], y.mant[i], y.exps[i], attn ? kHD / 64 : kMaxNb, sub, lane);
    };
    auto linear = [&](int l) { return l < a.n && layers[a.idx[l]].linear; };
    auto barriers = [&](int n) {
        for (int i = 0; i < n; ++i) lds_barrier();
    };
    // a layer's description into the scalar cache, for everyone, during a wait
    // (read cold, it holds up a layer's first loads by more than 1 us)
    auto touch = [&](int l) {
        const auto* p = reinterpret_cast<const volatile __attribute__((address_space(4))) uint32_t*>(
            &layers[a.idx[min(l, a.n - 1)]]);
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = p[min(16 * i, (int)sizeof(RtChainLayer) / 4 - 1)];
        asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]));
    };
    static_assert(sizeof(RtChainLayer) <= 256, "four lines");
    load_first(0, linear(0), 0);
    load_second(0, linear(0), 0);
    touch(1);
    int t = 0;
    for (int l = 0; l < a.n; ++l) {
        if (linear(l)) {
            __builtin_amdgcn_s_waitcnt(kWaitLoads);
            barriers(1);
            load_first(l, false, t + 1);
            barriers(2);  // norm
            load_second(l, false, t + 1);
            barriers(2);  // terms, q / k / v
            barriers(2);  // the attention step, all heads' outputs
            load_first(l + 1, linear(l + 1), t + 2);  // (into this step's buffer, read a barrier ago)
            barriers(2);  // activation, terms
            ++t;
        }
        __builtin_amdgcn_s_waitcnt(kWaitLoads);
        barriers(1);
        if (!linear(l)) load_first(l + 1, linear(l + 1), t + 1);
        load_second(l + 1, linear(l + 1), t + 1);
        barriers(3);  // norm (2), terms
        touch(l + 2);
        barriers(2);  // activation, terms
        ++t;
    }
    __builtin_amdgcn_s_waitcnt(kWaitLoads);  // nothing lands after the workgroup's end
}

}  // namespace

extern "C" __global__ __launch_bounds__(kThreads + 64) void rt_chain_kernel(
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

    lds_barrier();  // L.fail
    if (w == kWaves) {
        loader(L, a, layers, sub, lane, g);
        return;
    }
    const int t4 = 4 * (tid & 255);

    // the hidden state, elements 4 tid + j of threads below 256
    float h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
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
        h[0] = word_lo(v[0]);
        h[1] = word_hi(v[0]);
        h[2] = word_lo(v[1]);
        h[3] = word_hi(v[1]);
    }

    // h += the vector at `words` (add_residual)
    auto add_words = [&](const uint64_t* words) {
        uint64_t v[2];
        if (!await(v, {words + kRowWords * (tid & 255), words + kRowWords * (tid & 255) + 1}, tid < 256, deadline)) give_up();
        h[0] = h[0] + word_lo(v[0]);
        h[1] = h[1] + word_hi(v[0]);
        h[2] = h[2] + word_lo(v[1]);
        h[3] = h[3] + word_hi(v[1]);
    };

    int t = 0;  // step
    for (int l = 0; l < a.n; ++l) {
        ChainLayer& y = layers[a.idx[l]];
        uint64_t* const X = a.xch + (size_t)l * kWEnd;
        const uint32_t cur = (a.cur >> l) & 1u, rcur = (a.rcur >> l) & 1u;
        if (l > 0) add_words(a.xch + (size_t)(l - 1) * kWEnd + kWDown);
        if (y.linear) {
            // ---- rmsnorm, then qkv and z (04/qwen_kernels_opt.c:925-941) ----
            // loads for the gates, the attention step and o
            const float4 gwt = *reinterpret_cast<const float4*>((tid < 256 ? y.wa : y.wb) + (size_t)head * RT_HIDDEN + t4);
            // (through the vector path: a scalar load in flight holds up every LDS wait)
            int zero;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
            const float nea = y.nea[head + zero], dt = y.dt[head + zero];
            const int sect = min(tid >> 6, 2), ch = sect * kHD + head * RT_HEAD_DIM + 2 * lane;  // two channels (tid < 192)
            const float* ci = y.conv[cur];
            const float2 c0 = *reinterpret_cast<const float2*>(ci + ch);
            const float2 c1 = *reinterpret_cast<const float2*>(ci + RT_CONV_CH + ch);
            const float2 c2 = *reinterpret_cast<const float2*>(ci + 2 * RT_CONV_CH + ch);
            const float4 cw0 = *reinterpret_cast<const float4*>(y.conv_w + (size_t)ch * 4);
            const float4 cw1 = *reinterpret_cast<const float4*>(y.conv_w + (size_t)ch * 4 + 4);
            // four rows of one of this workgroup's eight state columns (blocked layout): wavefronts
            // 0 .. 3 have columns 2w and 2w + 1
            const int scol = 2 * (w & 3) + (lane & 1);
            const size_t so = (size_t)head * RT_HEAD_DIM * RT_HEAD_DIM + (size_t)part * kCols * RT_HEAD_DIM +
                              ((scol >> 2) * (RT_HEAD_DIM / 4) + (lane >> 1)) * 16 + (scol & 3) * 4;
            float4 S;
            if (w < kCols / 2) S = *reinterpret_cast<const float4*>(y.rec[rcur] + so);
            const float4 gnw = *reinterpret_cast<const float4*>(y.norm_w + ((4 * tid) & (RT_HEAD_DIM - 1)));
            if (!norm_step(L, h, L.big[t & 1].nw, a.eps, tid, lane, w)) return;
            {
                const float4 n4 = *reinterpret_cast<const float4*>(&L.normed[t4]);
                float(*pg)[kChunk / 4 + 4] = L.pg[tid >> 8];
                pg[0][tid & 255] = gwt.x * n4.x;
                pg[1][tid & 255] = gwt.y * n4.y;
                pg[2][tid & 255] = gwt.z * n4.z;
                pg[3][tid & 255] = gwt.w * n4.w;
            }
            big_terms(L, L.big[t & 1], w, lane);
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
            // (each of the four wavefronts by itself, no barrier: both scales, then the two
            // columns' sums and q . k as one chain of adds over its lanes)
            if (w < kCols / 2) {
                const int c8 = lane & 7;  // k (0 .. 3) and q (4 .. 7) squares of a residue
                const float sq = lanes4_combine(chain_n<RT_HEAD_DIM / 4>(&L.lq[c8 >> 2][c8 & 3][0]));
                // 1 / sqrtf(D): both steps of normal constants, so the instructions are exact
                const float q_scale = __fdiv_rn(1.0f, (float)__builtin_sqrt((double)RT_HEAD_DIM));
                const float sc = div_sqrt_add(c8 < 4 ? 1.0f : q_scale, sq, 1e-6f);
                const float ks = readlane_f(sc, 0), qs = readlane_f(sc, 4);
                const int i4 = lane >> 1;
                float4 k4 = *reinterpret_cast<const float4*>(&L.kq[0][4 * i4]);
                float4 q4 = *reinterpret_cast<const float4*>(&L.kq[1][4 * i4]);
                k4 = make_float4(k4.x * ks, k4.y * ks, k4.z * ks, k4.w * ks);
                q4 = make_float4(q4.x * qs, q4.y * qs, q4.z * qs, q4.w * qs);
                *reinterpret_cast<float4*>(&L.sp[0][scol][4 * i4]) = make_float4(S.x * k4.x, S.y * k4.y, S.z * k4.z, S.w * k4.w);
                *reinterpret_cast<float4*>(&L.sp[1][scol][4 * i4]) = make_float4(S.x * q4.x, S.y * q4.y, S.z * q4.z, S.w * q4.w);
                if ((lane & 1) == 0) {
                    L.qk[w][0][i4] = q4.x * k4.x;
                    L.qk[w][1][i4] = q4.y * k4.y;
                    L.qk[w][2][i4] = q4.z * k4.z;
                    L.qk[w][3][i4] = q4.w * k4.w;
                }
                wave_lds_sync();
                // lanes 0 .. 3: k . S and q . S of the two columns; 4 .. 7: q . k's residues,
                // whose 32 terms are the first quarter (the rest of theirs is not used)
                const float* row = &L.sp[(c8 >> 1) & 1][2 * w + (c8 & 1)][0];
                const float s32 = chain_n<RT_HEAD_DIM / 4>(c8 < 4 ? row : &L.qk[w][c8 & 3][0]);
                const float acc = chain_n<3 * RT_HEAD_DIM / 4>(row + RT_HEAD_DIM / 4, s32);
                const float qk = readlane_f(lanes4_combine(s32), 4);
                const float alpha = L.sc[0], beta = L.sc[1];
                const float2 v2 = *reinterpret_cast<const float2*>(&L.vv[part * kCols + 2 * w]);
                const float d0 = (v2.x - readlane_f(acc, 0) * alpha) * beta, d1 = (v2.y - readlane_f(acc, 1) * alpha) * beta;
                const float o0 = readlane_f(acc, 2) * alpha + qk * d0, o1 = readlane_f(acc, 3) * alpha + qk * d1;
                if (lane == 0) *reinterpret_cast<float2*>(&L.ocol[2 * w]) = make_float2(o0, o1);
                const float d = (lane & 1) ? d1 : d0;
                S = make_float4(S.x * alpha + d * k4.x, S.y * alpha + d * k4.y, S.z * alpha + d * k4.z, S.w * alpha + d * k4.w);
            }
            lds_barrier();  // (also: no polls before there can be something, they get in the way)
            // (one store of 32 bytes: four of 8, one by each wavefront, arrive 0.9 us later)
            if (w == 0 && lane < kCols / 2)
                publish(X + kWAttn + (head * RT_HEAD_DIM + part * kCols) / 2 + lane, L.ocol[2 * lane], L.ocol[2 * lane + 1]);
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
            // (behind the exchange: its reads would wait for the store)
            if (w < kCols / 2) *reinterpret_cast<float4*>(y.rec[rcur ^ 1] + so) = S;
            lds_barrier();  // (for the loader: the exchange is over)
            if (L.fail) return;
            {
                // wavefront w has heads 2w and 2w + 1; lane & 7 = head * 4 + residue of their squares
#pragma unroll
                for (int j = 0; j < 4; ++j) L.gp[tid >> 5][j][tid & 31] = at[j] * at[j];
                wave_lds_sync();
                const float ss = lanes4_combine(chain_n<RT_HEAD_DIM / 4>(&L.gp[2 * w + ((lane >> 2) & 1)][lane & 3][0]));
                const float sc = rms_scale(ss, RT_HEAD_DIM, a.eps);
                const float gr = lane < 32 ? readlane_f(sc, 0) : readlane_f(sc, 4);
                float v[4];
                gated4(v, at, gr, gnw, zs);
                bfp8_quant4_store_lds(v, tid & 15, &L.xsc[tid >> 4], &L.xs[(tid >> 4) * 32], true);
            }
            lds_barrier();
            small_terms<kHD / 64>(L, L.small[t & 1], w, lane);
            lds_barrier();
            if (w == 0) small_sums<kHD / 64>(L, X + kWO + kRowWords * sub, lane);
            add_words(X + kWO);
            ++t;
        }
        // ---- rmsnorm, gate and up, swiglu (:987-1001) ----
        if (!norm_step(L, h, L.big[t & 1].nw, a.eps, tid, lane, w)) return;
        if (g < kMlpRows / 16) big_terms(L, L.big[t & 1], w, lane);
        lds_barrier();
        if (g < kMlpRows / 16 && w == 0) mlp_sums(L, X + kWMlp + g * 8, lane);
        // ---- down (:1002-1004) ----
        if (w < kMlpRows / 512) {
            uint64_t v[4];
            const uint64_t* p = X + kWMlp + 4 * tid;
            if (!await(v, {p, p + 1, p + 2, p + 3}, true, deadline)) give_up();
            const float x[8] = {word_lo(v[0]), word_hi(v[0]), word_lo(v[1]), word_hi(v[1]),
                                word_lo(v[2]), word_hi(v[2]), word_lo(v[3]), word_hi(v[3])};
            quant8_store_lds(x, tid & 7, &L.xsc[tid >> 3], &L.xs[(tid >> 3) * 32]);
        }
        lds_barrier();
        if (L.fail) return;
        small_terms<kMaxNb>(L, L.small[t & 1], w, lane);
        lds_barrier();
        if (w == 0) small_sums<kMaxNb>(L, X + kWDown + kRowWords * sub, lane);
        ++t;
    }

    // the other set's words, for the launch after this one
    for (int i = g * kThreads + tid; i < a.clear_words; i += RT_CHAIN_WGS * kThreads) a.xch_clear[i] = kNotYet;
    // one workgroup finishes the hidden state (and the final norm)
    if (g != 0) return;
    add_words(a.xch + (size_t)(a.n - 1) * kWEnd + kWDown);
    if (tid < 256) *reinterpret_cast<float4*>(a.h_out + 4 * tid) = make_float4(h[0], h[1], h[2], h[3]);
    if (a.y_norm) {
        if (!norm_step(L, h, reinterpret_cast<const float4*>(a.final_w), a.eps, tid, lane, w)) return;
        if (tid < 256) *reinterpret_cast<float4*>(a.y_norm + 4 * tid) = *reinterpret_cast<const float4*>(&L.normed[4 * tid]);
    }
}

// Whether the device runs the chain's workgroups all at once.
bool rt_chain_fits() {
    static const bool fits = [] {
        int occ = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(rt_chain_kernel), kThreads + 64, 0) !=
            hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return occ >= 1 && bfp8_cu_count() >= RT_CHAIN_WGS;
    }();
    return fits;
}

hipError_t rt_launch_chain(const RtChainArgs& a, hipStream_t s) {
    if (!a.layers || a.n < 1 || a.n > RT_CHAIN_MAX_LAYERS || (!a.table && !a.h_in) || !a.h_out || !a.status || !a.xch ||
        a.xch == a.xch_clear || (a.y_norm && !a.final_w))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(rt_chain_kernel, dim3(RT_CHAIN_WGS), dim3(kThreads + 64), 0, s, a);
    return hipGetLastError();
}
