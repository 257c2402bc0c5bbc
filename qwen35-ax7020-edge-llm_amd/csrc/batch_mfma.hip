// batch_mfma.hip -- the batched BFP8 GEMV (up to 16 activation vectors against
// one weight matrix, weights read once) on the matrix cores, f32 flush-to-zero
// like the reference's Advanced SIMD epilogue.
//
// The reference has no batched GEMV: a batch is B calls of bfp8_gemv
// (04/qwen_kernels_opt.c:207-278), each keeping four int32 residue lanes per
// row and block (elements k = q mod 4), S_q = sum of mantissa * xq, and a
// float epilogue per block  fs_q += (float(S_q) * 2^(e-134)) * xscale,
// y = (fs_0 + fs_2) + (fs_1 + fs_3).
//
// Integer part on v_mfma_i32_32x32x16_i8, whose K of 16 is exactly the 16
// elements of one residue of one block.  With xq = 256*xh + xl (xh, xl int8,
// bfp8_layout.h) one MFMA computes, for 32 weight rows and residue q,
//   D[(v, p)][row] = sum over the residue's 16 elements of x_p[v] * m[row]
// for the 16 vectors v and both parts p (h, l) as its 32 rows: the A operand
// is the batch's split activations, the B operand the weight plane's
// residue-q slice.  A lane of D holds column `row` and rows 8(i/4) + 4(l/32)
// + i%4 (i < 16), so its registers i and i + 8 are the h and l sums of the same
// vector: S_q = 256 * D[i] + D[i + 8] exactly, in the lane, for 8 vectors.
// Integer sums are exact in any order.
//
// Float part, per (row, vector, block, residue), in the reference's order:
// float(S_q) * es * xs with es = 2^(e-134) a power of two.  float(S_q) * es is
// exact whenever it is a normal float (e in 8..236: |S_q| <= 2^25), so the two
// products round once, on S_q * es * xs.  When c = es * xs is itself a normal
// float it is exact too, and float(S_q) * c rounds the same real number: one
// product instead of two.  Each block checks that c is normal for every
// vector of the batch (a range of e computed from the batch's block scales)
// and takes the two products otherwise; e < 8 (es = 0) and zero, infinite or
// NaN scales give the same result either way.
//
// Work split, by what batch_form at the end picks for the sizes: a workgroup of 16
// wavefronts per 32-row half and group of vectors, a wavefront per residue and
// quarter of the blocks (bfp8_gemv_batch_span_kernel); a workgroup per tile, a
// wavefront per half and two residues, or per half, a wavefront per residue
// (bfp8_gemv_batch_mfma_kernel); a workgroup per four tiles, a wavefront per half
// with all 4 residues (bfp8_gemv_batch_cu_kernel); for two vectors also without
// the matrix cores (bfp8_gemv_batch_dot_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfp8_internal.h"
#include "bfp8_layout.h"
#include "gemv_dev.h"

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMfVec = 16;   // vectors (the MFMA's rows are vector x part)
constexpr int kMfGroup = 2;  // blocks per weight-load group

// CH: blocks of split activations staged in LDS at a time (16: the whole K in
// one staging; 8: half the LDS and the staging registers, for the kernel whose
// occupancy they limit).
template <int CH>
struct MfLds {
    // A operands: [block][residue][k half][part][vector], 8 bytes each: the
    // 64 lanes of one (block, residue) read 512 contiguous bytes
    uint64_t xa[CH][4][64];
    float xs[CH][kMfVec];      // [block][vector] block scales
    int lo[CH], hi[CH];        // per block: e range of the one-product epilogue
    // the end's exchange: 3 residue groups x 2 halves x 8 values x 64 lanes at most
    static_assert(CH * 4 * 64 * sizeof(uint64_t) >= 3 * 2 * 8 * 64 * sizeof(float),
                  "the fs exchange fits in the staging area");
};

// Staging of blocks c0 .. c0+nbc-1 of the B split activations and scales
// (vectors >= B and blocks >= nbc as zeros) into LDS, with each block's
// exponent range [lo, hi] inside which es * xs is a normal float for every
// normal scale xs of the batch: biased exponent of es * xs = e - 134 + E(xs),
// normal for 1..254, and e <= 236 keeps float(S) * es finite.  In two halves
// so that a caller can issue other loads between them: mf_stage_load issues
// every load of the NT threads (one round trip to L2 for all of them),
// mf_stage_store waits for them, writes LDS and synchronizes the workgroup.
template <int NT, int CH>
struct MfStaged {
    static constexpr int kItems = CH * 4 * 2 * kMfVec;  // 16-byte pieces of split activations
    static constexpr int kScales = CH * kMfVec;
    static_assert(kItems % NT == 0, "whole staging rounds");
    static constexpr int kScaleRounds = (kScales + NT - 1) / NT;
    u32x4 val[kItems / NT];
    float xs[kScaleRounds];
};

// 16 bytes of xsplit = one part of one residue (both k halves): item
// ((u * 4 + q) * 2 + p) * 16 + v, vectors fastest, so the LDS stores of
// consecutive threads are consecutive
// kVH: -1 every vector, else only vectors 8 kVH .. 8 kVH + 7 (the others
// staged as zeros: their MFMA rows are computed and not used).
template <int NT, int kVH, int CH>
__device__ __forceinline__ void mf_stage_load(MfStaged<NT, CH>& S, const uint32_t* __restrict__ xsplit,
                                              const float* __restrict__ xscale, int nb, int B, int c0, int nbc) {
#pragma unroll
    for (int j = 0; j < MfStaged<NT, CH>::kItems / NT; ++j) {
        const int i = threadIdx.x + j * NT;
        const int v = i % kMfVec, p = (i / kMfVec) % 2, q = (i / (2 * kMfVec)) % 4, u = i / (8 * kMfVec);
        S.val[j] = u32x4{0u, 0u, 0u, 0u};
        if (v < B && (kVH < 0 || (v >> 3) == kVH) && u < nbc)
            S.val[j] = *reinterpret_cast<const u32x4*>(
                xsplit + ((size_t)v * nb + c0 + u) * BFP8_XSPLIT_WORDS_PER_BLOCK + q * 8 + p * 4);
    }
#pragma unroll
    for (int j = 0; j < MfStaged<NT, CH>::kScaleRounds; ++j) {
        const int i = threadIdx.x + j * NT, v = i % kMfVec, u = i / kMfVec;
        S.xs[j] = (i < MfStaged<NT, CH>::kScales && v < B && (kVH < 0 || (v >> 3) == kVH) && u < nbc) ? xscale[(size_t)v * nb + c0 + u]
                                                                                        : 0.0f;
    }
}

template <int NT, int CH, bool kSync = true>
__device__ __forceinline__ void mf_stage_store(MfLds<CH>& L, const MfStaged<NT, CH>& S) {
#pragma unroll
    for (int j = 0; j < MfStaged<NT, CH>::kItems / NT; ++j) {
        const int i = threadIdx.x + j * NT;
        const int v = i % kMfVec, p = (i / kMfVec) % 2, q = (i / (2 * kMfVec)) % 4, u = i / (8 * kMfVec);
        L.xa[u][q][p * 16 + v] = ((uint64_t)S.val[j].y << 32) | S.val[j].x;       // k half 0: bytes 0..7
        L.xa[u][q][32 + p * 16 + v] = ((uint64_t)S.val[j].w << 32) | S.val[j].z;  // k half 1: bytes 8..15
    }
#pragma unroll
    for (int j = 0; j < MfStaged<NT, CH>::kScaleRounds; ++j) {
        const int i = threadIdx.x + j * NT;
        if (i < MfStaged<NT, CH>::kScales) {  // whole wavefronts (a multiple of 64)
            const int v = i % kMfVec, u = i / kMfVec;
            const float xs = S.xs[j];
            L.xs[u][v] = xs;
            const int E = (int)((__float_as_uint(xs) >> 23) & 0xffu);
            const bool normal = E >= 1 && E <= 254;
            int emin = normal ? E : 255, emax = normal ? E : 0;
#pragma unroll
            for (int m = 1; m < kMfVec; m <<= 1) {  // over the 16 lanes of block u
                emin = min(emin, __shfl_xor(emin, m, 64));
                emax = max(emax, __shfl_xor(emax, m, 64));
            }
            if (v == 0) {
                L.lo[u] = 135 - emin;
                L.hi[u] = min(236, 388 - emax);
            }
        }
    }
    if (kSync) __syncthreads();
}

// A lane's result slots: register i of the MFMA result (and i + 8, the low
// parts) is vector 8(i/4) + 4*kh + i%4 of the lane's row; every vector: slots
// i = 0..7; vector half kVH: slots i = 4 kVH .. 4 kVH + 3.
template <int kVH>
struct MfSlots {
    static constexpr int n = kVH < 0 ? 8 : 4;
    static constexpr int i0 = kVH < 0 ? 0 : 4 * kVH;
};

template <int kRes, int kVH>
struct MfState {
    float fs[kRes][MfSlots<kVH>::n];  // [residue of the group][slot]
};

template <int kRes>
struct MfLoads {
    uint64_t w[kMfGroup][kRes];  // [block][residue of the group]
    uint32_t e;
};

// One block: an MFMA per residue of the group and the epilogue.
template <int kRes, int kVH, int CH>
__device__ __forceinline__ void mf_block(MfState<kRes, kVH>& st, const MfLds<CH>& L, const uint64_t (&w)[kRes], uint32_t e,
                                         int u, int q0, int lane) {
    constexpr int NS = MfSlots<kVH>::n, I0 = MfSlots<kVH>::i0;
    i32x16 d[kRes];
    const i32x16 zero = {};
#pragma unroll
    for (int r = 0; r < kRes; ++r)
        d[r] = __builtin_amdgcn_mfma_i32_32x32x16_i8((long)L.xa[u][q0 + r][lane], (long)w[r], zero, 0, 0, 0);
    const int kh = lane >> 5;
    float xs[NS];
#pragma unroll
    for (int h = 0; h < NS / 4; ++h) {  // slots 4h..4h+3: vectors 8 (I0 / 4 + h) + 4 kh ..
        const f32x4 x4 = *reinterpret_cast<const f32x4*>(&L.xs[u][8 * (I0 / 4 + h) + 4 * kh]);
#pragma unroll
        for (int m = 0; m < 4; ++m) xs[4 * h + m] = x4[m];
    }
    const float es = exp_scale_ftz(e);
    const int lo = L.lo[u], hi = L.hi[u];
    const bool one_product = (e < 8u) | ((uint32_t)((int)e - lo) <= (uint32_t)(hi - lo));
    if (__builtin_amdgcn_ballot_w64(!one_product) == 0) {
        float c[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) c[k] = es * xs[k];
#pragma unroll
        for (int r = 0; r < kRes; ++r)
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int S = (int)((uint32_t)d[r][I0 + k] << 8) + d[r][I0 + k + 8];
                st.fs[r][k] = st.fs[r][k] + (float)S * c[k];
            }
    } else {
#pragma unroll
        for (int r = 0; r < kRes; ++r)
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int S = (int)((uint32_t)d[r][I0 + k] << 8) + d[r][I0 + k + 8];
                const float t1 = (float)S * es;
                st.fs[r][k] = st.fs[r][k] + t1 * xs[k];
            }
    }
}

// Weights of group gi (blocks kMfGroup*gi ..) for the lane's row, k half and
// the group's residues, and the row's exponent dword holding them (4 blocks
// per dword).  The whole offset goes in the per-lane offset, which the buffer
// range check covers: groups past the tile read zeros without touching memory.
static_assert(4 % kMfGroup == 0, "a group's exponents share one dword");
template <int kRes>
__device__ __forceinline__ void mf_issue(MfLoads<kRes>& ld, __amdgpu_buffer_rsrc_t wrs, __amdgpu_buffer_rsrc_t ers, int wv,
                                         int ev, int gi) {
#pragma unroll
    for (int uu = 0; uu < kMfGroup; ++uu)
#pragma unroll
        for (int r = 0; r < kRes; ++r) {
            const u32x2 v = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_raw_buffer_load_b64(wrs, wv + (gi * kMfGroup + uu) * 4096 + r * 1024, 0,
                                                            kNonTemporal));
            ld.w[uu][r] = ((uint64_t)v.y << 32) | v.x;
        }
    ld.e = load_e(ers, ev + (gi * kMfGroup / 4) * 256, 0);
}

template <int kRes, int NT, int kVH, int CH>
__device__ __forceinline__ void mf_group(MfState<kRes, kVH>& st, MfLds<CH>& L, const MfLoads<kRes>& ld, int gi, int nb,
                                         const uint32_t* __restrict__ xsplit, const float* __restrict__ xscale, int B,
                                         int q0, int lane) {
    const int b0 = gi * kMfGroup;
    if (b0 % CH == 0 && b0 > 0) {  // the first chunk is staged before the loop
        __syncthreads();  // every wavefront is done with the previous chunk
        MfStaged<NT, CH> S;
        mf_stage_load<NT, kVH, CH>(S, xsplit, xscale, nb, B, b0, min(CH, nb - b0));
        mf_stage_store<NT, CH>(L, S);
    }
#pragma unroll
    for (int uu = 0; uu < kMfGroup; ++uu) {
        if (b0 + uu >= nb) break;
        mf_block<kRes, kVH, CH>(st, L, ld.w[uu], (ld.e >> (8 * ((b0 + uu) & 3))) & 0xffu, (b0 + uu) % CH, q0, lane);
    }
}

// The work of one workgroup: tile t, its 32-row half s (kHalves == 1) or both
// (kHalves == 2, wavefront w takes half w & 1), the residues of group grp,
// the vectors of kVH (every vector, or one half of them).
// kDepth: weight-load groups in flight per wavefront (2: one group computed
// while the next loads; CH / kMfGroup: a chunk's every weight load issued at
// once, for GEMVs with too few tiles to fill the memory system otherwise).
template <int kRes, int kHalves, int kDepth, int kVH, int CH>
__device__ __forceinline__ void mf_body(MfLds<CH>& L, float* __restrict__ Y, const uint32_t* __restrict__ xsplit,
                                        const float* __restrict__ xscale, const uint8_t* __restrict__ mant,
                                        const uint8_t* __restrict__ exps, int M, int K, int B, int t, int s, int grp) {
    constexpr int NS = MfSlots<kVH>::n, I0 = MfSlots<kVH>::i0;
    const int lane = threadIdx.x & 63;
    const int q0 = grp * kRes;
    const int col = lane & 31, kh = lane >> 5;
    const int nb = K >> 6, nb4 = (nb + 3) >> 2;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mant + (size_t)t * nb * 4096u, (uint32_t)nb * 4096u);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)t * nb4 * 256u, (uint32_t)nb4 * 256u);
    const int wv = q0 * 1024 + (32 * s + col) * 16 + kh * 8;
    const int ev = (32 * s + col) * 4;
    MfState<kRes, kVH> st;
#pragma unroll
    for (int r = 0; r < kRes; ++r)
#pragma unroll
        for (int k = 0; k < NS; ++k) st.fs[r][k] = 0.0f;
    const int ng = (nb + kMfGroup - 1) / kMfGroup;
    // the first chunk's activation loads go out first, then the first
    // weight groups: the staging then waits for its own loads only (a
    // wavefront's loads complete in the order issued)
    constexpr int NT = 64 * kHalves * (4 / kRes);
    MfStaged<NT, CH> S0;
    mf_stage_load<NT, kVH, CH>(S0, xsplit, xscale, nb, B, 0, min(CH, nb));
    MfLoads<kRes> ld[kDepth];
#pragma unroll
    for (int d = 0; d < kDepth; ++d) mf_issue<kRes>(ld[d], wrs, ers, wv, ev, d);
    mf_stage_store<NT, CH>(L, S0);
    for (int gi = 0; gi < ng; gi += kDepth) {
        // kDepth load sets in turn: set d holds group gi + d, then gi + d + kDepth
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            if (gi + d < ng) mf_group<kRes, NT, kVH, CH>(st, L, ld[d], gi + d, nb, xsplit, xscale, B, q0, lane);
            mf_issue<kRes>(ld[d], wrs, ers, wv, ev, gi + d + kDepth);
        }
    }
    float (&fs)[kRes][NS] = st.fs;

    // y = (fs_0 + fs_2) + (fs_1 + fs_3): the other residue groups of the half
    // hand their sums to group 0 through the (no longer needed) staging area
    __syncthreads();
    float* xch = reinterpret_cast<float*>(&L.xa[0][0][0]);  // [group - 1][half][residue][slot][lane]
    if (grp > 0) {
#pragma unroll
        for (int r = 0; r < kRes; ++r)
#pragma unroll
            for (int k = 0; k < NS; ++k) xch[((((grp - 1) * 2 + s) * kRes + r) * NS + k) * 64 + lane] = fs[r][k];
    }
    __syncthreads();
    if (grp == 0) {
        const int row = t * 64 + 32 * s + col;
        const int pair_rows = M & ~1;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            float f[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gq = q / kRes, rq = q % kRes;
                f[q] = gq == 0 ? fs[rq][k] : xch[((((gq - 1) * 2 + s) * kRes + rq) * NS + k) * 64 + lane];
            }
            const int i = I0 + k;
            const int v = 8 * (i / 4) + 4 * kh + (i % 4);
            const float y = (f[0] + f[2]) + (f[1] + f[3]);
            if (v < B && row < pair_rows) Y[(size_t)v * M + row] = y;
        }
    }
}

// ---- many tiles, K <= 1024: a workgroup per CU's four tiles ------------------
// Eight wavefronts, two per SIMD; wavefront w takes tile 4 * blockIdx + w / 2,
// its 32-row half w % 2, and all four residues, so that the per-block work
// (exponent, one-product check, the eight scale products) is shared by 32
// values per lane.  Its weights are 8 VGPRs per block (four residue slices,
// 8 bytes per lane), loaded kAhead blocks ahead.  The batch's split
// activations and scales of every block are staged into LDS once, by the
// eight wavefronts together.  The staging's loads go out first, then the row
// exponents, then the first blocks' weights: a wavefront's vector loads
// complete in issue order, so the L2-resident staging never waits behind the
// HBM round trip, and the weights are in flight during the LDS stores.
// The two wavefronts of a SIMD run different tiles; the one issued first
// would win every issue slot and leave the other to finish alone, so each
// wavefront lowers its priority as it progresses (s_setprio 3 .. 0 over the
// blocks): the one behind is served first.
// Up to eight vectors finish four of the eight result slots per lane (NS = 4):
// 65536 x 1024, B = 4 17.3 us (a dot-product kernel) -> 12.2 (NS = 8) -> 11.6.
constexpr int kCuWaves = 8;
constexpr int kCuMaxNb = 16;

template <int NS>
struct CuOps {
    uint64_t a[4];    // MFMA A operands (split activations) per residue
    f32x4 x[NS / 4];  // block scales of the lane's slots 0..3 (and 4..7)
    int lo, hi;     // the block's one-product exponent range
};

// The epilogue of one block for the four residues (as mf_block's)
template <int NS>
__device__ __forceinline__ void cu_epilogue(float (&fs)[4][NS], const i32x16 (&d)[4], const CuOps<NS>& o, uint32_t e) {
    float xs[NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) xs[m] = o.x[m / 4][m % 4];
    const float es = exp_scale_ftz(e);
    const bool one_product = (e < 8u) | ((uint32_t)((int)e - o.lo) <= (uint32_t)(o.hi - o.lo));
    if (__builtin_amdgcn_ballot_w64(!one_product) == 0) {
        float c[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) c[k] = es * xs[k];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int S = (int)((uint32_t)d[r][k] << 8) + d[r][k + 8];
                fs[r][k] = fs[r][k] + (float)S * c[k];
            }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int S = (int)((uint32_t)d[r][k] << 8) + d[r][k + 8];
                const float t1 = (float)S * es;
                fs[r][k] = fs[r][k] + t1 * xs[k];
            }
    }
}

// s_setprio takes an immediate: level 3 for blocks 0..4, 2 for 5..9, 1 for
// 10..14, 0 after
__device__ __forceinline__ void cu_priority(int u) {
    const int level = u / 5;
    if (level == 0)
        __builtin_amdgcn_s_setprio(3);
    else if (level == 1)
        __builtin_amdgcn_s_setprio(2);
    else if (level == 2)
        __builtin_amdgcn_s_setprio(1);
    else
        __builtin_amdgcn_s_setprio(0);
}

template <int kAhead, int NS>
__global__ __launch_bounds__(64 * kCuWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void
bfp8_gemv_batch_cu_kernel(float* __restrict__ Y, const uint32_t* __restrict__ xsplit, const float* __restrict__ xscale,
                          const uint8_t* __restrict__ mant, const uint8_t* __restrict__ exps, int M, int K, int B) {
    static_assert(kAhead >= 1 && kAhead <= kCuMaxNb, "blocks in flight");
    __shared__ MfLds<kCuMaxNb> L;
    constexpr int NT = 64 * kCuWaves;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, col = lane & 31, kh = lane >> 5;
    const int nb = K >> 6, nb4 = (nb + 3) >> 2;  // nb <= kCuMaxNb (host-checked)
    const int t = (int)blockIdx.x * (kCuWaves / 2) + (w >> 1), s = w & 1;
    const bool live = t < bfp8_ntiles(M);  // the last workgroup may hold fewer tiles
    const int tt = live ? t : 0;
    // the staging's loads first (from L2), then the row's exponents and the
    // weights (from HBM): a wavefront's loads complete in issue order, so the
    // staging then waits for its own round trip only
    MfStaged<NT, kCuMaxNb> S0;
    mf_stage_load<NT, NS == 4 ? 0 : -1, kCuMaxNb>(S0, xsplit, xscale, nb, B, 0, nb);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)tt * nb4 * 256u, (uint32_t)nb4 * 256u);
    uint32_t ev[kCuMaxNb / 4];
#pragma unroll
    for (int g = 0; g < kCuMaxNb / 4; ++g) ev[g] = load_e(ers, (32 * s + col) * 4 + g * 256, 0);
    // residue q of block b for the lane's row and k half, through a buffer
    // range starting at the block (the lane offset stays fixed); blocks past
    // the tile, and wavefronts without a tile, have an empty range and read
    // zeros without touching memory
    const int wv = (32 * s + col) * 16 + kh * 8;
    uint64_t wq[kCuMaxNb][4];
    auto issue = [&](int b) {
        const __amdgpu_buffer_rsrc_t rs =
            make_rsrc(mant + ((size_t)tt * nb + b) * 4096u, live && b < nb ? (uint32_t)(nb - b) * 4096u : 0u);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x2 v =
                __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, wv + q * 1024, 0, kNonTemporal));
            wq[b][q] = ((uint64_t)v.y << 32) | v.x;
        }
    };
#pragma unroll
    for (int b = 0; b < kAhead; ++b) issue(b);
    mf_stage_store<NT, kCuMaxNb, false>(L, S0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the staging is in LDS; the weight loads stay in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (!live) return;

    float fs[4][NS];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < NS; ++k) fs[r][k] = 0.0f;
    const i32x16 zero = {};
    // block u's LDS operands are read behind block u - 1's MFMAs
    auto ops = [&](CuOps<NS>& o, int u) {
#pragma unroll
        for (int q = 0; q < 4; ++q) o.a[q] = L.xa[u][q][lane];
#pragma unroll
        for (int h = 0; h < NS / 4; ++h) o.x[h] = *reinterpret_cast<const f32x4*>(&L.xs[u][8 * h + 4 * kh]);
        o.lo = L.lo[u];
        o.hi = L.hi[u];
    };
    CuOps<NS> o[2];
    ops(o[0], 0);
#pragma unroll
    for (int u = 0; u < kCuMaxNb; ++u) {
        if (u + kAhead < kCuMaxNb) issue(u + kAhead);
        if (u >= nb) continue;  // (uniform; the loads above read nothing past the tile)
        cu_priority(u);
        i32x16 d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            d[r] = __builtin_amdgcn_mfma_i32_32x32x16_i8((long)o[u & 1].a[r], (long)wq[u][r], zero, 0, 0, 0);
        if (u + 1 < kCuMaxNb && u + 1 < nb) ops(o[(u + 1) & 1], u + 1);
        __builtin_amdgcn_sched_barrier(0);
        cu_epilogue(fs, d, o[u & 1], (ev[u >> 2] >> (8 * (u & 3))) & 0xffu);
    }

    // non-temporal stores: every wavefront writes its 2 KiB at its end, and
    // these leave the launch's last write burst sooner
    const int row = t * 64 + 32 * s + col;
    const int pair_rows = M & ~1;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int v = 8 * (k / 4) + 4 * kh + (k % 4);
        const float y = (fs[0][k] + fs[2][k]) + (fs[1][k] + fs[3][k]);
        if (v < B && row < pair_rows) __builtin_nontemporal_store(y, Y + (size_t)v * M + row);
    }
}

// ---- few tiles: a workgroup per 32-row half and group of vectors, each residue's
// blocks in four spans, one per wavefront ----------------------------------------
// Wavefront (q, j) computes residue q's terms of blocks jP .. jP + P - 1 (P =
// kP, a multiple of 4: whole exponent dwords) and keeps them in registers.  The
// in-order chain then visits the spans, j = 0 .. 3, one handing its sum to the
// next through LDS; with K <= 1024 (kP = 4) the sixteen terms of a sum go
// through LDS instead and wavefront (q, k) adds those of slot k, which needs
// two barriers instead of four (3584 x 1024, B = 16: 4.65 us against 4.82).
//
// Bound by latency (launch, the staging's round trip, the chain) and, with
// many vectors, by the epilogue's VALU work on the CUs that the launch
// reaches, so a workgroup takes few vectors when there are few tiles.  Result
// slot i < NS of a lane is MFMA row 4 * (lane / 32) + i: a workgroup of NS
// slots serves 2 NS vectors, and the MFMA rows of no slot read another
// vector's operand (their results are never used).
//
// Measured (us per call, back to back), against a dot-product kernel of four,
// two or one vectors per launch (B < 8) and a wavefront per residue and chain
// of all blocks (B >= 8, K > 1024) before: 2048 x 3584, B = 5 23.3 -> 7.0;
// 2048 x 3584, B = 16 15.7 -> 8.7; 3584 x 1024, B = 7 15.5 -> 3.9; 16384 x 1024,
// B = 4 8.7 -> 5.0; 16384 x 1024, B = 16 13.4 -> 9.4.
constexpr int kSpanMaxNb = 64;
template <int NS, int kP>
struct SpanLds {
    static constexpr int kV = 2 * NS, kNb = 4 * kP;
    // A operands: [block][residue][k half][part][vector], 8 bytes each
    __attribute__((aligned(16))) uint64_t xa[kNb][4][2][2][kV];
    __attribute__((aligned(16))) float xs[kNb][kV];  // [block][vector] block scales
    int2 range[kNb];            // per block: e range of the one-product epilogue
    float chain[4][NS][64];     // [residue][slot][lane]: a span's sums for the next; at the end fs_q
    float terms[4][NS][kP == 4 ? kNb : 1][64];  // kP = 4: [residue][slot][block][lane]
};

template <int NS, int kP>
__global__ __launch_bounds__(64 * 16) void bfp8_gemv_batch_span_kernel(
    float* __restrict__ Y, const uint32_t* __restrict__ xsplit, const float* __restrict__ xscale,
    const uint8_t* __restrict__ mant, const uint8_t* __restrict__ exps, int M, int K, int B, int ngroups) {
    using Lds = SpanLds<NS, kP>;
    constexpr int kV = Lds::kV, kNb = Lds::kNb, NT = 64 * 16;
    constexpr bool kExchange = kP == 4;
    __shared__ Lds L;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, kh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = w & 3, j = w >> 2;
    // the ngroups workgroups of a unit (tile, 32-row half) on one XCD (blocks
    // go to the 8 XCDs in turn): the first reads the weights, the rest find
    // them in that L2
    const int a = (int)blockIdx.x / (8 * ngroups), ar = (int)blockIdx.x % (8 * ngroups);
    const int unit = 8 * a + (ar & 7), v0 = (ar >> 3) * kV;
    if (unit >= 2 * bfp8_ntiles(M)) return;  // the whole workgroup: no barrier is left waiting
    const int t = unit >> 1, s = unit & 1;
    const int nb = K >> 6, nb4 = (nb + 3) >> 2;  // nb <= kNb (host-checked)

    // the group's split activations and scales (from L2) go out before the
    // exponents and weights (loads complete in issue order); piece i = one
    // part of one residue of one block of one vector, 16 bytes
    constexpr int kItems = kNb * 8 * kV, kRounds = (kItems + NT - 1) / NT;
    u32x4 xv[kRounds];
#pragma unroll
    for (int n = 0; n < kRounds; ++n) {
        const int i = tid + n * NT;
        const int v = v0 + i % kV, rp = (i / kV) % 8, b = i / (8 * kV);
        xv[n] = u32x4{0u, 0u, 0u, 0u};
        if (v < B && b < nb)
            xv[n] = *reinterpret_cast<const u32x4*>(xsplit + ((size_t)v * nb + b) * BFP8_XSPLIT_WORDS_PER_BLOCK + rp * 4);
    }
    float xsv = 0.0f;  // scale tid: block tid / kV, vector tid % kV
    static_assert(kNb * kV <= NT, "one scale per thread");
    if (tid < kNb * kV && v0 + tid % kV < B && tid / kV < nb) xsv = xscale[(size_t)(v0 + tid % kV) * nb + tid / kV];
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(exps + (size_t)t * nb4 * 256u, (uint32_t)nb4 * 256u);
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mant + (size_t)t * nb * 4096u, (uint32_t)nb * 4096u);
    const int wv = q * 1024 + (32 * s + col) * 16 + kh * 8;
    uint32_t ev[kP / 4];
    uint64_t wq[kP];  // blocks past the tile read zeros without touching memory
#pragma unroll
    for (int g = 0; g < kP / 4; ++g) ev[g] = load_e(ers, (32 * s + col) * 4 + (j * (kP / 4) + g) * 256, 0);
#pragma unroll
    for (int i = 0; i < kP; ++i) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wrs, wv + (kP * j + i) * 4096, 0, 0));
        wq[i] = ((uint64_t)v.y << 32) | v.x;
    }
#pragma unroll
    for (int n = 0; n < kRounds; ++n) {
        const int i = tid + n * NT;
        const int v = i % kV, p = (i / kV) % 2, rq = (i / (2 * kV)) % 4, b = i / (8 * kV);
        if (kItems % NT == 0 || i < kItems) {
            L.xa[b][rq][0][p][v] = ((uint64_t)xv[n].y << 32) | xv[n].x;
            L.xa[b][rq][1][p][v] = ((uint64_t)xv[n].w << 32) | xv[n].z;
        }
    }
    if (tid < kNb * kV) {  // whole wavefronts, or whole groups of kV lanes
        const int E = (int)((__float_as_uint(xsv) >> 23) & 0xffu);
        const bool normal = E >= 1 && E <= 254;
        int emin = normal ? E : 255, emax = normal ? E : 0;
#pragma unroll
        for (int m = 1; m < kV; m <<= 1) {
            emin = min(emin, __shfl_xor(emin, m, 64));
            emax = max(emax, __shfl_xor(emax, m, 64));
        }
        L.xs[tid / kV][tid % kV] = xsv;
        if (tid % kV == 0) L.range[tid / kV] = make_int2(135 - emin, min(236, 388 - emax));
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the staging is in LDS; the weight loads stay in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    // the span's terms
    const int pa = col >> 4, va = ((col >> 2) & 1) * NS + min(col & 3, NS - 1);  // this lane's A row: part, vector
    const i32x16 zero = {};
    float tv[kP][NS];
#pragma unroll
    for (int i = 0; i < kP; ++i) {
        const int b = kP * j + i;
        const i32x16 d = __builtin_amdgcn_mfma_i32_32x32x16_i8((long)L.xa[b][q][kh][pa][va], (long)wq[i], zero, 0, 0, 0);
        float xs[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) xs[k] = L.xs[b][kh * NS + k];
        const int2 range = L.range[b];
        const uint32_t e = (ev[i >> 2] >> (8 * (i & 3))) & 0xffu;
        const float es = exp_scale_ftz(e);
        const bool one_product = (e < 8u) | ((uint32_t)((int)e - range.x) <= (uint32_t)(range.y - range.x));
        if (__builtin_amdgcn_ballot_w64(!one_product) == 0) {
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const float c = es * xs[k];
                tv[i][k] = (float)((int)((uint32_t)d[k] << 8) + d[k + 8]) * c;
            }
        } else {
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const float t1 = (float)((int)((uint32_t)d[k] << 8) + d[k + 8]) * es;
                tv[i][k] = t1 * xs[k];
            }
        }
    }

    // the in-order chain (blocks past nb are in no sum)
    if constexpr (kExchange) {
#pragma unroll
        for (int i = 0; i < kP; ++i)
#pragma unroll
            for (int k = 0; k < NS; ++k) L.terms[q][k][kP * j + i][lane] = tv[i][k];
        __syncthreads();
        if (j < NS) {  // slot j of residue q
            float t[kNb], fs = 0.0f;
#pragma unroll
            for (int b = 0; b < kNb; ++b) t[b] = L.terms[q][j][b][lane];
#pragma unroll
            for (int b = 0; b < kNb; ++b)
                if (b < nb) fs = fs + t[b];
            L.chain[q][j][lane] = fs;
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int turn = 0; turn < 4; ++turn) {
            if (j == turn) {
                float fs[NS];
#pragma unroll
                for (int k = 0; k < NS; ++k) fs[k] = turn ? L.chain[q][k][lane] : 0.0f;
#pragma unroll
                for (int i = 0; i < kP; ++i) {
                    if (kP * turn + i < nb) {
#pragma unroll
                        for (int k = 0; k < NS; ++k) fs[k] = fs[k] + tv[i][k];
                    }
                }
#pragma unroll
                for (int k = 0; k < NS; ++k) L.chain[q][k][lane] = fs[k];
            }
            __syncthreads();
        }
    }
    if (w < NS) {  // wavefront w: slot w, y = (fs_0 + fs_2) + (fs_1 + fs_3)
        const float y = (L.chain[0][w][lane] + L.chain[2][w][lane]) + (L.chain[1][w][lane] + L.chain[3][w][lane]);
        const int row = t * 64 + 32 * s + col, v = v0 + kh * NS + w;
        if (v < B && row < (M & ~1)) __builtin_nontemporal_store(y, Y + (size_t)v * M + row);
    }
}

template <int NS>
hipError_t launch_span(float* Y, const uint32_t* xsplit, const float* xscale, const uint8_t* mant, const uint8_t* exps,
                       int M, int K, int B, hipStream_t s) {
    const int groups = (B + 2 * NS - 1) / (2 * NS);
    const dim3 grid(8 * groups * ((2 * bfp8_ntiles(M) + 7) / 8)), block(64 * 16);
    switch (((K >> 6) + 15) / 16) {
        case 1: hipLaunchKernelGGL((bfp8_gemv_batch_span_kernel<NS, 4>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B, groups); break;
        case 2: hipLaunchKernelGGL((bfp8_gemv_batch_span_kernel<NS, 8>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B, groups); break;
        case 3: hipLaunchKernelGGL((bfp8_gemv_batch_span_kernel<NS, 12>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B, groups); break;
        case 4: hipLaunchKernelGGL((bfp8_gemv_batch_span_kernel<NS, 16>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B, groups); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---- a workgroup per tile, or per 32-row half of one --------------------------------
// kHalves: halves of a tile per workgroup (2: both, workgroup per tile; 1:
// workgroup per 32-row half, twice the workgroups for GEMVs with few tiles).
// kSplit: 1, every vector in each workgroup; 2, a workgroup per half of the
// vectors, each wavefront then finishing 4 of the 8 result slots of its
// lanes -- half the epilogue per wavefront, on twice the wavefronts, for
// GEMVs whose wavefronts are too few to hide the epilogue's latencies.  The
// two workgroups of a unit are blocks 16a + x and 16a + 8 + x (x < 8), which
// go to the same XCD (blocks are dealt to the 8 XCDs in turn), so the second
// reads the unit's weights from that XCD's L2; unit 8a + x, blocks past the
// last unit exit at once.
template <int kRes, int kHalves, int kDepth, int kSplit, int CH>
__global__ __launch_bounds__(64 * kHalves * (4 / kRes)) __attribute__((amdgpu_waves_per_eu(kSplit == 2 ? 2 : 4))) void
bfp8_gemv_batch_mfma_kernel(float* __restrict__ Y, const uint32_t* __restrict__ xsplit,
                            const float* __restrict__ xscale, const uint8_t* __restrict__ mant,
                            const uint8_t* __restrict__ exps, int M, int K, int B) {
    __shared__ MfLds<CH> L;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int b = (int)blockIdx.x;
    const int bid = kSplit == 2 ? 8 * (b >> 4) + (b & 7) : b;
    const int nunits = kHalves == 2 ? bfp8_ntiles(M) : 2 * bfp8_ntiles(M);
    if (kSplit == 2 && bid >= nunits) return;  // the grid's last 16 blocks may hold fewer units
    // 32-row half, residue group, tile
    const int s = kHalves == 2 ? (w & 1) : (bid & 1), grp = kHalves == 2 ? (w >> 1) : w;
    const int t = kHalves == 2 ? bid : (bid >> 1);
    if (kSplit == 1)
        mf_body<kRes, kHalves, kDepth, -1, CH>(L, Y, xsplit, xscale, mant, exps, M, K, B, t, s, grp);
    else if (((b >> 3) & 1) == 0)
        mf_body<kRes, kHalves, kDepth, 0, CH>(L, Y, xsplit, xscale, mant, exps, M, K, B, t, s, grp);
    else
        mf_body<kRes, kHalves, kDepth, 1, CH>(L, Y, xsplit, xscale, mant, exps, M, K, B, t, s, grp);
}

// ---- two vectors (four with K <= 128), many tiles: dot products ------------------
// A workgroup per tile, wavefront = residue, lane = row: the residue sums by
// v_dot4_i32_i8.  Activations of a chunk of 8 blocks for all B vectors are
// staged in LDS (wave-uniform broadcast reads); each lane keeps B residue
// accumulators.  Its VALU work grows with B, and the matrix-core forms work for
// 8 or 16 vectors whatever B is, so it stands where two vectors (or few blocks)
// leave it the least to do: us by span / four tiles or one a workgroup / this,
// weights from HBM: 20480 x 256, B = 2 5.8 / 4.7 / 4.2; 32768 x 512, B = 2 7.7 /
// 6.3 / 6.3; 65536 x 1088, B = 2 21.5 / 17.2 / 16.3; 81920 x 128, B = 4 15.7 / 6.6 /
// 5.4.
constexpr int kBatchChunk = 8;  // blocks per LDS-staged step
template <int B>
__global__ __launch_bounds__(256) void bfp8_gemv_batch_dot_kernel(
    float* __restrict__ Y, const uint32_t* __restrict__ xsplit, const float* __restrict__ xscale,
    const uint8_t* __restrict__ mant, const uint8_t* __restrict__ exps, int M, int K) {
    __shared__ uint32_t xl[B * kBatchChunk * 32];
    __shared__ float xsl[B * kBatchChunk];  // the chunk's block scales (LDS, like the split words: no scalar loads,
                                            // whose out-of-order returns would make every LDS wait a full wait)
    float* red = reinterpret_cast<float*>(xl);  // the cross-wave sums reuse the staging space (4 * 64 * B floats)
    static_assert(kBatchChunk * 32 >= 4 * 64, "red fits in xl");
    const int q = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r = threadIdx.x & 63;
    const int t = blockIdx.x;
    const int nb = K >> 6;
    const int nb4 = (nb + 3) >> 2;
    const uint8_t* mtile = mant + (size_t)t * nb * 4096u;
    const uint8_t* etile = exps + (size_t)t * nb4 * 256u;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(mtile, (uint32_t)nb * 4096u);
    const __amdgpu_buffer_rsrc_t ers = make_rsrc(etile, (uint32_t)nb4 * 256u);
    const int wv = q * 1024 + r * 16;
    const int xwords = nb * 32;
    float fs[B];
#pragma unroll
    for (int v = 0; v < B; ++v) fs[v] = 0.0f;

    for (int b0 = 0; b0 < nb; b0 += kBatchChunk) {
        const int nbc = min(kBatchChunk, nb - b0);
        u32x4 w[kBatchChunk];
        uint32_t ew[kBatchChunk / 4] = {};
#pragma unroll
        for (int u = 0; u < kBatchChunk; ++u)
            if (u < nbc) w[u] = load_w(wrs, wv, (b0 + u) * 4096);
#pragma unroll
        for (int m = 0; m < kBatchChunk / 4; ++m)
            if (4 * m < nbc) ew[m] = load_e(ers, r * 4, ((b0 >> 2) + m) * 256);
        __syncthreads();  // previous chunk's LDS reads are done
        for (int i = threadIdx.x; i < B * nbc * 32; i += 256) {
            int v = i / (nbc * 32), o = i - v * nbc * 32;
            xl[v * kBatchChunk * 32 + o] = xsplit[(size_t)v * xwords + b0 * 32 + o];
        }
        for (int i = threadIdx.x; i < B * nbc; i += 256) {
            const int v = i / nbc, u = i - v * nbc;
            xsl[v * kBatchChunk + u] = xscale[(size_t)v * nb + b0 + u];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kBatchChunk; ++u) {
            if (u >= nbc) break;
            const uint32_t e = (ew[u >> 2] >> (8 * (u & 3))) & 0xffu;
            const float sc = exp_scale_ftz(e);
            // vectors in groups of four: the group's LDS reads go out together,
            // then its four dot-product chains interleave
            constexpr int kG = B < 4 ? B : 4;
#pragma unroll
            for (int v0 = 0; v0 < B; v0 += kG) {
                uint4 h[kG], l[kG];
                float xs[kG];
#pragma unroll
                for (int j = 0; j < kG; ++j) {
                    const uint32_t* xb = xl + ((v0 + j) * kBatchChunk + u) * 32 + q * 8;
                    h[j] = *reinterpret_cast<const uint4*>(xb);
                    l[j] = *reinterpret_cast<const uint4*>(xb + 4);
                    xs[j] = xsl[(v0 + j) * kBatchChunk + u];
                }
                int acc[kG];
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].x, (int)h[j].x, 0, false);
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].y, (int)h[j].y, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].z, (int)h[j].z, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].w, (int)h[j].w, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) {
                    acc[j] = (int)((uint32_t)acc[j] << 8);
                    acc[j] = __builtin_amdgcn_sdot4((int)w[u].x, (int)l[j].x, acc[j], false);
                }
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].y, (int)l[j].y, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].z, (int)l[j].z, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[j] = __builtin_amdgcn_sdot4((int)w[u].w, (int)l[j].w, acc[j], false);
#pragma unroll
                for (int j = 0; j < kG; ++j) {
                    const float t1 = (float)acc[j] * sc;
                    const float t2 = t1 * xs[j];
                    fs[v0 + j] = fs[v0 + j] + t2;
                }
            }
        }
    }
    __syncthreads();  // every wavefront is done with the staged activations
#pragma unroll
    for (int v = 0; v < B; ++v) red[(v * 4 + q) * 64 + r] = fs[v];
    __syncthreads();
    const int pair_rows = M & ~1;
    for (int i = threadIdx.x; i < B * 64; i += 256) {
        int v = i >> 6, rr = i & 63;
        int row = t * 64 + rr;
        const float* p = red + v * 256;
        float y = (p[rr] + p[128 + rr]) + (p[64 + rr] + p[192 + rr]);
        if (row < pair_rows) Y[(size_t)v * M + row] = y;
    }
}

// The form that a call takes.  One vector is a plain GEMV: 2.8 us against the span
// kernel's 3.4 at 3584 x 1024, 3.7 against 6.6 at 2048 x 3584, 11.7 against 12.2
// (a workgroup per four tiles) at 65536 x 1024.
//
// The span kernel's time goes up in steps of the workgroups that run at once (512,
// 256 with four slots) and with K rounded up to a multiple of 1024; the forms
// that read the weights once for all vectors cost more to start and then grow
// with the bytes.  The lines lie where the two cross, by the geometric mean of
// weights from HBM and weights from the cache (the span kernel is up to a
// quarter faster there: its weight loads are not non-temporal).  Each with both
// sides, us from HBM (from cache), lower side of the line first:
//   B <= 4, K <= 256: 128 tiles, B = 4 span 3.9, tile 4.1; 144 span 4.3 (4.4), tile 4.0 (4.1)
//   B = 2, K = 512: 256 span 4.7, dot 4.8; 320 span 6.0 (5.0), dot 5.6 (4.2); 1024 dot 9.2, four tiles 8.6
//   B = 4, K = 512: 256 span 4.9 (4.4), tile 5.1 (4.8); 400 span 7.8, tile 6.3; 640 tile 7.8, four tiles 7.4
//   B = 4, K = 1024: 512 span 9.6 (7.1), four tiles 9.2 (8.8); 576 10.9 (9.6), 9.5 (9.0)
//   B = 4, K = 768: 448 span 8.5 (6.8), four tiles 7.8 (7.5); 512 8.9 (7.0), 8.0 (7.6)
//   B = 2, K = 1088: 384 span 10.1 (7.4), dot 10.0 (9.3); 512 12.3 (9.5), 11.3 (10.1); 1024 21.5, 16.3
//   B = 4, K = 2048: 1024 span 27.9 (24.1), tile 27.4 (26.2); K = 2112: 832 tile 8 % faster, 1024 17 %
//   B = 8, K = 512: 128 span 4.2, tile 4.9; 144 6.9 (6.4), 5.0 (5.0); 512 tile 6.5, four tiles 7.2; 640 7.9, 7.5
//   B = 8, K = 768: 144 span 7.7, tile 7.0; 272 tile 8.4, four tiles 7.5
//   B = 8, K = 1024: 256 span 8.9 (7.2), four tiles 8.6 (8.3); 272 11.5 (9.8), 8.7 (8.4)
//   B = 8, K = 1088: 256 span 9.3, tile 9.6; 384 12.9 (10.5), 11.5 (11.1); 512 15.9, 11.9
//   B = 8, K = 3584: 320 span 26.8 (21.9), half 27.0 (26.3); 352 half 27.2, tile 30; 384 span 30.8, half 27.3;
//     448 half 33.2, tile 30.3
//   B = 16, K = 512: 64 span 4.0, tile 5.2; 128 6.9, 5.3; 1024 tile 10.1, four tiles 9.1
//   B = 16, K = 1024: 64 span 4.5; 128 span 8.1 (7.1), half 7.3 (6.7), tile 8.8; 192 tile 8.9, four tiles 11.0;
//     512 10.8, 11.2; 640 13.2, 11.4; 1088 tile 5 % faster, 1536 four tiles 10 %
//   B = 16, K = 1088: 128 span 8.7, tile 9.8; 160 11.5, 9.9; K = 2048: 256 span 16.5 (14.5), tile 16.4 (16.1);
//     384 22.9, 19.3
//   B = 16, K = 3584: 128 span 20.3 (18.0), half 19.0 (18.8); 192 span 28.1, half 23.0, tile 27.0; 224 half 33.9, tile 27.2
// (four tiles: bfp8_gemv_batch_cu_kernel; tile, half: bfp8_gemv_batch_mfma_kernel,
// whose half form runs 768 workgroups at once: 384 tiles, 192 above 8 vectors)
enum class BatchForm { kPlain, kDot, kSpan, kCu, kTile, kHalf };
BatchForm batch_form(int nt, int nb, int B) {
    if (B == 1) return BatchForm::kPlain;
    const int up = (nb + 15) & ~15, pad = up - nb;  // the span kernel's blocks, those past K
    if (nb <= kCuMaxNb) {
        const bool one_round = nt <= 1024;  // of the four-tile kernel
        if (nb <= 8) {
            if (nt <= (B > 8 ? 64 : B > 4 || (B > 2 && nb <= 4) ? 128 : 256)) return BatchForm::kSpan;
            if (nb > 4 && one_round && nt > (B == 2 || B > 8 ? 768 : 512)) return BatchForm::kCu;
            return B == 2 || (B == 4 && nb <= 2) ? BatchForm::kDot : BatchForm::kTile;
        }
        if (B <= 4) {
            if (nt < (nb <= 12 && B > 2 ? 480 : 544)) return BatchForm::kSpan;
            return B == 2 && !one_round && (nt < 1600 || nb <= 10) ? BatchForm::kDot : BatchForm::kCu;
        }
        if (B <= 8) return nt > 256 ? BatchForm::kCu : nt <= 128 || nb > 12 ? BatchForm::kSpan : BatchForm::kTile;
        if (nt <= 128) return nt <= 64 ? BatchForm::kSpan : BatchForm::kHalf;
        return nt <= 512 || (!one_round && nt <= 1280) ? BatchForm::kTile : BatchForm::kCu;
    }
    if (B <= 4) {
        if (nt * pad < 240 * up - 1100) return BatchForm::kSpan;
        return B == 2 ? BatchForm::kDot : BatchForm::kTile;
    }
    if (nb <= 32) {
        const int line = B <= 8 ? (pad >= 12 ? 340 : pad >= 6 ? 430 : pad >= 2 ? 520 : 900) : (pad >= 12 ? 128 : pad >= 6 ? 208 : 310);
        return nt <= line ? BatchForm::kSpan : BatchForm::kTile;
    }
    if (B <= 8) return nt <= 320 ? BatchForm::kSpan : nt <= 384 ? BatchForm::kHalf : BatchForm::kTile;
    if (B <= 12) return nt <= (nb <= 37 ? 176 : 208) ? BatchForm::kSpan : BatchForm::kTile;
    return nt <= (pad >= 8 ? 112 : 128) ? BatchForm::kSpan : nt <= 192 ? BatchForm::kHalf : BatchForm::kTile;
}

}  // namespace

const char* bfp8_batch_kernel_name(int M, int K, int B) {
    switch (batch_form(bfp8_ntiles(M), K >> 6, B)) {
        case BatchForm::kPlain: return bfp8_gemv_kernel_name(M, K);
        case BatchForm::kDot: return "bfp8_gemv_batch_dot_kernel";
        case BatchForm::kCu: return "bfp8_gemv_batch_cu_kernel";
        case BatchForm::kTile:
        case BatchForm::kHalf: return "bfp8_gemv_batch_mfma_kernel";
        default: return "bfp8_gemv_batch_span_kernel";
    }
}

hipError_t bfp8_launch_gemv_batch(float* Y, const uint32_t* xsplit, const float* xscale, const uint8_t* mant,
                                  const uint8_t* exps, int M, int K, int B, hipStream_t s) {
    const int nt = bfp8_ntiles(M);
    if (nt == 0) return hipSuccess;
    // a ragged K drops its last K % 64 elements, as every other GEMV path does
    // (nb = K / 64 blocks; the split activation's stride is nb blocks)
    if (B < 1 || B > kMfVec || K < 64 || K > 64 * kSpanMaxNb) return hipErrorInvalidValue;
    const int nb = K >> 6;
    switch (batch_form(nt, nb, B)) {
        case BatchForm::kPlain: {
            Bfp8GemvDesc d{};
            d.mant = mant;
            d.exps = exps;
            d.xsplit = xsplit;
            d.xscale = xscale;
            d.y = Y;
            d.M = M;
            d.K = K;
            d.pair_rows = M & ~1;
            return bfp8_launch_gemv(d, s);
        }
        case BatchForm::kCu: {
            const dim3 grid((nt + kCuWaves / 2 - 1) / (kCuWaves / 2)), block(64 * kCuWaves);
            if (B > 8)
                hipLaunchKernelGGL((bfp8_gemv_batch_cu_kernel<2, 8>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B);
            else
                hipLaunchKernelGGL((bfp8_gemv_batch_cu_kernel<2, 4>), grid, block, 0, s, Y, xsplit, xscale, mant, exps, M, K, B);
            return hipGetLastError();
        }
        case BatchForm::kDot:
            if (B == 2)
                hipLaunchKernelGGL(bfp8_gemv_batch_dot_kernel<2>, dim3(nt), dim3(256), 0, s, Y, xsplit, xscale, mant, exps, M, K);
            else
                hipLaunchKernelGGL(bfp8_gemv_batch_dot_kernel<4>, dim3(nt), dim3(256), 0, s, Y, xsplit, xscale, mant, exps, M, K);
            return hipGetLastError();
        case BatchForm::kTile:
            hipLaunchKernelGGL((bfp8_gemv_batch_mfma_kernel<2, 2, 2, 1, 8>), dim3(nt), dim3(256), 0, s, Y, xsplit, xscale,
                               mant, exps, M, K, B);
            return hipGetLastError();
        case BatchForm::kHalf:
            if (B > 8)  // a workgroup per half of the vectors too: 2 nt units, 16 blocks per 8
                hipLaunchKernelGGL((bfp8_gemv_batch_mfma_kernel<1, 1, 16 / kMfGroup, 2, 16>), dim3(16 * ((2 * nt + 7) / 8)),
                                   dim3(256), 0, s, Y, xsplit, xscale, mant, exps, M, K, B);
            else
                hipLaunchKernelGGL((bfp8_gemv_batch_mfma_kernel<1, 1, 16 / kMfGroup, 1, 16>), dim3(2 * nt), dim3(256), 0, s,
                                   Y, xsplit, xscale, mant, exps, M, K, B);
            return hipGetLastError();
        case BatchForm::kSpan: break;
    }
    // The fewest vectors per workgroup that still leave at most one workgroup
    // per CU; beyond that every vector in as few workgroups as hold them, but
    // with K > 2048 four at most (eight need 89 registers: one workgroup per CU
    // instead of two; 16384 x 3584, B = 16: 36.6 us against 33.5).
    const int units = 2 * nt, cus = bfp8_cu_count();
    int ns = 1;
    while (ns < 4 && units * ((B + 2 * ns - 1) / (2 * ns)) > cus) ns *= 2;
    if (units * ((B + 2 * ns - 1) / (2 * ns)) > cus) ns = B <= 2 ? 1 : (B <= 4 || nb > 32) ? 2 : 4;
    switch (ns) {
        case 1: return launch_span<1>(Y, xsplit, xscale, mant, exps, M, K, B, s);
        case 2: return launch_span<2>(Y, xsplit, xscale, mant, exps, M, K, B, s);
        default: return launch_span<4>(Y, xsplit, xscale, mant, exps, M, K, B, s);
    }
}
