// bfp8_ieee.hip -- kernels whose float arithmetic restates the reference's
// scalar (VFP) code, plus the integer-only kernels of the library.
//
// Compiled with IEEE f32 subnormals and -ffp-contract=off; every rounding
// step below is spelled with __fmul_rn / __fadd_rn / __fdiv_rn so that each
// C operation of the reference maps to one correctly rounded operation.
#include <hip/hip_runtime.h>

#include "bfp8_internal.h"
#include "quant_block.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---- activation quantizer, 04/qwen_kernels_opt.c:182-205 ------------------
// One wavefront per 64-element block (quant_block.h).
__device__ __forceinline__ void quantize_block(const Bfp8QuantDesc& d, int b) {
    const int nb = d.K >> 6;
    if (b >= nb) return;
    __shared__ uint32_t rec[32];
    const int i = threadIdx.x;
    bfp8_quant_block_wave(d.x[(size_t)b * 64 + i], i, d.xq ? d.xq + (size_t)b * 64 : nullptr, d.xscale + b,
                          d.xsplit + (size_t)b * 32, rec);
}

// Residue sum from a 16-byte residue chunk and the split activation record.
__device__ __forceinline__ int residue_sum_v(u32x4 w, const uint32_t* xb) {
    int acc = __builtin_amdgcn_sdot4((int)w.x, (int)xb[0], 0, false);
    acc = __builtin_amdgcn_sdot4((int)w.y, (int)xb[1], acc, false);
    acc = __builtin_amdgcn_sdot4((int)w.z, (int)xb[2], acc, false);
    acc = __builtin_amdgcn_sdot4((int)w.w, (int)xb[3], acc, false);
    acc = (int)((uint32_t)acc << 8);
    acc = __builtin_amdgcn_sdot4((int)w.x, (int)xb[4], acc, false);
    acc = __builtin_amdgcn_sdot4((int)w.y, (int)xb[5], acc, false);
    acc = __builtin_amdgcn_sdot4((int)w.z, (int)xb[6], acc, false);
    acc = __builtin_amdgcn_sdot4((int)w.w, (int)xb[7], acc, false);
    return acc;
}

__device__ __forceinline__ const u32x4* chunk_ptr(const uint8_t* mant, int nb, int row, int b, int q) {
    const int t = row >> 6, r = row & 63;
    return reinterpret_cast<const u32x4*>(mant + (((size_t)t * nb + b) * 4 + q) * 1024u + (size_t)r * 16u);
}

__device__ __forceinline__ uint32_t exp_byte(const uint8_t* exps, int nb, int row, int b) {
    const int t = row >> 6, r = row & 63, nb4 = (nb + 3) >> 2;
    return exps[(((size_t)t * nb4 + (b >> 2)) * 64 + r) * 4 + (b & 3)];
}

}  // namespace

extern "C" __global__ __launch_bounds__(64) void bfp8_quantize_kernel(const Bfp8QuantDesc* __restrict__ descs) {
    quantize_block(descs[blockIdx.y], blockIdx.x);
}

extern "C" __global__ __launch_bounds__(64) void bfp8_quantize1_kernel(Bfp8QuantDesc d) {
    quantize_block(d, blockIdx.x);
}

// ---- odd-M last row, 04/qwen_kernels_opt.c:279-306 ---------------------------
// Scalar VFP code: one int32 per block (lane sums added as integers), then
//   sum = sum + ((float(s) * EXP_SCALE[e]) * xscale[b])   in block order,
// IEEE subnormals (EXP_SCALE[e] is subnormal for e < 8).  K <= 4096 here.
extern "C" __global__ __launch_bounds__(64) void bfp8_tail_row_kernel(
    float* __restrict__ y, const uint32_t* __restrict__ xsplit, const float* __restrict__ xscale,
    const uint8_t* __restrict__ mant, const uint8_t* __restrict__ exps, int M, int K) {
    const int m = M - 1;
    const int nb = K >> 6;
    const int b = threadIdx.x;
    y += (size_t)blockIdx.x * M;  // a workgroup per activation
    xsplit += (size_t)blockIdx.x * nb * 32;
    xscale += (size_t)blockIdx.x * nb;
    __shared__ float prod[64];
    float p = 0.0f;
    if (b < nb) {
        int s = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) s += residue_sum_v(*chunk_ptr(mant, nb, m, b, q), xsplit + ((size_t)b * 4 + q) * 8);
        const float es = ldexpf(1.0f, (int)exp_byte(exps, nb, m, b) - 134);
        p = __fmul_rn(__fmul_rn((float)s, es), xscale[b]);
    }
    prod[b] = p;
    __syncthreads();
    if (b == 0) {
        float sum = 0.0f;
        for (int j = 0; j < nb; ++j) sum = __fadd_rn(sum, prod[j]);
        y[m] = sum;
    }
}

// ---- float path, 04/qwen_kernels_opt.c:311-325 (K > 4096 on the board) ------
// Unquantized x:  block_dot += (float)w * x  (64 sequential steps),
//                 sum += block_dot * EXP_SCALE[e]  (block order).
// One wavefront per row; lanes take blocks, lane 0 sums in order.
extern "C" __global__ __launch_bounds__(64) void bfp8_gemv_float_kernel(
    float* __restrict__ y, const float* __restrict__ x, const uint8_t* __restrict__ mant,
    const uint8_t* __restrict__ exps, int M, int K) {
    extern __shared__ float prods[];
    const int m = blockIdx.x;
    const int nb = K >> 6;
    for (int b = threadIdx.x; b < nb; b += 64) {
        u32x4 c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) c[q] = *chunk_ptr(mant, nb, m, b, q);
        const float* xb = x + (size_t)b * 64;
        float dot = 0.0f;
#pragma unroll
        for (int k = 0; k < 64; ++k) {
            // element k sits in residue chunk k&3, byte k>>2
            const int i = k >> 2;
            const uint32_t word = c[k & 3][i >> 2];
            const int w = (int)(int8_t)((word >> (8 * (i & 3))) & 0xffu);
            dot = __fadd_rn(dot, __fmul_rn((float)w, xb[k]));
        }
        const float es = ldexpf(1.0f, (int)exp_byte(exps, nb, m, b) - 134);
        prods[b] = __fmul_rn(dot, es);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float sum = 0.0f;
        for (int b = 0; b < nb; ++b) sum = __fadd_rn(sum, prods[b]);
        y[m] = sum;
    }
}

// ---- the engine's numpy fallback, 04/qwen_real_engine.py:1230-1238 ------------
// scales = 2^(e - 134) (float32, exact); products m * x rounded to float32;
// dots = np.sum(products, axis=-1) per block; y = np.sum(dots * scales, axis=-1).
// The summation order is numpy's (04/qwen_real_engine.py:323-329 names both):
//   pairwise (numpy >= 1.9): +0.0 + pairwise_sum(a, n), where pairwise_sum of
//     n < 8 elements adds them one by one from -0.0, of n <= 128 keeps eight
//     accumulators r[j] += a[8i + j], combines them as
//     ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7)) and adds the n % 8 rest
//     one by one, and above 128 splits at n/2 rounded down to a multiple of 8;
//   sequential (numpy 1.8.2, the board's): a[0] + a[1] + ... + a[n-1].
// One wavefront per row; lanes take blocks, lane 0 sums the block terms.
__device__ float np_pairwise(const float* a, int n) {
    if (n < 8) {
        float r = -0.0f;
        for (int i = 0; i < n; ++i) r = __fadd_rn(r, a[i]);
        return r;
    }
    if (n <= 128) {
        float r[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = a[j];
        int i = 8;
        for (; i < n - (n % 8); i += 8)
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = __fadd_rn(r[j], a[i + j]);
        float res = __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                              __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
        for (; i < n; ++i) res = __fadd_rn(res, a[i]);
        return res;
    }
    int n2 = n / 2;
    n2 -= n2 % 8;
    return __fadd_rn(np_pairwise(a, n2), np_pairwise(a + n2, n - n2));
}

__device__ __forceinline__ float np_sum(const float* a, int n, bool pairwise) {
    if (pairwise) return __fadd_rn(0.0f, np_pairwise(a, n));
    if (n == 0) return 0.0f;
    float r = a[0];
    for (int i = 1; i < n; ++i) r = __fadd_rn(r, a[i]);
    return r;
}

extern "C" __global__ __launch_bounds__(64) void bfp8_gemv_fallback_kernel(
    float* __restrict__ y, const float* __restrict__ x, const uint8_t* __restrict__ mant,
    const uint8_t* __restrict__ exps, int M, int K, int pairwise) {
    extern __shared__ float terms[];
    const int m = blockIdx.x;
    const int nb = K >> 6;
    for (int b = threadIdx.x; b < nb; b += 64) {
        u32x4 c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) c[q] = *chunk_ptr(mant, nb, m, b, q);
        const float* xb = x + (size_t)b * 64;
        float p[64];
#pragma unroll
        for (int k = 0; k < 64; ++k) {
            const int i = k >> 2;  // element k: residue chunk k & 3, byte k >> 2
            const uint32_t word = c[k & 3][i >> 2];
            p[k] = __fmul_rn((float)(int)(int8_t)((word >> (8 * (i & 3))) & 0xffu), xb[k]);
        }
        const float dot = np_sum(p, 64, pairwise != 0);
        terms[b] = __fmul_rn(dot, ldexpf(1.0f, (int)exp_byte(exps, nb, m, b) - 134));
    }
    __syncthreads();
    if (threadIdx.x == 0) y[m] = np_sum(terms, nb, pairwise != 0);
}

// ---- layout converter: reference planes <-> GPU planes ------------------------
// Row `row` of the mantissas starts at ms + row * ms_stride and its exponents
// at es + row * es_stride: the packer's SoA planes have strides K and K/64; the
// PL core's per-row stream (K/64 exponent bytes, then K mantissas per row) has
// K/64 + K for both.
//
// Bound by HBM: both directions move every byte once.  A workgroup takes a
// tile's four blocks of one exponent dword (16 KiB): wavefront w its rows
// 16w .. 16w + 15, lane 4r + d the 16-byte piece d of row r in each of the
// four blocks -- four 16-byte loads in flight per lane, a row's 256 bytes by
// one quad.  Piece d holds elements 16d + 4p + q (dword p, byte q), so its
// 4 x 4 bytes transposed are dword d of the four residue chunks; a 4 x 4
// exchange of dwords within the quad (DPP) then leaves lane 4r + q with the
// whole 16-byte residue chunk q, and the wavefront stores four 256-byte runs.
// The way back is the same steps in reverse (both transposes are their own
// inverse).  Mantissa rows start at any byte (a stream's row, a ragged K): those
// accesses are of a type with alignment 1, which this target does in one
// unaligned 16-byte access.  65536 x 1024: packed in 24.1 us (136 MB moved, 5.7
// TB/s), unpacked in 22.6; with a thread per block reading and writing its
// mantissas byte by byte, and the exponents in a launch of their own, 119.8.
typedef u32x4 u32x4_any __attribute__((aligned(1)));

// 4 x 4 bytes: byte q of word p -> byte p of word q.
__device__ __forceinline__ u32x4 transpose_bytes(u32x4 v) {
    const uint32_t a = __builtin_amdgcn_perm(v.y, v.x, 0x05010400u);  // x0 y0 x1 y1
    const uint32_t b = __builtin_amdgcn_perm(v.y, v.x, 0x07030602u);  // x2 y2 x3 y3
    const uint32_t c = __builtin_amdgcn_perm(v.w, v.z, 0x05010400u);  // z0 w0 z1 w1
    const uint32_t d = __builtin_amdgcn_perm(v.w, v.z, 0x07030602u);  // z2 w2 z3 w3
    return u32x4{__builtin_amdgcn_perm(c, a, 0x05040100u), __builtin_amdgcn_perm(c, a, 0x07060302u),
                 __builtin_amdgcn_perm(d, b, 0x05040100u), __builtin_amdgcn_perm(d, b, 0x07060302u)};
}

// The value of the quad's lane (lane ^ kXor).
template <int kXor>
__device__ __forceinline__ uint32_t quad_xor(uint32_t v) {
    constexpr int kCtrl = kXor == 1 ? 0xB1 : 0x4E;  // quad_perm [1,0,3,2] / [2,3,0,1]
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xf, 0xf, true);
}

// Across a quad: word q of lane d -> word d of lane q.
__device__ __forceinline__ u32x4 transpose_quad(u32x4 v, int lane) {
    const bool odd = lane & 1, high = lane & 2;
    // pairs of lanes exchange words (0, 1) and (2, 3), then pairs of pairs (0, 2) and (1, 3)
    const uint32_t s0 = quad_xor<1>(odd ? v.x : v.y), s1 = quad_xor<1>(odd ? v.z : v.w);
    v = odd ? u32x4{s0, v.y, s1, v.w} : u32x4{v.x, s0, v.z, s1};
    const uint32_t t0 = quad_xor<2>(high ? v.x : v.z), t1 = quad_xor<2>(high ? v.y : v.w);
    return high ? u32x4{t0, t1, v.z, v.w} : u32x4{v.x, v.y, t0, t1};
}

extern "C" __global__ __launch_bounds__(256) void bfp8_pack_kernel(
    uint8_t* __restrict__ mg, uint8_t* __restrict__ eg, const int8_t* __restrict__ ms, size_t ms_stride,
    const uint8_t* __restrict__ es, size_t es_stride, int M, int K) {
    const int nb = K >> 6, nb4 = (nb + 3) >> 2;
    const int lane = threadIdx.x & 63, j = lane & 3;
    const int r = 16 * ((int)threadIdx.x >> 6) + (lane >> 2);
    const size_t total = (size_t)bfp8_ntiles(M) * nb4;
    for (size_t u = blockIdx.x; u < total; u += gridDim.x) {
        const int t = (int)(u / nb4), b0 = (int)(u % nb4) * 4, row = t * 64 + r;
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = u32x4(0u);
            if (row < M && b0 + i < nb)
                v[i] = *reinterpret_cast<const u32x4_any*>(ms + (size_t)row * ms_stride + (size_t)(b0 + i) * 64 + 16 * j);
        }
        uint32_t word = 0;  // exponents: thread x < 64 takes row x of the tile
        const int erow = t * 64 + (int)threadIdx.x;
        if (threadIdx.x < 64 && erow < M)
            for (int p = 0; p < 4 && b0 + p < nb; ++p) word |= (uint32_t)es[(size_t)erow * es_stride + b0 + p] << (8 * p);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 c = transpose_quad(transpose_bytes(v[i]), lane);
            if (b0 + i < nb)
                *reinterpret_cast<u32x4*>(mg + (((size_t)t * nb + b0 + i) * 4 + j) * 1024u + (size_t)r * 16u) = c;
        }
        if (threadIdx.x < 64) reinterpret_cast<uint32_t*>(eg)[u * 64 + threadIdx.x] = word;
    }
}

extern "C" __global__ __launch_bounds__(256) void bfp8_unpack_kernel(
    int8_t* __restrict__ ms, uint8_t* __restrict__ es, const uint8_t* __restrict__ mg,
    const uint8_t* __restrict__ eg, int M, int K) {
    const int nb = K >> 6, nb4 = (nb + 3) >> 2;
    const int lane = threadIdx.x & 63, j = lane & 3;
    const int r = 16 * ((int)threadIdx.x >> 6) + (lane >> 2);
    const size_t total = (size_t)bfp8_ntiles(M) * nb4;
    for (size_t u = blockIdx.x; u < total; u += gridDim.x) {
        const int t = (int)(u / nb4), b0 = (int)(u % nb4) * 4, row = t * 64 + r;
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = u32x4(0u);
            if (b0 + i < nb)
                v[i] = *reinterpret_cast<const u32x4*>(mg + (((size_t)t * nb + b0 + i) * 4 + j) * 1024u + (size_t)r * 16u);
        }
        const int erow = t * 64 + (int)threadIdx.x;
        uint32_t word = 0;
        if (threadIdx.x < 64) word = reinterpret_cast<const uint32_t*>(eg)[u * 64 + threadIdx.x];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 c = transpose_bytes(transpose_quad(v[i], lane));
            if (row < M && b0 + i < nb)
                *reinterpret_cast<u32x4_any*>(ms + (size_t)row * K + (size_t)(b0 + i) * 64 + 16 * j) = c;
        }
        if (threadIdx.x < 64 && erow < M)
            for (int p = 0; p < 4 && b0 + p < nb; ++p) es[(size_t)erow * nb + b0 + p] = (uint8_t)(word >> (8 * p));
    }
}

// ---- synthetic reference-format planes (counter-based, host-reproducible) ----
extern "C" __global__ __launch_bounds__(256) void bfp8_synth_kernel(
    int8_t* __restrict__ ms, uint8_t* __restrict__ es, size_t nm, size_t ne, uint64_t seed, int lo, int hi) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nm; i += stride)
        ms[i] = bfp8_synth_mant(seed, i);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < ne; i += stride)
        es[i] = bfp8_synth_exp(seed, i, lo, hi);
}

// ---- bandwidth probes -----------------------------------------------------------
// Read-only ceiling: each workgroup streams one contiguous chunk with eight
// non-temporal dwordx4 loads in flight per thread; the folded value is stored
// only if it hits a magic constant, which keeps the loads live without any
// atomic traffic.
// Read-bandwidth probe: wavefront v's step s reads the 2 KiB run at
// (s * wavefronts + v) * 2 KiB (two 1 KiB loads, non-temporal), one step in
// flight per wavefront, 4096 wavefronts.  Of the patterns measured (blocked
// per workgroup with eight loads in flight per lane: 6.8-6.95 TB/s; runs of
// 1-8 KiB, one to four steps in flight) this one reads fastest: 7.14-7.20 TB/s
// over 1 GiB and 128 MiB.
extern "C" __global__ __launch_bounds__(256) void bfp8_read_probe_kernel(const u32x4* __restrict__ src, size_t n16,
                                                                         uint32_t* __restrict__ out) {
    const size_t nw = (size_t)gridDim.x * 4;
    const size_t wv = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    u32x4 acc = u32x4(0u);
    for (size_t st = 0;; ++st) {
        const size_t i0 = (st * nw + wv) * 128 + lane, i1 = i0 + 64;
        const u32x4 v0 = i0 < n16 ? __builtin_nontemporal_load(src + i0) : u32x4(0u);
        const u32x4 v1 = i1 < n16 ? __builtin_nontemporal_load(src + i1) : u32x4(0u);
        acc ^= v0 ^ v1;
        if (!__builtin_amdgcn_ballot_w64(i0 < n16)) break;  // every lane past the end: the wavefront is done
    }
    const uint32_t v = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (v == 0x9E3779B9u) out[0] = v;
}

extern "C" __global__ __launch_bounds__(256) void bfp8_copy_probe_kernel(
    u32x4* __restrict__ dst, const u32x4* __restrict__ src, size_t n16) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

// ---- launchers ----------------------------------------------------------------------
static int grid_for(size_t work, int per_block) {
    size_t g = (work + per_block - 1) / per_block;
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (int)g;
}

hipError_t bfp8_launch_quantize(const Bfp8QuantDesc* descs_dev, int ndesc, int max_nb, hipStream_t s) {
    if (ndesc <= 0 || max_nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_quantize_kernel, dim3(max_nb, ndesc), dim3(64), 0, s, descs_dev);
    return hipGetLastError();
}

hipError_t bfp8_launch_quantize1(const Bfp8QuantDesc& d, hipStream_t s) {
    const int nb = bfp8_nblocks(d.K);
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_quantize1_kernel, dim3(nb), dim3(64), 0, s, d);
    return hipGetLastError();
}

hipError_t bfp8_launch_tail_row(float* y, const uint32_t* xsplit, const float* xscale,
                                const uint8_t* mant, const uint8_t* exps, int M, int K, hipStream_t s, int nvec) {
    if (M <= 0 || !(M & 1) || nvec <= 0) return hipSuccess;
    if (bfp8_nblocks(K) > 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bfp8_tail_row_kernel, dim3(nvec), dim3(64), 0, s, y, xsplit, xscale, mant, exps, M, K);
    return hipGetLastError();
}

hipError_t bfp8_launch_gemv_float(float* y, const float* x, const uint8_t* mant, const uint8_t* exps,
                                  int M, int K, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    const int nb = bfp8_nblocks(K);
    if (nb > 16384) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bfp8_gemv_float_kernel, dim3(M), dim3(64), (size_t)(nb > 0 ? nb : 1) * 4, s, y, x,
                       mant, exps, M, K);
    return hipGetLastError();
}

hipError_t bfp8_launch_gemv_fallback(float* y, const float* x, const uint8_t* mant, const uint8_t* exps, int M,
                                     int K, int pairwise, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    const int nb = bfp8_nblocks(K);
    if (nb > 16384) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bfp8_gemv_fallback_kernel, dim3(M), dim3(64), (size_t)(nb > 0 ? nb : 1) * 4, s, y, x, mant,
                       exps, M, K, pairwise);
    return hipGetLastError();
}

hipError_t bfp8_launch_pack_strided(uint8_t* mant_gpu, uint8_t* exps_gpu, const int8_t* mant_src, size_t mant_stride,
                                    const uint8_t* exps_src, size_t exps_stride, int M, int K, hipStream_t s) {
    const int nb = bfp8_nblocks(K);
    if (M <= 0 || nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_pack_kernel, dim3(grid_for((size_t)bfp8_ntiles(M) * bfp8_nb4(nb), 1)), dim3(256), 0, s,
                       mant_gpu, exps_gpu, mant_src, mant_stride, exps_src, exps_stride, M, K);
    return hipGetLastError();
}

hipError_t bfp8_launch_pack(uint8_t* mant_gpu, uint8_t* exps_gpu, const int8_t* mant_soa,
                            const uint8_t* exps_soa, int M, int K, hipStream_t s) {
    return bfp8_launch_pack_strided(mant_gpu, exps_gpu, mant_soa, (size_t)K, exps_soa, (size_t)bfp8_nblocks(K), M,
                                    K, s);
}

hipError_t bfp8_launch_unpack(int8_t* mant_soa, uint8_t* exps_soa, const uint8_t* mant_gpu,
                              const uint8_t* exps_gpu, int M, int K, hipStream_t s) {
    const int nb = bfp8_nblocks(K);
    if (M <= 0 || nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_unpack_kernel, dim3(grid_for((size_t)bfp8_ntiles(M) * bfp8_nb4(nb), 1)), dim3(256), 0, s, mant_soa, exps_soa, mant_gpu,
                       exps_gpu, M, K);
    return hipGetLastError();
}

hipError_t bfp8_launch_synth_planes(int8_t* mant_soa, uint8_t* exps_soa, int M, int K, uint64_t seed,
                                    int e_lo, int e_hi, hipStream_t s) {
    if (M <= 0 || K <= 0) return hipSuccess;
    const size_t nm = (size_t)M * K, ne = (size_t)M * bfp8_nblocks(K);
    hipLaunchKernelGGL(bfp8_synth_kernel, dim3(grid_for(nm, 256 * 16)), dim3(256), 0, s, mant_soa, exps_soa, nm,
                       ne, seed, e_lo, e_hi);
    return hipGetLastError();
}

hipError_t bfp8_launch_read_probe(const void* buf, size_t bytes, uint32_t* out, hipStream_t s) {
    const size_t n16 = bytes / 16;
    if (n16 == 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_read_probe_kernel, dim3(1024), dim3(256), 0, s, (const u32x4*)buf, n16, out);
    return hipGetLastError();
}

hipError_t bfp8_launch_copy_probe(void* dst, const void* src, size_t bytes, hipStream_t s) {
    const size_t n16 = bytes / 16;
    if (n16 == 0) return hipSuccess;
    hipLaunchKernelGGL(bfp8_copy_probe_kernel, dim3(grid_for(n16, 256 * 4)), dim3(256), 0, s, (u32x4*)dst,
                       (const u32x4*)src, n16);
    return hipGetLastError();
}
