// GEMM of a few tokens (5 and more) on the integer matrix cores:
//   out[t][o] = [resid[t][o] +] (bias[o] + sum_b dx[t][b] * (W block b of row o . codes))
// for Q4_K, Q6_K (Q8_K activations) and Q8_0 (Q8_0 activations) weights read
// as they lie, up to four matrices of one input in a launch, or a gate / up
// pair that leaves as silu(gate) * up.
//
// What bounds it: not yet the weights, read once per 64 tokens, but waits on
// memory with few waves (counted on layers of 8 and 45 tokens: waves wait 42-72 %
// of their time, VALU 13-31 % and MFMA 3-10 % busy, 1 to 2.6 waves a SIMD).  The
// 8-token GEMV
// this replaces dots every weight byte with every token on the VALU; the
// 128-token GEMM tiles leave most of the chip idle on these sizes and add the
// K split's partial tiles through memory.  Here a workgroup owns 16 (or 32)
// weight rows for all its tokens and splits K over its wavefronts, so 4096
// rows are 256 workgroups without any partial leaving the CU: each wave walks
// its own super-blocks, weights straight into registers one super-block
// ahead, and the waves' f32 tiles are added in LDS in wave order.  RMSNorm,
// SiLU-mul and quantization are one pack launch before it, residual and
// silu(gate) * up its store: two launches where the steps took four to six.
// Measured, the four calls of a layer: 8 tokens of Q4_K 4096 / 14336 200 us
// before (GEMV), 73 us so; 45 tokens of Q4_K 2560 with Q6_K 9728 243 us before
// (128-token tiles, K split over workgroups), 79 us so.  Gate and up of 8
// tokens (2 x 14336 rows of 4096, 66 MB) 77 us before, 21.6 us so, 3.1 TB/s.
//
// Arithmetic: v_mfma_i32_16x16x32_i8 gives every sub-block's integer sum
// exactly, the K-quants' sub-block scales multiply it in 32-bit integers
// (24-bit products), and one f32 combination per super-block follows,
//   acc += dx * (sumi * d - mn * dmin),
// with mn = sum_j m_j * bsum_j (exact, v_mfma_f32_16x16x16_f16; |mn| < 2^23).
// The block formulas are those of dot_q4_k_q8_k, dot_q6_k_q8_k and
// dot_q8_0_q8_0 (src/gguf_dot_q8.c:603-666, 897-1002, 436-601).
//
// Operand layout of the 16x16 shapes: lane l supplies row l % 16 of A (a
// token) and column l % 16 of B (a weight row), K slots of group g = l / 16
// (8 bytes, or 4 fp16); accumulator register r of lane l holds
// C[4 (l / 16) + r][l % 16] = C[token][row].
//
// K order: a lane reads 16 bytes of Q4_K quants, g = 0..3 covering 64
// contiguous bytes of the row; v_permlane32_swap then leaves lane group g
// with piece {0, 2, 1, 3}[g] (8 bytes) of each 32-byte chunk.  The pack and
// the Q6_K loads use the same piece order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "common.h"
#include "gemm_small.h"
#include "q8k.h"

namespace exq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

__device__ __forceinline__ long pack2(uint32_t lo, uint32_t hi) {
    return (long)((uint64_t)lo | ((uint64_t)hi << 32));
}
__device__ __forceinline__ v4i mfma_i8(long a, long b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma_h(v4h a, v4h b) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// 8-byte piece of each 32-byte chunk that lane group g holds (its own inverse).
__device__ __forceinline__ int piece_of(int g) { return ((g & 1) << 1) | (g >> 1); }

// --------------------------------------------------------------- packing
//
// K-quant pack, kSmPackK bytes per (super-block, 16-token tile):
//   codes [j 4][lane 64][16 B]  lane t + 16 g: the int8 codes of elements
//         64 j + 8 piece(g) .. + 7 and 64 j + 32 + 8 piece(g) .. + 7
//   bsums [lane 64][4 fp16]     lane t + 16 g: 16-element sums 4 g .. 4 g + 3
//   dx    [16] f32
// Q8_0 pack, kSmPack0 bytes per (pair of 32-element blocks, tile):
//   codes [lane 64][16 B]       lane t + 16 g: elements 8 piece(g) .. + 7 of
//         the even and of the odd block
//   dx    [2][16] f32
// (an odd last block leaves its partner's places unwritten, and unread).
// Tokens of a tile past m are not written: a token's column of the product
// touches no other, and theirs is never stored.
constexpr int kSmBs = 4096, kSmDx = 4608, kSmDx0 = 1024;

// The prologue of one value: RMSNorm (x * scale) * w, silu(x) * x2, or x.
template <int PRO>
__device__ __forceinline__ float prologue(float x, float y, float scale) {
    if (PRO == 1) {
        const float v = x * scale;
        return v * y;
    }
    if (PRO == 2) return silu_f32(x) * y;
    return x;
}

__device__ __forceinline__ void load8(const float *p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// RMSNorm scale of a row of n elements (a multiple of 32) by the workgroup's
// first 256 threads: the sum of rmsnorm_kernel, term for term, so that a layer
// call gives the words of its steps.
constexpr int kRmsThreads = 256;
__device__ __forceinline__ float row_rms_scale(const float *x, int n, float eps) {
    __shared__ double part[kRmsThreads / 64];
    constexpr int kTogether = 4;
    const float4 *x4 = reinterpret_cast<const float4 *>(x);
    const int tid = threadIdx.x, n4 = n >> 2;
    if (tid < kRmsThreads) {
        double s = 0.0;
        for (int i0 = tid; i0 < n4; i0 += kTogether * kRmsThreads) {
            float4 v[kTogether];  // loaded together
#pragma unroll
            for (int k = 0; k < kTogether; ++k) v[k] = x4[min(i0 + k * kRmsThreads, n4 - 1)];
#pragma unroll
            for (int k = 0; k < kTogether; ++k) s += i0 + k * kRmsThreads < n4 ? square4(v[k]) : 0.0;
        }
        s = wave_sum_f64(s);
        if ((tid & 63) == 0) part[tid >> 6] = s;
    }
    __syncthreads();
    return rms_scale((part[0] + part[1]) + (part[2] + part[3]), n, eps);
}

__device__ __forceinline__ uint32_t bytes4(const int *q) {
    return (uint32_t)(q[0] & 0xff) | ((uint32_t)(q[1] & 0xff) << 8) | ((uint32_t)(q[2] & 0xff) << 16) |
           ((uint32_t)q[3] << 24);
}

__device__ __forceinline__ uint32_t half2_bits(int lo, int hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)lo) |
           ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)hi) << 16);
}

// One token per blockIdx.x; 16 lanes hold a super-block: lane 4 j + q its
// elements 64 j + 8 q .. + 7 and 64 j + 32 + 8 q .. + 7, one code vector.
// PRO 1: the workgroup holds the whole row (the RMSNorm's sum of squares);
// otherwise blockIdx.y counts chunks of blockDim.x / 16 super-blocks.
template <int PRO>
__global__ __launch_bounds__(1024) void small_pack_k_kernel(const float *__restrict__ x, const float *__restrict__ y,
                                                            float eps, int nsb, int ntt, uint8_t *__restrict__ pack) {
    const int t = (int)blockIdx.x;
    const int r = threadIdx.x & 15, j = r >> 2, q = r & 3;
    const int per = (int)(blockDim.x >> 4);
    const int first = (int)blockIdx.y * per + (int)(threadIdx.x >> 4);
    const int K = nsb * kQKK;
    const float *xr = x + (size_t)t * K;
    const int e0 = 64 * j + 8 * q;
    float scale = 0.0f;
    if (PRO == 1) scale = row_rms_scale(xr, K, eps);
    const int last = PRO == 1 ? nsb : min(nsb, ((int)blockIdx.y + 1) * per);
    for (int sb = first; sb < last; sb += per) {
        float xs[16];
        {
            float a[8], b[8], c[8], d[8];
            const int o = sb * kQKK + e0;
            load8(xr + o, a);
            load8(xr + o + 32, b);
            if (PRO != 0) {
                const float *yr = PRO == 2 ? y + (size_t)t * K : y;
                load8(yr + o, c);
                load8(yr + o + 32, d);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                xs[i] = prologue<PRO>(a[i], PRO != 0 ? c[i] : 0.0f, scale);
                xs[8 + i] = prologue<PRO>(b[i], PRO != 0 ? d[i] : 0.0f, scale);
            }
        }
        int qv[16];
        const Q8KRow16 k = q8k_quantize_row16(xs, qv);
        uint8_t *blk = pack + ((size_t)sb * ntt + (t >> 4)) * kSmPackK;
        const int tl = t & 15;
        *reinterpret_cast<uint4 *>(blk + j * 1024 + (tl + 16 * piece_of(q)) * 16) =
            make_uint4(bytes4(qv), bytes4(qv + 4), bytes4(qv + 8), bytes4(qv + 12));
        if (q == 0)  // the 16-element sums 4 j .. 4 j + 3
            *reinterpret_cast<uint2 *>(blk + kSmBs + (tl + 16 * j) * 8) =
                make_uint2(half2_bits(k.lo, k.lo_next), half2_bits(k.hi, k.hi_next));
        if (r == 0) *reinterpret_cast<float *>(blk + kSmDx + 4 * tl) = k.d;
    }
}

// The same pack from Q8_K blocks.
__global__ __launch_bounds__(256) void small_pack_k_blocks_kernel(const uint8_t *__restrict__ xq, size_t xq_stride,
                                                                  int nsb, int ntt, uint8_t *__restrict__ pack) {
    const int t = (int)blockIdx.x;
    const int r = threadIdx.x & 15, j = r >> 2, q = r & 3;
    const int sb = (int)blockIdx.y * 16 + (int)(threadIdx.x >> 4);
    if (sb >= nsb) return;
    const uint8_t *src = xq + (size_t)t * xq_stride + (size_t)sb * kBytesQ8_K;
    uint8_t *blk = pack + ((size_t)sb * ntt + (t >> 4)) * kSmPackK;
    const int tl = t & 15;
    const uint2 a = ldg8(src + 4 + 64 * j + 8 * q), b = ldg8(src + 4 + 64 * j + 32 + 8 * q);
    *reinterpret_cast<uint4 *>(blk + j * 1024 + (tl + 16 * piece_of(q)) * 16) = make_uint4(a.x, a.y, b.x, b.y);
    if (q == 0) {
        const uint2 s = ldg8(src + 260 + 8 * j);
        *reinterpret_cast<uint2 *>(blk + kSmBs + (tl + 16 * j) * 8) =
            make_uint2(half2_bits((int16_t)(s.x & 0xffffu), (int16_t)(s.x >> 16)),
                       half2_bits((int16_t)(s.y & 0xffffu), (int16_t)(s.y >> 16)));
    }
    if (r == 0) *reinterpret_cast<uint32_t *>(blk + kSmDx + 4 * tl) = ldg4(src);
}

// Q8_0: 4 lanes hold a block of 32, 8 elements each; the quantizer is that of
// quantize_q8_0_kernel.
template <int PRO>
__global__ __launch_bounds__(1024) void small_pack_0_kernel(const float *__restrict__ x, const float *__restrict__ y,
                                                            float eps, int nb, int ntt, uint8_t *__restrict__ pack) {
    const int t = (int)blockIdx.x;
    const int g = threadIdx.x & 3;
    const int per = (int)(blockDim.x >> 2);
    const int first = (int)blockIdx.y * per + (int)(threadIdx.x >> 2);
    const int K = nb * kQK8_0;
    const float *xr = x + (size_t)t * K;
    float scale = 0.0f;
    if (PRO == 1) scale = row_rms_scale(xr, K, eps);
    const int last = PRO == 1 ? nb : min(nb, ((int)blockIdx.y + 1) * per);
    for (int b = first; b < last; b += per) {
        float a[8], c[8];
        const int o = b * kQK8_0 + 8 * g;
        load8(xr + o, a);
        if (PRO != 0) load8((PRO == 2 ? y + (size_t)t * K : y) + o, c);
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            a[i] = prologue<PRO>(a[i], PRO != 0 ? c[i] : 0.0f, scale);
            amax = fmaxf(amax, fabsf(a[i]));
        }
        amax = fmaxf(amax, __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(amax))));
        amax = fmaxf(amax, __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(amax))));
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        int qv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float v = rintf(a[i] * id);
            const int k = (v >= -2147483648.0f && v < 2147483648.0f) ? (int)v : INT32_MIN;
            qv[i] = k < -128 ? -128 : (k > 127 ? 127 : k);
        }
        uint8_t *blk = pack + ((size_t)(b >> 1) * ntt + (t >> 4)) * kSmPack0;
        const int tl = t & 15, odd = b & 1;
        *reinterpret_cast<uint2 *>(blk + (tl + 16 * piece_of(g)) * 16 + 8 * odd) =
            make_uint2(bytes4(qv), bytes4(qv + 4));
        if (g == 0)
            *reinterpret_cast<float *>(blk + kSmDx0 + 4 * (16 * odd + tl)) =
                f16_bits_to_f32(f32_to_f16_rne(amax / 127.0f));
    }
}

// The same pack from Q8_0 blocks.
__global__ __launch_bounds__(256) void small_pack_0_blocks_kernel(const uint8_t *__restrict__ xq, size_t xq_stride,
                                                                  int nb, int ntt, uint8_t *__restrict__ pack) {
    const int t = (int)blockIdx.x;
    const int g = threadIdx.x & 3;
    const int b = (int)blockIdx.y * 64 + (int)(threadIdx.x >> 2);
    if (b >= nb) return;
    const uint8_t *src = xq + (size_t)t * xq_stride + (size_t)b * kBytesQ8_0;
    uint8_t *blk = pack + ((size_t)(b >> 1) * ntt + (t >> 4)) * kSmPack0;
    const int tl = t & 15, odd = b & 1;
    *reinterpret_cast<uint2 *>(blk + (tl + 16 * piece_of(g)) * 16 + 8 * odd) = ldg8(src + 2 + 8 * g);
    if (g == 0)
        *reinterpret_cast<float *>(blk + kSmDx0 + 4 * (16 * odd + tl)) = f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(src));
}

// --------------------------------------------------------------- formats
//
// A format supplies: W, the raw registers of one K unit of a lane's row; Op,
// its decoded operand; A, a token tile's operand; load_w, decode, load_a and
// dot (one unit of one row tile and token tile into the f32 accumulators).

struct SmallQ4K {
    static constexpr int kType = kTypeQ4_K;
    static constexpr int kUnits = 1;  // super-blocks per step
    struct W {
        uint4 hd, q0, q1;
    };
    struct Op {
        uint32_t lo[8], hi[8];  // chunk j: words 2 j, 2 j + 1 of its low and high nibbles
        int sc[8];
        v4h mn;
        float d, nd;
    };
    struct A {
        uint4 c[4];
        v4h bs;
        float4 dx;
    };
    __device__ static __forceinline__ void load_w(W &w, const uint8_t *row, int u, int, int g) {
        const uint8_t *p = row + (size_t)u * kBytesQ4_K;
        w.hd = *reinterpret_cast<const uint4 *>(p);
        w.q0 = *reinterpret_cast<const uint4 *>(p + 16 + 16 * g);
        w.q1 = *reinterpret_cast<const uint4 *>(p + 80 + 16 * g);
    }
    __device__ static __forceinline__ void split(uint32_t *lo, uint32_t *hi, const uint4 &q) {
        const auto x = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
        const uint32_t v[4] = {(uint32_t)x[0], (uint32_t)y[0], (uint32_t)x[1], (uint32_t)y[1]};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[i] = v[i] & 0x0f0f0f0fu;
            hi[i] = (v[i] >> 4) & 0x0f0f0f0fu;
        }
    }
    // the six-bit scales and minima of get_scale_min_k4 (src/gguf_quant.c:212-220)
    __device__ static __forceinline__ void decode(Op &o, const W &w, int g) {
        split(o.lo, o.hi, w.q0);
        split(o.lo + 4, o.hi + 4, w.q1);
        const uint32_t w0 = w.hd.y, w1 = w.hd.z, w2 = w.hd.w;
        const uint32_t s0 = w0 & 0x3f3f3f3fu, s1 = (w2 & 0x0f0f0f0fu) | ((w0 >> 2) & 0x30303030u);
        const uint32_t m0 = w1 & 0x3f3f3f3fu, m1 = ((w2 >> 4) & 0x0f0f0f0fu) | ((w1 >> 2) & 0x30303030u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o.sc[i] = (int)((s0 >> (8 * i)) & 0xffu);
            o.sc[4 + i] = (int)((s1 >> (8 * i)) & 0xffu);
        }
        const uint32_t mm = ((g & 2) ? m1 : m0) >> (16 * (g & 1));  // minima 2 g, 2 g + 1
        const _Float16 ma = (_Float16)(float)(mm & 0xffu), mb = (_Float16)(float)((mm >> 8) & 0xffu);
        o.mn = v4h{ma, ma, mb, mb};
        o.d = f16_bits_to_f32(w.hd.x & 0xffffu);
        o.nd = -f16_bits_to_f32(w.hd.x >> 16);
    }
    __device__ static __forceinline__ void load_a(A &a, const uint8_t *pk, int u, int, int ntt, int tt, int lane) {
        const uint8_t *blk = pk + ((size_t)u * ntt + tt) * kSmPackK;
#pragma unroll
        for (int j = 0; j < 4; ++j) a.c[j] = *reinterpret_cast<const uint4 *>(blk + j * 1024 + lane * 16);
        a.bs = __builtin_bit_cast(v4h, *reinterpret_cast<const uint2 *>(blk + kSmBs + lane * 8));
        a.dx = *reinterpret_cast<const float4 *>(blk + kSmDx + 16 * (lane >> 4));
    }
    __device__ static __forceinline__ void dot(float (&acc)[4], const A &a, const Op &o, int, int, int) {
        int s[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4i p = mfma_i8(pack2(a.c[j].x, a.c[j].y), pack2(o.lo[2 * j], o.lo[2 * j + 1]), v4i{0, 0, 0, 0});
            const v4i q = mfma_i8(pack2(a.c[j].z, a.c[j].w), pack2(o.hi[2 * j], o.hi[2 * j + 1]), v4i{0, 0, 0, 0});
#pragma unroll
            for (int r = 0; r < 4; ++r)
                s[r] += __mul24(p[r], o.sc[2 * j]) + __mul24(q[r], o.sc[2 * j + 1]);
        }
        const v4f mn = mfma_h(a.bs, o.mn);
        const float dx[4] = {a.dx.x, a.dx.y, a.dx.z, a.dx.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float v = __builtin_fmaf(mn[r], o.nd, (float)s[r] * o.d);
            acc[r] = __builtin_fmaf(v, dx[r], acc[r]);
        }
    }
};

// Q6_K: sub-blocks are 16 elements, half of a K = 32 product: lane groups
// with even g hold the first of the two, odd g the second, so a second
// product with the odd groups' weights zeroed gives the first one's sum and
//   sc0 S0 + sc1 S1 = sc1 (S0 + S1) + (sc0 - sc1) S0.
// The codes stay unsigned, q6 in 0..63; q = q6 - 32 takes 32 sum_j sc_j
// bsum_j off the integer.  Blocks are 2-byte aligned: words are read from
// the 4-byte address below and joined by byte shifts (wide loads at 2 mod 4
// run several times slower here).
struct SmallQ6K {
    static constexpr int kType = kTypeQ6_K;
    static constexpr int kUnits = 1;
    struct W {
        uint32_t l[4][3], h[2][3];  // ql 0, ql 32, ql 64, ql 96; qh 0, qh 32 (+ 8 piece)
        uint32_t s[4], se, d;
        uint32_t sh;
    };
    struct Op {
        uint32_t b[8][2];
        int s1[8], s01[8];
        v4h mn;
        float d;
    };
    typedef SmallQ4K::A A;
    __device__ static __forceinline__ void load3(uint32_t (&v)[3], const uint8_t *p) {
        const uint32_t *q = reinterpret_cast<const uint32_t *>(p);
        v[0] = q[0], v[1] = q[1], v[2] = q[2];
    }
    __device__ static __forceinline__ void load_w(W &w, const uint8_t *row, int u, int, int g) {
        const uint8_t *b = row + (size_t)u * kBytesQ6_K;
        w.sh = (uint32_t)((uintptr_t)b & 3u);
        const uint8_t *p = b - w.sh;
        const int o = 8 * piece_of(g);
#pragma unroll
        for (int i = 0; i < 4; ++i) load3(w.l[i], p + 32 * i + o);
#pragma unroll
        for (int i = 0; i < 2; ++i) load3(w.h[i], p + 128 + 32 * i + o);
#pragma unroll
        for (int i = 0; i < 4; ++i) w.s[i] = reinterpret_cast<const uint32_t *>(p + 192)[i];
        w.se = *reinterpret_cast<const uint16_t *>(b + 206);
        w.d = *reinterpret_cast<const uint16_t *>(b + 208);
    }
    __device__ static __forceinline__ void decode(Op &o, const W &w, int g) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t l0 = __builtin_amdgcn_alignbyte(w.l[2 * hh][i + 1], w.l[2 * hh][i], w.sh);
                const uint32_t l1 = __builtin_amdgcn_alignbyte(w.l[2 * hh + 1][i + 1], w.l[2 * hh + 1][i], w.sh);
                const uint32_t h = __builtin_amdgcn_alignbyte(w.h[hh][i + 1], w.h[hh][i], w.sh);
                o.b[4 * hh][i] = (l0 & 0x0f0f0f0fu) | ((h << 4) & 0x30303030u);
                o.b[4 * hh + 1][i] = (l1 & 0x0f0f0f0fu) | ((h << 2) & 0x30303030u);
                o.b[4 * hh + 2][i] = ((l0 >> 4) & 0x0f0f0f0fu) | (h & 0x30303030u);
                o.b[4 * hh + 3][i] = ((l1 >> 4) & 0x0f0f0f0fu) | ((h >> 2) & 0x30303030u);
            }
        uint32_t s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = __builtin_amdgcn_alignbyte(i < 3 ? w.s[i + 1] : w.se, w.s[i], w.sh);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t v = s[e >> 1] >> (16 * (e & 1));
            const int a = (int)(int8_t)(v & 0xffu), b = (int)(int8_t)((v >> 8) & 0xffu);
            o.s1[e] = b;
            o.s01[e] = a - b;
        }
        const uint32_t sg = (g & 2) ? ((g & 1) ? s[3] : s[2]) : ((g & 1) ? s[1] : s[0]);  // scales 4 g .. 4 g + 3
#pragma unroll
        for (int i = 0; i < 4; ++i) o.mn[i] = (_Float16)(float)(int8_t)((sg >> (8 * i)) & 0xffu);
        o.d = f16_bits_to_f32(w.d);
    }
    __device__ static __forceinline__ void load_a(A &a, const uint8_t *pk, int u, int end, int ntt, int tt,
                                                  int lane) {
        SmallQ4K::load_a(a, pk, u, end, ntt, tt, lane);
    }
    __device__ static __forceinline__ void dot(float (&acc)[4], const A &a, const Op &o, int, int, int g) {
        const uint32_t first = (g & 1) ? 0u : ~0u;
        int s[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint4 c = a.c[e >> 1];
            const long av = (e & 1) ? pack2(c.z, c.w) : pack2(c.x, c.y);
            const v4i p = mfma_i8(av, pack2(o.b[e][0], o.b[e][1]), v4i{0, 0, 0, 0});
            const v4i q = mfma_i8(av, pack2(o.b[e][0] & first, o.b[e][1] & first), v4i{0, 0, 0, 0});
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += __mul24(p[r], o.s1[e]) + __mul24(q[r], o.s01[e]);
        }
        const v4f mn = mfma_h(a.bs, o.mn);
        const float dx[4] = {a.dx.x, a.dx.y, a.dx.z, a.dx.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
            acc[r] = __builtin_fmaf((float)(s[r] - 32 * (int)mn[r]) * o.d, dx[r], acc[r]);
    }
};

// Q8_0: a step takes two pairs of 32-element blocks.  Of a pair, lane groups
// 0 and 1 read the halves of the even block's codes and groups 2 and 3 those
// of the odd block's, and v_permlane32_swap deals them out as for Q4_K; group
// g reads the scale of block g of the step, and a lane takes the four of its
// row from there.  Five loads per step for 2176 bytes of 16 rows; an 8-byte
// load and a scale per block and lane were twelve, which bounded it (8 tokens
// of 14336 rows of 4096: 56 us).
struct SmallQ80 {
    static constexpr int kType = kTypeQ8_0;
    static constexpr int kUnits = 4;
    struct W {
        uint4 q[2];
        uint32_t d;
    };
    struct Op {
        uint32_t q[4][2];
        float d[4];
    };
    struct A {
        uint4 c[2];
        float4 dx[4];
    };
    __device__ static __forceinline__ void load_w(W &w, const uint8_t *row, int u, int end, int g) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            w.q[i] = ldg16_a2(row + (size_t)min(u + 2 * i + (g >> 1), end - 1) * kBytesQ8_0 + 2 + 16 * (g & 1));
        w.d = *reinterpret_cast<const uint16_t *>(row + (size_t)min(u + g, end - 1) * kBytesQ8_0);
    }
    __device__ static __forceinline__ void decode(Op &o, const W &w, int) {
        const int r16 = threadIdx.x & 15;
        const float d = f16_bits_to_f32(w.d);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const auto x = __builtin_amdgcn_permlane32_swap(w.q[i].x, w.q[i].z, false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(w.q[i].y, w.q[i].w, false, false);
            o.q[2 * i][0] = (uint32_t)x[0];
            o.q[2 * i][1] = (uint32_t)y[0];
            o.q[2 * i + 1][0] = (uint32_t)x[1];
            o.q[2 * i + 1][1] = (uint32_t)y[1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) o.d[i] = __shfl(d, r16 + 16 * i, 64);
    }
    __device__ static __forceinline__ void load_a(A &a, const uint8_t *pk, int u, int end, int ntt, int tt, int lane) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint8_t *blk = pk + ((size_t)(min(u + 2 * i, end - 1) >> 1) * ntt + tt) * kSmPack0;
            a.c[i] = *reinterpret_cast<const uint4 *>(blk + lane * 16);
            a.dx[2 * i] = *reinterpret_cast<const float4 *>(blk + kSmDx0 + 16 * (lane >> 4));
            a.dx[2 * i + 1] = *reinterpret_cast<const float4 *>(blk + kSmDx0 + 64 + 16 * (lane >> 4));
        }
    }
    __device__ static __forceinline__ void dot(float (&acc)[4], const A &a, const Op &o, int u, int end, int) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (u + i >= end) break;  // wave-uniform
            const uint4 c = a.c[i >> 1];
            const v4i p = mfma_i8((i & 1) ? pack2(c.z, c.w) : pack2(c.x, c.y), pack2(o.q[i][0], o.q[i][1]),
                                  v4i{0, 0, 0, 0});
            const float dx[4] = {a.dx[i].x, a.dx[i].y, a.dx[i].z, a.dx[i].w};
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf((float)p[r] * o.d[i], dx[r], acc[r]);
        }
    }
};

// --------------------------------------------------------------- product

// One step of a wave (NEXT: the weights of units un .. are requested too).
// Loads retire in order: for Q8_0 and Q6_K the token tiles' operands are
// requested before the next step's weights, so no product waits for those
// (Q8_0 576 / 1536 layer of 30 tokens 48 us the other way round, 37 us so;
// Q6_K 9728 down of 64 tokens 38 and 28 us).  Q4_K steps are short of
// registers instead: holding every operand of more than two tiles halves the
// waves per CU (gate and up of 64 tokens 54 us), so they take the weights first
// and the operands tile by tile (48 us).
template <class F, int RT, int TT, bool NEXT>
__device__ __forceinline__ void small_step(float (&acc)[RT][TT][4], typename F::W (&w)[RT],
                                           const uint8_t *const (&row)[RT], const uint8_t *pk, int u, int un, int end,
                                           int ntt, int lane) {
    const int g = lane >> 4;
    typename F::W wn[RT];
    if constexpr (F::kType != kTypeQ4_K) {
        typename F::A a[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) F::load_a(a[tt], pk, u, end, ntt, tt, lane);
        if (NEXT)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) F::load_w(wn[rt], row[rt], un, end, g);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            typename F::Op op;
            F::decode(op, w[rt], g);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) F::dot(acc[rt][tt], a[tt], op, u, end, g);
        }
    } else {
        if (NEXT)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) F::load_w(wn[rt], row[rt], un, end, g);
        typename F::Op op[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) F::decode(op[rt], w[rt], g);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            typename F::A a;
            F::load_a(a, pk, u, end, ntt, tt, lane);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) F::dot(acc[rt][tt], a, op[rt], u, end, g);
        }
    }
    if (NEXT)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) w[rt] = wn[rt];
}

struct SmallArgs {
    const uint8_t *w[4];
    const float *bias[4], *resid[4];
    float *out[4];
    int n_out[4];
    int tile0[4];  // first workgroup row of each matrix
    int nmat;
    size_t row_bytes;
    const uint8_t *pack;
    int nk;        // super-blocks (K-quants) or 32-element blocks
    int m, ntt;    // tokens, 16-token tiles of the pack
};

// PAIR: w[0] and w[1] are gate and up, RT = 2 the row tile of each (two waves
// of one row tile each would read the operands twice: 31 us against 26 us for
// 8 tokens of 2 x 14336 rows of 4096).
template <class F, int RT, int TT, bool PAIR, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void gemm_small_kernel(SmallArgs a) {
    __shared__ float4 red[MAXW][RT * TT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = (int)(blockDim.x >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int tile = (int)blockIdx.x;
    const int tt0 = (int)blockIdx.y * TT;
    int z = 0;
    if (!PAIR)
        while (z + 1 < a.nmat && tile >= a.tile0[z + 1]) ++z;
    const int row0 = PAIR ? 16 * tile : 16 * RT * (tile - a.tile0[z]);
    const int n_out = a.n_out[z];

    const uint8_t *row[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
        row[rt] = a.w[PAIR ? rt : z] + (size_t)min(row0 + (PAIR ? 0 : 16 * rt) + r16, n_out - 1) * a.row_bytes;
    constexpr int kGran = F::kType == kTypeQ8_0 ? 2 : 1;  // Q8_0 blocks go in pairs
    const int np = (a.nk + kGran - 1) / kGran;
    // in 64 bits: with 32-bit divisions the compiler schedules the Q4_K loops
    // of three and four token tiles into 30 % more registers (down of 64
    // tokens of 14336 x 4096 41 us, 31 us so)
    const int k0 = kGran * (int)((long long)np * wave / nw);
    const int k1 = min(a.nk, kGran * (int)((long long)np * (wave + 1) / nw));

    float acc[RT][TT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rt][tt][r] = 0.0f;

    if (k0 < k1) {
        constexpr int kPk = F::kUnits == 1 ? kSmPackK : kSmPack0;
        const uint8_t *pk = a.pack + (size_t)tt0 * kPk;
        typename F::W w[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) F::load_w(w[rt], row[rt], k0, k1, g);
        // The K-quants' last step requests its own weights again (they hit in
        // L1): a peeled last step doubles the code, which costs more (Q4_K
        // down of 64 tokens 38 us against 31 us).  Q8_0's shorter steps peel
        // it (layer of 8 tokens 40 us unpeeled, 34 us so).
        if constexpr (F::kUnits == 1) {
            for (int u = k0; u < k1; ++u)
                small_step<F, RT, TT, true>(acc, w, row, pk, u, u + 1 < k1 ? u + 1 : u, k1, a.ntt, lane);
        } else {
            int u = k0;
            for (; u + F::kUnits < k1; u += F::kUnits)
                small_step<F, RT, TT, true>(acc, w, row, pk, u, u + F::kUnits, k1, a.ntt, lane);
            small_step<F, RT, TT, false>(acc, w, row, pk, u, u, k1, a.ntt, lane);
        }
    }

    // the waves' tiles, added in wave order
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
            red[wave][rt * TT + tt][lane] =
                make_float4(acc[rt][tt][0], acc[rt][tt][1], acc[rt][tt][2], acc[rt][tt][3]);
    __syncthreads();
    const auto total = [&](int tile_i, int l) {
        float4 s = red[0][tile_i][l];
        for (int w = 1; w < nw; ++w) {
            const float4 v = red[w][tile_i][l];
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
        return s;
    };
    for (int i = threadIdx.x; i < (PAIR ? 1 : RT) * TT * 64; i += (int)blockDim.x) {
        const int l = i & 63, ti = i >> 6;
        const int tt = ti % TT, rt = ti / TT;
        const int o = row0 + 16 * rt + (l & 15);
        const int t0 = 16 * (tt0 + tt) + 4 * (l >> 4);
        if (o >= n_out || t0 >= a.m) continue;
        const float4 s = total(rt * TT + tt, l);
        const float v[4] = {s.x, s.y, s.z, s.w};
        // bias after the whole dot (the reference's b + dot)
        const float b = a.bias[z] != nullptr ? a.bias[z][o] : 0.0f;
        if (PAIR) {
            const float4 su = total(TT + tt, l);
            const float u[4] = {su.x, su.y, su.z, su.w};
            const float bu = a.bias[1] != nullptr ? a.bias[1][o] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (t0 + r < a.m) a.out[0][(size_t)(t0 + r) * n_out + o] = silu_f32(b + v[r]) * (bu + u[r]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (t0 + r >= a.m) continue;
                const size_t at = (size_t)(t0 + r) * n_out + o;
                const float y = b + v[r];
                a.out[z][at] = a.resid[z] != nullptr ? a.resid[z][at] + y : y;
            }
        }
    }
}

}  // namespace exq

using namespace exq;

// True when a matrix of n_out rows of K elements takes this GEMM at m tokens:
// Q4_K, Q6_K and Q8_0 from kSmallMinTokens tokens.  Up to 64 tokens always
// (Q4_K to 32), beyond that while rows x K x (64-token blocks, each of which
// reads the weights again) stays below the line where the 128-token tiles of
// the prefill GEMMs catch up.  Theirs is one workgroup's walk through K, split
// four ways at most, whatever the rows: the line rises with K.  Swept over 44
// shapes of 33 to 768 tokens; nearest the line, few-token / prefill us:
//   Q4_K 9728 x 2560 (rows x K), 192 tokens (75 M) 42 / 45, 256 (100 M) 51 / 46;
//     4096 x 4096, 512 (134 M) 47 / 51, 768 (201 M) 66 / 62; 14336 x 4096, 128
//     (117 M) 49 / 49, 192 (176 M) 69 / 59; 8192 x 8192, 128 (134 M) 48 / 61,
//     192 (201 M) 68 / 65; 4096 x 14336, 192 (176 M) 69 / 83
//   Q4_K, one block of 33 to 64 tokens: 32000 x 4096 (131 M) 53 / 61, 28672 x
//     8192 (235 M) 94 / 89 (48 tokens 81 / 87); 40000 x 2560 (102 M) 54 / 52,
//     65536 x 2560 (168 M) 83 / 57
//   Q6_K 2560 x 2560, 384 (39 M) 40 / 40, 448 (46 M) 48 / 42; 4096 x 4096, 192
//     (50 M) 38 / 45, 256 (67 M) 50 / 47; 2560 x 9728, 192 (75 M) 49 / 58, 256
//     (100 M) 67 / 62; 4096 x 14336, 128 (117 M) 64 / 84, 256 (235 M) 120 / 108
//   Q8_0 2560 x 2560, 384 (39 M) 39 / 41, 448 (46 M) 47 / 42; 4096 x 4096, 192
//     (50 M) 42 / 49, 256 (67 M) 54 / 50; 49152 x 576, 128 (57 M) 66 / 57;
//     4096 x 14336, 128 (117 M) 87 / 92, 192 (176 M) 125 / 119
// Below 8 tokens the GEMV is as fast or faster for one matrix of few rows: 5
// tokens of Q8_0 1024 x 4096 9.8 us there, 11.4 here, 1024 x 28672 37 and 46
// (of 4096 rows 17 and 12); a group's other matrices would pay for a second
// quantization.
constexpr int kSmallMinTokens = 5;
bool gemm_small_take(int type, int n_out, int K, int m) {
    static const int lo = tuning_knob("EXQ_SM_LO", kSmallMinTokens), hi = tuning_knob("EXQ_SM_HI", 0);
    if ((type != kTypeQ8_0 && type != kTypeQ6_K && type != kTypeQ4_K) || m < lo) return false;
    if (hi != 0) return m <= hi;
    const int blocks = (m + 63) / 64;
    if (m <= 32 || (blocks == 1 && type != kTypeQ4_K)) return true;
    if (blocks > 4096) return false;  // (token blocks are a launch's y dimension)
    double line = type == kTypeQ4_K ? fmin(25e6 + 27e3 * K, 200e6) : type == kTypeQ6_K ? 20e6 + 7.5e3 * K : 25e6 + 7.5e3 * K;
    if (blocks == 1) line *= 1.3;  // (its 33 to 64 tokens are 54 on the average)
    return (double)n_out * K * blocks <= line;
}

size_t gemm_small_pack_bytes(int type, int m, int K) {
    const size_t ntt = (size_t)(m + 15) / 16 + 3;  // a launch reads whole groups of up to four tiles
    return type == kTypeQ8_0 ? (size_t)(K / kQK8_0 + 1) / 2 * ntt * kSmPack0 : (size_t)(K / kQKK) * ntt * kSmPackK;
}

static int small_tiles(int m) { return (m + 15) / 16; }

hipError_t launch_small_pack(int type, const float *x, const float *y, float eps, int pro, int m, int K,
                             uint8_t *pack, hipStream_t st) {
    const bool q80 = type == kTypeQ8_0;
    const int nu = q80 ? K / kQK8_0 : K / kQKK, lanes = q80 ? 4 : 16, ntt = small_tiles(m);
    // the RMSNorm holds a row per workgroup; otherwise 256 threads share it out
    int threads = 256;
    if (pro == 1) {
        threads = (nu * lanes + 63) / 64 * 64;
        threads = threads > 1024 ? 1024 : threads < kRmsThreads ? kRmsThreads : threads;
    }
    const dim3 grid((unsigned)m, pro == 1 ? 1u : (unsigned)((nu * lanes + threads - 1) / threads));
    if (q80) {
        auto k = pro == 1 ? small_pack_0_kernel<1> : pro == 2 ? small_pack_0_kernel<2> : small_pack_0_kernel<0>;
        hipLaunchKernelGGL(k, grid, dim3(threads), 0, st, x, y, eps, nu, ntt, pack);
    } else {
        auto k = pro == 1 ? small_pack_k_kernel<1> : pro == 2 ? small_pack_k_kernel<2> : small_pack_k_kernel<0>;
        hipLaunchKernelGGL(k, grid, dim3(threads), 0, st, x, y, eps, nu, ntt, pack);
    }
    return hipGetLastError();
}

hipError_t launch_small_pack_blocks(int type, const uint8_t *xq, size_t xq_stride, int m, int K, uint8_t *pack,
                                    hipStream_t st) {
    const int ntt = small_tiles(m);
    if (type == kTypeQ8_0) {
        const int nb = K / kQK8_0;
        hipLaunchKernelGGL(small_pack_0_blocks_kernel, dim3((unsigned)m, (unsigned)((nb + 63) / 64)), dim3(256), 0, st,
                           xq, xq_stride, nb, ntt, pack);
    } else {
        const int nsb = K / kQKK;
        hipLaunchKernelGGL(small_pack_k_blocks_kernel, dim3((unsigned)m, (unsigned)((nsb + 15) / 16)), dim3(256), 0,
                           st, xq, xq_stride, nsb, ntt, pack);
    }
    return hipGetLastError();
}

// Waves of a workgroup: 16 (128 registers each) where the operands fit in
// them, 8 for Q6_K's 6-bit operands and for more than two token tiles.
constexpr int small_max_waves(int type, int tt) { return type == kTypeQ6_K || tt > 2 ? 8 : 16; }

template <class F, int RT, int TT, bool PAIR>
static void small_launch(const SmallArgs &a, int tiles, int nw, hipStream_t st) {
    constexpr int kMaxW = small_max_waves(F::kType, TT);
    const dim3 grid((unsigned)tiles, (unsigned)((a.ntt + TT - 1) / TT));
    hipLaunchKernelGGL((gemm_small_kernel<F, RT, TT, PAIR, kMaxW>), grid, dim3((unsigned)(64 * nw)), 0, st, a);
}

template <class F>
static hipError_t small_dispatch(const SmallArgs &a, int rt, int tt, bool pair, int tiles, int nw, hipStream_t st) {
#define SM_CASE(T)                                                      \
    case T:                                                             \
        if (pair)                                                       \
            small_launch<F, 2, T, true>(a, tiles, nw, st);              \
        else if (rt == 2)                                               \
            small_launch<F, 2, T, false>(a, tiles, nw, st);             \
        else                                                            \
            small_launch<F, 1, T, false>(a, tiles, nw, st);             \
        break;
    switch (tt) {
        SM_CASE(1)
        SM_CASE(2)
        SM_CASE(3)
        SM_CASE(4)
    }
#undef SM_CASE
    return hipGetLastError();
}

// out[z] = [resid[z] +] (bias[z] + W[z] . pack), or with pair
// out[0] = silu(bias[0] + W[0] . pack) * (bias[1] + W[1] . pack).
hipError_t launch_gemm_small(int type, int nmat, const uint8_t *const *w, const int *n_out, const float *const *bias,
                             const float *const *resid, float *const *out, bool pair, size_t row_bytes, int K, int m,
                             const uint8_t *pack, hipStream_t st) {
    SmallArgs a{};
    a.nmat = nmat;
    a.row_bytes = row_bytes;
    a.pack = pack;
    a.m = m;
    a.ntt = small_tiles(m);
    a.nk = type == kTypeQ8_0 ? K / kQK8_0 : K / kQKK;
    // token tiles per workgroup: all of them up to four, then the count that
    // leaves the fewest empty ones
    const int nblk = (a.ntt + 3) / 4;
    const int tt = (a.ntt + nblk - 1) / nblk;
    // waves: as few K units each as fit (at least two super-blocks, four
    // 32-element blocks: a wave's loads of the second hide behind the first)
    const int maxw = small_max_waves(type, tt);
    static const int k_min = tuning_knob("EXQ_SM_PER", 2), k_max = tuning_knob("EXQ_SM_MAXW", 16);
    const int min_per = type == kTypeQ8_0 ? 4 : k_min;
    const int cap = maxw < k_max ? maxw : k_max;
    int per = (a.nk + cap - 1) / cap;
    per = per < min_per ? min_per : per;
    const int nw = (a.nk + per - 1) / per;
    long long rows = 0;
    for (int z = 0; z < nmat; ++z) rows += n_out[z];
    static const int k_rt = tuning_knob("EXQ_SM_RT", 0);
    // two row tiles a wave where there are workgroups enough: the operands are
    // loaded once for both.  Q6_K from the second token tile keeps one: twice
    // the operands and accumulators leave half the waves per CU (9728 rows of
    // 2560: 20 tokens 26.5 us with two, 21.9 with one; 64 tokens 46.8 and 30.5;
    // 16 tokens of 8192 rows 12.1 and 13.0)
    const bool wide = rows >= 16 * 512 && (type != kTypeQ6_K || tt == 1);
    const int rt = pair ? 2 : k_rt ? k_rt : wide ? 2 : 1;
    int tiles = 0;
    for (int z = 0; z < nmat; ++z) {
        a.w[z] = w[z];
        a.n_out[z] = n_out[z];
        a.bias[z] = bias != nullptr ? bias[z] : nullptr;
        a.resid[z] = resid != nullptr ? resid[z] : nullptr;
        a.out[z] = out[z];
        a.tile0[z] = tiles;
        tiles += (n_out[z] + 16 * rt - 1) / (16 * rt);
    }
    if (pair) tiles = (n_out[0] + 15) / 16;
    if (type == kTypeQ8_0) return small_dispatch<SmallQ80>(a, rt, tt, pair, tiles, nw, st);
    if (type == kTypeQ6_K) return small_dispatch<SmallQ6K>(a, rt, tt, pair, tiles, nw, st);
    return small_dispatch<SmallQ4K>(a, rt, tt, pair, tiles, nw, st);
}
