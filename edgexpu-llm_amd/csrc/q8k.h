// Q8_K quantization of one 256-element block by one wavefront (lane l owns
// elements 4l..4l+3): edgexpu_gguf_quantize_q8_k, src/gguf_dot_q8.c:360-412.
//   maxv   = signed value of the first element with the largest |x| (strict '>'
//            from amax = 0, so zeros and NaN never win)
//   iscale = -127 / maxv, q = clamp(lrintf(iscale * x), -127, 127)
//   bsums  = int16 sums of 16 consecutive q, d = 1 / iscale
//   an all-zero block (maxv == 0) is stored as zeros.
// Shared by the Q8_K block writer (quantize.hip) and the prefill GEMM's
// operand packers (gemm.hip, gemm_small.hip), so all produce the same codes
// bit for bit.
#pragma once

#include "common.h"

namespace exq {

struct Q8KLane {
    uint32_t word;  // the lane's 4 codes, element 4l+e in byte e
    int q[4];       // the same codes as integers
    int sum4;       // sum of the lane's 4 codes
    float d;        // block scale (0 for an all-zero block)
    bool zero;      // all-zero block
};

__device__ __forceinline__ Q8KLane q8k_quantize_lane(const float4 v, int lane) {
    const float xs[4] = {v.x, v.y, v.z, v.w};
    // First-index signed maximum of |x| (zeros and NaN never enter): the
    // largest magnitude over the wave as bits (non-negative floats order as
    // their bits), then the first lane holding it (ballot) and its first
    // element there; the sign is that element's.
    uint32_t b[4], amax_bits = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float av = fabsf(xs[e]);
        b[e] = av > 0.0f ? __float_as_uint(av) : 0u;
        amax_bits = max(amax_bits, b[e]);
    }
    amax_bits = row16_max_u32(amax_bits);
    amax_bits = max(amax_bits, (uint32_t)__shfl_xor((int)amax_bits, 16, 64));
    amax_bits = max(amax_bits, (uint32_t)__shfl_xor((int)amax_bits, 32, 64));
    bool hit = false, neg = false;
#pragma unroll
    for (int e = 3; e >= 0; --e) {  // the first element of this lane wins
        const bool h = amax_bits != 0u && b[e] == amax_bits;
        neg = h ? xs[e] < 0.0f : neg;
        hit = hit || h;
    }
    const unsigned long long hits = __ballot(hit);
    const int first = hits != 0ull ? __ffsll((long long)hits) - 1 : 0;
    const bool negative = __shfl((int)neg, first, 64) != 0;
    (void)lane;
    Q8KLane r;
    r.zero = amax_bits == 0u;
    r.word = 0u;
    r.sum4 = 0;
    r.d = 0.0f;
    r.q[0] = r.q[1] = r.q[2] = r.q[3] = 0;
    if (r.zero) return r;  // wavefront-uniform
    const float amax = __uint_as_float(amax_bits);
    const float maxv = negative ? -amax : amax;
    const float iscale = -127.0f / maxv;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float p = iscale * xs[e];
        // lrintf: a NaN or infinite product gives LONG_MIN, whose low 32 bits are 0.
        int q = fabsf(p) < 2147483648.0f ? (int)rintf(p) : 0;
        q = q > 127 ? 127 : (q < -127 ? -127 : q);
        r.q[e] = q;
        r.sum4 += q;
        r.word |= (uint32_t)(q & 0xff) << (8 * e);
    }
    r.d = 1.0f / iscale;
    return r;
}

// One 256-element block by 16 lanes of a DPP row: lane 4 j + q holds its
// elements 64 j + 8 q .. + 7 in xs[0..7] and 64 j + 32 + 8 q .. + 7 in
// xs[8..15], and gets their codes in qv.  The largest |x| (zeros and NaN never
// enter) by a row max, then iscale = -127 / max|x| and each code as above.
// The reference's max carries the sign of the first element of largest |x|;
// where that is negative, this block is the reference's with codes, sums and
// d negated, which a product dx * (C d - mn dmin), with C and mn integer sums
// of the codes, leaves word for word (sum |q| is the same either way).
struct Q8KRow16 {
    float d;
    int sq;                        // sum |q| of the block, in every lane
    int lo, lo_next, hi, hi_next;  // lanes q = 0: the 16-element sums 4 j .. 4 j + 3
};

__device__ __forceinline__ Q8KRow16 q8k_quantize_row16(const float (&xs)[16], int (&qv)[16]) {
    uint32_t amax_bits = 0u;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float av = fabsf(xs[i]);
        amax_bits = max(amax_bits, av > 0.0f ? __float_as_uint(av) : 0u);  // non-negative floats order as their bits
    }
    amax_bits = row16_max_u32(amax_bits);
    const bool zero = amax_bits == 0u;
    const float iscale = -127.0f / __uint_as_float(amax_bits);
    Q8KRow16 r;
    r.lo = r.hi = r.sq = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float pv = iscale * xs[i];
        // lrintf: a NaN or infinite product gives LONG_MIN, whose low 32 bits are 0
        int c = fabsf(pv) < 2147483648.0f ? (int)rintf(pv) : 0;
        c = c > 127 ? 127 : (c < -127 ? -127 : c);
        c = zero ? 0 : c;
        qv[i] = c;
        if (i < 8)
            r.lo += c;
        else
            r.hi += c;
        r.sq += abs(c);
    }
    r.d = zero ? 0.0f : 1.0f / iscale;
    // lanes q and q ^ 1 share the 16-element groups 4 j + q / 2 (low) and
    // 4 j + 2 + q / 2 (high); lane q = 0 then takes groups 4 j + 1 and 4 j + 3
    // from lane q = 2
    r.lo += (int)dpp_u32<kDppXor1>((uint32_t)r.lo);
    r.hi += (int)dpp_u32<kDppXor1>((uint32_t)r.hi);
    r.lo_next = (int)dpp_u32<kDppXor2>((uint32_t)r.lo);
    r.hi_next = (int)dpp_u32<kDppXor2>((uint32_t)r.hi);
    r.sq += (int)dpp_u32<kDppXor1>((uint32_t)r.sq);
    r.sq += (int)dpp_u32<kDppXor2>((uint32_t)r.sq);
    r.sq += (int)dpp_u32<kDppHalfMirror>((uint32_t)r.sq);
    r.sq += (int)dpp_u32<kDppMirror>((uint32_t)r.sq);
    return r;
}

}  // namespace exq
