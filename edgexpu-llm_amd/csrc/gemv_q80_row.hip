// One token of short Q8_0 rows (up to 2048 elements) against a few thousand
// rows: q/k/v, o, gate / up and down of a small model's decode step, where a
// launch is a chain of latencies and nothing is bound by bytes.
//
// The fused GEMV (gemv_fused_kernel.h) gives these shapes 18 to 96 workgroups
// of eight waves with two to four rows a lane slot, and its general schedule
// is several times the code; a step of 123 such launches, each kernel entered
// anew, ran at 5.4 us a launch where an empty kernel takes 1.6.  Here a wave
// has 64 / G rows (G lanes a row, one 32-element block a lane), a workgroup
// four waves, every load of the launch goes out before the first wait, and
// there is no loop: 3 to 4 times the workgroups and a short straight path.
// Measured back to back: o [576 x 576] 3.9 us before, 2.6 us so, q/k/v with
// the RMSNorm 4.4 and 2.9, gate / up 5.0 and 3.7, down [576 x 1536] 4.7 and
// 2.7; the SmolLM2-135M decode step 602 us before, 420 us so.
//
// Arithmetic as the fused GEMV's, word for word: the Q8_0 quantizer of
// quantize_q8_0_kernel on the (RMSNorm-ed, SiLU-multiplied or plain) input,
// each block (d * dx) * (int dot), lanes summed by partners ^ G/2 .. ^ 1, then
// residual + (bias + dot), or silu(gate) * up.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "common.h"

namespace exq {

constexpr int kRowWaves = 4;
constexpr int kRowThreads = 64 * kRowWaves;
constexpr int kRowMaxK = 8 * kRowThreads;  // the input is staged in one round, 8 elements a thread

struct RowArgs {
    const uint8_t *w[4];
    const float *bias[4], *resid[4];
    float *out[4];
    int n_out[4];
    int tile0[4];  // first workgroup of each matrix
    int nmat;
    int row_bytes, nb;
    const float *x, *y;  // y: RMSNorm weight (PRO 1) or the SiLU's factor (PRO 2)
    float eps;
};

__device__ __forceinline__ void row_load8(const float *p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// PAIR: w[0] is gate, w[1] up, out[0] = silu(gate) * up.
template <int G, int PRO, bool PAIR>
__global__ __launch_bounds__(kRowThreads) void gemv_q80_row_kernel(RowArgs a) {
    __shared__ __align__(16) uint32_t codes[kRowMaxK / 4];
    __shared__ float scales[kRowMaxK / kQK8_0];
    constexpr int S = 64 / G, R = PAIR ? 2 : 1;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int tile = (int)blockIdx.x;
    int z = 0;
    if (!PAIR)
        while (z + 1 < a.nmat && tile >= a.tile0[z + 1]) ++z;
    const int n_out = a.n_out[z];
    const int row = (tile - a.tile0[z]) * (kRowWaves * S) + wave * S + lane / G;
    const int gl = lane & (G - 1);

    // the thread's 8 elements (clamped: a thread past the row repeats its last
    // block's), then the lane's weight blocks
    const int blk = (int)threadIdx.x >> 2;
    const bool stages = blk < a.nb;
    const int e0 = min(blk, a.nb - 1) * kQK8_0 + 8 * (threadIdx.x & 3);
    float v[8], y[8];
    row_load8(a.x + e0, v);
    if (PRO != 0) row_load8(a.y + e0, y);
    uint4 q0[R], q1[R];
    uint32_t wd[R];
    float bias[R];
    const int rc = min(row, n_out - 1), bc = min(gl, a.nb - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint8_t *p = a.w[PAIR ? r : z] + (size_t)rc * a.row_bytes + (size_t)bc * kBytesQ8_0;
        q0[r] = ldg16_a2(p + 2);
        q1[r] = ldg16_a2(p + 18);
        wd[r] = *reinterpret_cast<const uint16_t *>(p);
        const float *b = a.bias[PAIR ? r : z];
        bias[r] = b != nullptr ? b[rc] : 0.0f;
    }
    const float *rs = PAIR ? nullptr : a.resid[z];
    const float res = rs != nullptr ? rs[rc] : 0.0f;
    __builtin_amdgcn_sched_barrier(0);

    if (PRO == 1) {
        // the fused GEMV's sum, whose thread f holds elements 4 f .. 4 f + 3: this
        // thread's two such sums, each over 32 lanes here by the partners of its
        // 64, then their sum
        __shared__ double part[2 * kRowWaves];
        double s[2] = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i >> 2] += (double)v[i] * (double)v[i];  // a float square is exact in double
        const double sum = wave_sum_f64<32>(stages ? s[0] : 0.0) + wave_sum_f64<32>(stages ? s[1] : 0.0);
        if ((lane & 31) == 0) part[threadIdx.x >> 5] = sum;
        __syncthreads();
        double ss = 0.0;
#pragma unroll
        for (int w = 0; w < 2 * kRowWaves; ++w) ss += part[w];
        const float scale = rms_scale(ss, a.nb * kQK8_0, a.eps);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float t = v[i] * scale;
            v[i] = t * y[i];
        }
    } else if (PRO == 2) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = silu_f32(v[i]) * y[i];
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(amax))));
    amax = fmaxf(amax, __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(amax))));
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    uint32_t word[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float t = rintf(v[i] * id);
        int c = (t >= -2147483648.0f && t < 2147483648.0f) ? (int)t : INT32_MIN;
        c = c < -128 ? -128 : (c > 127 ? 127 : c);
        word[i >> 2] |= (uint32_t)(c & 0xff) << (8 * (i & 3));
    }
    if (stages) {
        *reinterpret_cast<uint2 *>(codes + 2 * threadIdx.x) = make_uint2(word[0], word[1]);
        if ((threadIdx.x & 3) == 0) scales[blk] = f16_bits_to_f32(f32_to_f16_rne(amax / 127.0f));
    }
    __syncthreads();

    const uint4 x0 = *reinterpret_cast<const uint4 *>(codes + 8 * bc);
    const uint4 x1 = *reinterpret_cast<const uint4 *>(codes + 8 * bc + 4);
    const float dx = scales[bc];
    float sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int s = sdot4(q0[r].x, x0.x, 0);
        s = sdot4(q0[r].y, x0.y, s);
        s = sdot4(q0[r].z, x0.z, s);
        s = sdot4(q0[r].w, x0.w, s);
        s = sdot4(q1[r].x, x1.x, s);
        s = sdot4(q1[r].y, x1.y, s);
        s = sdot4(q1[r].z, x1.z, s);
        s = sdot4(q1[r].w, x1.w, s);
        sum[r] = gl < a.nb ? (f16_bits_to_f32(wd[r]) * dx) * (float)s : 0.0f;
#pragma unroll
        for (int off = G / 2; off > 0; off >>= 1) sum[r] += reduce_partner(sum[r], off);
    }
    if (gl != 0 || row >= n_out) return;
    const float o = bias[0] + sum[0];
    if (PAIR)
        a.out[0][row] = silu_f32(o) * (bias[R - 1] + sum[R - 1]);
    else
        a.out[z][row] = rs != nullptr ? res + o : o;
}

}  // namespace exq

using namespace exq;

// One token of Q8_0 rows, staged, of at most kRowMaxK elements, up to 8192 of
// them: a workgroup stages the input for 4 to 16 rows only, which long launches
// get nothing for (fused / this, us: 8192 rows of 576 5.3 / 4.0, of 2048 6.6 /
// 5.7; 16384 rows of 256 5.4 / 6.4, of 576 5.9 / 5.5, of 2048 9.6 / 8.9; 131072
// rows of 2048 54 / 55).
bool gemv_q80_row_take(int type, int K, int m, long long rows, bool staged) {
    static const long long max_rows = tuning_knob("EXQ_ROW_MAX", 8192);
    return type == kTypeQ8_0 && staged && m == 1 && K <= kRowMaxK && rows <= max_rows;
}

hipError_t launch_gemv_q80_row(int nmat, const uint8_t *const *w, const int *n_out, const float *const *bias,
                               const float *const *resid, float *const *out, int K, const float *x, const float *x2,
                               const float *nw, float eps, int pro, bool pair, hipStream_t st) {
    RowArgs a{};
    a.nmat = nmat;
    a.nb = K / kQK8_0;
    a.row_bytes = a.nb * kBytesQ8_0;
    a.x = x;
    a.y = pro == 1 ? nw : x2;
    a.eps = eps;
    const int g = a.nb <= 16 ? 16 : a.nb <= 32 ? 32 : 64;
    const int rows_wg = kRowWaves * (64 / g);
    int tiles = 0;
    for (int z = 0; z < nmat; ++z) {
        a.w[z] = w[z];
        a.n_out[z] = n_out[z];
        a.bias[z] = bias != nullptr ? bias[z] : nullptr;
        a.resid[z] = resid != nullptr ? resid[z] : nullptr;
        a.out[z] = out[z];
        a.tile0[z] = tiles;
        if (!pair || z == 0) tiles += (n_out[z] + rows_wg - 1) / rows_wg;
    }
    const auto launch = [&](auto lanes) {
        constexpr int kG = decltype(lanes)::value;
        auto k = pair ? (pro == 1 ? gemv_q80_row_kernel<kG, 1, true> : gemv_q80_row_kernel<kG, 0, true>)
                      : (pro == 1   ? gemv_q80_row_kernel<kG, 1, false>
                         : pro == 2 ? gemv_q80_row_kernel<kG, 2, false>
                                    : gemv_q80_row_kernel<kG, 0, false>);
        hipLaunchKernelGGL(k, dim3((unsigned)tiles), dim3(kRowThreads), 0, st, a);
    };
    if (g == 16)
        launch(std::integral_constant<int, 16>());
    else if (g == 32)
        launch(std::integral_constant<int, 32>());
    else
        launch(std::integral_constant<int, 64>());
    return hipGetLastError();
}
