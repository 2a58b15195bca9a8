// prep_batch.hip -- RMSNorm, sign flip, blockwise WHT and absmax INT8 of many token rows, one wave a row.
//
// prep_spec_kernel (qlinear.hip) spreads a row over 10 to 16 waves, which suits one row: the chain a wave runs is short.
// A batch of rows is bound by memory instead, and there most of a workgroup's time was its launch, two barriers and
// a chain of dependent loads and reductions with little in flight. Here a wave holds a whole row in registers: all of
// its loads are in flight at once, nothing is shared and there is no barrier.
//
// Lane l holds columns 512 c + 8 l .. + 7 of chunk c. The butterflies, maxima and codes do not depend on which lane
// holds a column; the RMSNorm's sum of squares does, and is added in prep_spec_kernel's order (its threads' 4
// columns, butterflies over 16 of its lanes, the four row sums of its wave, butterflies over its waves), so that codes
// and scales have the bits of that kernel and of the fused prep.
#include <type_traits>

#include "qdev.h"
#include "prep_batch.h"

namespace {

constexpr int kRowsWg = 4;   // rows (waves) of a workgroup

// NCH chunks of 512 columns cover ldq; LB as in prep_finish.
template <int NCH, int LB>
__global__ __launch_bounds__(64 * kRowsWg) void prep_batch_kernel(eif::PrepBatch p)
{
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * kRowsWg + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (m >= p.M) return;   // uniform over the wave; no barrier in this kernel
    const int block = LB >= 0 ? (LB > 0 ? 1 << LB : 0) : p.block;
    const float *xr = p.x + (size_t)m * p.ldx;
    float v[NCH][8];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int i0 = 512 * c + 8 * lane;
        load4<8>(xr, i0 < p.K ? i0 : 0, v[c]);
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
        if (512 * c + 8 * lane >= p.K) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] = 0.0f;
        }
    // W[w]: the sum of wave w of prep_spec_kernel (256 columns), then the butterfly over its waves
    static_assert(2 * NCH <= 16, "the waves of its workgroup");
    float W[16];
#pragma unroll
    for (int w = 0; w < 16; ++w) W[w] = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        float a = 0.0f, b = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) a = fmaf(v[c][e], v[c][e], a), b = fmaf(v[c][4 + e], v[c][4 + e], b);
        float s = a + b;   // its lanes 2l, 2l + 1
        s = s + xlane<1>(s);
        s = s + xlane<2>(s);
        s = s + xlane<4>(s);   // 8 lanes here, 16 there
        float q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 8 * i));
        W[2 * c] = ((q[0] + q[1]) + q[2]) + q[3];
        W[2 * c + 1] = ((q[4] + q[5]) + q[6]) + q[7];
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1)
#pragma unroll
        for (int w = 0; w < 16; w += 2 * o) W[w] = W[w] + W[w + o];
    const float ss = ((W[0] + 0.0f) + 0.0f) + 0.0f;
    const float r = 1.0f / sqrtf(ss / (float)p.K + p.eps);
    auto mul = [&](const float *f) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int i0 = 512 * c + 8 * lane;
            float u[8];
            load4<8>(f, i0 < p.K ? i0 : 0, u);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] = v[c][e] * u[e];
        }
    };
    if (p.nw) mul(p.nw);
    if (block > 0 && p.signs) mul(p.signs);
    float amax = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        float(&u)[8] = v[c];
#pragma unroll
        for (int h = 1; h < 8; h <<= 1) {
            if (h < block) {   // uniform
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if ((e & h) == 0) {
                        const float a = u[e], b = u[e + h];
                        u[e] = a + b;
                        u[e + h] = a - b;
                    }
            }
        }
        if (block > 8) wht_cross<1>(u, lane);
        if (block > 16) wht_cross<2>(u, lane);
        if (block > 32) wht_cross<4>(u, lane);
        if (block > 64) wht_cross<8>(u, lane);
        if (block > 128) wht_cross<16>(u, lane);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (block > 0) u[e] = u[e] * p.norm;
            amax = fmaxf(amax, fabsf(u[e]));
        }
    }
    amax = wave_max_dpp(amax);
    const float amax_n = amax * r;
    const bool zero = amax_n < 1e-12f;
    const float inv = zero ? 0.0f : 127.0f / amax;
    if (lane == 0) p.xs[m] = zero ? 1.0f : amax_n * (1.0f / 127.0f);
    int8_t *q = p.xq + (size_t)m * p.ldq;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int i0 = 512 * c + 8 * lane;
        if (i0 >= p.ldq) continue;   // ldq is a multiple of 16
        uint32_t d[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            uint32_t u = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) u |= ((uint32_t)quant1(v[c][4 * k + b], inv) & 0xFFu) << (8 * b);
            d[k] = u;
        }
        *reinterpret_cast<uint2 *>(q + i0) = make_uint2(d[0], d[1]);
    }
}

template <int NCH, int LB>
int go(const eif::PrepBatch &p, hipStream_t st)
{
    prep_batch_kernel<NCH, LB><<<eif_ceil_div(p.M, kRowsWg), 64 * kRowsWg, 0, st>>>(p);
    EIF_HIP_LAUNCHED();
    return EIF_HIP_OK;
}

}  // namespace

namespace eif {

// RMSNorm rows where this form is ahead of prep_spec_kernel with 4 columns a thread, which it replaces (kernel times, us,
// one workgroup a row / one wave a row, inputs rotated past the Infinity Cache):
// - without rotation from 1024 rows on up to five chunks of columns, from 2048 on up to eight, where a wave's registers
//   leave fewer of them on a SIMD (K = 896 at 1024 / 3001 rows 4.6 / 4.2, 8.1 / 7.1; 1280 5.4 / 5.3, 9.4 / 8.2; 2048 6.8 /
//   6.3, 11.2 / 9.8; 2560 8.6 / 7.3, 16.3 / 11.4, at 512 5.3 / 5.6; 3584 at 1500 rows 12.0 / 12.5, at 2048 13.6 / 11.5; 4096
//   at 1300 rows 11.9 / 12.3, at 2048 14.0 / 12.7);
// - with rotation for 2305 to 2560 columns from 1024 rows on, where the other form's ten waves a row no longer fill a CU
//   evenly (K = 2432 at 1024 / 3001 rows 9.9 / 9.2, 19.5 / 15.4; 2560 9.9 / 9.2, 19.5 / 15.8; WHT-64 10.7 / 9.5, 21.5 / 15.6;
//   2336 with WHT-32 10.3 / 9.0, 20.9 / 14.1). For fewer columns (K = 2304 at 1024 / 2300 rows 8.4 / 9.1, 13.0 / 13.6; 1536
//   6.6 / 7.2, 10.7 / 11.5) or more (2688 at 1024 rows 9.4 / 10.2, 3584 11.0 / 12.9) a lane's chain of butterflies is too
//   long for its few waves.
// Without a norm the two are level; the SwiGLU pre-op's 108 exponentials a lane are too long a chain (K = 6912, 512 rows 9.9 /
// 21.0, 3001 rows 47.4 / 46.9).
int launch_prep_batch(const PrepBatch &p, hipStream_t st)
{
    if (p.pre != EIF_HIP_PRE_RMS || p.M < 1024 || p.block > 256) return 1;
    if (p.block > 0) {
        if (p.ldq <= 2304 || p.ldq > 2560) return 1;
        return p.block == 128 ? go<5, 7>(p, st) : go<5, -1>(p, st);
    }
    if (p.ldq > 4096 || (p.ldq > 2560 && p.M < 2048)) return 1;
    const int nch = eif_ceil_div(p.ldq, 512);
    if (nch <= 2) return go<2, 0>(p, st);
    if (nch <= 4) return go<4, 0>(p, st);
    if (nch <= 5) return go<5, 0>(p, st);
    if (nch <= 6) return go<6, 0>(p, st);
    return go<8, 0>(p, st);
}

}  // namespace eif
