// attn_prefill.hip -- causal softmax attention of a prompt batch (the token loop of src/eif_tinyllm.c:1020-1500) over the
// fp16 KV cache, on f16 MFMAs with FP32 precision.
//
// On FP32 MFMAs (32 times fewer operations a cycle than f16 ones) the matrix products alone took a third of the time, and
// 16-query x 16-key tiles spent the rest on reductions across lanes, on LDS traffic and on shares written per 128 keys.
// Here the keys and values, which the cache holds in fp16, are MFMA operands as they are, and the FP32 side (the
// queries; the probabilities) is split exactly into two f16 terms, hi = f16(x), lo = f16(x - hi): 22 bits, whose
// remainder of 2^-23 or less of an element is below what FP32 accumulation rounds. Products of f16 are exact in FP32 and
// the sums are FP32, so nothing is held in 16 bits that was not before. Error against 64 bits (2-norm, queries and keys
// normal, 20 heads of 128): 1900 tokens 3.6e-7 on FP32 MFMAs, 2.6e-7 here; queries 4 times as large 1.07e-6, 7.2e-7;
// 511 tokens 3.6e-7, 2.1e-7; a tenth as large at positions 1100 .. 1999 2.2e-7, 2.3e-7. (Three terms: 2.6e-7, 7.2e-7, 2.1e-7,
// 2.3e-7, 15% slower.)
//
// A wave takes 32 queries of one head. S^T = K Q^T (v_mfma_f32_32x32x16_f16, rows = keys) leaves lane (c, h) =
// (lane % 32, lane / 32) with scores of query c alone, so the softmax needs one exchange between the halves per 32
// keys, and the probabilities are already the B operand of O^T += V^T P^T: lane half h holds keys 8 q + 4 h + i (q =
// 0 .. 3, i = 0 .. 3), and the staged values are laid out in that order of keys. The four waves of a workgroup are the
// query heads of a kv head (or more queries of it) on the same staged keys and values.
//
// Measured (us a layer, 20 query and 5 kv heads of 128, both kernels of it): 1900 tokens 389 on FP32 MFMAs, 111 here;
// 1024 142, 52; 511 50, 31; 256 29, 20; 64 14.4, 10.6; 900 at position 1100 314, 84. Up to 16 tokens, one block of the FP32
// kernel, that one is ahead (16 tokens 6.9 against 7.8) and stays (decode.hip).
#include <algorithm>

#include "attn_prefill.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kTerms = 2;
constexpr int kKeys = eif::kPfKeys;
constexpr float kPScale = 16384.0f;   // P is split times 2^14, so that its low terms stay normal f16 numbers

// Eight FP32 values as a sum of kTerms f16 vectors (each the rounded remainder of those before it).
EIF_DEV void split8(const float (&x)[8], v8h (&o)[kTerms])
{
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float r = x[e];
#pragma unroll
        for (int t = 0; t < kTerms; ++t) {
            const _Float16 hv = (_Float16)r;
            o[t][e] = hv;
            r = r - (float)hv;
        }
    }
}

template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void attn_prefill_kernel(eif::PrefillAttn a, int heads_wg, int qb, int ct, int s_call, float inv_sqrt_hd)
{
    constexpr int CH = HD / 16, DT = HD / 32, KP = HD / 8;   // dim chunks of S, dim tiles of O, 16-byte pieces of a row
    constexpr int KSW = KP >= 8 ? 7 : 3;
    __shared__ __align__(16) uint8_t k_l[2][kKeys * HD * 2];   // [key][piece ^ swizzle]
    __shared__ __align__(16) uint8_t v_l[2][HD * kKeys * 2];   // [dim][piece ^ swizzle]: keys in the order P's lanes hold them
    auto vswz = [](int dim) { return ((dim >> 1) + (dim >> 3)) & 3; };
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c32 = lane & 31, h = lane >> 5;
    const int kv_mul = a.n_heads / a.n_kv, parts = (kv_mul + heads_wg - 1) / heads_wg;
    const int g = blockIdx.x / parts, part = blockIdx.x - g * parts;
    const int hw = part * heads_wg + w % heads_wg, qs = w / heads_wg;
    const int nblk = gridDim.y / s_call, by = blockIdx.y / s_call, sp = blockIdx.y - by * s_call;
    const int b = nblk - 1 - by;                     // the longest ranges first
    const int ib = b * 32 * qb, i0 = ib + 32 * qs;   // the workgroup's and this wave's first query
    const bool active = qs < qb && hw < kv_mul && i0 < a.n;   // uniform over the wave
    const int head = g * kv_mul + (hw < kv_mul ? hw : 0);
    const int n_keys = a.pos0 + min(ib + 32 * qb, a.n), all_tiles = (n_keys + kKeys - 1) / kKeys;
    const int t0 = sp * ct, t1 = min(t0 + ct, all_tiles);
    if (t0 >= t1) return;   // uniform over the workgroup
    const bool split = all_tiles > ct;
    const __half *kg = a.kc + (size_t)g * a.seq_len * HD, *vg = a.vc + (size_t)g * a.seq_len * HD;

    // the wave's queries: lane (c32, h) holds dims 16 c + 8 h .. + 7 of query i0 + c32, times a power of two that
    // brings the row's largest element to 2^13 .. 2^14 (an exact scaling), split into f16 terms
    v8h q[CH][kTerms];
    float sinv;
    {
        const float *qp = a.qkv + (size_t)min(i0 + c32, a.n - 1) * a.ldqkv + head * HD + 8 * h;
        float x[CH][8], mx = 0.0f;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const float4 f0 = *reinterpret_cast<const float4 *>(qp + 16 * c), f1 = *reinterpret_cast<const float4 *>(qp + 16 * c + 4);
            x[c][0] = f0.x, x[c][1] = f0.y, x[c][2] = f0.z, x[c][3] = f0.w;
            x[c][4] = f1.x, x[c][5] = f1.y, x[c][6] = f1.z, x[c][7] = f1.w;
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[c][e]));
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const int ex = (int)(__float_as_uint(mx) >> 23) & 255;
        const int se = ex == 255 ? 127 : min(267 - ex, 253);
        const float sc = __uint_as_float((uint32_t)se << 23), rs = __uint_as_float((uint32_t)(254 - se) << 23);
        sinv = inv_sqrt_hd * rs;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[c][e] *= sc;
            split8(x[c], q[c]);
        }
    }

    // staging of a tile: thread t takes pieces t, t + 256, ... of the keys, and the 4 keys x 8 dims units of the values
    constexpr int KN = (kKeys * KP + 255) / 256, VU = kKeys / 2 * KP;   // key pieces a thread, value units of a tile
    v4u kr[KN], vr[2];
    const int vu = min(t, VU - 1), ve = vu % KP, vc = vu / KP;   // dims 8 ve .. + 7 of keys 2 vc and 2 vc + 1
    auto fetch = [&](int kt) __attribute__((always_inline)) {
        const int k0 = kKeys * kt;
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const int idx = min(t + 256 * i, kKeys * KP - 1), key = idx / KP, p = idx - key * KP;
            kr[i] = *reinterpret_cast<const v4u *>(kg + (size_t)min(k0 + key, n_keys - 1) * HD + 8 * p);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
            vr[i] = *reinterpret_cast<const v4u *>(vg + (size_t)min(k0 + 2 * vc + i, n_keys - 1) * HD + 8 * ve);
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const int idx = min(t + 256 * i, kKeys * KP - 1), key = idx / KP, p = idx - key * KP;
            const int sw = KP >= 8 ? key & KSW : (key >> 1) & KSW;
            *reinterpret_cast<v4u *>(&k_l[buf][key * HD * 2 + 16 * (p ^ sw)]) = kr[i];
        }
        if (t < VU) {
            // dim 8 ve + d's two keys are 4 bytes of its row, where P's lanes hold these keys
            const int kk = 2 * vc, qd = kk >> 3, piece = (qd >> 1) * 2 + ((kk >> 2) & 1), byte = 8 * (qd & 1) + 2 * (kk & 3);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const int dim = 8 * ve + d;
                *reinterpret_cast<uint32_t *>(&v_l[buf][dim * kKeys * 2 + 16 * (piece ^ vswz(dim)) + byte]) =
                    __builtin_amdgcn_perm(vr[1][d >> 1], vr[0][d >> 1], d & 1 ? 0x07060302u : 0x05040100u);
            }
        }
    };

    v16f O[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) O[d] = v16f{};
    float m = -INFINITY, l = 0.0f;   // of query c32; l over this half's keys
    const int qpos = a.pos0 + i0 + c32, wlast = a.pos0 + min(i0 + 31, a.n - 1);
    const int ksw = KP >= 8 ? c32 & KSW : (c32 >> 1) & KSW;

    fetch(t0);
    stage(t0 & 1);
    __syncthreads();
    for (int kt = t0; kt < t1; ++kt) {
        const int buf = kt & 1, k0 = kKeys * kt;
        fetch(min(kt + 1, t1 - 1));
        if (active && k0 <= wlast) {   // uniform over the wave
            v16f S = v16f{};
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const v8h kf = *reinterpret_cast<const v8h *>(&k_l[buf][c32 * HD * 2 + 16 * ((2 * c + h) ^ ksw)]);
#pragma unroll
                for (int tm = kTerms - 1; tm >= 0; --tm) S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, q[c][tm], S, 0, 0, 0);
            }
            float mx = -INFINITY;
            if (k0 + 31 > a.pos0 + i0) {   // uniform: keys past some query (also past the last key)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = k0 + 8 * (v / 4) + 4 * h + v % 4;
                    S[v] = key <= qpos ? S[v] * sinv : -INFINITY;
                    mx = fmaxf(mx, S[v]);
                }
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v) S[v] = S[v] * sinv, mx = fmaxf(mx, S[v]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m, mx);
            const bool none = mn == -INFINITY;   // no key of the range at or before the query yet
            if (__any(mn > m)) {
                const float sc = none ? 1.0f : expf(m - mn);
                l = l * sc;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int v = 0; v < 16; ++v) O[d][v] *= sc;
                m = mn;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float pw = none ? 0.0f : expf(S[8 * j + e] - mn);
                    l += pw;
                    p[e] = pw * kPScale;
                }
                v8h pt[kTerms];
                split8(p, pt);
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const int dim = 32 * d + c32;
                    const v8h vf = *reinterpret_cast<const v8h *>(
                        &v_l[buf][dim * kKeys * 2 + 16 * ((2 * j + h) ^ vswz(dim))]);
#pragma unroll
                    for (int tm = kTerms - 1; tm >= 0; --tm)
                        O[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pt[tm], O[d], 0, 0, 0);
                }
            }
        }
        stage(buf ^ 1);
        __syncthreads();
    }
    if (!active) return;
    const float lt = l + __shfl_xor(l, 32, 64);
    const int qi = i0 + c32;
    if (qi >= a.n) return;
    if (split) {   // share (b, sp): [b][sp][head][32 qb rows]
        const size_t e = (((size_t)b * s_call + sp) * a.n_heads + head) * (32 * qb) + 32 * qs + c32;
        float *op = a.po + e * HD + 4 * h;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int v = 0; v < 16; v += 4)
                *reinterpret_cast<float4 *>(op + 32 * d + 2 * v) =
                    make_float4(O[d][v] * (1.0f / kPScale), O[d][v + 1] * (1.0f / kPScale), O[d][v + 2] * (1.0f / kPScale),
                                O[d][v + 3] * (1.0f / kPScale));
        if (h == 0) a.pml[2 * e] = m, a.pml[2 * e + 1] = lt;
    } else {
        float *op = a.out + (size_t)qi * a.ldo + head * HD + 4 * h;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int v = 0; v < 16; v += 4)
                *reinterpret_cast<float4 *>(op + 32 * d + 2 * v) =
                    make_float4(O[d][v] * (1.0f / kPScale) / lt, O[d][v + 1] * (1.0f / kPScale) / lt,
                                O[d][v + 2] * (1.0f / kPScale) / lt, O[d][v + 3] * (1.0f / kPScale) / lt);
    }
}

// Blocks whose causal range was split: out = sum_s e^(m_s - M) O_s / sum_s e^(m_s - M) l_s over the block's shares,
// M = max_s m_s (a share with m_s = -inf weighs 0). Workgroup (token i, head), HD threads.
template <int HD>
__global__ __launch_bounds__(128) void attn_prefill_combine_kernel(eif::PrefillAttn a, int qb, int ct, int s_call)
{
    const int i = blockIdx.x, h = blockIdx.y, d = threadIdx.x, rows = 32 * qb;
    const int b = i / rows, row = i - rows * b;
    const int all_tiles = (a.pos0 + min(rows * (b + 1), a.n) + kKeys - 1) / kKeys;
    if (all_tiles <= ct) return;   // written by the attention kernel
    const int ns = (all_tiles + ct - 1) / ct;
    const size_t e0 = ((size_t)b * s_call * a.n_heads + h) * rows + row, es = (size_t)a.n_heads * rows;
    float mx = -INFINITY;
    for (int s = 0; s < ns; ++s) mx = fmaxf(mx, a.pml[2 * (e0 + s * es)]);
    float os = 0.0f, ls = 0.0f;
    for (int s = 0; s < ns; ++s) {
        const size_t e = e0 + s * es;
        const float ms = a.pml[2 * e];
        const float wgt = ms == -INFINITY ? 0.0f : expf(ms - mx);
        os = fmaf(wgt, a.po[e * HD + d], os);
        ls = fmaf(wgt, a.pml[2 * e + 1], ls);
    }
    a.out[(size_t)i * a.ldo + h * HD + d] = os / ls;
}

// Query heads and 32-query sub-blocks of a workgroup's four waves: heads of one kv head share its staged keys and
// values; a kv head of one or two query heads takes more queries instead.
void shape(int kv_mul, int *heads_wg, int *qb)
{
    *heads_wg = kv_mul >= 3 ? std::min(kv_mul, 4) : kv_mul;
    *qb = kv_mul >= 3 ? 1 : 4 / kv_mul;
}

int cus()
{
    static const int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
            return 256;
        return v;
    }();
    return n;
}

template <int HD>
int launch(const eif::PrefillAttn &a, hipStream_t st)
{
    int hw, qb;
    const int kv_mul = a.n_heads / a.n_kv;
    shape(kv_mul, &hw, &qb);
    const int parts = eif_ceil_div(kv_mul, hw), nblk = eif_ceil_div(a.n, 32 * qb);
    const int tiles = eif_ceil_div(a.pos0 + a.n, kKeys);   // of the longest block
    const int cols = a.n_kv * parts;
    // Tiles per share: a power of two near the work of a workgroup when two of them a CU share it evenly, within 4 ..
    // 32 (us at 20 / 5 heads of 128, tiles 4 / 8 / 16 / 32: 511 tokens, even share 1.3, 30.8 / 29.8 / 35.3 / 34.8; 1024,
    // 5.2, 66 / 52 / 48 / 62; 1900, 17.6, 158 / 128 / 111 / 112; 900 at position 1100, 14, 123 / 94 / 84 / 106).
    long work = 0;
    for (int b = 0; b < nblk; ++b) work += eif_ceil_div(a.pos0 + std::min(32 * qb * (b + 1), a.n), kKeys);
    const double even = (double)work * cols / (2 * cus());
    int ct = eif::kPfMinTiles;
    while (ct < 32 && ct < 0.85 * even) ct *= 2;
    const int s_call = eif_ceil_div(tiles, ct);
    if (s_call > 1 && (size_t)nblk * s_call * a.n_heads * (32 * qb) > a.shares) return EIF_HIP_E_ARG;
    attn_prefill_kernel<HD><<<dim3(cols, nblk * s_call), 256, 0, st>>>(a, hw, qb, ct, s_call, 1.0f / sqrtf((float)HD));
    EIF_HIP_LAUNCHED();
    if (s_call > 1) {
        attn_prefill_combine_kernel<HD><<<dim3(a.n, a.n_heads), HD, 0, st>>>(a, qb, ct, s_call);
        EIF_HIP_LAUNCHED();
    }
    return EIF_HIP_OK;
}

}  // namespace

namespace eif {

size_t prefill_attn_shares(int n, int n_heads, int n_kv, int seq_len)
{
    int hw, qb;
    shape(n_heads / n_kv, &hw, &qb);
    const size_t scap = ((size_t)(seq_len + kKeys - 1) / kKeys + kPfMinTiles - 1) / kPfMinTiles;
    return scap > 1 ? (size_t)eif_ceil_div(n, 32 * qb) * scap * n_heads * (32 * qb) : 0;
}

int launch_attn_prefill(const PrefillAttn &a, hipStream_t st)
{
    switch (a.head_dim) {
    case 128: return launch<128>(a, st);
    case 64: return launch<64>(a, st);
    case 32: return launch<32>(a, st);
    default: return EIF_HIP_E_ARG;
    }
}

}  // namespace eif
