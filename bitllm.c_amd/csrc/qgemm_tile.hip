// qgemm_tile.hip -- register-tiled int8-MFMA GEMM of ternary weights for large token batches.
//
// The GEMM forms of qlinear.hip give a wave 16 weight rows and up to 64 tokens on 16x16x64 MFMAs: each decoded weight
// step is used for few MFMAs, every MFMA reads 1 KB of activations from LDS, and a group combine (a conversion and an
// FMA per sum) follows every two of them. Here a wave takes 32 weight rows and 32 MT tokens on v_mfma_i32_32x32x32_i8.
//
// What bounds it: a g128 group costs a wave 4 MFMAs of 32 cycles per 32 x 32 outputs, and 16 conversions, 16 FMAs and
// the decode's share of vector instructions, which the SIMD overlaps with MFMAs only in part (measured: one MFMA and
// 12 vector instructions take 60 cycles with two waves on the SIMD, 32 and 26 alone). So at thousands of tokens the vector
// unit bounds the group-scaled form, not the matrix cores (gate|up 13824x2560 at 3001 tokens: vector instructions in 66% of the
// cycles, MFMAs in 35%, half of these beside vector instructions); at 512 tokens (40 and 22%) and with row scales it is the
// chain of a step and the ends of a launch. Four waves per SIMD (128 registers) hide the LDS reads and the barrier of
// each step. Measured (us, one launch; the forms of qlinear.hip against this one): g128 13824x2560 at 512 / 3001 tokens
// 37.8 / 229 against 28.2 / 159, 3840x2560 at 512 / 3001 15.3 / 59 against 12.3 / 44.7; g96 2560x6912 at 3001 tokens 163
// against 79.6; row scales 13824x2560 at 200 / 3001 tokens 20.7 / 193 against 13.1 / 116.
//
// Operands: lane (r, h) = (lane % 32, lane / 32) supplies 16 bytes of token / weight row r; the 32 columns of an MFMA
// are the 16 of half 0 and the 16 of half 1. Half h takes slots 2h and 2h + 1 of a step (qdev.h's layouts), whose
// columns of a unit (a group; row scales: half a step) are consecutive, so the activations are read in natural order:
// piece i of half h of unit u is bytes 32 UD u + 16 UD h + 16 i of the step. Every group size takes UD MFMAs a group, also
// the odd ones (a g96 group is three, where 16x16x64 pairs need four). The accumulator lane (r, h) holds outputs of weight row
// r and tokens 8 (v / 4) + 4 h + v % 4, v = 0 .. 15.
//
// The sums of each group are exact and are combined in group order, F = fmaf((float)acc, s, F), as the oracle does, and
// the row-scaled epilogue and the split along K are qlinear.hip's: the same bits. The linears of a BitNet-2B layer with
// their preps, at 512 tokens 115 -> 101 us, at 3001 503 -> 391; with row scales at 200 tokens 61.9 -> 55.7.
#include <algorithm>
#include <type_traits>

#include "qdev.h"
#include "qgemm_tile.h"

namespace {

using eif::TileGemm;
typedef int v16i __attribute__((ext_vector_type(16)));

// A workgroup of WN waves takes 32 MT tokens and 32 WN weight rows. Per step of K (64 UD columns) it stages the tokens'
// bytes in LDS (double-buffered, one barrier a step) and every wave loads its own codes and group scales; both are
// loaded one step ahead. (Three and five steps ahead measured the same: a step's chain of LDS reads, MFMAs and combine,
// not memory, is what a lone wave waits for.)
template <int UD, bool GROUPED, int MT, int WN>
__global__ __launch_bounds__(64 * WN) __attribute__((amdgpu_waves_per_eu(2)))
void qgemm_tile_kernel(const int8_t *__restrict__ xq, const uint8_t *__restrict__ W, const float *__restrict__ scales,
                       int wld, int ldq, int M, int nsteps, int G, int N, TileGemm a)
{
    using GE = Geo<kTern, UD>;
    constexpr int SC = GE::SC, SB = GE::SB;
    constexpr int RB = SC == 192 ? 256 : SC;       // LDS bytes of a token row
    constexpr int GP = SC / 16;                    // 16-byte pieces of it
    constexpr int THREADS = 64 * WN, TM = 32 * MT, TN = 32 * WN;
    constexpr int NL = (TM * GP + THREADS - 1) / THREADS;   // pieces a thread stages; past the last one it repeats it
    __shared__ __align__(16) int8_t xa[2][TM * RB];
    __shared__ __align__(16) float xs_l[TM];
    static_assert(TM <= THREADS, "one thread per token scale");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r32 = lane & 31, h = lane >> 5;
    // Workgroup ids b, b + 8, ... run on one XCD: each XCD takes a contiguous run of the tiles, a row block's token
    // blocks first, so that the codes of a row block are read through one L2.
    const int ntb = (M + TM - 1) / TM;
    const int q8 = gridDim.x >> 3, r8 = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int id = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
    const int rb = id / (ntb * a.ks), rz = id - rb * (ntb * a.ks), z = rz / ntb, m0 = (rz - z * ntb) * TM;
    // split along K (a.ks > 1): this workgroup's steps [s0, s1)
    const int s0 = z * nsteps / a.ks, s1 = (z + 1) * nsteps / a.ks;
    const bool live = rb * TN + 32 * wave < N;     // the last row block's spare waves repeat its last rows
    const int row0 = min(rb * TN + 32 * wave, a.rows_pad - 32), row = row0 + r32;

    // Activations. 32-bit byte offsets from the uniform bases (the launcher keeps rows and codes below 4 GiB), token
    // rows clamped into the batch. In LDS a row's pieces are permuted so that the same piece of eight consecutive
    // rows lies in eight bank groups.
    auto swz = [](int t) { return RB >= 128 ? t & 7 : (t >> 1) & 3; };
    uint32_t xo[NL], lo[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int pc = min((int)threadIdx.x + i * THREADS, TM * GP - 1), t = pc / GP, p = pc - t * GP;
        xo[i] = (uint32_t)min(m0 + t, M - 1) * (uint32_t)ldq + (uint32_t)(16 * p);
        lo[i] = (uint32_t)(t * RB + 16 * (p ^ swz(t)));
    }
    auto store_x = [&](int b, const v4i (&r)[NL]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<v4i *>(&xa[b][lo[i]]) = r[i];
    };
    const uint32_t wo = wt_base<kTern, UD>(row, 2 * h, wld), so = GROUPED ? gs_base(row, G) : 0u;

    // register buffer k: step k of a pair
    v4i xr[2][NL];
    uint32_t wr[2][2][UD];   // slots 2h and 2h + 1
    float cr[2][2];          // the step's two group scales of the row
    const int last = s1 - 1;
    auto load = [&](int st, int k) __attribute__((always_inline)) {
        st = min(st, last);   // past the last step its loads again, so that every round has the same in flight
#pragma unroll
        for (int i = 0; i < NL; ++i) xr[k][i] = *reinterpret_cast<const v4i *>(xq + (xo[i] + (uint32_t)(st * SC)));
        load_words<UD>(W + (wo + (uint32_t)(st * 64 * SB)), wr[k][0]);
        load_words<UD>(W + (wo + (uint32_t)(st * 64 * SB + 16 * SB)), wr[k][1]);
        if constexpr (GROUPED) {
            cr[k][0] = scales[so + 16u * (uint32_t)(2 * st)];
            cr[k][1] = scales[so + 16u * (uint32_t)min(2 * st + 1, G - 1)];
        }
    };

    // grouped: FP32 outputs; row-scaled: int32 sums
    float F[GROUPED ? MT : 1][16];
    v16i C[GROUPED ? 1 : MT];
#pragma unroll
    for (int m = 0; m < (GROUPED ? MT : 1); ++m)
#pragma unroll
        for (int v = 0; v < 16; ++v) F[m][v] = 0.0f;
#pragma unroll
    for (int m = 0; m < (GROUPED ? 1 : MT); ++m) C[m] = v16i{};

    // The MFMA sums carry the codes' 2^6; the combine takes them against the scale times 2^-6 (exact, see qgemm_kernel),
    // and 0 for a group past the row's last one (a ragged last step), which adds nothing.
    constexpr float kUnshift = 1.0f / (float)(1 << GE::SHIFT);
    const int ao = r32 * RB, as = swz(r32);
    auto compute = [&](int b, int st, const uint32_t (&w)[2][UD], const float (&c)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            long b0[GE::NMF], b1[GE::NMF], bb[2 * UD];
            decode<kTern, UD>(w[0], b0);
            decode<kTern, UD>(w[1], b1);
#pragma unroll
            for (int i = 0; i < UD; ++i) bb[i] = b0[u * UD + i], bb[UD + i] = b1[u * UD + i];
            v4i B[UD];
#pragma unroll
            for (int i = 0; i < UD; ++i)
                B[i] = v4i{(int)bb[2 * i], (int)(bb[2 * i] >> 32), (int)bb[2 * i + 1], (int)(bb[2 * i + 1] >> 32)};
            const float cu = 2 * st + u < G ? c[u] * kUnshift : 0.0f;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                v4i A[UD];
#pragma unroll
                for (int i = 0; i < UD; ++i)
                    A[i] = *reinterpret_cast<const v4i *>(&xa[b][ao + m * 32 * RB + 16 * (((2 * u + h) * UD + i) ^ as)]);
                v16i cc = GROUPED ? v16i{} : C[GROUPED ? 0 : m];
#pragma unroll
                for (int i = 0; i < UD; ++i) cc = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[i], B[i], cc, 0, 0, 0);
                if constexpr (GROUPED) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) F[m][v] = fmaf((float)cc[v], cu, F[m][v]);
                } else {
                    C[m] = cc;
                }
            }
        }
    };

    load(s0, 0);
    load(s0 + 1, 1);
    if ((int)threadIdx.x < TM) xs_l[threadIdx.x] = a.xs[min(m0 + (int)threadIdx.x, M - 1)];
    store_x(0, xr[0]);
    __syncthreads();
    for (int st = s0; st < last; st += 2) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            compute(k, st + k, wr[k], cr[k]);
            load(st + k + 2, k);
            store_x(k ^ 1, xr[k ^ 1]);
            __syncthreads();
        }
    }
    if ((s1 - s0) & 1) compute(0, last, wr[0], cr[0]);

    // Split along K, as qlinear.hip's gemm_finish: every split leaves its partial sums with device-coherent stores and
    // counts its arrival on the tile; the last one adds all of them in split order and goes on to the epilogue.
    if (a.ks > 1) {
        const int ntile = gridDim.x / a.ks, tile = rb * ntb + m0 / TM;
        auto pz = [&](int j) { return a.part + ((size_t)j * ntile + tile) * (16 * MT * THREADS) + threadIdx.x; };
        float *own = pz(z);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                st_coh(own + (16 * m + v) * THREADS, GROUPED ? F[GROUPED ? m : 0][v] : __int_as_float(C[GROUPED ? 0 : m][v]));
        __builtin_amdgcn_s_waitcnt(0);
        __shared__ int last_l;
        __syncthreads();
        if (threadIdx.x == 0)
            last_l = __hip_atomic_fetch_add(a.cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.ks - 1;
        __syncthreads();
        if (!last_l) return;
        if (threadIdx.x == 0) st_coh_i(a.cnt + tile, 0);   // zero again for the next launch
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float q[2][16];   // a split's partials while the next one's are loaded (past the last split its own again)
#pragma unroll
            for (int v = 0; v < 16; ++v) q[0][v] = ld_coh(pz(0) + (16 * m + v) * THREADS);
            for (int j = 0; j < a.ks; ++j) {
                const float *p = pz(min(j + 1, a.ks - 1));
#pragma unroll
                for (int v = 0; v < 16; ++v) q[1][v] = ld_coh(p + (16 * m + v) * THREADS);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if constexpr (GROUPED) F[m][v] = j == 0 ? q[0][v] : F[m][v] + q[0][v];
                    else C[m][v] = (j == 0 ? 0 : C[m][v]) + __float_as_int(q[0][v]);
                    q[0][v] = q[1][v];
                }
            }
        }
    }
    if (!live || row >= N) return;

    const float bb = a.bias ? a.bias[row] : 0.0f;
    const float rs = !GROUPED && scales ? scales[row] : 1.0f;
    auto epilogue = [&](auto full_c) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_c)::value;   // every token of the block in the batch
        const size_t t0 = (size_t)(m0 + 4 * h);
        float *yp = a.y + t0 * a.ldy + row;
        const float *rp = a.res ? a.res + t0 * a.ldr + row : nullptr;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int lt = 32 * m + 8 * q;
                const float4 x4 = *reinterpret_cast<const float4 *>(&xs_l[lt + 4 * h]);
                const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (!FULL && m0 + lt + 4 * h + v >= M) continue;
                    float out;
                    if constexpr (GROUPED) out = F[m][4 * q + v] * xv[v];
                    else out = ((float)(C[m][4 * q + v] >> GE::SHIFT) * xv[v]) * rs;
                    if (a.bias) out = out + bb;
                    if (rp) out = out + rp[(size_t)(lt + v) * a.ldr];
                    yp[(size_t)(lt + v) * a.ldy] = out;
                }
            }
    };
    if (m0 + TM <= M) epilogue(std::true_type{});
    else epilogue(std::false_type{});
}

// Workgroups (before the split along K) and partial sums of a shape.
struct Shape {
    int mt, wn;
    int tiles(const TileGemm &g) const { return eif_ceil_div(g.M, 32 * mt) * eif_ceil_div(g.rows_pad, 32 * wn); }
    size_t part_bytes(const TileGemm &g) const
    {
        return g.ks > 1 ? (size_t)g.ks * tiles(g) * (16 * mt * 64 * wn) * sizeof(float) : 0;
    }
};
constexpr Shape kSmall{1, 4}, kLarge{2, 8};

template <int UD, bool GROUPED, int MT, int WN>
int go(const TileGemm &g, hipStream_t st)
{
    const int grid = Shape{MT, WN}.tiles(g) * g.ks;
    qgemm_tile_kernel<UD, GROUPED, MT, WN><<<grid, 64 * WN, 0, st>>>(g.xq, g.W, g.scales, g.wld, g.ldq, g.M, g.nsteps,
                                                                     g.G, g.N, g);
    EIF_HIP_LAUNCHED();
    return EIF_HIP_OK;
}

// Two shapes: "small", 32 tokens x 128 rows on four waves, and "large", 64 tokens x 256 rows on eight (half the
// decode a token, half the activation reads a row). Small from one workgroup per CU on (row scales: from five eighths of
// that); below, the forms of qlinear.hip, which split K and give a lone wave shorter chains (us, them / small: g128
// 3840x2560 at 256 tokens, 240 workgroups, 8.9 / 9.3, at 512, 480 workgroups, 15.3 / 12.3; 13824x2560 at 64, 216, 9.0 / 9.2, at
// 128, 432, 15.0 / 11.9; g96 2560x6912 at 256, 160, 20.2 / 22.1, at 512, 320, 31.8 / 27.5; row scales 2560x6912 at 256, 160,
// 13.8 / 12.6). Large where its workgroups fill the CUs about once or from one and a half times on; between, some CUs
// run two while the others wait (us, small / large: g128 13824x2560 at 256 tokens, 216 large workgroups, 19.1 / 18.2, at
// 768, 648, 45.1 / 39.7; 2560x2560 at 1900, 300, 24.7 / 28.2, at 3001, 470, 36.7 / 31.7; g96 2560x6912 at 1900, 300,
// 59.0 / 69.1, at 3001, 470, 97.5 / 79.6; 3840x2560 at 768, 180, 16.0 / 17.4).
const Shape *pick(const TileGemm &g)
{
    if (g.fmt != kTern || g.M < 1) return nullptr;
    // the kernel's 32-bit offsets (the other forms refuse such shapes)
    if ((size_t)g.M * g.ldq >= ((size_t)1 << 32) || (size_t)g.rows_pad * g.wld >= ((size_t)1 << 32)) return nullptr;
    const int C = eif_device_cus(), small = kSmall.tiles(g) * g.ks, large = kLarge.tiles(g) * g.ks;
    if (8 * small < (g.grouped ? 8 : 5) * C) return nullptr;
    return 2 * large >= 3 * C || (large <= C && 4 * large >= 3 * C) ? &kLarge : &kSmall;
}

template <int UD, bool GROUPED>
int launch(const TileGemm &g, const Shape &s, hipStream_t st)
{
    return s.mt == kLarge.mt ? go<UD, GROUPED, kLarge.mt, kLarge.wn>(g, st) : go<UD, GROUPED, kSmall.mt, kSmall.wn>(g, st);
}

}  // namespace

namespace eif {

bool gemm_tile_takes(const TileGemm &g, int *tiles, size_t *part_bytes)
{
    const Shape *s = pick(g);
    if (!s) return false;
    *tiles = s->tiles(g);
    *part_bytes = s->part_bytes(g);
    return true;
}

int launch_gemm_tile(const TileGemm &g, hipStream_t st)
{
    const Shape *s = pick(g);
    if (!s || (g.ks > 1 && (!g.part || !g.cnt))) return EIF_HIP_E_ARG;
    if (!g.grouped) return launch<4, false>(g, *s, st);
    switch (g.ud) {
    case 1: return launch<1, true>(g, *s, st);
    case 2: return launch<2, true>(g, *s, st);
    case 3: return launch<3, true>(g, *s, st);
    case 4: return launch<4, true>(g, *s, st);
    case 8: return launch<8, true>(g, *s, st);
    default: return EIF_HIP_E_ARG;
    }
}

}  // namespace eif
