// mdx_prefill_long.hip — batch prefill of more than 64 rows, gfx950.
//
// The kernels of mdx_prefill.hip take 64 rows per pass over the weights and
// give every query row an attention block of its own.  A longer prompt has
// enough rows to tile both operands: here the projections are LDS-tiled MFMA
// GEMMs over all rows (each weight read once per row tile, int8/int4 widened
// to fp16 once per block as they are staged), and attention runs 64 query
// rows of one KV head against each staged K/V tile on MFMA.  A prompt alone,
// through 4 layers of hidden 1024, against chunks of 64 rows: fp16 65 rows 381
// -> 240 us, 200 853 -> 317, 1500 7783 -> 960; int4 65 337 -> 262, 1500 7381
// -> 1020.
#include <hip/hip_runtime.h>

#include <cmath>

#include "mdx_common.h"
#include "mdx_device.h"
#include "mdx_gemm_tile.h"

using namespace mdx;

namespace {

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kKT = 64;            // k per LDS stage
constexpr int kStageChunks = kKT / 8;   // 16-byte chunks per LDS row

// Where a tile's 16-byte chunk of row r goes: chunks are permuted within the
// row by the row index, so the rows of an MFMA fragment read spread over the
// banks without padding (padded rows instead: M = 2000 projections 141 -> 146
// us a layer).
__device__ __forceinline__ int lds_chunk(int row, int chunk) {
    return row * kStageChunks + (chunk ^ (row & 7));
}

// Block id -> work item: ids id, id + 8, ... run on one XCD (one L2); each XCD
// takes a contiguous run of items.  A bijection for any count.
__device__ __forceinline__ int xcd_item(int id, int n) {
    const int q = n >> 3, r = n & 7, x = id & 7, i = id >> 3;
    return x * q + min(x, r) + i;
}

enum LongEpi { LE_STORE = 0, LE_PART = 1, LE_SWIGLU = 2, LE_ROPE = 3 };

struct LongArgs {
    const uint16_t* x16;      // [M][K]
    const uint8_t* w;         // W^T rows
    const float* scale;       // [N] or NULL
    int M, K, N;
    int tiles_m, tiles_n, splits, per_split;   // per_split: LDS stages per split
    int run;                  // stages per partial sum
    float* out;               // LE_STORE [M][N]; LE_PART [splits][M][N], unscaled
    uint16_t* out16;          // LE_SWIGLU [M][N/2]
    // LE_ROPE
    int pos0, nq, nkv, style;
    const float* q_norm;
    const float* k_norm;
    float eps;
    const float* cos_t;
    const float* sin_t;
    float* q_out;             // [M][nq*hd]
    uint16_t* kc;             // [max_seq][nkv*hd]
    uint16_t* vc;
};

// Weight row of tile row c (0..BN-1): consecutive rows, or for SwiGLU
// alternating runs of 16 gate rows and the 16 up rows of the same features.
template <int BN>
__device__ __forceinline__ int long_row(int tile, int c, bool swiglu, int N) {
    if (!swiglu) return tile * BN + c;
    const int f = tile * (BN / 2) + (c >> 5) * 16 + (c & 15);
    return f < N / 2 ? ((c & 16) ? N / 2 + f : f) : N;
}

// QK-norm + RoPE + append of the head slices a wave holds.  acc[t][j]: weight
// columns 16t + 4g + i (t within the wave's NT tiles) of row m; a head is HD
// consecutive columns, all in this lane and its three g-partners.
template <int HD, int NT>
__device__ __forceinline__ void rope_store(const LongArgs& a, float4_t (&v)[NT], int col0, int m, int g,
                                           bool store) {
    constexpr int TH = HD / 16;               // tiles per head
    const int qd = a.nq * HD, kvd = a.nkv * HD;
    const size_t pos = (size_t)a.pos0 + m;
#pragma unroll
    for (int h = 0; h < NT / TH; h++) {
        const int c0 = col0 + h * HD;         // the head's first column
        if (c0 >= a.N) break;
        float4_t* x = v + h * TH;
        if (c0 >= qd + kvd) {
            uint16_t* dst = a.vc + pos * kvd + (c0 - qd - kvd);
#pragma unroll
            for (int t = 0; t < TH; t++) {
                uint2 o;
                o.x = (uint32_t)f32_to_f16_bits(x[t][0]) | ((uint32_t)f32_to_f16_bits(x[t][1]) << 16);
                o.y = (uint32_t)f32_to_f16_bits(x[t][2]) | ((uint32_t)f32_to_f16_bits(x[t][3]) << 16);
                if (store) *reinterpret_cast<uint2*>(dst + 16 * t + 4 * g) = o;
            }
            continue;
        }
        const bool is_q = c0 < qd;
        const float* nw = is_q ? a.q_norm : a.k_norm;
        if (nw) {
            float ss = 0.0f;
#pragma unroll
            for (int t = 0; t < TH; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) ss += x[t][i] * x[t][i];
            ss = rows_sum4(ss);
            const float rms = 1.0f / sqrtf(ss / (float)HD + a.eps);
#pragma unroll
            for (int t = 0; t < TH; t++) {
                const float4 w = *reinterpret_cast<const float4*>(nw + 16 * t + 4 * g);
                x[t][0] = (x[t][0] * rms) * w.x;
                x[t][1] = (x[t][1] * rms) * w.y;
                x[t][2] = (x[t][2] * rms) * w.z;
                x[t][3] = (x[t][3] * rms) * w.w;
            }
        }
        const float* cr = a.cos_t + pos * (HD / 2);
        const float* sr = a.sin_t + pos * (HD / 2);
        if (a.style == 0) {
            // pairs (2i, 2i+1)
#pragma unroll
            for (int t = 0; t < TH; t++) {
                const float2 c = *reinterpret_cast<const float2*>(cr + 8 * t + 2 * g);
                const float2 s = *reinterpret_cast<const float2*>(sr + 8 * t + 2 * g);
                const float a0 = x[t][0], b0 = x[t][1], a1 = x[t][2], b1 = x[t][3];
                x[t][0] = a0 * c.x - b0 * s.x;
                x[t][1] = b0 * c.x + a0 * s.x;
                x[t][2] = a1 * c.y - b1 * s.y;
                x[t][3] = b1 * c.y + a1 * s.y;
            }
        } else {
            // pairs (i, i + HD/2)
#pragma unroll
            for (int t = 0; t < TH / 2; t++) {
                const float4 c = *reinterpret_cast<const float4*>(cr + 16 * t + 4 * g);
                const float4 s = *reinterpret_cast<const float4*>(sr + 16 * t + 4 * g);
                const float cc[4] = {c.x, c.y, c.z, c.w}, sc[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x0 = x[t][i], x1 = x[t + TH / 2][i];
                    x[t][i] = x0 * cc[i] - x1 * sc[i];
                    x[t + TH / 2][i] = x1 * cc[i] + x0 * sc[i];
                }
            }
        }
        if (!store) continue;
        if (is_q) {
            float* dst = a.q_out + (size_t)m * qd + c0;
#pragma unroll
            for (int t = 0; t < TH; t++)
                *reinterpret_cast<float4*>(dst + 16 * t + 4 * g) = make_float4(x[t][0], x[t][1], x[t][2], x[t][3]);
        } else {
            uint16_t* dst = a.kc + pos * kvd + (c0 - qd);
#pragma unroll
            for (int t = 0; t < TH; t++) {
                uint2 o;
                o.x = (uint32_t)f32_to_f16_bits(x[t][0]) | ((uint32_t)f32_to_f16_bits(x[t][1]) << 16);
                o.y = (uint32_t)f32_to_f16_bits(x[t][2]) | ((uint32_t)f32_to_f16_bits(x[t][3]) << 16);
                *reinterpret_cast<uint2*>(dst + 16 * t + 4 * g) = o;
            }
        }
    }
}

// ---- projections: LDS-tiled MFMA GEMM -----------------------------------------
//
// Block = 4 waves, one BN (weight rows) x BM (activation rows) tile; a stage
// is 64 k of both panels in LDS (fp16, two buffers), staged through registers
// PD stages ahead.  The weights are the MFMA A operand, the activations the B
// operand, so a lane ends with 4 consecutive output columns of one row:
// 16-byte stores, SwiGLU pairs and RoPE pairs in one lane.  Waves split the
// tile WN x (4/WN).  Lane group g takes k 16g + 8s .. +7 of a stage at step s
// for both operands.
template <int KIND, int BM, int BN, int WN, int PD, int EPI, int HD>
__global__ __launch_bounds__(256, 2) void k_long_gemm(LongArgs a) {
    constexpr int WM = 4 / WN;
    constexpr int NT = BN / WN / 16, MT = BM / WM / 16;   // 16x16 tiles per wave
    constexpr int XU = BM * kStageChunks / 256;           // 16-byte loads per thread, activations
    constexpr int KPU = KIND == MDX_W_F16 ? 8 : (KIND == MDX_W_I8 ? 16 : 32);   // k per weight load
    constexpr int UPR = kKT / KPU;                        // weight loads per row
    constexpr int WUN = BN * UPR, WU = (WUN + 255) / 256;
    constexpr bool SWIGLU = EPI == LE_SWIGLU;
    __shared__ uint4 xs[2][BM * kStageChunks];
    __shared__ uint4 ws[2][BN * kStageChunks];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int g = lane >> 4, c16 = lane & 15;
    const int wn = wave % WN, wm = wave / WN;
    const int item = xcd_item(blockIdx.x, gridDim.x);
    const int tm = item % a.tiles_m, rest = item / a.tiles_m;
    const int tn = rest % a.tiles_n, split = rest / a.tiles_n;
    const int nst_all = (a.K + kKT - 1) / kKT;
    const int s0 = split * a.per_split, s1 = min(nst_all, s0 + a.per_split);
    const size_t row_bytes = KIND == MDX_W_F16 ? (size_t)a.K * 2 : (KIND == MDX_W_I8 ? (size_t)a.K : (size_t)a.K / 2);

    // This thread's loads.  None is conditional, so the compiler can count the
    // ones in flight and waits for no younger stage than the one it needs (a
    // load under a branch makes it wait for all: M = 203, K = 1024 took 1 us a
    // stage whatever PD).  Rows past the edge repeat the last row (their
    // results are not stored), stages past the last repeat it, and k past K
    // repeat the row's last load and become zeros on their way to LDS, in both
    // operands: a repeated weight may be an infinity (fp16 ones only).
    const uint16_t* xp[XU];
    int xk[XU], xl[XU];
#pragma unroll
    for (int i = 0; i < XU; i++) {
        const int u = tid + 256 * i, row = u / kStageChunks, ch = u % kStageChunks;
        xk[i] = 8 * ch;
        xl[i] = lds_chunk(row, ch);
        xp[i] = a.x16 + (size_t)min(tm * BM + row, a.M - 1) * a.K;
    }
    const uint8_t* wp[WU];
    int wk[WU], wr[WU];
#pragma unroll
    for (int i = 0; i < WU; i++) {
        const int u = min(tid + 256 * i, WUN - 1), row = u / UPR, ch = u % UPR;
        wk[i] = KPU * ch;
        wr[i] = row;
        wp[i] = a.w + (size_t)min(long_row<BN>(tn, row, SWIGLU, a.N), a.N - 1) * row_bytes;
    }
    u32x4_t xv[PD][XU], wv[PD][WU];
    auto load = [&](int d, int st) __attribute__((always_inline)) {
        const int k0 = min(st, s1 - 1) * kKT;
#pragma unroll
        for (int i = 0; i < XU; i++)
            xv[d][i] = *reinterpret_cast<const u32x4_t*>(xp[i] + (unsigned)min(k0 + xk[i], a.K - 8));
#pragma unroll
        for (int i = 0; i < WU; i++) {
            const unsigned k = (unsigned)min(k0 + wk[i], a.K - KPU);
            wv[d][i] = *reinterpret_cast<const u32x4_t*>(wp[i] + (KIND == MDX_W_F16 ? 2 * k : KIND == MDX_W_I8 ? k : k / 2));
        }
    };
    auto stash = [&](int d, int buf, int st) __attribute__((always_inline)) {
        if ((st + 1) * kKT > a.K) {       // K ends inside this stage
#pragma unroll
            for (int i = 0; i < XU; i++)
                if (st * kKT + xk[i] >= a.K) xv[d][i] = u32x4_t{0u, 0u, 0u, 0u};
            if constexpr (KIND == MDX_W_F16) {
#pragma unroll
                for (int i = 0; i < WU; i++)
                    if (st * kKT + wk[i] >= a.K) wv[d][i] = u32x4_t{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int i = 0; i < XU; i++) xs[buf][xl[i]] = __builtin_bit_cast(uint4, xv[d][i]);
#pragma unroll
        for (int i = 0; i < WU; i++) {
            if (WUN % 256 != 0 && tid + 256 * i >= WUN) break;
            half8_t b[KPU / 8];
            widen_b<KIND>(__builtin_bit_cast(uint4, wv[d][i]), b);
#pragma unroll
            for (int s = 0; s < KPU / 8; s++)
                ws[buf][lds_chunk(wr[i], wk[i] / 8 + s)] = __builtin_bit_cast(uint4, b[s]);
        }
    };

    // sums of a.run stages (long_run) are added to a second set
    float4_t acc[NT][MT], tot[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < MT; j++) acc[t][j] = tot[t][j] = float4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int d = 0; d < PD; d++) load(d, s0 + d);
    stash(0, 0, s0);
    load(0, s0 + PD);
    __syncthreads();
    int left = a.run;
    for (int sb = s0; sb < s1; sb += PD) {
#pragma unroll
        for (int d = 0; d < PD; d++) {
            const int st = sb + d;
            if (st >= s1) break;
            const int buf = (st - s0) & 1;
            // the next stage's LDS writes and a later one's loads are issued
            // before this one's products
            const int dn = (d + 1) % PD;
            stash(dn, buf ^ 1, st + 1);
            load(dn, st + 1 + PD);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                half8_t xb[MT];
#pragma unroll
                for (int j = 0; j < MT; j++)
                    xb[j] = __builtin_bit_cast(half8_t, xs[buf][lds_chunk((wm * MT + j) * 16 + c16, 2 * g + s)]);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const half8_t wa = __builtin_bit_cast(half8_t, ws[buf][lds_chunk((wn * NT + t) * 16 + c16, 2 * g + s)]);
#pragma unroll
                    for (int j = 0; j < MT; j++)
                        acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa, xb[j], acc[t][j], 0, 0, 0);
                }
            }
            if (--left == 0) {
                left = a.run;
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int j = 0; j < MT; j++) {
                        tot[t][j] += acc[t][j];
                        acc[t][j] = float4_t{0.f, 0.f, 0.f, 0.f};
                    }
            }
            __syncthreads();
        }
    }

#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < MT; j++) acc[t][j] += tot[t][j];

    // acc[t][j]: output columns 16 (wn NT + t) + 4g + i of row 16 (wm MT + j) + c16
#pragma unroll
    for (int j = 0; j < MT; j++) {
        const int m = tm * BM + (wm * MT + j) * 16 + c16;
        const bool mv = m < a.M;
        if constexpr (EPI == LE_ROPE) {
            float4_t v[NT];
            const int col0 = tn * BN + wn * NT * 16;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                v[t] = acc[t][j];
                if (a.scale) {
                    const float4 sc = *reinterpret_cast<const float4*>(a.scale + min(col0 + 16 * t, a.N - 16) + 4 * g);
                    v[t][0] *= sc.x; v[t][1] *= sc.y; v[t][2] *= sc.z; v[t][3] *= sc.w;
                }
            }
            // the lanes of rows past M take part in the row sums; their table
            // reads repeat the last row's
            rope_store<HD, NT>(a, v, col0, mv ? m : a.M - 1, g, mv);
        } else if constexpr (SWIGLU) {
            const int F = a.N / 2;
#pragma unroll
            for (int t = 0; t < NT; t += 2) {
                const int f = tn * (BN / 2) + (wn * NT + t) * 8 + 4 * g;
                if (!mv || f >= F) continue;
                float4 sg = make_float4(1.f, 1.f, 1.f, 1.f), su = sg;
                if (a.scale) {
                    sg = *reinterpret_cast<const float4*>(a.scale + f);
                    su = *reinterpret_cast<const float4*>(a.scale + F + f);
                }
                const float4_t gt = acc[t][j], up = acc[t + 1][j];
                uint2 o;
                o.x = (uint32_t)f32_to_f16_bits(silu_mul(gt[0] * sg.x, up[0] * su.x)) |
                      ((uint32_t)f32_to_f16_bits(silu_mul(gt[1] * sg.y, up[1] * su.y)) << 16);
                o.y = (uint32_t)f32_to_f16_bits(silu_mul(gt[2] * sg.z, up[2] * su.z)) |
                      ((uint32_t)f32_to_f16_bits(silu_mul(gt[3] * sg.w, up[3] * su.w)) << 16);
                *reinterpret_cast<uint2*>(a.out16 + (size_t)m * F + f) = o;
            }
        } else {
            float* orow = a.out + ((size_t)split * a.M + (mv ? m : 0)) * a.N;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int n = tn * BN + (wn * NT + t) * 16 + 4 * g;
                if (!mv || n >= a.N) continue;
                float4_t y = acc[t][j];
                if (n + 4 <= a.N && a.N % 4 == 0) {
                    if (EPI == LE_STORE && a.scale) {
                        const float4 sc = *reinterpret_cast<const float4*>(a.scale + n);
                        y[0] *= sc.x; y[1] *= sc.y; y[2] *= sc.z; y[3] *= sc.w;
                    }
                    *reinterpret_cast<float4*>(orow + n) = make_float4(y[0], y[1], y[2], y[3]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (n + i < a.N) orow[n + i] = EPI == LE_STORE && a.scale ? y[i] * a.scale[n + i] : y[i];
                }
            }
        }
    }
}

// ---- attention ------------------------------------------------------------------
//
// Block = one KV head x 64 query rows (64/G consecutive positions x the G
// heads of the group), 16 rows per wave and two groups of four waves, which
// take alternate K/V tiles of 64 positions and are merged at the end: the
// causal rows make the last blocks twice as long as the average one, and
// nothing else is left to run beside them, so a block's own length is what
// counts (one group, two blocks per CU: 67 us at M = 2000 within a prefill, 55
// with two).  Tiles are staged in LDS (V transposed), the group's next one in
// registers meanwhile.  S^T = K . Q^T, so a lane holds scores of one query row
// and its running maximum and sum are its own; P^T is then already the B operand
// of O^T = V^T . P^T (the k order of that product is the order in which a lane
// holds its scores).
//
// Queries and probabilities are fp32: each goes in as the sum of two fp16
// values, both rounded to nearest (23 bits), the queries scaled per row so that
// neither part leaves the fp16 range, the probabilities by 2^6.  What this must
// not lose against fp32 arithmetic (k_attn_prefill) is kept by the order of the
// sums: a product's second parts go first, the scores are summed over 64
// dimensions at a time (32 at 64 dimensions), the tile's P.V is summed from
// zero and then added, and the exponent's offset is the reference score alone
// (an offset of 6 more rounds every exponent at 2^-22).  Outputs rounded
// otherwise than the exact result rounds, per thousand, before these / now /
// k_attn_prefill, normal inputs, 16 heads of 128 over 8: M = 515 1.87 / 0.98 /
// 1.03, M = 2000 2.11 / 1.11 / 1.16, equal scores 1.13 / 0.49 / 0.62; 8 of 256
// over 2, M = 515: 2.10 / 0.98 / 0.98.  Their cost, launched alone on cold
// inputs, M = 2000: 69.3 -> 70.2 us; 256 dimensions 159 -> 135 us (independent
// sums).
//
// The vector unit is what bounds it (at M = 2000 the longest block's tile took
// 2.9 us with expf and a rescale per tile): the exponentials are v_exp_f32 of
// one fma (the row's scale, the softmax scale and log2 e are one factor, as
// exact as the fp32 score), the reference score only moves, and the sums are
// only rescaled, when a row's maximum has outgrown it by 2^8, and addresses are
// clamped instead of values selected.  16 query heads of 128 over 8 KV heads,
// M = 2000: 92 -> 67 us by these.
//
// Infinities and NaN: scores that come out as NaN are recomputed in fp32 (an
// infinite key times the two parts of a query may be inf - inf), and a V tile
// that holds any takes the products of its own positions only, in fp32, so
// that a position beyond a row's own never reaches that row.
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_exp(uint32_t m, u32x4_t v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++)
        m = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, m),
                                                                   __builtin_bit_cast(u16x2_t, w[i] & 0x7fff7fffu)));
    return m;
}
__device__ __forceinline__ bool exp_nonfinite(uint32_t m) { return (m & 0xffffu) >= 0x7c00u || (m >> 16) >= 0x7c00u; }

// fp32 values as the sums of two fp16 values.
__device__ __forceinline__ void split16(const float (&v)[8], half8_t& hi, half8_t& lo) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (_Float16)v[e];
        lo[e] = (_Float16)(v[e] - (float)hi[e]);
    }
}

template <int HD, int G>
__global__ __launch_bounds__(512, 2) void k_attn_long(int pos0, int M, const float* __restrict__ q,
                                                      const uint16_t* __restrict__ kc,
                                                      const uint16_t* __restrict__ vc, int nkv, int n_tb,
                                                      uint16_t* __restrict__ out16) {
    constexpr int TB = 64 / G;             // positions per block
    constexpr int KB = HD == 256 ? 32 : 64;   // keys per tile (32: no spills at 256 dimensions)
    constexpr int DS = HD / 32;            // k-steps of a score
    constexpr int NS = HD == 256 ? 4 : 2;  // sums of a score
    constexpr int DT = HD / 16;            // 16-row tiles of O^T
    constexpr int KS = HD / 8 + 1;         // uint4 per LDS row of K (16-byte pad)
    constexpr int VS = KB / 8 + 1;         // uint4 per LDS row of V^T
    constexpr int KU = KB * (HD / 8) / 256;        // K loads per thread
    constexpr int VUN = (KB / 4) * (HD / 8);       // V units: 4 keys x 8 dims
    constexpr int VU = (VUN + 255) / 256;
    // a group's K tile, or the fp32 probabilities of a non-finite V tile (64 rows x KB)
    constexpr int KN = KB * KS > 16 * KB ? KB * KS : 16 * KB;
    constexpr int MN = (4 * DT + 2) * 256 / 4;     // uint4 of a group's sums in the merge
    static_assert(2 * (KN + HD * VS) >= MN, "the merge fits the tiles");
    __shared__ uint4 lds[2 * (KN + HD * VS)];

    const int grp = threadIdx.x >> 8, tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
    uint4* const ks = lds + grp * (KN + HD * VS);
    uint4* const vs = ks + KN;
    const int g = lane >> 4, c16 = lane & 15;
    const int kvh = blockIdx.x % nkv;
    const int t0 = (n_tb - 1 - blockIdx.x / nkv) * TB;   // the longest blocks first
    const int nq = nkv * G, kvd = nkv * HD;
    const int r = wave * 16 + c16;                       // this lane's query row
    const int t = t0 + r / G, hq = kvh * G + r % G;
    const bool tv = t < M;
    const int L = pos0 + (tv ? t : M - 1) + 1;           // positions this row attends over
    const int Lmax = pos0 + min(t0 + TB, M);             // and the block
    const float* qrow = q + ((size_t)(tv ? t : M - 1) * nq + hq) * HD;

    // K/V tile loads of this thread
    u32x4_t kr[KU], vr[VU][4];
    auto load = [&](int p0) __attribute__((always_inline)) {
        // positions past the block's last repeat it (their scores are masked)
        const int pb = min(p0, Lmax - 1), last = Lmax - 1 - pb;
        const uint16_t* kp = kc + (size_t)pb * kvd + kvh * HD;
        const uint16_t* vp = vc + (size_t)pb * kvd + kvh * HD;
#pragma unroll
        for (int i = 0; i < KU; i++) {
            const int u = tid + 256 * i, key = u / (HD / 8), ch = u % (HD / 8);
            kr[i] = *reinterpret_cast<const u32x4_t*>(kp + (unsigned)(min(key, last) * kvd + 8 * ch));
        }
#pragma unroll
        for (int i = 0; i < VU; i++) {
            const int u = tid + 256 * i, kg = u % (KB / 4), db = u / (KB / 4);
            if (VUN % 256 != 0 && db >= HD / 8) break;
#pragma unroll
            for (int j = 0; j < 4; j++)
                vr[i][j] = *reinterpret_cast<const u32x4_t*>(vp + (unsigned)(min(4 * kg + j, last) * kvd + 8 * db));
        }
    };
    load(grp * KB);

    // the query row as fp16 pairs, scaled by 2^e to a maximum in [2^14, 2^15);
    // a score times c is its exponent in base 2
    half8_t qh[DS], ql[DS];
    float up, c;
    {
        float qv[DS][8], mx = 0.0f;
#pragma unroll
        for (int s = 0; s < DS; s++) {
            const float4 lo = *reinterpret_cast<const float4*>(qrow + 32 * s + 8 * g);
            const float4 hi = *reinterpret_cast<const float4*>(qrow + 32 * s + 8 * g + 4);
            qv[s][0] = lo.x; qv[s][1] = lo.y; qv[s][2] = lo.z; qv[s][3] = lo.w;
            qv[s][4] = hi.x; qv[s][5] = hi.y; qv[s][6] = hi.z; qv[s][7] = hi.w;
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(qv[s][e]));
        }
        mx = rows_max4(mx);
        int ex = 0;
        if (mx > 0.0f && mx < INFINITY) {
            ex = 14 - ilogbf(mx);
            ex = ex > 100 ? 100 : ex;
        }
        up = ldexpf(1.0f, ex);
        c = ldexpf(1.44269504088896340736f / sqrtf((float)HD), -ex);
#pragma unroll
        for (int s = 0; s < DS; s++) {
#pragma unroll
            for (int e = 0; e < 8; e++) qv[s][e] *= up;
            split16(qv[s], qh[s], ql[s]);
        }
    }

    float4_t o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++) o[d] = float4_t{0.f, 0.f, 0.f, 0.f};
    float ref = -INFINITY, runL = 0.0f;       // ref: base-2 exponent of the reference score

    // the groups' tiles of a round; the last one of group 1 may be all masked
    for (int pr0 = 0; pr0 < Lmax; pr0 += 2 * KB) {
        const int p0 = pr0 + grp * KB;
        uint32_t vmax = 0;
#pragma unroll
        for (int i = 0; i < KU; i++) {
            const int u = tid + 256 * i;
            ks[(u / (HD / 8)) * KS + u % (HD / 8)] = __builtin_bit_cast(uint4, kr[i]);
        }
#pragma unroll
        for (int i = 0; i < VU; i++) {
            const int u = tid + 256 * i, kg = u % (KB / 4), db = u / (KB / 4);
            if (VUN % 256 != 0 && db >= HD / 8) break;
            // key 4 kg + j lies at offset 32 (kg/8) + 8 (kg%4) + 4 (kg/4 % 2) + j of
            // its row: the order of the second product
            const int off = 32 * (kg >> 3) + 8 * (kg & 3) + 4 * ((kg >> 2) & 1);
            uint32_t wd[4][4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                vmax = max_exp(vmax, vr[i][j]);
                wd[j][0] = vr[i][j].x; wd[j][1] = vr[i][j].y; wd[j][2] = vr[i][j].z; wd[j][3] = vr[i][j].w;
            }
            uint16_t* vb = reinterpret_cast<uint16_t*>(vs) + off;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
                uint2 w2;
                w2.x = __builtin_amdgcn_perm(wd[1][e / 2], wd[0][e / 2], sel);
                w2.y = __builtin_amdgcn_perm(wd[3][e / 2], wd[2][e / 2], sel);
                *reinterpret_cast<uint2*>(vb + (8 * db + e) * (VS * 8)) = w2;
            }
        }
        const bool slow = __syncthreads_or(exp_nonfinite(vmax));
        load(p0 + 2 * KB);

        // scores: s[kt][i] = key p0 + 16 kt + 4 g + i, then 2^6 times their
        // exponentials relative to the reference (ls: the sum of these, unscaled)
        float4_t s[KB / 16];
        float ls, next;
        auto softmax = [&]() __attribute__((always_inline)) {
            if (p0 + KB > pos0 + t0 + 1) {      // some row of the block ends inside this tile
#pragma unroll
                for (int kt = 0; kt < KB / 16; kt++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (p0 + 16 * kt + 4 * g + i >= L) s[kt][i] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < KB / 16; kt++)
                mx = fmaxf(mx, fmaxf(fmaxf(s[kt][0], s[kt][1]), fmaxf(s[kt][2], s[kt][3])));
            const float m2 = rows_max4(mx) * c;
            next = m2 > ref + 8.0f ? m2 : ref;          // (the first score: ref is -inf)
            const float off = next == -INFINITY ? 0.0f : -next;
            ls = 0.0f;
#pragma unroll
            for (int kt = 0; kt < KB / 16; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s[kt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][i], c, off));
                    ls = ls + s[kt][i];
                    s[kt][i] = s[kt][i] * 64.0f;
                }
        };
#pragma unroll
        for (int kt = 0; kt < KB / 16; kt++) {
            float4_t sum[NS];
            half8_t k8[DS];
#pragma unroll
            for (int n = 0; n < NS; n++) sum[n] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < DS; d++) {
                k8[d] = __builtin_bit_cast(half8_t, ks[(16 * kt + c16) * KS + 4 * d + g]);
                sum[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[d], ql[d], sum[0], 0, 0, 0);
            }
#pragma unroll
            for (int d = 0; d < DS; d++)
                sum[d * NS / DS] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[d], qh[d], sum[d * NS / DS], 0, 0, 0);
#pragma unroll
            for (int n = 1; n < NS; n *= 2)
#pragma unroll
                for (int e = 0; e < NS; e += 2 * n) sum[e] += sum[e + n];
            s[kt] = sum[0];
        }
        softmax();
        if (__any(ls != ls)) {
            const uint16_t* kb = reinterpret_cast<const uint16_t*>(ks);
#pragma unroll
            for (int kt = 0; kt < KB / 16; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint16_t* kk = kb + (16 * kt + 4 * g + i) * (KS * 8);
                    float sum = 0.0f;
#pragma unroll 1
                    for (int d = 0; d < HD; d++) sum = sum + qrow[d] * f16_bits_to_f32(kk[d]);
                    s[kt][i] = sum * up;
                }
            softmax();
        }
        if (__any(next != ref)) {
            const float alpha = next == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ref - next);
            runL = runL * alpha;
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[d][i] = o[d][i] * alpha;
            ref = next;
        }
        runL = runL + ls;
        if (!slow) {
            half8_t ph[KB / 32], pl[KB / 32];
#pragma unroll
            for (int pr = 0; pr < KB / 32; pr++) {
                const float pv[8] = {s[2 * pr][0], s[2 * pr][1], s[2 * pr][2], s[2 * pr][3],
                                     s[2 * pr + 1][0], s[2 * pr + 1][1], s[2 * pr + 1][2], s[2 * pr + 1][3]};
                split16(pv, ph[pr], pl[pr]);
            }
#pragma unroll
            for (int d = 0; d < DT; d++) {
                float4_t t = float4_t{0.f, 0.f, 0.f, 0.f};
                half8_t v8[KB / 32];
#pragma unroll
                for (int pr = 0; pr < KB / 32; pr++) {
                    v8[pr] = __builtin_bit_cast(half8_t, vs[(16 * d + c16) * VS + 4 * pr + g]);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(v8[pr], pl[pr], t, 0, 0, 0);
                }
#pragma unroll
                for (int pr = 0; pr < KB / 32; pr++)
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(v8[pr], ph[pr], t, 0, 0, 0);
                o[d] += t;
            }
        } else {
            __syncthreads();                // every wave is done with the K tile
            float* pf = reinterpret_cast<float*>(ks) + (size_t)wave * 16 * KB;   // [16 rows][KB]
#pragma unroll
            for (int kt = 0; kt < KB / 16; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) pf[c16 * KB + 16 * kt + 4 * g + i] = s[kt][i];
            __syncthreads();
            const uint16_t* vb = reinterpret_cast<const uint16_t*>(vs);
#pragma unroll 1
            for (int key = 0; key < KB; key++) {
                if (p0 + key >= L) break;
                const float p = pf[c16 * KB + key];
                const int off = 32 * (key >> 5) + 8 * ((key >> 2) & 3) + 4 * ((key >> 4) & 1) + (key & 3);
#pragma unroll
                for (int d = 0; d < DT; d++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        o[d][i] = o[d][i] + p * f16_bits_to_f32(vb[(16 * d + 4 * g + i) * (VS * 8) + off]);
            }
        }
        __syncthreads();                    // the tile is rewritten
    }
    // group 1's sums, brought to a common reference
    float* const mg = reinterpret_cast<float*>(lds) + tid;
    if (grp == 1) {
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int i = 0; i < 4; i++) mg[(4 * d + i) * 256] = o[d][i];
        mg[4 * DT * 256] = ref;
        mg[(4 * DT + 1) * 256] = runL;
    }
    __syncthreads();
    if (grp == 1 || !tv) return;
    const float ref1 = mg[4 * DT * 256], top = fmaxf(ref, ref1);
    // (a reference of -inf: no score above -inf, sums of zero or NaN)
    const float a0 = ref == top ? 1.0f : __builtin_amdgcn_exp2f(ref - top);
    const float a1 = ref1 == top ? 1.0f : __builtin_amdgcn_exp2f(ref1 - top);
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int i = 0; i < 4; i++) o[d][i] = o[d][i] * a0 + mg[(4 * d + i) * 256] * a1;
    const float l = 64.0f * rows_sum4(runL * a0 + mg[(4 * DT + 1) * 256] * a1);
    uint16_t* dst = out16 + ((size_t)t * nq + hq) * HD + 4 * g;
#pragma unroll
    for (int d = 0; d < DT; d++) {
        uint2 w;
        w.x = (uint32_t)f32_to_f16_bits(o[d][0] / l) | ((uint32_t)f32_to_f16_bits(o[d][1] / l) << 16);
        w.y = (uint32_t)f32_to_f16_bits(o[d][2] / l) | ((uint32_t)f32_to_f16_bits(o[d][3] / l) << 16);
        *reinterpret_cast<uint2*>(dst + 16 * d) = w;
    }
}

// ---- tile choice ------------------------------------------------------------------

struct LongTile {
    int bm, bn, splits;
};

int cdiv(int a, int b) { return (a + b - 1) / b; }

// Tiles of 128 x 128 once there are 256 of them, one per CU, else 64-row or 64
// x 64 ones; the residual projections (which can sum partials) also split K
// into runs of at least 256 until there are about 512 blocks.  64 x 64 / 128 x
// 128, us: fp16 K = 1024, N = 4096: M = 512 (128 tiles of 128) 14.8 / 22.4, 896
// (224) 23.5 / 24.2, 1024 (256) 24.3 / 24.7, 1500 (384) 32.9 / 30.2, 2000 (512)
// 42.1 / 31.5; N = 6144: 640 (240) 24.2 / 24.4, 896 (336) 32.2 / 30.5, 2000
// (768) 62.2 / 53.7.  int8 and int4 break even later: int8 N = 4096 1024 (256)
// 24.2 / 27.8, 1500 33.2 / 33.0, 2000 42.1 / 33.7.  The tile is chosen before
// the split: N = 1024 with split and norm, fp16 K = 3072: M = 1000 (64) 24.9 /
// 27.6, 2000 (128) 40.8 / 36.6; K = 2048 20.3 / 25.8, 31.1 / 31.1.
constexpr int kMaxLongSplits = 8;
int long_splits(int tiles) {
    const int ns = 512 / tiles;
    return ns > kMaxLongSplits ? kMaxLongSplits : (ns < 1 ? 1 : ns);
}
LongTile long_tile(int M, int N, int K, bool can_split, bool wide) {
    LongTile t;
    t.splits = 1;
    if (cdiv(M, 128) * cdiv(N, 128) >= 256) t.bm = t.bn = 128;
    else if (wide) t.bm = 64, t.bn = 128;
    else t.bm = t.bn = 64;
    if (can_split) {
        const int nst = cdiv(K, kKT);
        int ns = long_splits(cdiv(M, t.bm) * cdiv(N, t.bn));
        if (ns > K / 256) ns = K / 256;
        if (ns < 1) ns = 1;
        const int per = cdiv(nst, ns);
        t.splits = cdiv(nst, per);          // none is empty
    }
    return t;
}

// Stages per partial sum.  A chain of sums rounds at the size it has reached,
// so few long ones and many short ones both lose, and products of 4-bit
// weights, short enough to be summed almost exactly inside an MFMA, want the
// longest.  Off the exact sums by (2-norm, 1e-8) at 1 / 2 / 4 stages, and the
// eight interleaved sums of the 64-row kernels, which these must not exceed:
// fp16 K = 256 7.0 / 8.0 / 10.4, 7.1; 576 8.2 / 8.8 / -, 8.4; 1024 9.6 / 9.5 /
// 11.2, 9.5; 3072 14.0 / 12.0 / 12.5, 13.9; 4096 - / 13.1 / 13.0, 15.7; int8 K
// = 512 7.4 / 7.5 / 9.3, 7.4; 1024 9.1 / 8.4 / 9.7, 8.4; 4096 - / 12.4 / 11.8,
// 14.0; int4, at 2 / 4 / this rule: K = 1536 7.2 / 6.5 / 6.5, 6.5; 4096 11.0 /
// 8.9 / 8.2, 8.2.  One chain over 3072 of fp16: 35.  The additions do not show
// in the time (fp16 2000 x 1024 x 6144 at 1 / 2 / 4: 52.4 / 55.2 / 54.3 us).
int long_run(int kind, int stages) {
    if (kind == MDX_W_I4) return 2 * cdiv(stages, 16);
    return stages <= (kind == MDX_W_F16 ? 12 : 8) ? 1 : (stages <= 48 ? 2 : 4);
}

template <int KIND, int EPI, int HD>
int long_launch_kind(const LongArgs& a, const LongTile& t, hipStream_t s) {
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n * a.splits)), block(256);
    if constexpr (EPI == LE_ROPE) {
        if (t.bm == 128) hipLaunchKernelGGL((k_long_gemm<KIND, 128, 128, 1, 1, EPI, HD>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_long_gemm<KIND, 64, 128, 1, 2, EPI, HD>), grid, block, 0, s, a);
    } else {
        if (t.bm == 128) hipLaunchKernelGGL((k_long_gemm<KIND, 128, 128, 2, 1, EPI, 0>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_long_gemm<KIND, 64, 64, 2, 2, EPI, 0>), grid, block, 0, s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int EPI, int HD>
int long_launch(LongArgs& a, int kind, const LongTile& t, void* stream) {
    a.tiles_m = cdiv(a.M, t.bm);
    a.tiles_n = EPI == LE_SWIGLU ? cdiv(a.N / 2, t.bn / 2) : cdiv(a.N, t.bn);
    a.splits = t.splits;
    a.per_split = cdiv(cdiv(a.K, kKT), t.splits);
    a.run = long_run(kind, a.per_split);
    if ((long long)a.tiles_m * a.tiles_n * a.splits > 0x7fffffffLL) return -1;
    hipStream_t s = (hipStream_t)stream;
    switch (kind) {
        case MDX_W_F16: return long_launch_kind<MDX_W_F16, EPI, HD>(a, t, s);
        case MDX_W_I8: return long_launch_kind<MDX_W_I8, EPI, HD>(a, t, s);
        case MDX_W_I4: return long_launch_kind<MDX_W_I4, EPI, HD>(a, t, s);
        default: return -5;
    }
}

LongArgs long_args(const uint16_t* x16, int M, const mdx_wdesc* w) {
    LongArgs a = {};
    a.x16 = x16;
    a.w = (const uint8_t*)w->w;
    a.scale = w->scale;
    a.M = M;
    a.K = w->K;
    a.N = w->N;
    return a;
}

}  // namespace

extern "C" {

int mdx_long_ok(const mdx_wdesc* w) {
    return w->kind >= MDX_W_F16 && w->kind <= MDX_W_I4 && w->K > 0 && w->K % 32 == 0 && w->N > 0;
}

int mdx_launch_long_gemm(const uint16_t* x16, int M, const mdx_wdesc* w, int swiglu, void* out, void* stream) {
    if (M <= 0 || !out || !mdx_long_ok(w) || (swiglu && w->N % 8)) return -1;
    LongArgs a = long_args(x16, M, w);
    const LongTile t = long_tile(M, w->N, w->K, false, false);
    if (swiglu) {
        a.out16 = (uint16_t*)out;
        return long_launch<LE_SWIGLU, 0>(a, w->kind, t, stream);
    }
    a.out = (float*)out;
    return long_launch<LE_STORE, 0>(a, w->kind, t, stream);
}

size_t mdx_long_scratch_floats(int M, int N) {
    /* the most that any launch of up to M rows leaves, whatever its K (hidden
     * 1024, 2048 rows: 8.4 MB) */
    size_t most = 0;
    for (int m = 1; m <= M; m++) {
        const LongTile t = long_tile(m, N, 256, false, false);
        const size_t n = (size_t)long_splits(cdiv(m, t.bm) * cdiv(N, t.bn)) * m * N;
        if (n > most) most = n;
    }
    return most;
}

int mdx_launch_long_residual_norm(const uint16_t* x16, int M, const mdx_wdesc* w, float* hidden,
                                  const float* norm_w, float eps, uint16_t* x16_out, float* scratch,
                                  void* stream) {
    if (M <= 0 || !mdx_long_ok(w) || w->N % 4) return -1;
    LongArgs a = long_args(x16, M, w);
    const LongTile t = long_tile(M, w->N, w->K, true, false);
    a.out = scratch;
    const int rc = long_launch<LE_PART, 0>(a, w->kind, t, stream);
    return rc ? rc : mdx_launch_residual_norm(scratch, t.splits, M, M, w->N, w->scale, hidden, norm_w, eps,
                                              x16_out, stream);
}

int mdx_launch_long_qkv_rope(const uint16_t* x16, int M, const mdx_wdesc* w, int pos0, const float* q_norm,
                             const float* k_norm, float eps, const float* cos_t, const float* sin_t, int nq,
                             int nkv, int hd, int rope_style, float* q_out, uint16_t* k_cache,
                             uint16_t* v_cache, void* stream) {
    if (M <= 0 || pos0 < 0 || !mdx_long_ok(w) || w->N != (nq + 2 * nkv) * hd) return -1;
    LongArgs a = long_args(x16, M, w);
    a.pos0 = pos0;
    a.nq = nq;
    a.nkv = nkv;
    a.style = rope_style;
    a.q_norm = q_norm;
    a.k_norm = k_norm;
    a.eps = eps;
    a.cos_t = cos_t;
    a.sin_t = sin_t;
    a.q_out = q_out;
    a.kc = k_cache;
    a.vc = v_cache;
    const LongTile t = long_tile(M, w->N, w->K, false, true);
    if (hd == 64) return long_launch<LE_ROPE, 64>(a, w->kind, t, stream);
    if (hd == 128) return long_launch<LE_ROPE, 128>(a, w->kind, t, stream);
    return -5;
}

int mdx_launch_long_attn(int pos0, const float* q, int M, const uint16_t* k_cache, const uint16_t* v_cache,
                         int nq, int nkv, int hd, uint16_t* out16, void* stream) {
    if (nkv <= 0 || nq % nkv || M <= 0 || pos0 < 0) return -1;
    const int G = nq / nkv;
    if (G < 1 || G > 4 || (G & (G - 1))) return -5;
    const int n_tb = cdiv(M, 64 / G);
    dim3 grid((unsigned)(n_tb * nkv));
#define MDX_LATTN(HD_, G_)                                                                                 \
    if (hd == HD_ && G == G_) {                                                                            \
        hipLaunchKernelGGL((k_attn_long<HD_, G_>), grid, dim3(512), 0, (hipStream_t)stream, pos0, M, q,    \
                           k_cache, v_cache, nkv, n_tb, out16);                                            \
        return hipGetLastError() == hipSuccess ? 0 : -4;                                                   \
    }
    MDX_LATTN(64, 1) MDX_LATTN(64, 2) MDX_LATTN(64, 4)
    MDX_LATTN(128, 1) MDX_LATTN(128, 2) MDX_LATTN(128, 4)
    MDX_LATTN(256, 1) MDX_LATTN(256, 2) MDX_LATTN(256, 4)
#undef MDX_LATTN
    return -5;
}

}  // extern "C"
