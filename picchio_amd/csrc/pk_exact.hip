// pk_exact.hip — the prompt path's dense arithmetic in the reference's order.
//
// forward_prefill (picchio.c:1795-1932) runs the attention projections,
// the sink attention and the router on every prompt position. Here those
// steps follow the reference operation by operation, so that the prompt's
// hidden states (and the KV rows the decode steps read) carry no rounding
// of their own:
//  * matmul_f32 (quant.h:117-148, AVX2 branch) and matmul_q8 (quant.h:152-186),
//    also behind matmul_qt for those formats: per (row, output) eight fp32
//    FMA chains, chain j over columns j, 8+j, ..., folded with hsum256's tree
//    ((c0+c4)+(c2+c6))+((c1+c5)+(c3+c7)) (quant.h:94-103), then the ragged
//    tail as gcc builds quant.h:138 (a block of four products added one by
//    one, then contracted FMAs); bias and residual added afterwards as
//    gqa_attention (picchio.c:530-532, :613) and forward_token (:1691) do.
//  * gqa_attention's softmax with sink (picchio.c:569-607): in-order score
//    dots (products added one by one), the maximum over sink and scores,
//    the sum of expf terms in position order starting from the sink's, each
//    weight divided by the sum, and the value rows accumulated in position
//    order, oh = fma(w, v, oh).
//  * the prompt router (picchio.c:1840-1844): the dot starts at the bias and
//    adds the products one by one.
// expf is evaluated as the double exp rounded to float (pk_expf_cr), which
// equals glibc's expf except where glibc's result is not the correctly
// rounded one (about 8e-5 of inputs).
#include "pk_dev.h"
#include "pk_engine.h"
#include "pk_i4_device.h"

#include <algorithm>
#include <type_traits>

namespace {

// ───────────────────────── matmul_f32 for S rows ─────────────────────────
// fp32 matrix instructions with K = 1 are one correctly rounded fused
// multiply-add per element (denormals kept: checked against fmaf over 12
// million random operands), so their accumulators are the reference's
// chains. They share the VALU's multipliers (28 ns per 2048 products and
// SIMD, v_fma 40), so what bounds these kernels is the weight stream for a
// few rows, the multipliers and how evenly the waves cover the SIMDs for
// many; a chain is serial over the columns, so K is never split.
//
// k_gemm_chain8, few rows: a workgroup of two waves computes 16 outputs of 16
// input rows (MF) or of NS = 1 or 2. The weights and inputs pass through LDS
// in chunks of 128 columns (two buffers, one barrier per chunk, two chunks'
// loads in flight in registers). Lane l = 16 b + r of wave h reads column
// 8k + 4h + b of weight row r and input row r (the row pitch of 4 mod 64
// floats puts the 64 lanes on 64 banks).
//  * MF: v_mfma_f32_16x16x1_4b_f32, the four blocks being chains 4h .. 4h + 3.
//  * NS: the same chains as v_fma, one per lane and input row.
// The second wave's chains join the first's through LDS for hsum256's tree.
// Measured (us, fp32, against the kernel before it: 64 rows x 32 outputs per
// workgroup on v_fma): 5120 x 2880, 1 row 179 -> 12.2, 64 rows 178 -> 44;
// INT8 201088 x 2880, 1 row 4100 -> 234 (k_gemv_chain8_q8: 130).
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

constexpr int CH_OUTS = 16;
constexpr int CH_THREADS = 128;
constexpr int CH_KC = 128;                // columns per staged chunk
constexpr int CH_MAX_Y = 65535;           // grid.y; further rows in grid.z

// Sixteen stored int8 weights as floats at d.
__device__ __forceinline__ void ch_put_i8(float *d, uint4 w) {
    const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int k = 0; k < 4; ++k)
        *reinterpret_cast<float4 *>(d + 4 * k) = make_float4((float)(int8_t)v[k], (float)(int8_t)(v[k] >> 8),
                                                             (float)(int8_t)(v[k] >> 16), (float)(int8_t)(v[k] >> 24));
}

// Output (s, o) from the tree a of its chains: the columns past the last
// whole 8, the row scale, bias and residual.
template <typename TW>
__device__ __forceinline__ void ch_finish(const float *X, int64_t ldx, const TW *W, const float *rscale,
                                          const float *bias, float *out, int64_t ldo, int S, int I, int O,
                                          int add_res, float a, int s, int o) {
    if (s >= S || o >= O) return;
    const TW *wr = W + (int64_t)o * I;
    const float *xr = X + (int64_t)s * ldx;
    int c = I & ~7;
    if constexpr (sizeof(TW) == 4) {
        if (I - c >= 4) {
            const float p0 = xr[c] * wr[c], p1 = xr[c + 1] * wr[c + 1];
            const float p2 = xr[c + 2] * wr[c + 2], p3 = xr[c + 3] * wr[c + 3];
            a = a + p0; a = a + p1; a = a + p2; a = a + p3;
            c += 4;
        }
    }
    for (; c < I; ++c) a = __builtin_fmaf(xr[c], (float)wr[c], a);
    if (rscale) a = a * rscale[o];
    if (bias) a = a + bias[o];
    float *y = out + (int64_t)s * ldo + o;
    *y = add_res ? *y + a : a;
}

// TW = int8_t: matmul_q8 (quant.h:152-186), the same chains over the weights
// converted to float, the tail as contracted FMAs, the sum times the row scale.
// VEC: 16-byte loads (16-byte aligned rows of X and W, I a multiple of 4, or
// of 16 for int8 weights).
template <typename TW, bool VEC, bool MF, int NS>
__global__ __launch_bounds__(CH_THREADS) void k_gemm_chain8(const float *__restrict__ X, int64_t ldx,
                                                            const TW *__restrict__ W,
                                                            const float *__restrict__ rscale,
                                                            const float *__restrict__ bias, float *out, int64_t ldo,
                                                            int S, int I, int O, int add_res) {
    constexpr int KC = CH_KC, P = KC + 4, XR = MF ? 16 : NS;
    constexpr int WV = VEC ? 16 / sizeof(TW) : 1, XV = VEC ? 4 : 1;     // values per load
    constexpr int WN = (CH_OUTS * KC / WV + CH_THREADS - 1) / CH_THREADS;
    constexpr int XN = (XR * KC / XV + CH_THREADS - 1) / CH_THREADS;
    constexpr int BUF = (CH_OUTS + XR) * P;
    __shared__ __attribute__((aligned(16))) float lds[2 * BUF];
    const int tid = threadIdx.x, lane = tid & 63;
    const int h = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int o0 = blockIdx.x * CH_OUTS;
    const int s0 = ((int)blockIdx.y + CH_MAX_Y * (int)blockIdx.z) * XR;
    const int I8 = I & ~7, chunks = (I8 + KC - 1) / KC;

    struct stage {
        typename std::conditional<VEC, uint4, TW>::type w[WN];
        typename std::conditional<VEC, float4, float>::type x[XN];
    };
    // load e of a chunk: row e / (KC / V), columns V (e % (KC / V)) .. (rows
    // and columns past the end repeat the last ones; they are not used)
    auto load = [&](stage &st, int c0) {
        const int nc = min(KC, I8 - c0);
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int e = min(tid + CH_THREADS * u, CH_OUTS * KC / WV - 1), r = e / (KC / WV);
            const int c = min(WV * (e % (KC / WV)), nc - WV);
            const TW *p = W + (int64_t)min(o0 + r, O - 1) * I + c0 + c;
            if constexpr (VEC) st.w[u] = pk_load_nt(reinterpret_cast<const uint4 *>(p));
            else st.w[u] = *p;
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int e = min(tid + CH_THREADS * u, XR * KC / XV - 1), r = e / (KC / XV);
            const int c = min(XV * (e % (KC / XV)), nc - XV);
            const float *p = X + (int64_t)min(s0 + r, S - 1) * ldx + c0 + c;
            if constexpr (VEC) st.x[u] = *reinterpret_cast<const float4 *>(p);
            else st.x[u] = *p;
        }
    };
    auto store = [&](const stage &st, float *wl, float *xl) {
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int e = tid + CH_THREADS * u, r = e / (KC / WV), c = WV * (e % (KC / WV));
            if (WN * CH_THREADS > CH_OUTS * KC / WV && e >= CH_OUTS * KC / WV) break;
            float *d = wl + r * P + c;
            if constexpr (VEC && sizeof(TW) == 4) {
                *reinterpret_cast<uint4 *>(d) = st.w[u];
            } else if constexpr (VEC) {
                ch_put_i8(d, st.w[u]);
            } else {
                *d = (float)st.w[u];
            }
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int e = tid + CH_THREADS * u, r = e / (KC / XV), c = XV * (e % (KC / XV));
            if (XN * CH_THREADS > XR * KC / XV && e >= XR * KC / XV) break;
            if constexpr (VEC) *reinterpret_cast<float4 *>(xl + r * P + c) = st.x[u];
            else xl[r * P + c] = st.x[u];
        }
    };

    const int r = lane & 15, b = lane >> 4;
    f32x16 acc;
    float a1[NS ? NS : 1];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < NS; ++t) a1[t] = 0.0f;
    auto multiply = [&](const float *wl, const float *xl, int steps) {
        const float *wp = wl + r * P + 4 * h + b, *xp = xl + (MF ? r * P : 0) + 4 * h + b;
        auto step = [&](int k) {
            const float w = wp[8 * k];
            if constexpr (MF) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(xp[8 * k], w, acc, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < NS; ++t) a1[t] = __builtin_fmaf(xp[t * P + 8 * k], w, a1[t]);
        };
        if (steps == KC / 8) {
#pragma unroll
            for (int k = 0; k < KC / 8; ++k) step(k);
        } else {
            for (int k = 0; k < steps; ++k) step(k);
        }
    };
    stage st[2];
    if (chunks > 0) {
        load(st[0], 0);
        load(st[1], min(1, chunks - 1) * KC);
    }
    const auto chunk = [&](stage &sv, int n, float *wl, bool refill) {
        float *xl = wl + CH_OUTS * P;
        store(sv, wl, xl);
        if (refill) load(sv, min(n + 2, chunks - 1) * KC);
        __syncthreads();
        multiply(wl, xl, min(KC, I8 - n * KC) / 8);
    };
    // pairs without guards (a guarded refill would make every wait one for all
    // outstanding loads), then the last
    int n = 0;
    for (; n + 2 <= chunks; n += 2) {
        chunk(st[0], n, lds, true);
        chunk(st[1], n + 1, lds + BUF, true);
    }
    if (n < chunks) chunk(st[0], n, lds, false);
    // hsum256: ((c0+c4)+(c2+c6))+((c1+c5)+(c3+c7)); wave 1 holds c4 .. c7
    __syncthreads();
    if (h == 1) {
        if constexpr (MF) {
#pragma unroll
            for (int i = 0; i < 16; ++i) lds[i * 64 + lane] = acc[i];
        }
#pragma unroll
        for (int t = 0; t < NS; ++t) lds[t * 64 + lane] = a1[t];
    }
    __syncthreads();
    if (h == 1) return;
    if constexpr (MF) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // register 4 b + i: chain b, input row 4 (lane / 16) + i, output lane % 16
            const float b0 = acc[i] + lds[i * 64 + lane], b1 = acc[4 + i] + lds[(4 + i) * 64 + lane];
            const float b2 = acc[8 + i] + lds[(8 + i) * 64 + lane], b3 = acc[12 + i] + lds[(12 + i) * 64 + lane];
            ch_finish(X, ldx, W, rscale, bias, out, ldo, S, I, O, add_res, (b0 + b2) + (b1 + b3), s0 + 4 * b + i,
                      o0 + r);
        }
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        float v = a1[t] + lds[t * 64 + lane];        // lane 16 b + r: c_b + c_{b+4}
        v = v + __shfl_xor(v, 32, 64);
        v = v + __shfl_xor(v, 16, 64);
        if (b == 0) ch_finish(X, ldx, W, rscale, bias, out, ldo, S, I, O, add_res, v, s0 + t, o0 + r);
    }
}

// One to four rows of many int8 outputs: a wave computes 64 outputs, lane =
// weight row with its eight chains in registers, the inputs in scalar
// registers. The wave's 64 x 128 byte chunk passes through its own LDS (rows
// 144 bytes apart: 16-byte reads of 16 rows on distinct banks), the next
// chunk's loads in flight. Per weight one conversion and NS fused
// multiply-adds (2.2 + 1.25 NS ns per 64 and SIMD), so it is bound by the
// weight stream. 201088 x 2880, 1 row: 130 us = 4.5 TB/s;
// k_gemm_chain8 234 (it keeps the weights in LDS as floats).
constexpr int GQ_KC = 128, GQ_P = GQ_KC + 16;
template <int NS>
__global__ __launch_bounds__(64) void k_gemv_chain8_q8(const float *__restrict__ X, const int8_t *__restrict__ W,
                                                       const float *__restrict__ rscale, float *out, int S, int I,
                                                       int O) {
    __shared__ __attribute__((aligned(16))) uint8_t wl[64 * GQ_P];
    const int lane = threadIdx.x, o0 = blockIdx.x * 64;
    const int chunks = (I + GQ_KC - 1) / GQ_KC;      // (I % 16 == 0)
    uint4 st[8];
    // load u: rows 8 u + lane / 8, 16 bytes at 16 (lane % 8)
    const int lr = lane >> 3, lc = 16 * (lane & 7);
    auto load = [&](int c0) {
        const int c = min(c0 + lc, I - 16);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            st[u] = pk_load_nt(reinterpret_cast<const uint4 *>(W + (int64_t)min(o0 + 8 * u + lr, O - 1) * I + c));
    };
    float acc[NS][8];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[t][j] = 0.0f;
    const pk_cptr<float> x = pk_const(X);
    load(0);
    for (int n = 0; n < chunks; ++n) {
        const int c0 = n * GQ_KC;
#pragma unroll
        for (int u = 0; u < 8; ++u) *reinterpret_cast<uint4 *>(wl + (8 * u + lr) * GQ_P + lc) = st[u];
        pk_wave_lds_order();
        load(min(n + 1, chunks - 1) * GQ_KC);
        const int pieces = min(GQ_KC, I - c0) / 16;
        for (int m = 0; m < pieces; ++m) {
            const uint4 v = *reinterpret_cast<const uint4 *>(wl + lane * GQ_P + 16 * m);
            const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float w = (float)(int8_t)(d[q] >> (8 * i));
#pragma unroll
                    for (int t = 0; t < NS; ++t) {
                        const int j = 4 * (q & 1) + i;
                        acc[t][j] = __builtin_fmaf(x[(int64_t)min(t, S - 1) * I + c0 + 16 * m + 4 * q + i], w, acc[t][j]);
                    }
                }
        }
        pk_wave_lds_order();
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        const float b0 = acc[t][0] + acc[t][4], b1 = acc[t][1] + acc[t][5];
        const float b2 = acc[t][2] + acc[t][6], b3 = acc[t][3] + acc[t][7];
        ch_finish<int8_t>(X, I, W, rscale, nullptr, out, O, S, I, O, 0, (b0 + b2) + (b1 + b3), t, o0 + lane);
    }
}

// Many rows (fp32 or int8 weights, 16-byte loads): a workgroup of four waves
// computes 64 outputs of 64 input rows, wave (p, q) outputs 32 p .. and rows
// 32 q .. with v_mfma_f32_32x32x1_2b_f32: lane l = 32 b + r reads columns
// 8k + 4b .. + 3 of weight row r and input row r as one float4 each, and
// instruction i multiplies component i, its two blocks being chains i and
// 4 + i. Chunks of 32 columns, staged as above. 5120 x 2880, 512 rows: 164 us
// (92 TFLOP/s; 349 in 16-row tiles).
constexpr int CT_TILE = 64, CT_KC = 32, CT_P = CT_KC + 4;
template <typename TW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_chain8_tile(
    const float *__restrict__ X, int64_t ldx, const TW *__restrict__ W, const float *__restrict__ rscale,
    const float *__restrict__ bias, float *out, int64_t ldo, int S, int I, int O, int add_res) {
    constexpr int WV = 16 / sizeof(TW);
    constexpr int WN = CT_TILE * CT_KC / WV / 256 > 0 ? CT_TILE * CT_KC / WV / 256 : 1, XN = CT_TILE * CT_KC / 4 / 256;
    constexpr int BUF = 2 * CT_TILE * CT_P;
    __shared__ __attribute__((aligned(16))) float lds[2 * BUF];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = wave & 1, q = wave >> 1;
    const int o0 = blockIdx.x * CT_TILE, s0 = blockIdx.y * CT_TILE;
    const int I8 = I & ~7, chunks = (I8 + CT_KC - 1) / CT_KC;
    const int we = min(tid, CT_TILE * CT_KC / WV - 1);          // (int8: 128 loads of 16 columns)
    struct stage {
        pk_f32x4 w[WN];
        pk_f32x4 x[XN];
    };
    auto load = [&](stage &st, int c0) {
        const int nc = min(CT_KC, I8 - c0);
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int e = we + 256 * u, r = e / (CT_KC / WV), c = min(WV * (e % (CT_KC / WV)), nc - WV);
            st.w[u] = *reinterpret_cast<const pk_f32x4 *>(W + (int64_t)min(o0 + r, O - 1) * I + c0 + c);
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int e = tid + 256 * u, r = e / (CT_KC / 4), c = min(4 * (e % (CT_KC / 4)), nc - 4);
            st.x[u] = *reinterpret_cast<const pk_f32x4 *>(X + (int64_t)min(s0 + r, S - 1) * ldx + c0 + c);
        }
    };
    auto store = [&](const stage &st, float *wl, float *xl) {
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int e = we + 256 * u, r = e / (CT_KC / WV);
            float *d = wl + r * CT_P + WV * (e % (CT_KC / WV));
            if constexpr (sizeof(TW) == 4) {
                *reinterpret_cast<pk_f32x4 *>(d) = st.w[u];
            } else if (tid == we) {
                ch_put_i8(d, __builtin_bit_cast(uint4, st.w[u]));
            }
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int e = tid + 256 * u;
            *reinterpret_cast<pk_f32x4 *>(xl + e / (CT_KC / 4) * CT_P + 4 * (e % (CT_KC / 4))) = st.x[u];
        }
    };
    f32x32 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 32; ++k) acc[i][k] = 0.0f;
    const int r = lane & 31, b = lane >> 5;
    stage st[2];
    if (chunks > 0) {
        load(st[0], 0);
        load(st[1], min(1, chunks - 1) * CT_KC);
    }
    const auto chunk = [&](stage &sv, int n, float *wl, bool refill) {
        float *xl = wl + CT_TILE * CT_P;
        store(sv, wl, xl);
        if (refill) load(sv, min(n + 2, chunks - 1) * CT_KC);
        __syncthreads();
        const int steps = min(CT_KC, I8 - n * CT_KC) / 8;
        const float *wp = wl + (32 * p + r) * CT_P + 4 * b, *xp = xl + (32 * q + r) * CT_P + 4 * b;
#pragma unroll
        for (int k = 0; k < CT_KC / 8; ++k) {
            if (k < steps) {
                const float4 w = *reinterpret_cast<const float4 *>(wp + 8 * k);
                const float4 x = *reinterpret_cast<const float4 *>(xp + 8 * k);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(x.x, w.x, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x1f32(x.y, w.y, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_32x32x1f32(x.z, w.z, acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f32_32x32x1f32(x.w, w.w, acc[3], 0, 0, 0);
            }
        }
    };
    // pairs without guards, then the last
    int n = 0;
    for (; n + 2 <= chunks; n += 2) {
        chunk(st[0], n, lds, true);
        chunk(st[1], n + 1, lds + BUF, true);
    }
    if (n < chunks) chunk(st[0], n, lds, false);
    // registers k / 16 + k: block k / 16 (chains i, 4 + i), input row
    // 8 (k % 16 / 4) + 4 b + k % 4, output r
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const float b0 = acc[0][k] + acc[0][16 + k], b1 = acc[1][k] + acc[1][16 + k];
        const float b2 = acc[2][k] + acc[2][16 + k], b3 = acc[3][k] + acc[3][16 + k];
        ch_finish(X, ldx, W, rscale, bias, out, ldo, S, I, O, add_res, (b0 + b2) + (b1 + b3),
                  s0 + 32 * q + 8 * (k >> 2) + 4 * b + (k & 3), o0 + 32 * p + r);
    }
}

// ───────────────────── gqa_attention of prompt rows ─────────────────────
// One wave per (head, row). Scores of the row's window into LDS, the max,
// the exp terms, their sum in position order (one lane), the weights, then
// lane i < hd accumulates column i of the values in position order.
__global__ __launch_bounds__(64) void k_attn_rows_exact(int pos_base, const float *qkv, int64_t qkv_stride,
                                                        const float *Kl, const float *Vl, int H, int KVH, int hd,
                                                        int ctx, int sliding, int window, const float *sinks,
                                                        float *att) {
    extern __shared__ float sc[];              // [window positions]
    __shared__ float s_sum;
    const int h = blockIdx.x, r = blockIdx.y, lane = threadIdx.x;
    const int pos = pos_base + r;
    int end = pos < ctx ? pos : ctx - 1;
    int start = 0;
    if (sliding) {
        start = end - window + 1;
        if (start < 0) start = 0;
    }
    const int n = end - start + 1;
    const int kv_dim = KVH * hd, kvh = h / (H / KVH);
    const float *qh = qkv + (int64_t)r * qkv_stride + h * hd;
    const float scale = 1.0f / sqrtf((float)hd);
    for (int t = lane; t < n; t += 64) {
        // (the K cache's chunk layout: a position's float4 columns cs apart)
        const int tk = start + t;
        const int cs = pk_k_cs(tk, ctx);
        const float4 *kt = reinterpret_cast<const float4 *>(Kl + pk_k_off(tk, kvh, 0, ctx, KVH, hd));
        const float4 *q4 = reinterpret_cast<const float4 *>(qh);
        float dot = 0.0f;
        for (int i = 0; i < hd / 4; ++i) {
            const float4 k4 = kt[(int64_t)i * cs], qq = q4[i];
            float p;
            p = qq.x * k4.x; dot = dot + p;
            p = qq.y * k4.y; dot = dot + p;
            p = qq.z * k4.z; dot = dot + p;
            p = qq.w * k4.w; dot = dot + p;
        }
        sc[t] = dot * scale;
    }
    __syncthreads();
    // max over the sink and the scores (a comparison: order-free)
    float mx = -INFINITY;
    for (int t = lane; t < n; t += 64) mx = fmaxf(mx, sc[t]);
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    const float sink = sinks[h];
    if (sink > mx) mx = sink;
    for (int t = lane; t < n; t += 64) sc[t] = pk_expf_cr(sc[t] - mx);
    __syncthreads();
    if (lane == 0) {
        float sum = pk_expf_cr(sink - mx);
        for (int t = 0; t < n; ++t) sum += sc[t];
        s_sum = sum;
    }
    __syncthreads();
    const float sum = s_sum;
    for (int t = lane; t < n; t += 64) sc[t] = sc[t] / sum;
    __syncthreads();
    for (int i = lane; i < hd; i += 64) {
        const float *vc = Vl + (int64_t)start * kv_dim + kvh * hd + i;
        float o = 0.0f;
        for (int t = 0; t < n; ++t) o = __builtin_fmaf(sc[t], vc[(int64_t)t * kv_dim], o);
        att[(int64_t)r * H * hd + h * hd + i] = o;
    }
}

// ───────────────────────── prompt router ─────────────────────────
// logits[s][e] = bias[e] + x[s][0]*w[e][0] + ... in order (products
// rounded, then added). 128 threads: lane t takes expert t % E of row
// s0 + t / E; the router rows are staged transposed in LDS, 64 columns at a
// time, the input rows beside them.
constexpr int RS_KC = 64;

__global__ __launch_bounds__(128) void k_router_seq(const float *__restrict__ X, const float *__restrict__ R,
                                                    const float *__restrict__ bias, int S, int D, int E,
                                                    float *logits) {
    extern __shared__ float lds_rs[];
    const int rows = 128 / E;                  // rows per block (E <= 128)
    float *wt = lds_rs;                        // [RS_KC][E]
    float *xt = lds_rs + RS_KC * E;            // [rows][RS_KC]
    const int tid = threadIdx.x;
    const int e = tid % E, rr = tid / E;
    const int s = blockIdx.x * rows + rr;
    const bool live = rr < rows && s < S;
    float acc = live ? bias[e] : 0.0f;
    for (int c0 = 0; c0 < D; c0 += RS_KC) {
        const int nc = min(RS_KC, D - c0);
        __syncthreads();
        for (int q = tid; q < E * RS_KC; q += 128) {
            const int ee = q / RS_KC, c = q - ee * RS_KC;
            wt[c * E + ee] = c < nc ? R[(int64_t)ee * D + c0 + c] : 0.0f;
        }
        for (int q = tid; q < rows * RS_KC; q += 128) {
            const int r2 = q / RS_KC, c = q - r2 * RS_KC;
            const int s2 = blockIdx.x * rows + r2;
            xt[r2 * RS_KC + c] = (c < nc && s2 < S) ? X[(int64_t)s2 * D + c0 + c] : 0.0f;
        }
        __syncthreads();
        if (live)
            for (int c = 0; c < nc; ++c) {
                const float p = xt[rr * RS_KC + c] * wt[c * E + e];
                acc = acc + p;
            }
    }
    if (live) logits[(int64_t)s * E + e] = acc;
}

// The same sums with 16-byte loads (D % 4 == 0, aligned rows): one wave per
// block of EB experts and 64 / EB rows, lane t taking expert t % EB of row t /
// EB. What bounds it is the chain of dependent adds (2880 x 1.6 ns, each
// after its product) and the latency of the router rows: a 64-column chunk is
// multiplied in ~0.3 us, so RQ_PF chunks' loads are in flight in registers.
// A chunk passes through the wave's own LDS (rows 4 mod 64 floats apart, read
// as float4): several waves of one workgroup would share the loads but are
// bound by their LDS reads. 64 rows x 32 experts x 2880: 30 us; 38 with four
// waves per workgroup, 70 with two and one chunk in flight.
constexpr int RQ_P = RS_KC + 4;          // padded LDS row (floats)
constexpr int RQ_PF = 4;                 // chunks in flight
template <int EB>
__global__ __launch_bounds__(64) void k_router_seq4(const float *__restrict__ X, const float *__restrict__ R,
                                                    const float *__restrict__ bias, int S, int D, int E,
                                                    float *logits) {
    constexpr int ROWS = 64 / EB, C4 = RS_KC / 4;
    constexpr int WN = EB * C4 / 64, XN = (ROWS * C4 + 63) / 64;     // 16-byte loads per lane and chunk
    __shared__ __attribute__((aligned(16))) float lds[2][(EB + ROWS) * RQ_P];
    const int lane = threadIdx.x;
    const int e0 = blockIdx.y * EB, s0 = blockIdx.x * ROWS;
    const int e = e0 + lane % EB, s = s0 + lane / EB;
    float acc = bias[min(e, E - 1)];
    const int chunks = (D + RS_KC - 1) / RS_KC;
    struct stage {
        pk_f32x4 w[WN], x[XN];
    };
    // (rows and columns past the end repeat the last ones; they are not used)
    auto load = [&](stage &st, int n) {
        const int c0 = min(n, chunks - 1) * RS_KC, last = min(RS_KC, D - c0) / 4 - 1;
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int q = lane + 64 * u;
            st.w[u] = *reinterpret_cast<const pk_f32x4 *>(R + (int64_t)min(e0 + q / C4, E - 1) * D + c0 +
                                                          4 * min(q % C4, last));
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int q = min(lane + 64 * u, ROWS * C4 - 1);
            st.x[u] = *reinterpret_cast<const pk_f32x4 *>(X + (int64_t)min(s0 + q / C4, S - 1) * D + c0 +
                                                          4 * min(q % C4, last));
        }
    };
    stage st[RQ_PF];
#pragma unroll
    for (int u = 0; u < RQ_PF; ++u) load(st[u], u);
    // (the bias is waited for here: inside the loop the compiler would wait
    // for every outstanding load before the first add)
    asm volatile("" ::"v"(acc));
    const auto chunk = [&](stage &sv, int n, float *wt, bool refill) {
        float *xt = wt + EB * RQ_P;
#pragma unroll
        for (int u = 0; u < WN; ++u) {
            const int q = lane + 64 * u;
            *reinterpret_cast<pk_f32x4 *>(wt + q / C4 * RQ_P + 4 * (q % C4)) = sv.w[u];
        }
#pragma unroll
        for (int u = 0; u < XN; ++u) {
            const int q = lane + 64 * u;
            if (q < ROWS * C4) *reinterpret_cast<pk_f32x4 *>(xt + q / C4 * RQ_P + 4 * (q % C4)) = sv.x[u];
        }
        if (refill) load(sv, n + RQ_PF);
        __syncthreads();                          // (one wave: orders the LDS writes and reads)
        const int nc4 = min(RS_KC, D - n * RS_KC) / 4;
        const float *wp = wt + lane % EB * RQ_P, *xp = xt + lane / EB * RQ_P;
        const auto add4 = [&](const pk_f32x4 &w, const pk_f32x4 &x) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float p = x[k] * w[k];
                acc = acc + p;
            }
        };
        if (nc4 == C4) {
            // every LDS read goes out before the first add
            pk_f32x4 w[C4], x[C4];
#pragma unroll
            for (int j = 0; j < C4; ++j) {
                w[j] = *reinterpret_cast<const pk_f32x4 *>(wp + 4 * j);
                x[j] = *reinterpret_cast<const pk_f32x4 *>(xp + 4 * j);
            }
#pragma unroll
            for (int j = 0; j < C4; ++j) add4(w[j], x[j]);
        } else {
            for (int j = 0; j < nc4; ++j)
                add4(*reinterpret_cast<const pk_f32x4 *>(wp + 4 * j), *reinterpret_cast<const pk_f32x4 *>(xp + 4 * j));
        }
    };
    // whole rounds without guards (a guarded refill would make every wait one
    // for all outstanding loads), then the rest
    int n = 0;
    for (; n + RQ_PF <= chunks; n += RQ_PF) {
#pragma unroll
        for (int v = 0; v < RQ_PF; ++v) chunk(st[v], n + v, lds[v & 1], true);
    }
#pragma unroll
    for (int v = 0; v < RQ_PF; ++v)
        if (n + v < chunks) chunk(st[v], n + v, lds[v & 1], false);
    if (e < E && s < S) logits[(int64_t)s * E + e] = acc;
}

}  // namespace

// Whether more than 32 rows (16-byte loads) run in 64 x 64 tiles: where the
// 16-row tiles take longer. At 2880 columns those take 8.6 us per workgroup (16
// outputs x 16 rows) and CU, the 64 x 64 tiles 12 us and 52 per round of the CUs.
// fp32, 16-row / 64 x 64 tiles, us: 5120 x 2880, 96 rows (7.5 per CU, one round)
// 61 / 64, 128 rows 87 / 64, 512 rows 349 / 164; 2880 x 4096, 160 rows (7.0) 88 /
// 90, 192 rows (8.4) 108 / 90; 16000 x 2880, 33 rows 98 / 65, 65 rows 169 / 111;
// 1000 x 2880, 320 rows (4.9) 51 / 64, 512 rows (7.9) 75 / 65. int8, whose 64 x 64
// tiles also convert the weights: 5120 x 2880, 96 rows 62 / 72; 1000 x 2880, 512
// rows 66 / 72; 2880 x 4096, 192 rows 104 / 101.
static bool chain8_tiled(int S, int O, bool i8) {
    const int64_t cus = pk_device_cus();
    const int64_t tiles = (int64_t)((O + CT_TILE - 1) / CT_TILE) * ((S + CT_TILE - 1) / CT_TILE);
    const int64_t few = (int64_t)((O + CH_OUTS - 1) / CH_OUTS) * ((S + 15) / 16), rounds = (tiles + cus - 1) / cus;
    return S > 32 && 2 * few > ((i8 ? 5 : 3) + 12 * rounds) * cus;
}

// (16-row tiles: one or two rows on v_fma)
template <typename TW>
static int launch_chain8(const float *X, int64_t ldx, const TW *W, const float *rscale, const float *bias, float *out,
                         int64_t ldo, int S, int I, int O, bool add_res, hipStream_t st) {
    PK_CHECK(S > 0 && I > 0 && O > 0, PK_ERR_ARG, "gemm chain8: bad shape");
    PK_CHECK((S + 63) / 64 <= CH_MAX_Y, PK_ERR_UNSUPPORTED, "gemm chain8: %d rows", S);
    const bool vec = (ldx & 3) == 0 && I % (16 / (int)sizeof(TW)) == 0 && (((uintptr_t)X | (uintptr_t)W) & 15) == 0;
    const int64_t ot = (O + CT_TILE - 1) / CT_TILE, rt = (S + CT_TILE - 1) / CT_TILE;
    if (vec && chain8_tiled(S, O, sizeof(TW) == 1)) {
        hipLaunchKernelGGL(k_gemm_chain8_tile<TW>, dim3((unsigned)ot, (unsigned)rt), dim3(256), 0, st, X, ldx, W,
                           rscale, bias, out, ldo, S, I, O, add_res ? 1 : 0);
        PK_HIP(hipGetLastError());
        return PK_OK;
    }
    const int tiles = S <= 2 ? 1 : (S + 15) / 16;
    const dim3 grid((O + CH_OUTS - 1) / CH_OUTS, std::min(tiles, CH_MAX_Y), (tiles + CH_MAX_Y - 1) / CH_MAX_Y);
#define PK_CH8(V, M, N)                                                                                             \
    hipLaunchKernelGGL((k_gemm_chain8<TW, V, M, N>), grid, dim3(CH_THREADS), 0, st, X, ldx, W, rscale, bias, out, ldo, \
                       S, I, O, add_res ? 1 : 0)
    if (S == 1) {
        if (vec) PK_CH8(true, false, 1); else PK_CH8(false, false, 1);
    } else if (S == 2) {
        if (vec) PK_CH8(true, false, 2); else PK_CH8(false, false, 2);
    } else {
        if (vec) PK_CH8(true, true, 0); else PK_CH8(false, true, 0);
    }
#undef PK_CH8
    PK_HIP(hipGetLastError());
    return PK_OK;
}

int pk_launch_gemm_chain8(const float *X, int64_t ldx, const float *W, const float *bias, float *out, int64_t ldo,
                          int S, int I, int O, bool add_res, hipStream_t st) {
    return launch_chain8<float>(X, ldx, W, nullptr, bias, out, ldo, S, I, O, add_res, st);
}

int pk_launch_gemm_chain8_q8(const float *X, const int8_t *W, const float *scale, float *out, int S, int I, int O,
                             hipStream_t st) {
    PK_CHECK(S > 0 && I > 0 && O > 0 && scale, PK_ERR_ARG, "gemm chain8 q8: bad argument");
    // a wave per 64 outputs from three waves per CU on (k_gemm_chain8 / here, us at
    // 2880 columns: 16000 outputs, 1 row 23 / 32; 32000, 1 row 42 / 37, 4 rows 63 /
    // 71; 50000, 1 row 66 / 40, 4 rows 102 / 73; 201088, 1 row 234 / 130)
    if (S <= 4 && (I & 15) == 0 && (((uintptr_t)X | (uintptr_t)W) & 15) == 0 &&
        (O + 63) / 64 >= 3 * pk_device_cus()) {
        const dim3 grid((O + 63) / 64);
        if (S == 1) hipLaunchKernelGGL(k_gemv_chain8_q8<1>, grid, dim3(64), 0, st, X, W, scale, out, S, I, O);
        else if (S == 2) hipLaunchKernelGGL(k_gemv_chain8_q8<2>, grid, dim3(64), 0, st, X, W, scale, out, S, I, O);
        else hipLaunchKernelGGL(k_gemv_chain8_q8<4>, grid, dim3(64), 0, st, X, W, scale, out, S, I, O);
        PK_HIP(hipGetLastError());
        return PK_OK;
    }
    return launch_chain8<int8_t>(X, I, W, scale, nullptr, out, O, S, I, O, false, st);
}

int pk_launch_attn_rows_exact(int pos_base, int n, const float *qkv, int64_t qkv_stride, const float *Kl,
                              const float *Vl, int H, int KVH, int hd, int ctx, int sliding, int window,
                              const float *sinks, float *att, hipStream_t st) {
    PK_CHECK(n > 0 && n <= 65535 && H % KVH == 0, PK_ERR_ARG, "attention rows: bad shape");
    const int last = pos_base + n - 1;
    int span = (last < ctx ? last : ctx - 1) + 1;
    if (sliding && span > window) span = window;
    PK_CHECK((size_t)span * 4 <= 64 * 1024, PK_ERR_UNSUPPORTED, "attention rows: window of %d positions", span);
    hipLaunchKernelGGL(k_attn_rows_exact, dim3(H, n), dim3(64), (size_t)span * 4, st, pos_base, qkv, qkv_stride,
                       Kl, Vl, H, KVH, hd, ctx, sliding, window, sinks, att);
    PK_HIP(hipGetLastError());
    return PK_OK;
}

int pk_launch_router_seq(const float *X, const float *R, const float *bias, int S, int D, int E, float *logits,
                         hipStream_t st) {
    PK_CHECK(S > 0 && D > 0 && E > 0 && E <= 128, PK_ERR_ARG, "router: bad shape");
    if ((D & 3) == 0 && (((uintptr_t)X | (uintptr_t)R) & 15) == 0) {
        if (E <= 8)
            hipLaunchKernelGGL(k_router_seq4<8>, dim3((S + 7) / 8), dim3(64), 0, st, X, R, bias, S, D, E, logits);
        else
            hipLaunchKernelGGL(k_router_seq4<32>, dim3((S + 1) / 2, (E + 31) / 32), dim3(64), 0, st, X, R, bias, S, D,
                               E, logits);
        PK_HIP(hipGetLastError());
        return PK_OK;
    }
    const int rows = 128 / E;
    const size_t lds = ((size_t)RS_KC * E + (size_t)rows * RS_KC) * 4;
    hipLaunchKernelGGL(k_router_seq, dim3((S + rows - 1) / rows), dim3(128), lds, st, X, R, bias, S, D, E, logits);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
