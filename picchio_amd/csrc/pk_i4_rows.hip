// pk_i4_rows.hip — the INT4 gs64 GEMV of several input rows on the fp32
// matrix instructions, bit-identical to quant.h:259-319 (matmul_i4_gs).
//
// A wave owns one 64-row block of a matrix (lane = row, as in the tile
// layout) and up to 8 input rows, and walks the row's groups in order. Each
// weight nibble is decoded once (v_cvt_off_f32_i4) and multiplies four input
// rows per v_mfma_f32_4x4x1_16b_f32: 16 blocks of 4 lanes hold 64 weight rows
// (operand B), the A operand's block `abid` (four input rows at one column)
// is broadcast to all of them (cbsz = 4), and the result has one weight row
// per lane and one input row per register. With K = 1 the instruction is a
// single fused multiply-add per element, correctly rounded and with
// denormals kept (checked against fmaf over 12 million random operands), so
// the eight accumulators per input row are exactly the eight FMA chains of
// the AVX2 loop, and their fold and the fold over groups are the same
// operations as k_i4_gemv's.
//
// What bounds it: the multipliers. A group costs a wave of 8 input rows 128
// matrix instructions (3.9 ns each), 64 decodes (2.2) and 64 additions of the
// chains' trees (1.6), none of which overlap: fp32 matrix instructions run
// on the VALU's multipliers (a probe's times add up at 1 to 4 waves per
// SIMD). The per-row kernel k_i4_gemv_stream pays 64 decodes, 64 fused
// multiply-adds and 8 additions per input row and reads the expert's block
// once per (row, expert) pair. Measured, 64 tokens x top-4 of 32 experts
// (20B shape): gate_up 431 -> 160, down 247 -> 88 us; one wave per row block
// walking all 45 groups took 175 and 114 (an uneven last round of long
// waves), with the decodes between the products 199 and 132.
#include "pk_internal.h"

#include "pk_i4_device.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int RW_M = PK_ROWS_TILE;   // input rows per tile (two sets of 4)
constexpr int RW_PF = 2;         // groups in flight per wave
constexpr int RW_WAVES = 4;      // waves per workgroup, sharing a row block's groups
constexpr int RW_GW = 12;        // consecutive groups per wave (4 x 12 cover a 2880-wide row's 45)

// Byte `BYTE` of w, its low nibble as a signed 4-bit value, / 16.
template <int BYTE>
__device__ __forceinline__ float rw_q16(uint32_t w) {
    return __builtin_amdgcn_cvt_off_f32_i4((int)((w >> (8 * BYTE)) & 0xffu));
}

template <int NS>
struct rw_stage {
    uint4 wa, wb;
    float s;
    float4 x[NS];
};

__device__ __forceinline__ float rw_comp(const float4 &v, int c) {
    return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
}

// The eight weights of a stored dword (columns 8D .. 8D + 7).
__device__ __forceinline__ void rw_decode(uint32_t w, float (&q)[8]) {
    uint32_t h = w >> 4;
    asm("" : "+v"(h));           // (kept as one shift, so that each byte below is an operand select)
    q[0] = rw_q16<0>(w);
    q[1] = rw_q16<0>(h);
    q[2] = rw_q16<1>(w);
    q[3] = rw_q16<1>(h);
    q[4] = rw_q16<2>(w);
    q[5] = rw_q16<2>(h);
    q[6] = rw_q16<3>(w);
    q[7] = rw_q16<3>(h);
}

// Columns 8D .. 8D + 7, column 8D + j on chain j. The A registers hold column
// 4k + c in block k of component c.
template <int NS, int D, int J>
__device__ __forceinline__ void rw_column(float q, const float4 (&x)[NS], f32x4 (&c)[NS][8]) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
        c[s][J] = __builtin_amdgcn_mfma_f32_4x4x1f32(rw_comp(x[s], J & 3), q,
                                                     D == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : c[s][J], 4,
                                                     2 * D + (J >> 2), 0);
}

template <int NS, int D>
__device__ __forceinline__ void rw_dword(const float (&q)[8], const float4 (&x)[NS], f32x4 (&c)[NS][8]) {
    rw_column<NS, D, 0>(q[0], x, c);
    rw_column<NS, D, 1>(q[1], x, c);
    rw_column<NS, D, 2>(q[2], x, c);
    rw_column<NS, D, 3>(q[3], x, c);
    rw_column<NS, D, 4>(q[4], x, c);
    rw_column<NS, D, 5>(q[5], x, c);
    rw_column<NS, D, 6>(q[6], x, c);
    rw_column<NS, D, 7>(q[7], x, c);
}

// The group sums of 4 NS input rows, one row of the block per lane. The
// decodes and the products each run as one stretch of 32 columns: a VALU
// instruction between matrix instructions costs about twice one among its
// like, since both run on the same multipliers and do not overlap.
template <int NS>
__device__ __forceinline__ void rw_group(const rw_stage<NS> &st, f32x4 (&p)[NS]) {
    f32x4 c[NS][8];
    float q[4][8];
    rw_decode(st.wa.x, q[0]);
    rw_decode(st.wa.y, q[1]);
    rw_decode(st.wa.z, q[2]);
    rw_decode(st.wa.w, q[3]);
    __builtin_amdgcn_sched_barrier(0);
    rw_dword<NS, 0>(q[0], st.x, c);
    rw_dword<NS, 1>(q[1], st.x, c);
    rw_dword<NS, 2>(q[2], st.x, c);
    rw_dword<NS, 3>(q[3], st.x, c);
    __builtin_amdgcn_sched_barrier(0);
    rw_decode(st.wb.x, q[0]);
    rw_decode(st.wb.y, q[1]);
    rw_decode(st.wb.z, q[2]);
    rw_decode(st.wb.w, q[3]);
    __builtin_amdgcn_sched_barrier(0);
    rw_dword<NS, 4>(q[0], st.x, c);
    rw_dword<NS, 5>(q[1], st.x, c);
    rw_dword<NS, 6>(q[2], st.x, c);
    rw_dword<NS, 7>(q[3], st.x, c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float b0 = c[s][0][i] + c[s][4][i], b1 = c[s][1][i] + c[s][5][i];
            const float b2 = c[s][2][i] + c[s][6][i], b3 = c[s][3][i] + c[s][7][i];
            p[s][i] = (b0 + b2) + (b1 + b3);
        }
}

// Results of input rows j (v0) and j + 1 (v1) of the tile at weight row
// `row`: the SwiGLU of two input rows at once (even lanes finish the first's
// pair of rows (row, row + 1), odd lanes the second's), or both values.
template <int EPI, typename PAIR>
__device__ __forceinline__ void rw_put2(const pk_i4_items &it, PAIR pair_of, int j, int cnt, int row, int O, float v0,
                                        float v1, float lim, float alpha) {
    if constexpr (EPI == PK_EPI_SWIGLU) {
        const bool even = (row & 1) == 0;
        const float other = __shfl_xor(even ? v1 : v0, 1, 64);
        const float v = pk_swiglu(even ? v0 : other, even ? other : v1, lim, alpha);
        const int jj = even ? j : j + 1;
        if (jj < cnt && (row | 1) < O) it.y[(int64_t)pair_of(jj) * it.y_stride + (row >> 1)] = v;
    } else if (row < O) {
        if (j < cnt) it.y[(int64_t)pair_of(j) * it.y_stride + row] = v0;
        if (j + 1 < cnt) it.y[(int64_t)pair_of(j + 1) * it.y_stride + row] = v1;
    }
}

template <int NS, int EPI>
__device__ __forceinline__ void rw_body(const pk_i4_items &it, const int32_t *pairs, int beg, int cnt,
                                        const uint8_t *base, int rb, int O, int NG, float lim, float alpha,
                                        float (&accs)[RW_M][64]) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint4 *tiles =
        reinterpret_cast<const uint4 *>(base + it.off_tiles) + (int64_t)rb * NG * (PK_TILE_BYTES / 16);
    constexpr bool RS = EPI == PK_EPI_ROW_SCALED;
    const float *sc = reinterpret_cast<const float *>(base + it.off_scales) + (int64_t)rb * (RS ? 1 : NG) * 64;
    auto pair_of = [&](int j) { return pairs ? pairs[beg + j] : beg + j; };
    // lane l loads input row l % 4 of each set, columns 4 (l / 4) .. + 3
    // (rows past the tile's last repeat it; their results are not stored)
    const float *xp[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
        xp[s] = it.x + (int64_t)(pair_of(min(4 * s + (lane & 3), cnt - 1)) / it.x_div) * it.x_stride + 4 * (lane >> 2);
    const int row = rb * 64 + lane;
    const float bias =
        it.off_bias >= 0 ? reinterpret_cast<const float *>(base + it.off_bias)[min(row, O - 1)] : 0.0f;
    const float rs = RS ? sc[lane] : 0.0f;
    rw_stage<NS> st[RW_PF];
    auto load = [&](rw_stage<NS> &d, int g) {
        d.wa = pk_load_nt(&tiles[g * 128 + lane]);
        d.wb = pk_load_nt(&tiles[g * 128 + 64 + lane]);
        d.s = RS ? 0.0f : sc[g * 64 + lane];
#pragma unroll
        for (int s = 0; s < NS; ++s) d.x[s] = *reinterpret_cast<const float4 *>(xp[s] + g * 64);
    };
    // the row's sum so far, handed from wave to wave (and span to span) in
    // group order: a = fma(partial, scale, a). With a scale per row (no
    // prescribed order) each wave's groups are summed pairwise, unscaled, and
    // added; the scale comes last.
    f32x4 acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int b0 = 0; b0 < NG; b0 += RW_WAVES * RW_GW) {
        const int g0 = b0 + wave * RW_GW;
        f32x4 p[RW_GW][NS];
        float sv[RW_GW];
#pragma unroll
        for (int u = 0; u < RW_PF; ++u) load(st[u], min(g0 + u, NG - 1));
#pragma unroll
        for (int u = 0; u < RW_GW; ++u) {
            if (g0 + u < NG) rw_group<NS>(st[u % RW_PF], p[u]);
            sv[u] = st[u % RW_PF].s;
            if (u + RW_PF < RW_GW) load(st[u % RW_PF], min(g0 + u + RW_PF, NG - 1));
        }
        for (int w = 0; w < RW_WAVES; ++w) {
            if (w == wave) {
                f32x4 prev[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        prev[s][i] = b0 + w > 0 ? accs[4 * s + i][lane] : 0.0f;
                        acc[s][i] = prev[s][i];
                    }
                if constexpr (RS) {
                    // (pairwise, in eights and fours)
                    static_assert(RW_GW == 12, "");
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v[RW_GW];
#pragma unroll
                            for (int u = 0; u < RW_GW; ++u) v[u] = g0 + u < NG ? p[u][s][i] : 0.0f;
                            const float lo[8] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
                            acc[s][i] = prev[s][i] + (pk_add8(lo) + ((v[8] + v[9]) + (v[10] + v[11])));
                        }
                } else {
#pragma unroll
                    for (int u = 0; u < RW_GW; ++u)
                        if (g0 + u < NG) {
#pragma unroll
                            for (int s = 0; s < NS; ++s)
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    acc[s][i] = __builtin_fmaf(p[u][s][i], sv[u], acc[s][i]);
                        }
                }
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) accs[4 * s + i][lane] = acc[s][i];
            }
            __syncthreads();
        }
    }
    // wave w finishes rows 2w, 2w + 1 of the tile
    const int j = 2 * wave;
    if (j >= cnt) return;
    float a0 = accs[j][lane], a1 = accs[j + 1][lane];
    if constexpr (RS) {
        a0 = (float)(16.0 * (double)a0 * (double)rs);
        a1 = (float)(16.0 * (double)a1 * (double)rs);
    }
    if (it.off_bias >= 0 && row < O) { a0 = a0 + bias; a1 = a1 + bias; }
    rw_put2<EPI>(it, pair_of, j, cnt, row, O, a0, a1, lim, alpha);
}

// grid (RB, tiles): workgroup (rb, t) is row block rb of tile t, its waves
// taking runs of RW_GW groups. tl.pairs: the tiles of k_group_pairs; null:
// rows tile * t .. of n_items consecutive ones, all of slot slot_base.
template <int EPI>
__global__ __launch_bounds__(RW_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2))) void k_i4_rows(
    pk_i4_items it, pk_i4_tiles tl, int tile, int O, int NG, float lim, float alpha) {
    __shared__ float accs[RW_M][64];
    const int rb = blockIdx.x, t = blockIdx.y;
    int beg, cnt, slot = it.slot_base;
    if (tl.pairs) {
        if (t >= *tl.n_tiles) return;
        beg = tl.tile_beg[t];
        cnt = tl.tile_cnt[t];
        slot += tl.tile_exp[t];
    } else {
        beg = t * tile;
        cnt = min(tile, it.n_items - beg);
    }
    const uint8_t *base = it.base + (int64_t)slot * it.slot_stride;
    if (cnt > 4) rw_body<2, EPI>(it, tl.pairs, beg, cnt, base, rb, O, NG, lim, alpha, accs);
    else rw_body<1, EPI>(it, tl.pairs, beg, cnt, base, rb, O, NG, lim, alpha, accs);
}

// ───────────────────── tiles of 16 rows ─────────────────────
// Many pairs per expert: a wave walks all groups of one row block and folds
// them as it goes. More than 8 rows of a tile run on
// v_mfma_f32_16x16x1_4b_f32, its four blocks being the row block's quarters
// (operand B, lane = weight row) times 16 input rows at one column, broadcast
// to the blocks (cbsz = 2): 14.2 ns per 64 x 16 products against 15.5 on the
// 4 x 4 form, and each decode serves 16 rows. Register 4 q + i of lane l is
// weight row 16 q + l % 16, input row 4 (l / 16) + i.
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int D, int J>
__device__ __forceinline__ void rw16_column(float q, const float4 (&x)[4], f32x16 (&c)[8]) {
    constexpr f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    c[J] = __builtin_amdgcn_mfma_f32_16x16x1f32(rw_comp(x[D >> 1], J & 3), q, D == 0 ? zero : c[J], 2,
                                                2 * (D & 1) + (J >> 2), 0);
}

template <int D>
__device__ __forceinline__ void rw16_dword(const float (&q)[8], const float4 (&x)[4], f32x16 (&c)[8]) {
    rw16_column<D, 0>(q[0], x, c);
    rw16_column<D, 1>(q[1], x, c);
    rw16_column<D, 2>(q[2], x, c);
    rw16_column<D, 3>(q[3], x, c);
    rw16_column<D, 4>(q[4], x, c);
    rw16_column<D, 5>(q[5], x, c);
    rw16_column<D, 6>(q[6], x, c);
    rw16_column<D, 7>(q[7], x, c);
}

struct rw16_stage {
    uint4 wa, wb;
    float s[4];
    float4 x[4];
};

__device__ __forceinline__ void rw16_group(const rw16_stage &st, f32x16 &acc) {
    f32x16 c[8];
    float q[4][8];
    rw_decode(st.wa.x, q[0]);
    rw_decode(st.wa.y, q[1]);
    rw_decode(st.wa.z, q[2]);
    rw_decode(st.wa.w, q[3]);
    __builtin_amdgcn_sched_barrier(0);
    rw16_dword<0>(q[0], st.x, c);
    rw16_dword<1>(q[1], st.x, c);
    rw16_dword<2>(q[2], st.x, c);
    rw16_dword<3>(q[3], st.x, c);
    __builtin_amdgcn_sched_barrier(0);
    rw_decode(st.wb.x, q[0]);
    rw_decode(st.wb.y, q[1]);
    rw_decode(st.wb.z, q[2]);
    rw_decode(st.wb.w, q[3]);
    __builtin_amdgcn_sched_barrier(0);
    rw16_dword<4>(q[0], st.x, c);
    rw16_dword<5>(q[1], st.x, c);
    rw16_dword<6>(q[2], st.x, c);
    rw16_dword<7>(q[3], st.x, c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float b0 = c[0][i] + c[4][i], b1 = c[1][i] + c[5][i];
        const float b2 = c[2][i] + c[6][i], b3 = c[3][i] + c[7][i];
        acc[i] = __builtin_fmaf((b0 + b2) + (b1 + b3), st.s[i >> 2], acc[i]);
    }
}

constexpr int RW16_PF = 2;

template <int EPI>
__device__ __forceinline__ void rw16_body(const pk_i4_items &it, const int32_t *pairs, int beg, int cnt,
                                          const uint8_t *base, int rb, int O, int NG, float lim, float alpha) {
    const int lane = threadIdx.x & 63;
    const uint4 *tiles =
        reinterpret_cast<const uint4 *>(base + it.off_tiles) + (int64_t)rb * NG * (PK_TILE_BYTES / 16);
    const float *sc = reinterpret_cast<const float *>(base + it.off_scales) + (int64_t)rb * NG * 64;
    auto pair_of = [&](int j) { return pairs[beg + j]; };
    // lane l loads input row l % 16, columns 4 (l / 16) .. + 3 of each 16
    const float *xp = it.x + (int64_t)(pair_of(min(lane & 15, cnt - 1)) / it.x_div) * it.x_stride + 4 * (lane >> 4);
    rw16_stage st[RW16_PF];
    auto load = [&](rw16_stage &d, int g) {
        d.wa = pk_load_nt(&tiles[g * 128 + lane]);
        d.wb = pk_load_nt(&tiles[g * 128 + 64 + lane]);
#pragma unroll
        for (int q = 0; q < 4; ++q) d.s[q] = sc[g * 64 + 16 * q + (lane & 15)];
#pragma unroll
        for (int m = 0; m < 4; ++m) d.x[m] = *reinterpret_cast<const float4 *>(xp + g * 64 + 16 * m);
    };
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int u = 0; u < RW16_PF; ++u) load(st[u], min(u, NG - 1));
    for (int g = 0; g < NG; g += RW16_PF) {
#pragma unroll
        for (int u = 0; u < RW16_PF; ++u) {
            if (g + u < NG) rw16_group(st[u], acc);
            load(st[u], min(g + u + RW16_PF, NG - 1));
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = rb * 64 + 16 * q + (lane & 15);
        if (it.off_bias >= 0 && row < O) {
            const float bias = reinterpret_cast<const float *>(base + it.off_bias)[row];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[4 * q + i] = acc[4 * q + i] + bias;
        }
#pragma unroll
        for (int i = 0; i < 4; i += 2)
            rw_put2<EPI>(it, pair_of, 4 * (lane >> 4) + i, cnt, row, O, acc[4 * q + i], acc[4 * q + i + 1], lim, alpha);
    }
}

// The same walk for up to 8 rows on the 4 x 4 form.
template <int NS, int EPI>
__device__ __forceinline__ void rw_walk(const pk_i4_items &it, const int32_t *pairs, int beg, int cnt,
                                        const uint8_t *base, int rb, int O, int NG, float lim, float alpha) {
    const int lane = threadIdx.x & 63;
    const uint4 *tiles =
        reinterpret_cast<const uint4 *>(base + it.off_tiles) + (int64_t)rb * NG * (PK_TILE_BYTES / 16);
    const float *sc = reinterpret_cast<const float *>(base + it.off_scales) + (int64_t)rb * NG * 64;
    auto pair_of = [&](int j) { return pairs[beg + j]; };
    const float *xp[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
        xp[s] = it.x + (int64_t)(pair_of(min(4 * s + (lane & 3), cnt - 1)) / it.x_div) * it.x_stride + 4 * (lane >> 2);
    rw_stage<NS> st[RW16_PF];
    auto load = [&](rw_stage<NS> &d, int g) {
        d.wa = pk_load_nt(&tiles[g * 128 + lane]);
        d.wb = pk_load_nt(&tiles[g * 128 + 64 + lane]);
        d.s = sc[g * 64 + lane];
#pragma unroll
        for (int s = 0; s < NS; ++s) d.x[s] = *reinterpret_cast<const float4 *>(xp[s] + g * 64);
    };
    f32x4 acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < RW16_PF; ++u) load(st[u], min(u, NG - 1));
    for (int g = 0; g < NG; g += RW16_PF) {
#pragma unroll
        for (int u = 0; u < RW16_PF; ++u) {
            if (g + u < NG) {
                f32x4 p[NS];
                rw_group<NS>(st[u], p);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[s][i] = __builtin_fmaf(p[s][i], st[u].s, acc[s][i]);
            }
            load(st[u], min(g + u + RW16_PF, NG - 1));
        }
    }
    const int row = rb * 64 + lane;
    const float bias = it.off_bias >= 0 && row < O ? reinterpret_cast<const float *>(base + it.off_bias)[row] : 0.0f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (it.off_bias >= 0 && row < O) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[s][i] = acc[s][i] + bias;
        }
#pragma unroll
        for (int i = 0; i < 4; i += 2)
            rw_put2<EPI>(it, pair_of, 4 * s + i, cnt, row, O, acc[s][i], acc[s][i + 1], lim, alpha);
    }
}

// grid (ceil(RB / 4), tiles): wave w of a workgroup takes row block 4 x + w of
// tile y of tl (at most 16 pairs).
template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_i4_rows16(
    pk_i4_items it, pk_i4_tiles tl, int O, int NG, int RB, float lim, float alpha) {
    const int rb = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = blockIdx.y;
    if (rb >= RB || t >= *tl.n_tiles) return;
    const int beg = tl.tile_beg[t], cnt = tl.tile_cnt[t], slot = it.slot_base + tl.tile_exp[t];
    const uint8_t *base = it.base + (int64_t)slot * it.slot_stride;
    if (cnt > 8) rw16_body<EPI>(it, tl.pairs, beg, cnt, base, rb, O, NG, lim, alpha);
    else if (cnt > 4) rw_walk<2, EPI>(it, tl.pairs, beg, cnt, base, rb, O, NG, lim, alpha);
    else rw_walk<1, EPI>(it, tl.pairs, beg, cnt, base, rb, O, NG, lim, alpha);
}

}  // namespace

bool pk_i4_rows_ok(const pk_i4_items &it, int epilogue) {
    return !it.xq && !it.yq && epilogue != PK_EPI_COMBINE && (it.x_stride & 3) == 0 && ((uintptr_t)it.x & 15) == 0;
}

// A workgroup per (row block, row) takes as long as its groups while a CU has
// at most two; beyond, each further one adds its time, and decoding a weight
// once per 4 rows pays. Here a row block takes a span of 48 groups at a time,
// whole spans' time whatever the last one holds, so that with one or two
// workgroups per CU it pays for rows that fill 3/4 of their spans. Per row /
// here, us: 1024 x 1024, 17 rows (272 workgroups) 6.4 / 9.8, 33 rows (528)
// 11.3 / 9.7; 5760 x 576, 3 rows 5.8 / 8.4, 6 rows 10.0 / 8.6; 4096 x 4096, 8
// rows (512) 15.4 / 16.6, 9 rows 20.3 / 16.8; 2048 x 2048, 9 rows 9.4 / 10.0;
// 2880 x 2880, 6 rows (270) 13.0 / 10.1; 5760 x 2880, 3 rows 12.4 / 10.0; 2880 x
// 5760, 6 rows 21.6 / 17.1; 2880 x 8192, 6 rows 28.5 / 24.0.
bool pk_i4_rows_pays(const pk_i4_shape &sh, int64_t n) {
    const int span = RW_WAVES * RW_GW, spans = (sh.NG + span - 1) / span;
    const int64_t blocks = n * sh.RB, n_cu = pk_device_cus();
    return blocks > 2 * n_cu || (blocks > n_cu && 4 * sh.NG >= 3 * span * spans);
}

int pk_launch_i4_rows(const pk_i4_items &it, const pk_i4_tiles *tl, const pk_i4_shape &sh, int epilogue, float lim,
                      float alpha, int max_tiles, hipStream_t st, int tile_rows) {
    PK_CHECK(pk_i4_rows_ok(it, epilogue), PK_ERR_ARG, "i4 rows: inputs not 16-byte aligned, or not the fp32 chains");
    PK_CHECK(sh.NG > 0 && sh.RB > 0 && it.n_items > 0 && it.x_div > 0, PK_ERR_ARG, "i4 rows: empty shape");
    PK_CHECK(sh.NG <= 128, PK_ERR_UNSUPPORTED, "i4 rows: I=%d above 8192", sh.I);     // (as for one row)
    PK_CHECK(!tl || (tl->pairs && tl->tile_exp && tl->tile_beg && tl->tile_cnt && tl->n_tiles), PK_ERR_ARG,
             "i4 rows: missing tiles");
    PK_CHECK(tile_rows == 8 || (tile_rows == 16 && tl && epilogue != PK_EPI_ROW_SCALED), PK_ERR_ARG,
             "i4 rows: tiles of %d", tile_rows);
    // one matrix: tiles of 8 rows, but of 4 where tiles of 8 would leave CUs
    // without a workgroup (5760 x 2880, 8 rows: 9.5 against 13.6 us)
    int tile = tile_rows;
    if (!tl && tile == 8 && (int64_t)sh.RB * ((it.n_items + 7) / 8) <= pk_device_cus()) tile = 4;
    const int tiles = tl ? max_tiles : (it.n_items + tile - 1) / tile;
    PK_CHECK(tiles > 0 && tiles <= 65535, PK_ERR_UNSUPPORTED, "i4 rows: %d tiles", tiles);
    const pk_i4_tiles none{};
    if (tile == 16) {
        const dim3 grid((sh.RB + 3) / 4, tiles);
        if (epilogue == PK_EPI_SWIGLU)
            hipLaunchKernelGGL(k_i4_rows16<PK_EPI_SWIGLU>, grid, dim3(256), 0, st, it, *tl, sh.O, sh.NG, sh.RB, lim,
                               alpha);
        else
            hipLaunchKernelGGL(k_i4_rows16<PK_EPI_PLAIN>, grid, dim3(256), 0, st, it, *tl, sh.O, sh.NG, sh.RB, lim,
                               alpha);
        PK_HIP(hipGetLastError());
        return PK_OK;
    }
    const dim3 grid(sh.RB, tiles);
    if (epilogue == PK_EPI_SWIGLU)
        hipLaunchKernelGGL(k_i4_rows<PK_EPI_SWIGLU>, grid, dim3(RW_WAVES * 64), 0, st, it, tl ? *tl : none, tile, sh.O,
                           sh.NG, lim, alpha);
    else if (epilogue == PK_EPI_ROW_SCALED)
        hipLaunchKernelGGL(k_i4_rows<PK_EPI_ROW_SCALED>, grid, dim3(RW_WAVES * 64), 0, st, it, none, tile, sh.O, sh.NG,
                           lim, alpha);
    else
        hipLaunchKernelGGL(k_i4_rows<PK_EPI_PLAIN>, grid, dim3(RW_WAVES * 64), 0, st, it, tl ? *tl : none, tile, sh.O,
                           sh.NG, lim, alpha);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
