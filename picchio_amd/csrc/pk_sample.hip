// pk_sample.hip — next-token sampling on the device (sample_logits,
// picchio.c:1509-1649), so that a decode loop with temperature / top-k /
// top-p / repetition penalty never leaves the GPU.
//
// A draw over a large vocabulary is spread over the device (the launches after
// k_sample below); greedy draws, small vocabularies, the exact-sum option and
// a top-k beyond CAND run in k_sample alone: one workgroup of 1024 threads,
// wave w owning the w-th sixteenth of the vocabulary in each pass, with 16
// loads in flight per lane. Steps, in the reference's order:
//   1. repetition penalty: once per history entry (a token that appears c
//      times is divided / multiplied c times, as the reference's loop does);
//   2. temperature below 1e-6: the first maximum (greedy), no draw;
//   3. logits * (1 / T);
//   4. top-k threshold = the K-th largest value, by a radix select on
//      order-preserving keys (exact; ties at the threshold stay). After the
//      first 8-bit pass the entries in or above the threshold's bucket are
//      gathered into LDS when they fit, and the rest of the selection and the
//      index order of the kept entries are worked out there; otherwise the
//      passes stay in global memory and a ballot compaction keeps index order;
//   5. softmax, top-p over the probabilities > 1e-10, the draw.
// A logit below the top-k threshold becomes -1e30 and then exactly 0 in the
// reference, so its float sums equal the same sums over the kept entries in
// index order, one term at a time. Up to SMALL kept entries one lane makes
// each sum in that order from LDS; beyond, a workgroup (order_sum) or, without
// a top-k, the device (om_sum) scans to the same bits. The top-p list is sorted descending with equal values by index (what glibc's
// merge sort leaves): in LDS for up to SMALL entries, beyond that chunk by
// chunk (a radix select on 64-bit (key, ~index) finds each chunk's bound) with
// the running sum carried across. The array left behind and the draw equal
// the reference's up to the device expf's last ulp.
// The opt-in fast_sums mode makes those sums exact instead (64-bit integers of
// the values scaled by a power of two, rounded once), which any order gives:
// the top-p cut is the shortest descending prefix whose exact sum reaches
// top_p (a radix descent carrying counts and exact sums, ties by index) and
// the pick the first index whose exact running sum reaches the draw. The
// reference's float rounding (about sqrt(n) * 2^-24 relative) then separates
// the two, so over a flat distribution a cut or a pick moves now and then.
#include "pk_dev.h"
#include "pk_engine.h"

#include <cstddef>

namespace {

constexpr int SNT = 1024;                 // threads of the sampling workgroup
constexpr int NW = SNT / 64;              // its waves
constexpr int U = 16;                     // loads in flight per lane in a pass
constexpr int SMALL = 4096;               // kept entries handled in LDS in the reference's order
constexpr int CAND = 4096;                // top-k candidates gathered into LDS after the first radix pass
constexpr int RANK_N = 512;               // entries placed by counting instead of a bitonic network
constexpr int FX_P = 62;                  // fixed-point bits for probabilities (sums <= ~1)

// Scratch of the launches that spread a draw over the device (zeroed when
// allocated; the counters are re-armed by the launch that reads them last).
constexpr int SB_BINS = 4096;
constexpr int SAMP_RUNS = 4096;
struct samp_ws {
    uint32_t hist[SB_BINS];
    uint32_t cur[SB_BINS * 16];           // a bucket's cursor, 64 bytes apart: neighbours do not share a line
    int32_t n_cand;                       // top-k candidates in cv / ci (0: none gathered)
    uint32_t mx_key;                      // key of the largest scaled logit
    float sum;                            // the ordered sum of the launch before
    int32_t m;                            // candidates of the top-p sort (0: top-p does nothing)
    int32_t cut;                          // 1: entries below tau go; 2: top-p is done
    float tau;
    uint32_t unsorted;                    // 1: a bucket exceeds what a workgroup sorts
    float cv[CAND];
    int32_t ci[CAND];
    float part[SAMP_RUNS];                // the ordered sum's runs: a plain sum,
    uint2 mv[SAMP_RUNS];                  // the pair of moves in one binade,
    int32_t mex[SAMP_RUNS];               // and that binade
};

__device__ __forceinline__ uint32_t key_of(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float float_of(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// v * 2^S truncated to an integer, for 0 <= v with v * 2^S < 2^64 (exact
// whenever v >= 2^(23 - S)); zero, denormals and negatives give 0.
__device__ __forceinline__ uint64_t fx(float v, int S) {
    const uint32_t b = __float_as_uint(v);
    const int e = (int)(b >> 23) & 255;
    if (e == 0 || (b >> 31)) return 0;
    const uint64_t m = (b & 0x7fffffu) | 0x800000u;
    const int sh = e - 150 + S;
    if (sh >= 0) return m << sh;
    return sh <= -24 ? 0 : m >> (-sh);
}
// an exact integer sum back to float: one rounding, then the exact scaling
__device__ __forceinline__ float unfx(uint64_t q, int S) { return ldexpf((float)q, -S); }

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m, 64);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m, 64);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t shfl_up_u64(uint64_t v, int d) {
    const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)v, d, 64);
    const uint32_t hi = (uint32_t)__shfl_up((int)(uint32_t)(v >> 32), d, 64);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
    for (int o = 32; o > 0; o >>= 1) v += shfl_xor_u64(v, o);
    return v;
}
__device__ __forceinline__ uint64_t wave_incl_scan_u64(uint64_t v) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t t = shfl_up_u64(v, d);
        if (lane >= d) v += t;
    }
    return v;
}
// Every thread of the workgroup calls these.
__device__ __forceinline__ uint64_t block_sum_u64(uint64_t v, uint64_t *s_q) {
    v = wave_sum_u64(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_q[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t t = 0;
    for (int w = 0; w < NW; ++w) t += s_q[w];
    return t;
}
// The same network ordering by index ascending (values carried along).
__device__ __forceinline__ void bitonic_by_index(float *sv, int *si, int P) {
    const int half = P >> 1;
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < half; t += SNT) {
                const int lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
                const int ia = si[lo], ib = si[hi];
                const bool rev = (lo & size) != 0;
                if ((ia < ib) == rev) {
                    const float va = sv[lo];
                    sv[lo] = sv[hi]; sv[hi] = va;
                    si[lo] = ib; si[hi] = ia;
                }
            }
            __syncthreads();
        }
}

__device__ __forceinline__ float block_max(float v, float *s_red) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = s_red[0];
    for (int w = 1; w < NW; ++w) m = fmaxf(m, s_red[w]);
    return m;
}
__device__ __forceinline__ int block_max_i(int v, int *s_redi) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_redi[threadIdx.x >> 6] = v;
    __syncthreads();
    int m = s_redi[0];
    for (int w = 1; w < NW; ++w) m = max(m, s_redi[w]);
    return m;
}

// This wave's share [b, e) of [0, n): 16 contiguous shares, multiples of 64.
struct seg_t { int b, e; };
__device__ __forceinline__ seg_t wave_seg(int n) {
    const int per = ((n + NW - 1) / NW + 63) & ~63;
    const int b = min(n, (int)(threadIdx.x >> 6) * per);
    return {b, min(n, b + per)};
}

// f(j, v, ok) for every j of this wave's share of src[0..n): 64-entry steps,
// U steps' loads issued before any is used (clamped, so every load is valid).
template <class F>
__device__ __forceinline__ void seg_for(const float *src, int n, F f) {
    const seg_t s = wave_seg(n);
    const int lane = threadIdx.x & 63;
    for (int base = s.b; base < s.e; base += 64 * U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = src[min(base + u * 64 + lane, n - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = base + u * 64 + lane;
            f(j, v[u], j < s.e);
        }
    }
}

// Entries of src[0..n) with keep(v), in index order, into dv / di as
// (map(v), j). Returns their number. Every thread of the workgroup calls it.
template <class Keep, class Map>
__device__ __forceinline__ int compact(const float *src, int n, Keep keep, Map map, float *dv, int *di, int *s_w) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int c = 0;
    seg_for(src, n, [&](int, float v, bool ok) { c += __popcll(__ballot(ok && keep(v))); });
    __syncthreads();
    if (lane == 0) s_w[wave] = c;
    __syncthreads();
    int off = 0, tot = 0;
    for (int w = 0; w < NW; ++w) {
        const int x = s_w[w];
        off += w < wave ? x : 0;
        tot += x;
    }
    const uint64_t lt = (1ull << lane) - 1ull;
    seg_for(src, n, [&](int j, float v, bool ok) {
        const bool p = ok && keep(v);
        const uint64_t m = __ballot(p);
        if (p) {
            const int o = off + __popcll(m & lt);
            dv[o] = map(v);
            di[o] = j;
        }
        off += __popcll(m);
    });
    __syncthreads();
    return tot;
}

// Bitonic network over LDS (sv, si)[0..P), P a power of two <= SMALL:
// value descending, then index ascending.
__device__ __forceinline__ void bitonic(float *sv, int *si, int P) {
    const int half = P >> 1;
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < half; t += SNT) {
                const int lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
                const float va = sv[lo], vb = sv[hi];
                const int ia = si[lo], ib = si[hi];
                const bool rev = (lo & size) != 0;     // second half of a merge runs backwards
                const bool a_first = va > vb || (va == vb && ia < ib);
                if (a_first == rev) {
                    sv[lo] = vb; sv[hi] = va;
                    si[lo] = ib; si[hi] = ia;
                }
            }
            __syncthreads();
        }
}

// f(v) for v = p[0], p[1], .. until it returns true; the index it did so at,
// or -1. LDS reads go out eight at a time ahead of the chain.
template <class F>
__device__ __forceinline__ int serial_scan(const float *p, int n, F f) {
    int j = 0;
    for (; j + 8 <= n; j += 8) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = p[j + u];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (f(t[u])) return j + u;
    }
    for (; j < n; ++j)
        if (f(p[j])) return j;
    return -1;
}
__device__ __forceinline__ float serial_sum(const float *p, int n) {
    float s = 0.0f;
    (void)serial_scan(p, n, [&](float v) { s = s + v; return false; });
    return s;
}

// Step 5 over kv / ki[0..n) in LDS (n <= SMALL), in the reference's order.
// Returns (to thread 0) the position picked, or -1; *r_out the draw.
__device__ __forceinline__ int finish_small(float *kv, int n, float top_p, pk_sampler_dev *sp, float *sv, int *si,
                            float *s_red, int *s_redi, float *s_sum, int *s_cut, float *r_out) {
    const int tid = threadIdx.x;
    float mx = -1e30f;
    for (int j = tid; j < n; j += SNT) mx = fmaxf(mx, kv[j]);
    mx = block_max(mx, s_red);
    for (int j = tid; j < n; j += SNT) kv[j] = expf(kv[j] - mx);
    __syncthreads();
    if (tid == 0) *s_sum = serial_sum(kv, n);
    __syncthreads();
    const float sum = *s_sum;
    for (int j = tid; j < n; j += SNT) kv[j] = kv[j] / sum;
    __syncthreads();
    if (top_p < 1.0f && top_p > 0.0f) {
        int c = 0;
        for (int j = tid; j < n; j += SNT) c += kv[j] > 1e-10f ? 1 : 0;
        // the candidates' count: a block sum of c
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
        __syncthreads();
        if ((tid & 63) == 0) s_redi[tid >> 6] = c;
        __syncthreads();
        int na = 0;
        for (int w = 0; w < NW; ++w) na += s_redi[w];
        if (na > 1) {
            // sorting every entry puts the candidates (> 1e-10) first, in order
            if (n <= RANK_N) {
                // each entry's place by counting those before it
                if (tid < n) {
                    const float x = kv[tid];
                    int at = 0;
                    for (int i = 0; i < n; ++i) at += kv[i] > x || (kv[i] == x && i < tid) ? 1 : 0;
                    sv[at] = x;
                    si[at] = tid;
                }
                __syncthreads();
            } else {
                int P = 1;
                while (P < n) P <<= 1;
                for (int j = tid; j < P; j += SNT) {
                    sv[j] = j < n ? kv[j] : -INFINITY;
                    si[j] = j < n ? j : 0x7fffffff;
                }
                __syncthreads();
                bitonic(sv, si, P);
            }
            if (tid == 0) {
                float cum = 0.0f;
                const int at = serial_scan(sv, na, [&](float v) { cum = cum + v; return cum >= top_p; });
                *s_cut = at < 0 ? na : at + 1;
            }
            __syncthreads();
            for (int j = *s_cut + tid; j < na; j += SNT) kv[si[j]] = 0.0f;
            __syncthreads();
            if (tid == 0) *s_sum = serial_sum(kv, n);
            __syncthreads();
            const float s2 = *s_sum;
            if (s2 > 0)
                for (int j = tid; j < n; j += SNT) kv[j] = kv[j] / s2;
            __syncthreads();
        }
    }
    int pick = -1;
    if (tid == 0) {
        uint64_t x = sp->rng;
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        sp->rng = x;
        const float r = (float)(x >> 33) / (float)(1ULL << 31);
        *r_out = r;
        float cum = 0.0f;
        pick = serial_scan(kv, n, [&](float v) { cum = cum + v; return cum >= r; });
        if (pick < 0)
            for (int j = n - 1; j >= 0; --j)
                if (kv[j] > 0) { pick = j; break; }
    }
    return pick;
}

struct lds_hist {
    uint32_t c[NW][256];
    uint64_t s[NW][256];
};

// ── the reference's float sum, in parallel ──
// s = 0; s = s + v_j in index order, every sum rounded to float (v_j >= 0).
// While s stays in one binade it is a multiple S of its last place u, S below
// 2^24, and adding v moves S by rint(v / u): the nearer integer, or, when v / u
// lies half way, the one that leaves S even. So an element is a pair of moves
// (d0, d1) for S even and S odd, a run of elements composes to such a pair,
// and a workgroup scans the pairs of OS_CHUNK elements at once: exact integer
// arithmetic that gives the serial sum's bits. Where S would reach 2^24 the
// thread that holds that element adds its own elements one by one in float,
// and the scan goes on from there in the new binade (a sum passes few: it has
// to double each time). NaN and infinite elements are added in float too.
constexpr int OS_E = 8;                   // elements per thread
constexpr int OS_CHUNK = OS_E * SNT;
constexpr int OS_BUF = OS_CHUNK + OS_CHUNK / OS_E;     // LDS floats (rows of 8 set 9 apart)
constexpr uint32_t OS_BIG = 1u << 25;     // a move past the binade
// The first OS_HEAD elements are added by one thread (2.4 ns each): a sum's
// first binades are short, and each costs a scan of the chunk (2.3 us). A draw
// in one workgroup, no cut, 5000 flat entries: 62 us with every element on one
// thread, 76 with the scan alone, 53 so (256 elements 55, 2048 60); 16000: 141,
// 87 and 65.
constexpr int OS_HEAD = 512;

// a's moves, then b's (the callers clamp to OS_BIG before 32 bits could
// overflow: 8 elements, 64 lanes, 16 waves)
__device__ __forceinline__ uint2 os_then(uint2 a, uint2 b) {
    return make_uint2(a.x + ((a.x & 1u) ? b.y : b.x), a.y + ((a.y & 1u) ? b.x : b.y));
}
__device__ __forceinline__ uint2 os_clamp(uint2 a) { return make_uint2(min(a.x, OS_BIG), min(a.y, OS_BIG)); }
// a lane's pair moved by a DPP control (lanes without a source: no moves)
template <int CTRL, int ROWS>
__device__ __forceinline__ uint2 os_dpp(uint2 a) {
    return make_uint2((uint32_t)__builtin_amdgcn_update_dpp(0, (int)a.x, CTRL, ROWS, 0xf, false),
                      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a.y, CTRL, ROWS, 0xf, false));
}
// Inclusive scan over the lanes of a row of 16, or of the wave.
template <bool WAVE>
__device__ __forceinline__ uint2 os_scan(uint2 a) {
    a = os_then(os_dpp<0x111, 0xf>(a), a);                 // row shifts by 1, 2, 4, 8
    a = os_then(os_dpp<0x112, 0xf>(a), a);
    a = os_then(os_dpp<0x114, 0xf>(a), a);
    a = os_then(os_dpp<0x118, 0xf>(a), a);
    if constexpr (WAVE) {
        a = os_then(os_dpp<0x142, 0xa>(a), a);             // lane 15 of rows 0, 2 to rows 1, 3
        a = os_then(os_dpp<0x143, 0xc>(a), a);             // lane 31 to rows 2, 3
    }
    return a;
}

// The pair of moves of a thread's OS_E elements in binade ex (s = S 2^(ex - 150)).
__device__ __forceinline__ uint2 os_moves(const float (&v)[OS_E], int ex) {
    uint2 d = make_uint2(0u, 0u);                          // (x: from S even, y: from S odd)
#pragma unroll
    for (int k = 0; k < OS_E; ++k) {
        // (past the binade, infinite or NaN: OS_BIG)
        const float t = fminf(ldexpf(v[k], 150 - ex), (float)OS_BIG);
        const float q = rintf(t), h = t - q;               // a tie goes to even: the move for S even
        const float qo = q + (fabsf(h) == 0.5f ? h + h : 0.0f);
        d = os_then(d, make_uint2((uint32_t)q, (uint32_t)qo));
    }
    return os_clamp(d);
}

// find: stop at the first index whose running sum is >= r. Leaves the sum (up
// to there) in *s_out and that index (or -1) in *hit_out; s0: where the sum
// starts. Every thread of the workgroup calls it (buf: OS_BUF floats).
__device__ __forceinline__ void order_sum(const float *src, int n, float *buf, bool find, float r, float *s_out,
                                          int *hit_out) {
    __shared__ uint2 s_wave[NW];
    __shared__ float os_s;
    __shared__ int os_start, os_hit;
    static_assert(OS_HEAD % (4 * OS_E) == 0 && OS_HEAD <= OS_CHUNK, "four rows of elements at a time");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float s = 0.0f;
    int hit = -1;
    float nx[OS_E];                       // the next chunk, in flight while this one is scanned
    const auto fetch = [&](int b) {
#pragma unroll
        for (int k = 0; k < OS_E; ++k) nx[k] = src[min(b + tid + SNT * k, n - 1)];
    };
    if (n > 0) fetch(0);
    for (int base = 0; base < n && hit < 0; base += OS_CHUNK) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < OS_E; ++k) {
            const int j = tid + SNT * k;
            buf[j + j / OS_E] = base + j < n ? nx[k] : 0.0f;              // (+ 0 leaves the sum as it is)
        }
        if (base + OS_CHUNK < n) fetch(base + OS_CHUNK);
        __syncthreads();
        float v[OS_E];
#pragma unroll
        for (int k = 0; k < OS_E; ++k) v[k] = buf[(OS_E + 1) * tid + k];
        int start = 0;                                     // the chunk's elements before it are in s
        if (base == 0) {
            if (tid == 0) {
                float x = 0.0f;
                int at = -1;
                for (int row = 0; row < OS_HEAD / OS_E && at < 0; row += 4) {      // (zeros past n: + 0)
                    float t[4 * OS_E];
#pragma unroll
                    for (int k = 0; k < 4 * OS_E; ++k) t[k] = buf[(OS_E + 1) * (row + k / OS_E) + k % OS_E];
                    const float x0 = x;
#pragma unroll
                    for (int k = 0; k < 4 * OS_E; ++k) x = x + t[k];
                    if (find && x >= r) {                  // (the sum only grows: the crossing is among these)
                        x = x0;
                        for (int k = 0; k < 4 * OS_E && at < 0; ++k) {
                            x = x + buf[(OS_E + 1) * (row + k / OS_E) + k % OS_E];
                            if (x >= r) at = OS_E * row + k;
                        }
                    }
                }
                os_s = x;
                os_hit = at;
            }
            __syncthreads();
            s = os_s;
            hit = os_hit;
            start = OS_HEAD;
            if (OS_E * tid < start) {
#pragma unroll
                for (int k = 0; k < OS_E; ++k) v[k] = 0.0f;
            }
            if (hit >= 0 || !(s < INFINITY)) break;
        }
        while (start < OS_CHUNK) {
            const uint32_t sb = __float_as_uint(s);
            const int ex = max((int)(sb >> 23), 1);        // s = S 2^(ex - 150)
            const uint32_t S = (sb & 0x7fffffu) | ((sb >> 23) ? 0x800000u : 0u);
            const uint2 d = os_moves(v, ex);
            const uint2 inc = os_scan<true>(d);
            __syncthreads();                               // (s_wave, os_* of the last round are read)
            if (lane == 63) s_wave[wave] = os_clamp(inc);
            if (tid == 0) { os_start = OS_CHUNK; os_hit = 0x7fffffff; }
            __syncthreads();
            // lane l < 16: the waves up to l
            const uint2 upto = os_scan<false>(lane < NW ? s_wave[lane & (NW - 1)] : make_uint2(0u, 0u));
            const uint2 all = make_uint2((uint32_t)__builtin_amdgcn_readlane((int)upto.x, NW - 1),
                                         (uint32_t)__builtin_amdgcn_readlane((int)upto.y, NW - 1));
            const int before = __builtin_amdgcn_readfirstlane(max(wave - 1, 0));
            uint2 pre = make_uint2((uint32_t)__builtin_amdgcn_readlane((int)upto.x, before),
                                   (uint32_t)__builtin_amdgcn_readlane((int)upto.y, before));
            if (wave == 0) pre = make_uint2(0u, 0u);
            pre = os_then(pre, os_dpp<0x138, 0xf>(inc));   // and the wave's lanes before this one
            const bool odd = S & 1u;
            const uint32_t S0 = S + (odd ? pre.y : pre.x);             // before this thread's elements
            const uint32_t S1 = S0 + ((S0 & 1u) ? d.y : d.x);
            const float a0 = ldexpf((float)min(S0, OS_BIG), ex - 150);
            const bool cross = S0 < 0x1000000u && S1 >= 0x1000000u;
            const bool hits = find && S0 < 0x1000000u && !cross && ldexpf((float)S1, ex - 150) >= r &&
                              (!(a0 >= r) || OS_E * tid <= start);
            if (cross || hits) {
                float x = a0;
                int at = -1;
                for (int k = 0; k < OS_E; ++k) {
                    x = x + v[k];
                    if (find && at < 0 && x >= r) {
                        at = OS_E * tid + k;
                        break;
                    }
                }
                if (at >= 0) atomicMin(&os_hit, at);
                if (cross) { os_s = x; os_start = OS_E * (tid + 1); }
            }
            __syncthreads();
            const int got = os_hit;
            if (got != 0x7fffffff) {
                hit = base + got;
                break;
            }
            start = os_start;
            if (start < OS_CHUNK || !(S + (odd ? all.y : all.x) < 0x1000000u)) s = os_s;
            else s = ldexpf((float)(S + (odd ? all.y : all.x)), ex - 150);
            if (!(s < INFINITY)) break;                    // NaN stays NaN, infinity stays (nothing later changes it)
            if (OS_E * tid < start) {                      // (whole threads: in s)
#pragma unroll
                for (int k = 0; k < OS_E; ++k) v[k] = 0.0f;
            }
        }
        if (!(s < INFINITY)) break;
    }
    __syncthreads();
    if (tid == 0) {
        *s_out = s;
        *hit_out = hit;
    }
    __syncthreads();
}

__device__ __forceinline__ uint64_t comp_key(float v, int j) {
    return ((uint64_t)key_of(v) << 32) | (uint64_t)(0xffffffffu - (uint32_t)j);
}

// Top-p in the reference's order over pv[0..n) (n > SMALL): the candidates
// (> 1e-10) are taken in descending (value, then index) order SMALL at a
// time: a radix select on 64-bit (key, ~index) finds each chunk's lower
// bound, the chunk is sorted in LDS and one lane continues the running float
// sum through it until it reaches top_p. Entries after the cut become 0; the
// rest is renormalised by the serial sum. Every thread calls it.
__device__ __forceinline__ void top_p_chunks(float *pv, int n, float top_p, lds_hist &H, float *sv, int *si,
                                             float *stage, int *s_redi, uint64_t *s_pfx, uint64_t *s_msk,
                                             uint32_t *s_k, int *s_cut, int *s_tp, float *s_sum, int *s_pick) {
    const int tid = threadIdx.x, wave = tid >> 6;
    int c = 0;
    seg_for(pv, n, [&](int, float v, bool ok) { c += (ok && v > 1e-10f) ? 1 : 0; });
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    __syncthreads();
    if ((tid & 63) == 0) s_redi[wave] = c;
    __syncthreads();
    int m = 0;
    for (int w = 0; w < NW; ++w) m += s_redi[w];
    if (m <= 1) return;                                   // the reference's n_active > 1
    uint64_t bound = ~0ull;                               // chunks so far: composite keys >= bound
    uint64_t cut_ck = 0;
    bool found = false;
    __shared__ float s_cum;
    __shared__ int s_cnt;
    if (tid == 0) s_cum = 0.0f;
    for (int taken = 0; taken < m && !found;) {
        const int C = min(SMALL, m - taken);
        if (tid == 0) { *s_pfx = 0; *s_msk = 0; *s_k = (uint32_t)C; }
        for (int shift = 56; shift >= 0; shift -= 8) {
            for (int b = tid; b < NW * 256; b += SNT) (&H.c[0][0])[b] = 0;
            __syncthreads();
            const uint64_t prefix = *s_pfx, mask = *s_msk;
            seg_for(pv, n, [&](int j, float v, bool ok) {
                const uint64_t k = comp_key(v, j);
                if (ok && v > 1e-10f && k < bound && (k & mask) == prefix)
                    atomicAdd(&H.c[wave][(k >> shift) & 255u], 1u);
            });
            __syncthreads();
            if (tid < 256) {
                uint32_t cc = 0;
                for (int w = 0; w < NW; ++w) cc += H.c[w][tid];
                H.c[0][tid] = cc;
            }
            __syncthreads();
            if (tid == 0) {
                uint32_t k = *s_k;
                int d = 255;
                for (; d > 0; --d) {
                    if (k <= H.c[0][d]) break;
                    k -= H.c[0][d];
                }
                *s_k = k;
                *s_pfx = prefix | ((uint64_t)d << shift);
                *s_msk = mask | (255ull << shift);
                s_cnt = 0;
            }
            __syncthreads();
        }
        const uint64_t lo = *s_pfx;                       // the chunk: lo <= key < bound, C entries
        seg_for(pv, n, [&](int j, float v, bool ok) {
            const uint64_t k = comp_key(v, j);
            if (ok && v > 1e-10f && k >= lo && k < bound) {
                const int o = atomicAdd(&s_cnt, 1);        // below C: the keys are distinct
                if (o < SMALL) {
                    sv[o] = v;
                    si[o] = j;
                }
            }
        });
        __syncthreads();
        int P = 1;
        while (P < C) P <<= 1;
        for (int j = C + tid; j < P; j += SNT) { sv[j] = -INFINITY; si[j] = 0x7fffffff; }
        __syncthreads();
        bitonic(sv, si, P);
        if (tid == 0) {
            float cum = s_cum;
            int at = -1;
            for (int j = 0; j < C; ++j) {
                cum = cum + sv[j];
                if (cum >= top_p) { at = j; break; }
            }
            s_cum = cum;
            *s_cut = at < 0 ? -1 : si[at];
            *s_tp = at < 0 ? 0 : __float_as_int(sv[at]);
        }
        __syncthreads();
        if (*s_cut >= 0) {
            found = true;
            cut_ck = comp_key(__int_as_float(*s_tp), *s_cut);
        }
        taken += C;
        bound = lo;
        __syncthreads();
    }
    if (found)
        seg_for(pv, n, [&](int j, float v, bool ok) {
            if (ok && v > 1e-10f && comp_key(v, j) < cut_ck) pv[j] = 0.0f;
        });
    __syncthreads();
    order_sum(pv, n, stage, false, 0.0f, s_sum, s_pick);
    const float s2 = *s_sum;
    if (s2 > 0)
        seg_for(pv, n, [&](int j, float v, bool ok) {
            if (ok) pv[j] = v / s2;
        });
    __syncthreads();
}

// Top-p with exact sums over pv[0..n): the shortest descending prefix of the
// candidates (> 1e-10) whose exact sum reaches top_p, by a radix descent over
// keys carrying counts and exact sums per digit; ties at the cut value are
// taken by index. Every thread calls it.
__device__ __forceinline__ void top_p_exact_sums(float *pv, int n, float top_p, lds_hist &H, int *s_w,
                                                 uint64_t *s_q, uint32_t *s_prefix, uint32_t *s_mask,
                                                 uint32_t *s_k, uint64_t *s_acc, int *s_cut, int *s_tp) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t target = fx(top_p, FX_P) + ((fx(top_p, FX_P) == 0) ? 1 : 0);
    if (tid == 0) { *s_prefix = 0; *s_mask = 0; *s_acc = 0; *s_cut = 1; *s_tp = 1; }
    __syncthreads();
    for (int shift = 24; shift >= 0 && *s_tp; shift -= 8) {
        for (int b = tid; b < NW * 256; b += SNT) {
            (&H.c[0][0])[b] = 0;
            (&H.s[0][0])[b] = 0;
        }
        __syncthreads();
        const uint32_t prefix = *s_prefix, mask = *s_mask;
        seg_for(pv, n, [&](int, float v, bool ok) {
            const uint32_t k = key_of(v);
            if (ok && v > 1e-10f && (k & mask) == prefix) {
                atomicAdd(&H.c[wave][(k >> shift) & 255u], 1u);
                atomicAdd((unsigned long long *)&H.s[wave][(k >> shift) & 255u], (unsigned long long)fx(v, FX_P));
            }
        });
        __syncthreads();
        if (tid < 256) {
            uint32_t c = 0;
            uint64_t sm = 0;
            for (int w = 0; w < NW; ++w) { c += H.c[w][tid]; sm += H.s[w][tid]; }
            H.c[0][tid] = c;
            H.s[0][tid] = sm;
        }
        __syncthreads();
        if (tid == 0 && shift == 24) {
            uint32_t na = 0;
            for (int d = 0; d < 256; ++d) na += H.c[0][d];
            *s_tp = na > 1;                               // the reference's n_active > 1
        }
        if (tid == 0 && *s_cut) {
            uint64_t acc = *s_acc;
            int d = 255;
            for (; d >= 0; --d) {
                if (acc + H.s[0][d] >= target) break;
                acc += H.s[0][d];
            }
            if (d < 0) {
                *s_cut = 0;                               // the candidates never reach top_p: no cut
            } else {
                *s_acc = acc;
                *s_prefix = prefix | ((uint32_t)d << shift);
                *s_mask = mask | (255u << shift);
                if (shift == 0) *s_k = H.c[0][d];         // entries equal to the cut value
            }
        }
        __syncthreads();
    }
    if (*s_tp && *s_cut) {
        const float tau = float_of(*s_prefix);
        const uint64_t tq = fx(tau, FX_P);
        // tied entries kept, in index order: the first `keep` of them
        const int keep = (int)((target - *s_acc + tq - 1) / tq);
        const int ties = (int)*s_k;
        int off = 0;
        if (keep < ties) {
            int c = 0;
            seg_for(pv, n, [&](int, float v, bool ok) { c += __popcll(__ballot(ok && v == tau)); });
            __syncthreads();
            if (lane == 0) s_w[wave] = c;
            __syncthreads();
            for (int w = 0; w < wave; ++w) off += s_w[w];
        }
        const uint64_t lt = (1ull << lane) - 1ull;
        seg_for(pv, n, [&](int j, float v, bool ok) {
            const bool tie = ok && v == tau;
            const uint64_t m = __ballot(tie);
            if (ok && v > 1e-10f && (v < tau || (tie && off + __popcll(m & lt) >= keep))) pv[j] = 0.0f;
            off += __popcll(m);
        });
        __syncthreads();
    }
    if (*s_tp) {
        // renormalised (also when nothing was cut, as the reference does)
        uint64_t q2 = 0;
        seg_for(pv, n, [&](int, float v, bool ok) {
            if (ok) q2 += fx(v, FX_P);
        });
        const float s2 = unfx(block_sum_u64(q2, s_q), FX_P);
        if (s2 > 0)
            seg_for(pv, n, [&](int j, float v, bool ok) {
                if (ok) pv[j] = v / s2;
            });
        __syncthreads();
    }
}

// The first index of pv[0..n) whose exact cumulative sum reaches r (> 0):
// exact sums per wave share, then per 64 chunks of the chosen share, then the
// chosen chunk entry by entry. -1 when the total stays below r.
__device__ __forceinline__ int pick_exact_sums(const float *pv, int n, float r, uint64_t *s_q, int *s_wsel,
                                               uint64_t *s_run, int *s_pick) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t qw = 0;
    seg_for(pv, n, [&](int, float v, bool ok) {
        if (ok) qw += fx(v, FX_P);
    });
    qw = wave_sum_u64(qw);
    __syncthreads();
    if (lane == 0) s_q[wave] = qw;
    __syncthreads();
    const uint64_t R = fx(r, FX_P);
    if (tid == 0) {
        uint64_t run = 0;
        int w = 0;
        for (; w < NW; ++w) {
            if (run + s_q[w] >= R) break;
            run += s_q[w];
        }
        *s_wsel = w < NW ? w : -1;
        *s_run = run;
        *s_pick = -1;
    }
    __syncthreads();
    if (wave == *s_wsel) {
        const seg_t sg = wave_seg(n);
        const int cs = (sg.e - sg.b + 63) / 64;
        const int c0 = min(sg.e, sg.b + lane * cs), c1 = min(sg.e, c0 + cs);
        uint64_t ql = 0;
        for (int j = c0; j < c1; j += 16) {
            float t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) t[u] = pv[min(j + u, c1 - 1)];
#pragma unroll
            for (int u = 0; u < 16; ++u) ql += j + u < c1 ? fx(t[u], FX_P) : 0;
        }
        const uint64_t incl = wave_incl_scan_u64(ql);
        const uint64_t run = *s_run;
        const uint64_t hit = __ballot(run + incl >= R);
        const int L = hit ? __ffsll((long long)hit) - 1 : 63;
        if (lane == L) {
            uint64_t acc = run + incl - ql;
            int pk = -1;
            for (int j = c0; j < c1; ++j) {
                acc += fx(pv[j], FX_P);
                if (acc >= R) { pk = j; break; }
            }
            *s_pick = pk;
        }
    }
    __syncthreads();
    return *s_pick;
}

// 1. repetition penalty: the first occurrence of each token applies it as
// many times as the token occurs (counts in ai[], reset first).
__device__ __forceinline__ void apply_penalty(float *lg, int V, const pk_sampler_dev *sp, int *ai) {
    const int tid = threadIdx.x;
    const float rep = sp->rep_penalty;
    if (rep > 1.0f) {
        const int hl = min(sp->history_len, PK_HISTORY_CAP);
        for (int i = tid; i < hl; i += SNT) {
            const int t = sp->history[i];
            if (t >= 0 && t < V) ai[t] = 0;
        }
        __syncthreads();
        unsigned own = 0;
#pragma unroll
        for (int q = 0; q < PK_HISTORY_CAP / SNT; ++q) {
            const int i = tid + q * SNT;
            if (i < hl) {
                const int t = sp->history[i];
                if (t >= 0 && t < V && atomicAdd(&ai[t], 1) == 0) own |= 1u << q;
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PK_HISTORY_CAP / SNT; ++q)
            if (own & (1u << q)) {
                const int t = sp->history[tid + q * SNT];
                const int c = atomicAdd(&ai[t], 0);
                float v = lg[t];
                for (int r = 0; r < c; ++r) v = v > 0 ? v / rep : v * rep;
                lg[t] = v;
            }
        __syncthreads();
    }
}

// The draw's last step: the id into the history, the decode state and `last`.
// tok < 0: the reference's final fall-through 0, which is not appended.
__device__ __forceinline__ void finish_draw(pk_sampler_dev *sp, pk_dstate *st, int32_t *out_toks, int out_cap, int tok) {
    if (tok >= 0 && sp->history_len < PK_HISTORY_CAP) sp->history[sp->history_len++] = tok;
    const int t = tok < 0 ? 0 : tok;
    if (st) {
        if (st->n_out < out_cap) out_toks[st->n_out] = t;
        st->n_out = st->n_out + 1;
        st->next = t;
        st->tok = t;
        st->pos = st->pos + 1;
    }
    sp->last = t;
}

// bmax[0..nb): optional maxima of disjoint blocks of lg as the GEMV wrote it
// (before the penalty, which only lowers values: an upper bound of the
// maximum, which is all the top-k window needs). write_back = 0: nobody
// reads lg afterwards, so a top-k draw leaves it as it is.
__global__ __launch_bounds__(SNT) void k_sample(float *lg, int V, pk_sampler_dev *sp, float *av, int *ai,
                                                pk_dstate *st, int32_t *out_toks, int out_cap,
                                                const float *bmax, int nb, int write_back, samp_ws *pre) {
    // radix histograms (counts, exact sums) and the small path's sort share one block
    __shared__ __align__(16) uint64_t lds_raw[sizeof(lds_hist) / 8];
    // the small path's kept entries double as the buffer of the ordered sums
    __shared__ __align__(16) float stage[OS_BUF > 2 * SMALL ? OS_BUF : 2 * SMALL];
    __shared__ float s_red[NW];
    __shared__ int s_redi[NW], s_w[NW];
    __shared__ uint64_t s_q[NW];
    __shared__ uint32_t s_prefix, s_mask, s_k;
    __shared__ uint64_t s_pfx64, s_msk64;
    __shared__ int s_tok, s_cut, s_tp, s_wsel, s_pick;
    __shared__ float s_sum, s_r;
    __shared__ uint64_t s_acc, s_run;
    lds_hist &H = *reinterpret_cast<lds_hist *>(lds_raw);
    float *sv = reinterpret_cast<float *>(lds_raw);
    int *si = reinterpret_cast<int *>(sv + SMALL);
    float *kv = stage;
    int *ki = reinterpret_cast<int *>(stage + SMALL);
    __shared__ float cv[CAND];                          // top-k candidates (value, index)
    __shared__ int ci[CAND];
    __shared__ int s_nc, s_cnt, s_win;
    __shared__ uint64_t s_q2[NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float T = sp->temperature, top_p = sp->top_p;
    const int K = sp->top_k;

    if (!pre) apply_penalty(lg, V, sp, ai);

    if (T < 1e-6f) {
        // 2. greedy: the first maximum (the reference moves on a strictly
        // greater value only, so ties and NaNs keep the earlier index)
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        seg_for(lg, V, [&](int j, float v, bool ok) {
            if (ok && (v > bv || (v == bv && j < bi))) { bv = v; bi = j; }
        });
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (lane == 0) { s_red[wave] = bv; s_redi[wave] = bi; }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < NW; ++w)
                if (s_red[w] > bv || (s_red[w] == bv && s_redi[w] < bi)) { bv = s_red[w]; bi = s_redi[w]; }
            s_tok = (bi == 0x7fffffff || !(bv > lg[0])) ? 0 : bi;
        }
        __syncthreads();
    } else {
        // 3. temperature (applied as each pass reads, and stored with the kept entries)
        const float inv_t = 1.0f / T;
        const auto scaled = [inv_t](float v) { return v * inv_t; };

        // 4. top-k threshold: the K-th largest key, 8 bits per pass from the top.
        // After the first pass (sign and exponent) the entries whose top byte
        // reaches the threshold's are few for any real top-k; when at most CAND,
        // they are gathered into LDS and the later passes, the kept set and its
        // index order are worked out there.
        const bool use_k = K > 0 && K < V;
        int n = V;
        bool direct = false;                                  // kept entries already in kv / ki
        if (use_k) {
            if (tid == 0) { s_prefix = 0; s_mask = 0; s_k = (uint32_t)K; }
            // histogram totals into H.c[0], then the digit holding the K-th largest
            const auto radix_walk = [&](int shift) {
                __syncthreads();
                if (tid < 256) {
                    uint32_t c = 0;
                    for (int w = 0; w < NW; ++w) c += H.c[w][tid];
                    H.c[0][tid] = c;
                }
                __syncthreads();
                if (tid == 0) {
                    uint32_t k = s_k;
                    int d = 255;
                    for (; d > 0; --d) {
                        if (k <= H.c[0][d]) break;
                        k -= H.c[0][d];
                    }
                    s_k = k;
                    s_prefix = s_prefix | ((uint32_t)d << shift);
                    s_mask = s_mask | (255u << shift);
                    // entries at or above the new bucket: K - k above it, and the bucket
                    s_nc = (int)((uint32_t)K - k + H.c[0][d]);
                    s_cnt = 0;
                }
                __syncthreads();
            };
            // candidates gathered by k_samp_gather: every entry at or above the
            // bucket of the K-th largest
            const int given = pre ? min(pre->n_cand, CAND) : 0;
            if (given > 0) {
                for (int i = tid; i < given; i += SNT) {
                    cv[i] = pre->cv[i];
                    ci[i] = pre->ci[i];
                }
                if (tid == 0) s_nc = given;
                __syncthreads();
            } else {
                // First 8 bits. The K-th largest nearly always lies within a few
                // binades of the maximum: the maximum key, then the counts of the 8
                // sign/exponent buckets at and below it in 16-bit fields of two
                // registers per lane (no atomics: a whole wave would hit the same
                // few LDS counters). Otherwise a full histogram pass.
                uint32_t mk = 0;
                if (bmax) {
                    for (int b = tid; b < nb; b += SNT) mk = max(mk, key_of(bmax[b] * inv_t));
                } else {
                    seg_for(lg, V, [&](int, float v, bool ok) {
                        if (ok) mk = max(mk, key_of(v * inv_t));
                    });
                }
                for (int o = 32; o > 0; o >>= 1) mk = max(mk, (uint32_t)__shfl_xor((int)mk, o, 64));
                if (lane == 0) s_w[wave] = (int)mk;
                __syncthreads();
                mk = 0;
                for (int w = 0; w < NW; ++w) mk = max(mk, (uint32_t)s_w[w]);
                const uint32_t tb = mk >> 24;
                uint64_t lo = 0, hi = 0;
                seg_for(lg, V, [&](int, float v, bool ok) {
                    const uint32_t d = tb - (key_of(v * inv_t) >> 24);
                    const uint64_t inc = (ok && d < 8u) ? (1ull << (16u * (d & 3u))) : 0ull;
                    lo += d < 4u ? inc : 0ull;
                    hi += d < 4u ? 0ull : inc;
                });
                lo = wave_sum_u64(lo);                        // per wave at most V/16 per field
                hi = wave_sum_u64(hi);
                if (lane == 0) { s_q[wave] = lo; s_q2[wave] = hi; }
                __syncthreads();
                if (tid == 0) {
                    uint32_t cum = 0, rank = 0;
                    int i = 0;
                    for (; i < 8; ++i) {
                        uint32_t c = 0;
                        for (int w = 0; w < NW; ++w)
                            c += (uint32_t)(((i < 4 ? s_q[w] : s_q2[w]) >> (16 * (i & 3))) & 0xffffu);
                        if (cum + c >= (uint32_t)K) {
                            rank = (uint32_t)K - cum;         // the K-th largest's rank inside bucket i
                            cum += c;
                            break;
                        }
                        cum += c;
                    }
                    s_win = i < 8 && (int)tb - i >= 0;
                    if (s_win) {
                        s_k = rank;
                        s_prefix = (tb - (uint32_t)i) << 24;
                        s_mask = 0xff000000u;
                        s_nc = (int)cum;
                        s_cnt = 0;
                    }
                }
                __syncthreads();
                if (!s_win) {
                    for (int b = tid; b < NW * 256; b += SNT) (&H.c[0][0])[b] = 0;
                    __syncthreads();
                    seg_for(lg, V, [&](int, float v, bool ok) {
                        if (ok) atomicAdd(&H.c[wave][key_of(v * inv_t) >> 24], 1u);
                    });
                    radix_walk(24);
                }
            }
            // the remaining 24 bits; as soon as the entries at or above the
            // current bucket fit in LDS they are gathered there and the rest runs on them
            bool in_lds = given > 0;
            int nc = given;
            const bool few = given > 0 && given <= RANK_N;
            if (few) {
                // the K-th largest by counting: entries above it < K <= those not below it
                if (tid < given) {
                    const uint32_t k = key_of(cv[tid]);
                    int above = 0, same = 0;
                    for (int i = 0; i < given; ++i) {
                        const uint32_t ki_ = key_of(cv[i]);
                        above += ki_ > k ? 1 : 0;
                        same += ki_ == k ? 1 : 0;
                    }
                    if (above < K && K <= above + same) s_prefix = k;      // (equal keys write the same)
                }
                __syncthreads();
            }
            for (int shift = few ? -16 : given > 0 ? 24 : 16; shift >= -8; shift -= 8) {
                if (!in_lds && s_nc <= CAND) {
                    nc = s_nc;
                    const uint32_t top = s_prefix;
                    seg_for(lg, V, [&](int j, float v, bool ok) {
                        const float x = v * inv_t;
                        if (ok && key_of(x) >= top) {
                            const int o = atomicAdd(&s_cnt, 1);   // below nc: counted by the passes
                            if (o < CAND) {
                                cv[o] = x;
                                ci[o] = j;
                            }
                        }
                    });
                    in_lds = true;
                    __syncthreads();
                }
                if (shift < 0) break;
                for (int b = tid; b < NW * 256; b += SNT) (&H.c[0][0])[b] = 0;
                __syncthreads();
                const uint32_t prefix = s_prefix, mask = s_mask;
                if (in_lds) {
                    for (int i = tid; i < nc; i += SNT) {
                        const uint32_t k = key_of(cv[i]);
                        if ((k & mask) == prefix) atomicAdd(&H.c[wave][(k >> shift) & 255u], 1u);
                    }
                } else {
                    seg_for(lg, V, [&](int, float v, bool ok) {
                        const uint32_t k = key_of(v * inv_t);
                        if (ok && (k & mask) == prefix) atomicAdd(&H.c[wave][(k >> shift) & 255u], 1u);
                    });
                }
                radix_walk(shift);
            }
            const float thr = float_of(s_prefix);
            // a zero threshold also keeps -0.0, whose key lies below the candidates'
            if (in_lds && thr != 0.0f) {
                // the kept candidates, then into index order
                if (tid == 0) s_cnt = 0;
                __syncthreads();
                for (int i = tid; i < nc; i += SNT)
                    if (!(cv[i] < thr)) {
                        const int o = atomicAdd(&s_cnt, 1);
                        kv[o] = cv[i];
                        ki[o] = ci[i];
                    }
                __syncthreads();
                n = s_cnt;
                if (n <= RANK_N) {
                    float x = 0.0f;
                    int id = 0, at = 0;
                    if (tid < n) {
                        x = kv[tid];
                        id = ki[tid];
                        for (int i = 0; i < n; ++i) at += ki[i] < id ? 1 : 0;
                    }
                    __syncthreads();
                    if (tid < n) { kv[at] = x; ki[at] = id; }
                    __syncthreads();
                } else {
                    int P = 1;
                    while (P < n) P <<= 1;
                    for (int j = n + tid; j < P; j += SNT) { kv[j] = 0.0f; ki[j] = 0x7fffffff; }
                    __syncthreads();
                    bitonic_by_index(kv, ki, P);
                }
                direct = true;
            } else {
                n = compact(lg, V, [inv_t, thr](float v) { return !(v * inv_t < thr); }, scaled, av, ai, s_w);
            }
        }

        if (n <= SMALL) {
            // 5a. in LDS, the reference's order
            if (!direct) {
                for (int j = tid; j < n; j += SNT) {
                    kv[j] = use_k ? av[j] : lg[j] * inv_t;
                    ki[j] = use_k ? ai[j] : j;
                }
                __syncthreads();
            }
            const int pick = finish_small(kv, n, top_p, sp, sv, si, s_red, s_redi, &s_sum, &s_cut, &s_r);
            if (tid == 0) {
                // a draw of 0 takes the first vocabulary entry even when it was dropped
                s_tok = s_r <= 0.0f ? 0 : (pick >= 0 ? ki[pick] : -1);
            }
            __syncthreads();
            // the array as the reference leaves it: probabilities, 0 elsewhere
            if (use_k && write_back && !(pre && pre->n_cand > 0)) {      // (k_samp_gather has zeroed it)
                for (int i = tid; i < V; i += SNT) lg[i] = 0.0f;
                __syncthreads();
            }
            if (!use_k || write_back)
                for (int j = tid; j < n; j += SNT) lg[ki[j]] = kv[j];
        } else {
            // 5b. over pv[0..n) in global memory (av after top-k, else lg in place)
            float *pv = use_k ? av : lg;
            const bool fast = sp->fast_sums != 0;
            float mx = -1e30f;
            seg_for(pv, n, [&](int j, float v, bool ok) {
                if (!ok) return;
                if (!use_k) {
                    v = v * inv_t;
                    pv[j] = v;
                }
                mx = fmaxf(mx, v);
            });
            mx = block_max(mx, s_red);
            const int se = 63 - (32 - __clz(n));           // n values <= 1 sum below 2^63
            uint64_t q = 0;
            seg_for(pv, n, [&](int j, float v, bool ok) {
                if (!ok) return;
                const float e = expf(v - mx);
                pv[j] = e;
                q += fx(e, se);
            });
            float sum;
            if (fast) {
                sum = unfx(block_sum_u64(q, s_q), se);
            } else {
                __syncthreads();
                order_sum(pv, n, stage, false, 0.0f, &s_sum, &s_pick);
                sum = s_sum;
            }
            seg_for(pv, n, [&](int j, float v, bool ok) {
                if (ok) pv[j] = v / sum;
            });
            __syncthreads();

            if (top_p < 1.0f && top_p > 0.0f) {
                if (fast)
                    top_p_exact_sums(pv, n, top_p, H, s_w, s_q, &s_prefix, &s_mask, &s_k, &s_acc, &s_cut, &s_tp);
                else
                    top_p_chunks(pv, n, top_p, H, sv, si, stage, s_redi, &s_pfx64, &s_msk64, &s_k, &s_cut,
                                 &s_tp, &s_sum, &s_pick);
            }

            // the draw
            if (tid == 0) {
                uint64_t x = sp->rng;
                x ^= x << 13;
                x ^= x >> 7;
                x ^= x << 17;
                sp->rng = x;
                s_r = (float)(x >> 33) / (float)(1ULL << 31);
            }
            __syncthreads();
            const float r = s_r;
            int pick;
            if (fast) {
                pick = pick_exact_sums(pv, n, r, s_q, &s_wsel, &s_run, &s_pick);
            } else {
                // the first index whose running float sum (in index order) reaches r
                order_sum(pv, n, stage, true, r, &s_sum, &s_pick);
                pick = s_pick;
            }
            if (pick < 0) {
                // nothing reached r: the last entry with probability > 0
                int last = -1;
                seg_for(pv, n, [&](int j, float v, bool ok) {
                    if (ok && v > 0) last = max(last, j);
                });
                pick = block_max_i(last, s_redi);
            }
            // a draw of 0 takes the first vocabulary entry even when it was dropped
            if (tid == 0) s_tok = r <= 0.0f ? 0 : (pick >= 0 ? (use_k ? ai[pick] : pick) : -1);
            __syncthreads();
            if (use_k && write_back) {
                for (int i = tid; i < V; i += SNT) lg[i] = 0.0f;
                __syncthreads();
                for (int j = tid; j < n; j += SNT) lg[ai[j]] = av[j];
            }
        }
    }
    if (tid == 0) finish_draw(sp, st, out_toks, out_cap, s_tok);
    if (pre) {                                         // re-armed for the next draw
        __syncthreads();
        for (int i = tid; i < SB_BINS; i += SNT) pre->hist[i] = 0;
        if (tid == 0) pre->n_cand = 0;
    }
}

// ───────────── a draw over the device: top-k up to CAND entries ─────────────
// One workgroup reads the vocabulary at ~60 GB/s, four times per draw (135 us
// at 201,088 entries). Here every CU takes a share: the keys' upper 12 bits are
// counted (k_samp_hist), every workgroup finds the bucket that holds the
// K-th largest from those counts and gathers its share's entries at or above
// it (k_samp_gather, which also zeroes the array), and k_sample finishes on
// the candidates. Where they exceed CAND, or the bucket holds zero (a zero
// threshold also keeps -0.0, below it), nothing is gathered or zeroed and
// k_sample does the whole draw.
constexpr int SH_T = 256, SH_E = 4;       // threads, entries per thread

__global__ __launch_bounds__(SNT) void k_samp_penalty(float *lg, int V, const pk_sampler_dev *sp, int *ai) {
    apply_penalty(lg, V, sp, ai);
}

__global__ __launch_bounds__(SH_T) void k_samp_hist(const float *lg, int V, const pk_sampler_dev *sp, samp_ws *ws) {
    __shared__ uint32_t h[SB_BINS];
    for (int i = threadIdx.x; i < SB_BINS; i += SH_T) h[i] = 0;
    const float inv_t = 1.0f / sp->temperature;
    float v[SH_E];
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SH_E; ++k)
        if (j0 + SH_T * k < V) atomicAdd(&h[key_of(v[k] * inv_t) >> 20], 1u);
    __syncthreads();
    for (int i = threadIdx.x; i < SB_BINS; i += SH_T)
        if (h[i]) atomicAdd(&ws->hist[i], h[i]);
}

__global__ __launch_bounds__(SH_T) void k_samp_gather(float *lg, int V, const pk_sampler_dev *sp, samp_ws *ws,
                                                      int write_back) {
    __shared__ uint32_t s_w[SH_T / 64];
    __shared__ int s_bin, s_cnt;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float inv_t = 1.0f / sp->temperature;
    const uint32_t K = (uint32_t)sp->top_k;
    float v[SH_E];
    const int j0 = blockIdx.x * SH_T * SH_E + tid;
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
    // thread t counts the 16 bins below the top t * 16; an inclusive scan
    // from the top finds the thread, then the bin, of the K-th largest
    constexpr int B = SB_BINS / SH_T;
    uint32_t c[B], sum = 0;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        c[i] = ws->hist[SB_BINS - 1 - (B * tid + i)];
        sum += c[i];
    }
    uint32_t inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_w[wave] = inc;
    if (tid == 0) {                                   // (no bin for top_k 0 or above V: k_sample takes the draw)
        s_bin = 0;
        s_cnt = CAND + 1;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) inc += s_w[w];
    if (inc >= K && inc - sum < K) {
        uint32_t cum = inc - sum;
        int i = 0;
        for (; i < B; ++i) {
            cum += c[i];
            if (cum >= K) break;
        }
        s_bin = SB_BINS - 1 - (B * tid + i);
        s_cnt = (int)cum;
    }
    __syncthreads();
    const int bin = s_bin;
    if (s_cnt > CAND || bin == (int)(key_of(0.0f) >> 20) || bin == (int)(key_of(-0.0f) >> 20)) return;
#pragma unroll
    for (int k = 0; k < SH_E; ++k) {
        const int j = j0 + SH_T * k;
        if (j >= V) continue;
        const float x = v[k] * inv_t;
        if ((int)(key_of(x) >> 20) >= bin) {
            const int o = atomicAdd(&ws->n_cand, 1);
            if (o < CAND) {                           // (o < s_cnt)
                ws->cv[o] = x;
                ws->ci[o] = j;
            }
        }
        if (write_back) lg[j] = 0.0f;
    }
}

// ───────────── a draw over the device: no top-k ─────────────
// The reference's steps as launches of their own: the elementwise ones on
// every CU, the ordered float sums as runs (om_sum). The top-p
// list is sorted by buckets: the candidates (> 1e-10) are counted by the
// upper bits of their value (64 buckets per binade, at most 2131), placed
// into their buckets, the largest first, and each bucket is sorted in LDS by
// its own workgroup (equal values need no order: a sum does not tell them
// apart, and the cut takes ties by index). Where a bucket exceeds SORT_CAP
// different values, one workgroup takes the list chunk by chunk instead.
// Measured, 201,088 entries of a peaked distribution, top-p 0.95: 252 us
// per draw against 5,000 to 6,000 in one workgroup; 396 with each ordered sum
// on one workgroup (100 us, 75 in the draw; 30 + 8 and 32 + 8 as runs).
constexpr int SORT_CAP = 4096;
constexpr uint32_t P_MIN = 0x2edbe6ffu;   // bits of 1e-10f
constexpr int P_SHIFT = 17;
constexpr int P_BINS = (int)((0x3f800000u - P_MIN) >> P_SHIFT) + 1;
static_assert(P_BINS <= SB_BINS, "top-p buckets");
__device__ __forceinline__ int p_bin(float p) {       // 0: the largest values
    return P_BINS - 1 - (int)min((__float_as_uint(p) - P_MIN) >> P_SHIFT, (uint32_t)P_BINS - 1u);
}

// lg = lg / T, and the largest
__global__ __launch_bounds__(SH_T) void k_samp_scale(float *lg, int V, const pk_sampler_dev *sp, samp_ws *ws) {
    __shared__ uint32_t s_w[SH_T / 64];
    const float inv_t = 1.0f / sp->temperature;
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
    float v[SH_E];
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
    float mx = -1e30f;
#pragma unroll
    for (int k = 0; k < SH_E; ++k) {
        const float x = v[k] * inv_t;
        if (j0 + SH_T * k < V) {
            lg[j0 + SH_T * k] = x;
            mx = fmaxf(mx, x);
        }
    }
    uint32_t mk = key_of(mx);
    for (int o = 32; o > 0; o >>= 1) mk = max(mk, (uint32_t)__shfl_xor((int)mk, o, 64));
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = mk;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SH_T / 64; ++w) mk = max(mk, s_w[w]);
        atomicMax(&ws->mx_key, mk);
    }
}

__global__ __launch_bounds__(SH_T) void k_samp_exp(float *lg, int V, const samp_ws *ws) {
    const float mx = float_of(ws->mx_key);
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
    float v[SH_E];
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
#pragma unroll
    for (int k = 0; k < SH_E; ++k)
        if (j0 + SH_T * k < V) lg[j0 + SH_T * k] = expf(v[k] - mx);
}

// The ordered sum over the device. order_sum walks the array with one
// workgroup (201,088 entries: 25 chunks of 8192 and a round per binade, 2.3 us
// each: 100 us). A run's pair of moves depends only on the binade of the sum
// before it, so every wave composes its run's pair for the binade that a plain
// float sum of the runs before it predicts (k_samp_part, k_samp_moves), and one
// wave then scans the pairs, 64 runs at a time, in the exact sum. A run whose
// prediction was wrong, or in which the sum passes a binade or the draw, is
// added element by element from the array, as order_sum adds it: the
// predictions decide what is fast, never the result.
constexpr int OM_RUN = 64 * OS_E;         // elements of a wave's pass; a run is `per` of them
static int om_per(int n) { return (n + OM_RUN * SAMP_RUNS - 1) / (OM_RUN * SAMP_RUNS); }
static int om_runs(int n) { return (n + OM_RUN * om_per(n) - 1) / (OM_RUN * om_per(n)); }

// part[c] = run c's sum, in any order
__global__ __launch_bounds__(SH_T) void k_samp_part(const float *src, int n, int per, int runs, samp_ws *ws) {
    const int lane = threadIdx.x & 63, c = blockIdx.x * (SH_T / 64) + (threadIdx.x >> 6);
    if (c >= runs) return;
    float sum = 0.0f;
    for (int p = 0; p < per; ++p) {
        const int64_t b = ((int64_t)c * per + p) * OM_RUN + lane;
        float v[OS_E];
#pragma unroll
        for (int k = 0; k < OS_E; ++k) v[k] = src[min(b + 64 * k, (int64_t)n - 1)];
#pragma unroll
        for (int k = 0; k < OS_E; ++k) sum += b + 64 * k < n ? v[k] : 0.0f;
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (lane == 0) ws->part[c] = sum;
}

// This lane's OS_E elements of the pass at b (zeros past n: + 0 leaves a sum as it is).
__device__ __forceinline__ void om_load(const float *src, int n, int64_t b, float (&v)[OS_E]) {
    const int64_t j = b + OS_E * (threadIdx.x & 63);
    float t[OS_E];
#pragma unroll
    for (int k = 0; k < OS_E; ++k) t[k] = src[min(j + k, (int64_t)n - 1)];
#pragma unroll
    for (int k = 0; k < OS_E; ++k) v[k] = j + k < n ? t[k] : 0.0f;
}

// mv[c], mex[c] = run c's pair of moves, and the binade it holds in
__global__ __launch_bounds__(SH_T) void k_samp_moves(const float *src, int n, int per, int runs, samp_ws *ws) {
    const int lane = threadIdx.x & 63, c = blockIdx.x * (SH_T / 64) + (threadIdx.x >> 6);
    if (c >= runs) return;
    float v[OS_E];
    om_load(src, n, (int64_t)c * per * OM_RUN, v);
    float s = 0.0f;
    for (int i = lane; i < c; i += 64) s += ws->part[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    const int ex = max((int)((__float_as_uint(s) >> 23) & 0xffu), 1);
    uint2 all = make_uint2(0u, 0u);
    for (int p = 0; p < per; ++p) {
        if (p) om_load(src, n, ((int64_t)c * per + p) * OM_RUN, v);
        const uint2 inc = os_scan<true>(os_moves(v, ex));
        all = os_clamp(os_then(all, make_uint2((uint32_t)__builtin_amdgcn_readlane((int)inc.x, 63),
                                               (uint32_t)__builtin_amdgcn_readlane((int)inc.y, 63))));
    }
    if (lane == 0) {
        ws->mv[c] = all;
        ws->mex[c] = ex;
    }
}

// The sum of src[0..n) in index order on one wave, over the runs' moves; find:
// stop at the first index whose running sum is >= r (-1: none).
__device__ __forceinline__ float om_sum(const float *src, int n, int per, int runs, const samp_ws *ws, bool find,
                                        float r, int &hit) {
    __shared__ uint2 mv[SAMP_RUNS];
    __shared__ int mex[SAMP_RUNS];
    const int lane = threadIdx.x & 63;
    for (int i = lane; i < runs; i += 64) {
        mv[i] = ws->mv[i];
        mex[i] = ws->mex[i];
    }
    pk_wave_lds_order();
    hit = -1;
    float s = 0.0f;
    for (int c = 0; c < runs;) {
        {
            const uint32_t sb = __float_as_uint(s);
            const int ex = max((int)(sb >> 23), 1);
            const uint32_t S = (sb & 0x7fffffu) | ((sb >> 23) ? 0x800000u : 0u);
            const int i = min(c + lane, runs - 1);
            const bool ok = c + lane < runs && mex[i] == ex;
            const uint2 inc = os_scan<true>(ok ? mv[i] : make_uint2(OS_BIG, OS_BIG));
            const uint32_t S1 = S + ((S & 1u) ? inc.y : inc.x);
            const uint64_t bad =
                __ballot(!ok || S1 >= 0x1000000u || (find && ldexpf((float)min(S1, OS_BIG), ex - 150) >= r));
            const int f = bad ? __builtin_ctzll(bad) : 64;
            if (f > 0) s = ldexpf((float)(uint32_t)__builtin_amdgcn_readlane((int)S1, f - 1), ex - 150);
            c += f;
            if (f == 64 || c >= runs) continue;
        }
        for (int p = 0; p < per; ++p) {
            const int64_t base = ((int64_t)c * per + p) * OM_RUN;
            if (base >= n) break;
            float v[OS_E];
            om_load(src, n, base, v);
            for (int start = 0; start < OM_RUN;) {         // the pass's elements before it are in s
                const uint32_t sb = __float_as_uint(s);
                const int ex = max((int)(sb >> 23), 1);
                const uint32_t S = (sb & 0x7fffffu) | ((sb >> 23) ? 0x800000u : 0u);
                const uint2 d = os_moves(v, ex);
                const uint2 inc = os_scan<true>(d), pre = os_dpp<0x138, 0xf>(inc);
                const bool odd = S & 1u;
                const uint32_t S0 = S + (odd ? pre.y : pre.x);         // before this lane's elements
                const uint32_t S1 = S0 + ((S0 & 1u) ? d.y : d.x);
                const float a0 = ldexpf((float)min(S0, OS_BIG), ex - 150);
                const bool cross = S0 < 0x1000000u && S1 >= 0x1000000u;
                const bool hits = find && S0 < 0x1000000u && !cross && ldexpf((float)S1, ex - 150) >= r &&
                                  (!(a0 >= r) || OS_E * lane <= start);
                float x = a0;
                int at = -1;
                if (cross || hits)
#pragma unroll
                    for (int k = 0; k < OS_E; ++k)
                        if (at < 0) {
                            x = x + v[k];
                            if (find && x >= r) at = k;
                        }
                const uint64_t got = __ballot(at >= 0), over = __ballot(cross);
                if (got) {
                    const int f = __builtin_ctzll(got);
                    hit = (int)base + OS_E * f + __builtin_amdgcn_readlane(at, f);
                    return s;
                }
                if (over) {
                    const int f = __builtin_ctzll(over);
                    s = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), f));
                    start = OS_E * (f + 1);
                } else {
                    s = ldexpf((float)(uint32_t)__builtin_amdgcn_readlane((int)S1, 63), ex - 150);
                    start = OM_RUN;
                }
                if (!(s < INFINITY)) return s;             // NaN stays NaN, infinity stays
                if (OS_E * lane < start) {                 // (whole lanes: in s)
#pragma unroll
                    for (int k = 0; k < OS_E; ++k) v[k] = 0.0f;
                }
            }
        }
        ++c;
    }
    return s;
}

// ws->sum = the ordered sum of src[0..n), after its k_samp_part and k_samp_moves
__global__ __launch_bounds__(64) void k_samp_sum(const float *src, int n, int per, int runs, samp_ws *ws) {
    if (ws->cut == 2) return;
    int hit;
    const float s = om_sum(src, n, per, runs, ws, false, 0.0f, hit);
    if (threadIdx.x == 0) {
        ws->sum = s;
        ws->mx_key = 0;                               // (read; re-armed)
    }
}

// lg = lg / sum. mode 1: the softmax's division, and the candidates' counts per
// bucket; 2: the division alone; 0: renormalising after the cut.
__global__ __launch_bounds__(SH_T) void k_samp_div(float *lg, int V, samp_ws *ws, int mode) {
    __shared__ uint32_t h[P_BINS];
    const float sum = ws->sum;
    const bool count = mode == 1;
    if (mode == 0 && (ws->m <= 1 || ws->cut == 2 || !(sum > 0))) return;    // (renormalising: the reference's conditions)
    if (count) {
        for (int i = threadIdx.x; i < P_BINS; i += SH_T) h[i] = 0;
        __syncthreads();
    }
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
    float v[SH_E];
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
#pragma unroll
    for (int k = 0; k < SH_E; ++k)
        if (j0 + SH_T * k < V) {
            const float p = v[k] / sum;
            lg[j0 + SH_T * k] = p;
            if (count && p > 1e-10f) atomicAdd(&h[p_bin(p)], 1u);
        }
    if (!count) return;
    __syncthreads();
    for (int i = threadIdx.x; i < P_BINS; i += SH_T)
        if (h[i]) atomicAdd(&ws->hist[i], h[i]);
}

// cur[b] = where bucket b starts (the cursors of k_samp_place), m
__global__ __launch_bounds__(SNT) void k_samp_offsets(samp_ws *ws) {
    __shared__ uint32_t s_w[NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int B = SB_BINS / SNT;
    uint32_t c[B], sum = 0;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        c[i] = ws->hist[B * tid + i];
        sum += c[i];
    }
    uint32_t inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    for (int w = 0; w < wave; ++w) inc += s_w[w];
    uint32_t off = inc - sum;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        ws->cur[(B * tid + i) * 16] = off;
        off += c[i];
    }
    if (tid == SNT - 1) {
        ws->m = (int)inc;
        ws->cut = 0;
        ws->unsorted = 0;
    }
}

__global__ __launch_bounds__(SH_T) void k_samp_place(const float *lg, int V, samp_ws *ws, float *sorted) {
    if (ws->m <= 1) return;
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
    float v[SH_E];
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
#pragma unroll
    for (int k = 0; k < SH_E; ++k)
        if (j0 + SH_T * k < V && v[k] > 1e-10f) sorted[atomicAdd(&ws->cur[p_bin(v[k]) * 16], 1u)] = v[k];
}

// bucket blockIdx.x, descending (cur[b] is its end once everything is placed);
// its count is re-armed
__global__ __launch_bounds__(SH_T) void k_samp_sort(samp_ws *ws, float *sorted) {
    __shared__ float x[SORT_CAP];
    __shared__ int s_diff;
    const int b = blockIdx.x, n = (int)ws->hist[b];
    __syncthreads();
    if (threadIdx.x == 0) {
        if (n) ws->hist[b] = 0;
        s_diff = 0;
    }
    if (n <= 1 || ws->m <= 1) return;
    float *p = sorted + (int)ws->cur[b * 16] - n;
    __syncthreads();
    if (n > SORT_CAP) {
        const float first = p[0];
        bool diff = false;
        for (int i = threadIdx.x; i < n; i += SH_T) diff |= p[i] != first;
        if (diff) s_diff = 1;
        __syncthreads();
        if (threadIdx.x == 0 && s_diff) ws->unsorted = 1;
        return;
    }
    int P = 2;
    while (P < n) P <<= 1;
    for (int i = threadIdx.x; i < P; i += SH_T) x[i] = i < n ? p[i] : -1.0f;
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < P / 2; t += SH_T) {
                const int lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
                const float a = x[lo], c = x[hi];
                if ((a < c) != ((lo & size) != 0)) { x[lo] = c; x[hi] = a; }
            }
            __syncthreads();
        }
    for (int i = threadIdx.x; i < n; i += SH_T) p[i] = x[i];
}

// The cut: the first position of the sorted list whose ordered running sum
// reaches top_p. Entries below its value go (k_samp_zero); of those equal to
// it the first `keep` by index stay.
__global__ __launch_bounds__(SNT) void k_samp_cut(float *lg, int V, const pk_sampler_dev *sp, samp_ws *ws,
                                                  const float *sorted) {
    __shared__ __align__(16) uint64_t lds_raw[sizeof(lds_hist) / 8];
    __shared__ __align__(16) float buf[OS_BUF];
    __shared__ float s_sum;
    __shared__ int s_hit, s_cut, s_tp, s_redi[NW], s_n[2];
    __shared__ uint64_t s_pfx64, s_msk64;
    __shared__ uint32_t s_k;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = ws->m;
    if (m <= 1) return;                               // the reference's n_active > 1
    const float top_p = sp->top_p;
    if (ws->unsorted) {
        float *sv = reinterpret_cast<float *>(lds_raw);
        top_p_chunks(lg, V, top_p, *reinterpret_cast<lds_hist *>(lds_raw), sv, reinterpret_cast<int *>(sv + SMALL), buf,
                     s_redi, &s_pfx64, &s_msk64, &s_k, &s_cut, &s_tp, &s_sum, &s_hit);
        if (tid == 0) ws->cut = 2;
        return;
    }
    order_sum(sorted, m, buf, true, top_p, &s_sum, &s_hit);
    const int hit = s_hit;
    if (hit < 0) return;                              // never reached: nothing goes
    const float tau = sorted[hit];
    // the run of entries equal to tau
    if (tid < 2) s_n[tid] = 0;
    __syncthreads();
    int above = 0, same = 0;
    seg_for(sorted, m, [&](int, float v, bool ok) {
        above += ok && v > tau ? 1 : 0;
        same += ok && v == tau ? 1 : 0;
    });
    for (int o = 32; o > 0; o >>= 1) {
        above += __shfl_xor(above, o, 64);
        same += __shfl_xor(same, o, 64);
    }
    if (lane == 0) {
        atomicAdd(&s_n[0], above);
        atomicAdd(&s_n[1], same);
    }
    __syncthreads();
    const int keep = hit + 1 - s_n[0];
    if (keep < s_n[1]) {
        int off = 0, c = 0;
        seg_for(lg, V, [&](int, float v, bool ok) { c += __popcll(__ballot(ok && v == tau)); });
        if (lane == 0) s_redi[wave] = c;
        __syncthreads();
        for (int w = 0; w < wave; ++w) off += s_redi[w];
        const uint64_t lt = (1ull << lane) - 1ull;
        seg_for(lg, V, [&](int j, float v, bool ok) {
            const bool tie = ok && v == tau;
            const uint64_t mk = __ballot(tie);
            if (tie && off + __popcll(mk & lt) >= keep) lg[j] = 0.0f;
            off += __popcll(mk);
        });
    }
    if (tid == 0) {
        ws->tau = tau;
        ws->cut = 1;
    }
}

__global__ __launch_bounds__(SH_T) void k_samp_zero(float *lg, int V, const samp_ws *ws) {
    if (ws->m <= 1 || ws->cut != 1) return;
    const float tau = ws->tau;
    const int j0 = blockIdx.x * SH_T * SH_E + threadIdx.x;
    float v[SH_E];
#pragma unroll
    for (int k = 0; k < SH_E; ++k) v[k] = lg[min(j0 + SH_T * k, V - 1)];
#pragma unroll
    for (int k = 0; k < SH_E; ++k)
        if (j0 + SH_T * k < V && v[k] > 1e-10f && v[k] < tau) lg[j0 + SH_T * k] = 0.0f;
}

// The draw: the first index whose ordered running sum reaches it.
__global__ __launch_bounds__(SNT) void k_samp_draw(const float *lg, int V, int per, int runs, pk_sampler_dev *sp,
                                                   samp_ws *ws, pk_dstate *st, int32_t *out_toks, int out_cap) {
    __shared__ float s_r;
    __shared__ int s_hit, s_redi[NW];
    const int tid = threadIdx.x;
    if (tid == 0) {
        uint64_t x = sp->rng;
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        sp->rng = x;
        s_r = (float)(x >> 33) / (float)(1ULL << 31);
        ws->m = 0;
        ws->cut = 0;
    }
    __syncthreads();
    const float r = s_r;
    if (tid < 64) {
        int hit;
        (void)om_sum(lg, V, per, runs, ws, true, r, hit);
        if (tid == 0) s_hit = hit;
    }
    __syncthreads();
    int pick = s_hit;
    if (pick < 0) {
        // nothing reached r: the last entry with probability > 0
        int last = -1;
        seg_for(lg, V, [&](int j, float v, bool ok) {
            if (ok && v > 0) last = max(last, j);
        });
        pick = block_max_i(last, s_redi);
    }
    // a draw of 0 takes the first vocabulary entry even when it was dropped
    if (tid == 0) finish_draw(sp, st, out_toks, out_cap, r <= 0.0f ? 0 : pick);
}

// Prompt ids into the history in order (valid ids only, up to its capacity).
__global__ void k_seed_history(pk_sampler_dev *sp, const int32_t *ids, int n, int V) {
    if (threadIdx.x != 0) return;
    int hl = sp->history_len;
    for (int i = 0; i < n && hl < PK_HISTORY_CAP; ++i) {
        const int t = ids[i];
        if (t >= 0 && t < V) sp->history[hl++] = t;
    }
    sp->history_len = hl;
}

}  // namespace

int pk_sample_reserve(pk_engine *e, int vocab) {
    PK_CHECK(vocab >= 1, PK_ERR_ARG, "vocab %d", vocab);
    if (!e->samp) {
        PK_CHECK(!e->capturing, PK_ERR_ARG, "sampling: call pk_set_sampling before capturing");
        PK_TRY(pk_dev_alloc(e, (void **)&e->samp, sizeof(pk_sampler_dev)));
        pk_sampler_dev h{};
        h.top_p = 1.0f;
        h.rep_penalty = 1.0f;
        e->samp_params = h;
        PK_HIP(hipMemcpyAsync(e->samp, &h, sizeof(h), hipMemcpyHostToDevice, e->stream));
        PK_HIP(hipStreamSynchronize(e->stream));
    }
    if (!e->samp_ws) {
        PK_CHECK(!e->capturing, PK_ERR_ARG, "sampling: call pk_set_sampling before capturing");
        PK_TRY(pk_dev_alloc(e, (void **)&e->samp_ws, sizeof(samp_ws)));
        PK_HIP(hipMemsetAsync(e->samp_ws, 0, sizeof(samp_ws), e->stream));
        PK_HIP(hipStreamSynchronize(e->stream));
    }
    if (vocab <= e->samp_cap) return PK_OK;
    PK_CHECK(!e->capturing, PK_ERR_ARG, "sampling: vocabulary %d beyond the scratch made before capture", vocab);
    PK_HIP(hipStreamSynchronize(e->stream));
    pk_drop_steps(e);                         // they address the old scratch
    pk_dev_free(e, e->samp_av);
    pk_dev_free(e, e->samp_ai);
    e->device_bytes -= (int64_t)e->samp_cap * 8;
    e->samp_av = nullptr;
    e->samp_ai = nullptr;
    e->samp_cap = 0;
    PK_TRY(pk_dev_alloc(e, (void **)&e->samp_av, (int64_t)vocab * 4));
    PK_TRY(pk_dev_alloc(e, (void **)&e->samp_ai, (int64_t)vocab * 4));
    e->samp_cap = vocab;
    return PK_OK;
}

// How a draw of the host's parameters runs: in one workgroup (greedy, small
// vocabularies, exact-sum draws, top-k beyond CAND), or over the device with
// or without a top-k.
enum { SAMP_ONE = 0, SAMP_TOPK = 1, SAMP_NUCLEUS = 2 };
constexpr int SAMP_MIN_V = 16384;         // (a share per CU would be under 64 entries)
static int samp_kind(const pk_sampler_dev &p, int vocab) {
    if (p.temperature < 1e-6f || vocab < SAMP_MIN_V) return SAMP_ONE;
    if (p.top_k > 0 && p.top_k < vocab) return p.top_k <= CAND ? SAMP_TOPK : SAMP_ONE;
    return p.fast_sums ? SAMP_ONE : SAMP_NUCLEUS;
}

int pk_launch_sample(pk_engine *e, float *logits, int vocab, pk_dstate *st, int32_t *out_toks, int out_cap,
                     const float *block_max, int n_blocks, bool write_back) {
    PK_CHECK(e->samp && vocab >= 1 && vocab <= e->samp_cap, PK_ERR_ARG,
             "sampling: vocabulary %d, scratch for %d", vocab, e->samp_cap);
    const int kind = samp_kind(e->samp_params, vocab);
    samp_ws *ws = (samp_ws *)e->samp_ws;
    if (kind != SAMP_ONE && e->samp_params.rep_penalty > 1.0f) {
        hipLaunchKernelGGL(k_samp_penalty, dim3(1), dim3(SNT), 0, e->stream, logits, vocab, e->samp, e->samp_ai);
        PK_HIP(hipGetLastError());
    }
    const dim3 grid((vocab + SH_T * SH_E - 1) / (SH_T * SH_E));
#define PK_SAMP(K, G, T, ...)                                                  \
    do {                                                                       \
        hipLaunchKernelGGL(K, dim3(G), dim3(T), 0, e->stream, __VA_ARGS__);    \
        PK_HIP(hipGetLastError());                                             \
    } while (0)
    if (kind == SAMP_NUCLEUS) {
        const bool cut = e->samp_params.top_p < 1.0f && e->samp_params.top_p > 0.0f;
        const int per = om_per(vocab), runs = om_runs(vocab);
        const dim3 waves((runs + SH_T / 64 - 1) / (SH_T / 64));
#define PK_SUM()                                                               \
    do {                                                                       \
        PK_SAMP(k_samp_part, waves, SH_T, logits, vocab, per, runs, ws);       \
        PK_SAMP(k_samp_moves, waves, SH_T, logits, vocab, per, runs, ws);      \
    } while (0)
        PK_SAMP(k_samp_scale, grid, SH_T, logits, vocab, e->samp, ws);
        PK_SAMP(k_samp_exp, grid, SH_T, logits, vocab, ws);
        PK_SUM();
        PK_SAMP(k_samp_sum, 1, 64, logits, vocab, per, runs, ws);
        PK_SAMP(k_samp_div, grid, SH_T, logits, vocab, ws, cut ? 1 : 2);
        if (cut) {
            PK_SAMP(k_samp_offsets, 1, SNT, ws);
            PK_SAMP(k_samp_place, grid, SH_T, logits, vocab, ws, e->samp_av);
            PK_SAMP(k_samp_sort, P_BINS, SH_T, ws, e->samp_av);
            PK_SAMP(k_samp_cut, 1, SNT, logits, vocab, e->samp, ws, e->samp_av);
            PK_SAMP(k_samp_zero, grid, SH_T, logits, vocab, ws);
            PK_SUM();
            PK_SAMP(k_samp_sum, 1, 64, logits, vocab, per, runs, ws);
            PK_SAMP(k_samp_div, grid, SH_T, logits, vocab, ws, 0);
        }
        PK_SUM();
        PK_SAMP(k_samp_draw, 1, SNT, logits, vocab, per, runs, e->samp, ws, st, out_toks, out_cap);
#undef PK_SUM
        return PK_OK;
    }
    if (kind == SAMP_TOPK) {
        PK_SAMP(k_samp_hist, grid, SH_T, logits, vocab, e->samp, ws);
        PK_SAMP(k_samp_gather, grid, SH_T, logits, vocab, e->samp, ws, write_back ? 1 : 0);
    }
    PK_SAMP(k_sample, 1, SNT, logits, vocab, e->samp, e->samp_av, e->samp_ai, st, out_toks, out_cap, block_max, n_blocks,
            write_back ? 1 : 0, kind == SAMP_TOPK ? ws : nullptr);
#undef PK_SAMP
    return PK_OK;
}

int pk_sample_seed_history(pk_engine *e, const int32_t *ids_dev, int n) {
    if (!e->samp_on || !(e->samp_params.rep_penalty > 1.0f) || n <= 0) return PK_OK;
    hipLaunchKernelGGL(k_seed_history, dim3(1), dim3(64), 0, e->stream, e->samp, ids_dev, n, e->c.vocab);
    PK_HIP(hipGetLastError());
    return PK_OK;
}

// Which of the captured steps serves these settings: a captured step's
// kernels read the values on the device, but not which kernels run.
static int step_key(const pk_sampler_dev &p, int vocab) {
    const int pen = p.rep_penalty > 1.0f, cut = p.top_p < 1.0f && p.top_p > 0.0f;
    // greedy without a penalty is the lm_head's own argmax (no draw, no history use)
    if (!(p.temperature >= 1e-6f) && !pen) return 0;
    static_assert(PK_STEPS == 8, "one workgroup, top-k, no top-k with and without a cut");
    switch (samp_kind(p, vocab)) {
    case SAMP_TOPK: return 2 + pen;
    case SAMP_NUCLEUS: return 4 + pen + 2 * cut;
    default: return 1;
    }
}

// Parameters into the device state; rng and history replaced only on reset
// (temperature .. top_k come before rng in the struct, so a short copy keeps them).
static int put_params(pk_engine *e, const pk_sampler_dev &p, bool reset) {
    PK_TRY(pk_sample_reserve(e, e->c.vocab > 0 ? e->c.vocab : 1));
    const size_t bytes = reset ? offsetof(pk_sampler_dev, history) : offsetof(pk_sampler_dev, rng);
    PK_HIP(hipMemcpyAsync(e->samp, &p, bytes, hipMemcpyHostToDevice, e->stream));
    PK_HIP(hipStreamSynchronize(e->stream));
    e->samp_params = p;
    e->step_key = step_key(p, e->c.vocab);
    e->samp_on = e->step_key != 0;
    return PK_OK;
}

extern "C" int pk_set_sampling(pk_engine *e, float temperature, float top_p, int top_k, float rep_penalty,
                               uint64_t seed) {
    PK_CHECK(e, PK_ERR_ARG, "null argument");
    PK_CHECK(!e->capturing, PK_ERR_ARG, "set_sampling: not available while capturing");
    pk_sampler_dev p{};
    p.temperature = temperature;
    p.top_p = top_p;
    p.top_k = top_k;
    p.rep_penalty = rep_penalty;
    p.rng = seed;
    p.history_len = 0;
    p.fast_sums = e->samp ? e->samp_params.fast_sums : 0;
    return put_params(e, p, true);
}

extern "C" int pk_set_sampling_fast_sums(pk_engine *e, int on) {
    PK_CHECK(e, PK_ERR_ARG, "null argument");
    PK_CHECK(!e->capturing, PK_ERR_ARG, "set_sampling_fast_sums: not available while capturing");
    PK_TRY(pk_sample_reserve(e, e->c.vocab > 0 ? e->c.vocab : 1));
    e->samp_params.fast_sums = on ? 1 : 0;
    e->step_key = step_key(e->samp_params, e->c.vocab);
    PK_HIP(hipMemcpyAsync((char *)e->samp + offsetof(pk_sampler_dev, fast_sums), &e->samp_params.fast_sums, 4,
                          hipMemcpyHostToDevice, e->stream));
    PK_HIP(hipStreamSynchronize(e->stream));
    return PK_OK;
}

extern "C" int pk_set_turn_sampling(pk_engine *e, float temperature, float top_p, int top_k) {
    PK_CHECK(e, PK_ERR_ARG, "null argument");
    PK_CHECK(!e->capturing, PK_ERR_ARG, "set_turn_sampling: not available while capturing");
    PK_TRY(pk_sample_reserve(e, e->c.vocab > 0 ? e->c.vocab : 1));
    pk_sampler_dev p = e->samp_params;
    // the TURN header's defensive clamp (picchio.c:2737-2743)
    if (temperature < 0.0f) temperature = 0.0f;
    if (temperature > 5.0f) temperature = 5.0f;
    if (top_p <= 0.0f || top_p > 1.0f) top_p = 1.0f;
    if (top_k < 0) top_k = 0;
    p.temperature = temperature;
    p.top_p = top_p;
    p.top_k = top_k;
    return put_params(e, p, false);
}

extern "C" int pk_reset_history(pk_engine *e) {
    PK_CHECK(e, PK_ERR_ARG, "null argument");
    PK_CHECK(!e->capturing, PK_ERR_ARG, "reset_history: not available while capturing");
    if (!e->samp) return PK_OK;
    static const int32_t zero = 0;
    PK_HIP(hipMemcpyAsync((char *)e->samp + offsetof(pk_sampler_dev, history_len), &zero, 4,
                          hipMemcpyHostToDevice, e->stream));
    PK_HIP(hipStreamSynchronize(e->stream));
    return PK_OK;
}

extern "C" int pk_sample_logits(pk_engine *e, float *logits_dev, int vocab, int32_t *tok_host) {
    PK_CHECK(e && logits_dev && tok_host, PK_ERR_ARG, "null argument");
    PK_CHECK(vocab >= 1, PK_ERR_ARG, "vocab %d", vocab);
    PK_CHECK(!e->capturing, PK_ERR_ARG, "sample_logits: host result; not available while capturing");
    PK_TRY(pk_sample_reserve(e, vocab));
    PK_TRY(pk_launch_sample(e, logits_dev, vocab, nullptr, nullptr, 0, nullptr, 0, true));
    int32_t last = 0;
    PK_HIP(hipMemcpyAsync(&last, (char *)e->samp + offsetof(pk_sampler_dev, last), 4, hipMemcpyDeviceToHost,
                          e->stream));
    PK_HIP(hipStreamSynchronize(e->stream));
    *tok_host = last;
    return PK_OK;
}

extern "C" int pk_sampler_state(pk_engine *e, uint64_t *rng, int32_t *history, int cap, int *history_len) {
    PK_CHECK(e && rng && history_len, PK_ERR_ARG, "null argument");
    PK_CHECK(!e->capturing, PK_ERR_ARG, "sampler_state: not available while capturing");
    PK_TRY(pk_sample_reserve(e, e->c.vocab > 0 ? e->c.vocab : 1));
    pk_sampler_dev *h = new pk_sampler_dev;
    hipError_t rc = hipMemcpyAsync(h, e->samp, sizeof(*h), hipMemcpyDeviceToHost, e->stream);
    if (rc == hipSuccess) rc = hipStreamSynchronize(e->stream);
    if (rc == hipSuccess) {
        *rng = h->rng;
        *history_len = h->history_len;
        if (history)
            for (int i = 0; i < h->history_len && i < cap; ++i) history[i] = h->history[i];
    }
    delete h;
    PK_HIP(rc);
    return PK_OK;
}
