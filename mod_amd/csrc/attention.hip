// Attention on the matrix cores in fp32: out = softmax(q k^T * scale) v for
// grouped-query heads, over all keys or causal, with an online softmax.
//
// The scores and the weighted sum are contractions, so they run on
// v_mfma_f32_32x32x2_f32: fp32 operands, products and sums, as the VALU loops
// this replaces (same inf / NaN behaviour), at twice the VALU's rate. Both are
// formed transposed: S^T = K Q^T and O^T = V^T P^T. A column of either is one
// (query, head) pair, held by lanes c and c + 32, so
//   - the softmax of a column is arithmetic inside a lane plus one exchange
//     between the two halves, and rescaling O^T is a multiply per register;
//   - accumulator register e of S^T (keys 8 (e / 4) + 4 h + e % 4 of the tile
//     for half h) is, after the exp, the B operand of step e of O^T: the keys of
//     that step are the ones the two halves hold, and V's rows are loaded to
//     match. The probabilities never leave their registers.
// The G query heads of a kv head are columns of the same tile, so K and V are
// read once for all of them.
//
// A workgroup owns 32 columns; its 4 waves take every 4th tile of 32 keys,
// loaded straight into registers in operand layout (32 KB of K and V per tile
// for 128 MFMAs of 64 cycles: 4 B per cycle and wave, far below what L2
// serves, so sharing tiles through LDS would buy nothing), the next K tile in
// flight during V's product, V during K's and the softmax, each in halves (all
// of both in flight spilled registers: 88 us against 72 in the first case
// below). The columns' q is in LDS. The waves' (max, sum, O) meet in LDS at
// the end. When there are too few column tiles
// for the CUs, the keys are split over workgroups as well and a second launch
// merges the partials. Steps of at most AT_VEC_COLS columns per kv head run on
// the VALU (attn_vec_kernel). Few rows over few keys have kernels of their own
// beside the callers (model_ops.hip, prefill.hip).
//
// Measured (MI355X; before: a workgroup per query row on the VALU, keys one by
// one): 777 queries and keys, 16 heads over 8, D 128: 909 -> 72 us; one query
// of 4 sequences over 2047 keys: 578 -> 27 us (18 on the VALU kernel); causal over 1021
// positions: 462 -> 57 us. Bound by the fp32 MFMA (35 us of it in the first)
// and by the softmax between its two products, which two waves per SIMD only
// partly cover. Error against 64 bits 3.1e-7 (was 5.2e-7) and 1.8e-7 (8.2e-7); with
// few keys see AT_FINE_KEYS.
#include "attention.hpp"
#include "wf_planes.hpp"

#include <algorithm>
#include <float.h>
#include <type_traits>

namespace pio {

typedef float at_f4 __attribute__((ext_vector_type(4)));
typedef float at_f2 __attribute__((ext_vector_type(2)));
typedef float at_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 at_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 at_h8 __attribute__((ext_vector_type(8)));

constexpr int AT_COLS = 32;    // (query, head) pairs per workgroup
constexpr int AT_KEYS = 32;    // keys per tile
constexpr int AT_WAVES = 4;
// Keys up to which a column tile's scores are summed in chains of 8 terms, added as
// a tree: with few keys their rounding is the larger part of the result's. Error
// against 64 bits (x 1e-7) at 2 / 16 / 32 / 64 / 96 keys of 128 dims: 0.61 / 1.24 /
// 1.52 / 1.62 / 1.68, and 0.75 / 1.50 / 1.82 / 1.94 / 2.00 in 4 chains, beside 0.62 /
// 1.24 / 1.52 / 1.89 / 2.18 of a kernel that adds a score's 128 products as a tree,
// which grows with the keys (5.9 at 1024; 4 chains 2.2). Costs 0.6 us (64 queries and
// keys), and all the prompt's tiles in 8 chains would cost 2 %.
constexpr int AT_FINE_KEYS = 96;
constexpr int AT_VEC_COLS = 4; // columns per kv head up to which the VALU kernel serves

struct AttnParams {
    AttnArgs a;
    int G, tiles;              // query heads per kv head; column tiles per (b, kv head)
    int splits, per_split;     // key tiles per split (a multiple of AT_WAVES)
    float* part_o;             // [splits][B * Hk * tiles * 32][D] when splits > 1
    float* part_ml;            // [splits][..][2]
};

template <int D>
constexpr size_t at_lds_bytes() { return (size_t)AT_WAVES * AT_COLS * (D + 4) * 4; }

// Vector types of a lane's loads: 16 bytes of a K row, D / 32 elements of a V row.
template <typename KT, int D> struct AtRaw;
template <> struct AtRaw<float, 128> { typedef at_f4 k, v; };
template <> struct AtRaw<float, 64> { typedef at_f4 k; typedef at_f2 v; };
template <> struct AtRaw<_Float16, 128> { typedef at_h8 k; typedef at_h4 v; };

// Dimension held by slot sl of a row (fp16 cache rows pair dims i and i + 64).
template <bool PAIR>
__device__ __forceinline__ int at_dim(int sl) { return PAIR ? (sl >> 1) + 64 * (sl & 1) : sl; }

// Slot of the first of the 4 steps in K group c of half h: a lane's 16-byte
// load covers one group of fp32 or two of fp16.
template <typename KT>
__device__ __forceinline__ int at_slot(int c, int h) {
    return sizeof(KT) == 4 ? 8 * c + 4 * h : 16 * (c >> 1) + 8 * h + 4 * (c & 1);
}

// 4 consecutive slots from sl of (row s of batch b, query head hd).
template <bool PAIR, bool CAUSAL>
__device__ __forceinline__ void at_store(const AttnArgs& a, int D, int b, int s, int hd, int sl, at_f4 v) {
    if constexpr (CAUSAL) {
        const int K = a.H * D;
        if constexpr (PAIR) {
            wf_put2(a.planes, s, hd * D + (sl >> 1), K, v[0], v[2]);
            wf_put2(a.planes, s, hd * D + (sl >> 1) + 64, K, v[1], v[3]);
        } else {
            wf_put4(a.planes, s, hd * D + sl, K, make_float4(v[0], v[1], v[2], v[3]));
        }
    } else {
        *(at_f4*)(a.out + b * a.o_b + (int64_t)s * a.o_s + hd * D + sl) = v;
    }
}

// A finished column's 4 slots from sl: r, the sum of exp(score - m) v over l, the
// sum of the weights; D / 4 consecutive lanes have one column. The first sum can
// leave the fp32 range where softmax(s) v does not (T keys with |v| above FLT_MAX / T),
// so a column with an inf or NaN among its outputs whose scores are in order
// (0 < l < inf) is formed again by its lanes alone, as softmax(s) v is written:
// the weights' sum, then normalised weights times v, over the keys that the column
// sees. (In a causal tile an inf or NaN in the value row of a later key meets the
// zero weights of earlier columns and makes them NaN: they come out right here.)
template <int D, typename KT, bool CAUSAL>
__device__ __forceinline__ at_f4 at_finish(const AttnArgs& a, int b, int g, int s, int hd, int sl, at_f4 r, float m,
                                           float l) {
    constexpr bool PAIR = sizeof(KT) == 2;
    constexpr int U = 4;                   // keys at a time
    bool odd = false;
#pragma unroll
    for (int j = 0; j < 4; j++) odd |= !(fabsf(r[j]) <= FLT_MAX);
    constexpr unsigned long long group = (1ull << (D / 4)) - 1;
    if (!(__ballot(odd) >> (threadIdx.x & 63 & ~(D / 4 - 1)) & group) || !(l > 0.f && l <= FLT_MAX)) return r;
    const int limit = CAUSAL ? a.pos0 + s + 1 : a.T;
    const float* qr = a.q + b * a.q_b + (int64_t)s * a.q_s + hd * D;
    const KT* kb = (const KT*)a.k + b * a.kv_b + g * a.kv_h + sl;
    const KT* vb = (const KT*)a.v + b * a.kv_b + g * a.kv_h + sl;
    float q[4], inv = 1.f;
#pragma unroll
    for (int j = 0; j < 4; j++) q[j] = qr[at_dim<PAIR>(sl + j)];
    for (int pass = 0; pass < 2; pass++) {
        float sum = 0.f;
        at_f4 o = {0.f, 0.f, 0.f, 0.f};
        for (int t0 = 0; t0 < limit; t0 += U) {
            float e[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const KT* kr = kb + (int64_t)min(t0 + u, limit - 1) * a.kv_t;
                e[u] = 0.f;
#pragma unroll
                for (int j = 0; j < 4; j++) e[u] = fmaf(q[j], (float)kr[j], e[u]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int x = D / 8; x >= 1; x >>= 1) e[u] += __shfl_xor(e[u], x, 64);
                e[u] = expf(e[u] * a.scale - m);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (t0 + u >= limit) break;
                if (pass == 0) {
                    sum += e[u];
                } else {
                    const KT* vr = vb + (int64_t)(t0 + u) * a.kv_t;
#pragma unroll
                    for (int j = 0; j < 4; j++) o[j] = fmaf(e[u] * inv, (float)vr[j], o[j]);
                }
            }
        }
        if (pass) return o;
        inv = 1.0f / sum;
    }
    return r;
}

template <int D, typename KT, bool CAUSAL>
__global__ __launch_bounds__(64 * AT_WAVES, 2) void attn_mfma_kernel(AttnParams p) {
    constexpr bool PAIR = sizeof(KT) == 2;
    constexpr int NT = D / 32;             // O^T tiles: row i of tile n is slot NT * i + n
    constexpr int NC = D / 8;              // K groups of 4 steps
    constexpr int OP = D + 4;              // LDS pitch of the merge (floats)
    extern __shared__ __attribute__((aligned(16))) float at_lds[];
    __shared__ float at_m[AT_WAVES][AT_COLS], at_l[AT_WAVES][AT_COLS];
    const AttnArgs& a = p.a;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;

    // kv heads fastest: with 8 of them each XCD's L2 holds one head's K and V
    int x = blockIdx.x;
    const int g = x % a.Hk;
    x /= a.Hk;
    const int b = x % a.B;
    int ct = x / a.B;
    if (CAUSAL) {
        // Later tiles see more keys. In dispatch order the first 256 workgroups
        // (one per CU) take tiles from the long end, the next 256 from the
        // short end, and so on, so that a CU's two have about the same sum.
        const int run = max(1, 256 / (a.B * a.Hk)), n = ct / run, r = (n >> 1) * run + ct - n * run;
        ct = n & 1 ? r : p.tiles - 1 - r;
    }
    const int ncols = a.S * p.G, c0 = ct * AT_COLS;
    const int last_s = (min(c0 + AT_COLS, ncols) - 1) / p.G;
    const int limit_all = CAUSAL ? a.pos0 + last_s + 1 : a.T;       // keys any column sees
    const int tiles_all = (limit_all + AT_KEYS - 1) / AT_KEYS;
    const int kt0 = blockIdx.y * p.per_split, kt1 = min(kt0 + p.per_split, tiles_all);

    // q of the columns -> LDS, in the order the S^T steps read it
    for (int i = tid; i < AT_COLS * (D / 4); i += 64 * AT_WAVES) {
        const int c = i / (D / 4), grp = i % (D / 4);              // group grp = 2 c4 + half
        const int cc = min(c0 + c, ncols - 1), s = cc / p.G, hd = g * p.G + cc - s * p.G;
        const float* qr = a.q + b * a.q_b + (int64_t)s * a.q_s + hd * D;
        const int sl = at_slot<KT>(grp >> 1, grp & 1);
        at_f4 v;
        if constexpr (PAIR) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = qr[at_dim<PAIR>(sl + e)];
        } else {
            v = *(const at_f4*)(qr + sl);
        }
        *(at_f4*)(at_lds + (grp * AT_COLS + c) * 4) = v;
    }
    __syncthreads();

    const KT* kb = (const KT*)a.k + b * a.kv_b + g * a.kv_h;
    const KT* vb = (const KT*)a.v + b * a.kv_b + g * a.kv_h;
    const int mycol = min(c0 + col, ncols - 1);
    const int limit = CAUSAL ? a.pos0 + mycol / p.G + 1 : a.T;

    at_v16f o[NT];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[n][e] = 0.f;
    float m = a.m_seed, l = 0.f;

    // A tile's K: 4 steps per group from the row of this lane's key; its V: the
    // rows of the 16 steps' keys, NT consecutive slots per lane. Raw bits, so
    // that fp16 is widened at its use and the loads stay in flight together.
    // Rows past the last key re-read it (their weights and V are zeroed below).
    typedef typename AtRaw<KT, D>::k at_kt;
    typedef typename AtRaw<KT, D>::v at_vt;
    constexpr int KL = D * (int)sizeof(KT) / 32;     // K loads of 16 bytes
    at_kt kr[KL];
    at_vt vr[16];
    const int k_lane = col * a.kv_t + h * (16 / (int)sizeof(KT));
    const int v_lane = 4 * h * a.kv_t + NT * col;
    auto load_k = [&](int kt, int half) {
        const int t0 = kt * AT_KEYS;
        const KT* r = t0 + AT_KEYS <= limit_all
                          ? kb + (int64_t)t0 * a.kv_t + k_lane
                          : kb + (int64_t)min(t0 + col, limit_all - 1) * a.kv_t + h * (16 / (int)sizeof(KT));
#pragma unroll
        for (int c = half * (KL / 2); c < (half + 1) * (KL / 2); c++)
            kr[c] = *(const at_kt*)(r + c * (32 / (int)sizeof(KT)));
    };
    auto load_v = [&](int kt, int half) {
        const int t0 = kt * AT_KEYS;
        if (t0 + AT_KEYS <= limit_all) {
            const KT* tb = vb + (int64_t)t0 * a.kv_t;
#pragma unroll
            for (int e = 8 * half; e < 8 * half + 8; e++)
                vr[e] = *(const at_vt*)(tb + (8 * (e >> 2) + (e & 3)) * a.kv_t + v_lane);
        } else {
#pragma unroll
            for (int e = 8 * half; e < 8 * half + 8; e++) {
                const int t = min(t0 + 8 * (e >> 2) + 4 * h + (e & 3), limit_all - 1);
                vr[e] = *(const at_vt*)(vb + (int64_t)t * a.kv_t + NT * col);
            }
        }
    };
    auto k_at = [&](int c, int e) {
        if constexpr (PAIR) return (float)kr[c >> 1][4 * (c & 1) + e];
        else return (float)kr[c][e];
    };

    // One chain of a score's terms: n groups of 8 from c.
    auto chain = [&](int c, int n) {
        at_v16f t;
#pragma unroll
        for (int e = 0; e < 16; e++) t[e] = 0.f;
#pragma unroll
        for (int i = c; i < c + n; i++) {
            const at_f4 qv = *(const at_f4*)(at_lds + ((2 * i + h) * AT_COLS + col) * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) t = __builtin_amdgcn_mfma_f32_32x32x2f32(k_at(i, e), qv[e], t, 0, 0, 0);
        }
        return t;
    };
    // (causal: of 16 terms, as its 8 partial sums of a score were before)
    const bool fine = limit_all <= AT_FINE_KEYS;
    auto scores_fine = [&] {
        constexpr int CG = CAUSAL ? 2 : 1, PAIRS = NC / CG / 2, LV = PAIRS == 8 ? 3 : 2;
        at_v16f level[LV], sum;
#pragma unroll
        for (int p2 = 0; p2 < PAIRS; p2++) {
            sum = chain(2 * p2 * CG, CG);
            sum += chain((2 * p2 + 1) * CG, CG);
#pragma unroll
            for (int i = 0; i < LV; i++) {
                asm volatile("" : "+v"(sum));   // formed here: sunk past the branches, all chains would be held
                if (!(p2 >> i & 1)) {
                    level[i] = sum;
                    break;
                }
                sum += level[i];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return sum;
    };
    // 4 chains: half the rounding of one
    auto scores = [&] {
        at_v16f s = chain(0, NC / 4);
#pragma unroll
        for (int ch = 1; ch < 4; ch++) s += chain(ch * (NC / 4), NC / 4);
        return s;
    };

    int kt = kt0 + w;
    if (kt < kt1) {
        load_k(kt, 0);
        load_k(kt, 1);
    }
    for (; kt < kt1; kt += AT_WAVES) {
        load_v(kt, 0);
        __builtin_amdgcn_sched_barrier(0);
        at_v16f s = fine ? scores_fine() : scores();
        __builtin_amdgcn_sched_barrier(0);
        load_v(kt, 1);
        __builtin_amdgcn_sched_barrier(0);
        const int t0 = kt * AT_KEYS;
        const bool more = kt + AT_WAVES < kt1;
        // wave-uniform: some key of the tile is past some column's last one
        const bool edge = t0 + AT_KEYS > (CAUSAL ? a.pos0 + c0 / p.G + 1 : a.T);
        float mt = m;
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] *= a.scale;
        if (edge) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int t = t0 + 8 * (e >> 2) + 4 * h + (e & 3);
                if (t < limit) mt = fmaxf(mt, s[e]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) mt = fmaxf(mt, s[e]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float corr = expf(m - mt);
        float sum[16];                     // added as a tree
#pragma unroll
        for (int e = 0; e < 16; e++) {
            s[e] = expf(s[e] - mt);
            if (edge && t0 + 8 * (e >> 2) + 4 * h + (e & 3) >= limit) s[e] = 0.f;
            sum[e] = s[e];
        }
#pragma unroll
        for (int n = 8; n >= 1; n >>= 1)
#pragma unroll
            for (int e = 0; e < n; e++) sum[e] += sum[e + n];
        l = l * corr + sum[0];
        if (__any(mt != m)) {
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[n][e] *= corr;
        }
        m = mt;
        // a key past the last one: its weight is zero, and what is read in its
        // place must not be inf or NaN. (A causal tile's later keys are rows of
        // this batch: see at_finish.)
        auto zero_v = [&](int e) {
            if (edge && t0 + 8 * (e >> 2) + 4 * h + (e & 3) >= limit_all)
#pragma unroll
                for (int n = 0; n < NT; n++) vr[e][n] = 0;
        };
#pragma unroll
        for (int e = 0; e < 8; e++) zero_v(e);
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
            for (int n = 0; n < NT; n++) o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32((float)vr[e][n], s[e], o[n], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_k(kt + AT_WAVES, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 8; e < 16; e++) zero_v(e);
#pragma unroll
        for (int e = 8; e < 16; e++)
#pragma unroll
            for (int n = 0; n < NT; n++) o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32((float)vr[e][n], s[e], o[n], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_k(kt + AT_WAVES, 1);
    }

    // the waves' columns meet in LDS: common maximum, scaled sums
    l += __shfl_xor(l, 32, 64);
    if (h == 0) {
        at_m[w][col] = m;
        at_l[w][col] = l;
    }
    __syncthreads();   // and every wave is done with q
    float mx = at_m[0][col];
#pragma unroll
    for (int i = 1; i < AT_WAVES; i++) mx = fmaxf(mx, at_m[i][col]);
    const float f = expf(m - mx);
    float* ob = at_lds + (w * AT_COLS + col) * OP;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int i = 8 * (e >> 2) + 4 * h + (e & 3);
#pragma unroll
        for (int n = 0; n < NT; n++) ob[NT * i + n] = o[n][e] * f;
    }
    __syncthreads();
    for (int i = tid; i < AT_COLS * (D / 4); i += 64 * AT_WAVES) {
        const int c = i / (D / 4), sl = (i % (D / 4)) * 4;
        if (c0 + c >= ncols) continue;
        at_f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < AT_WAVES; k++) v += *(const at_f4*)(at_lds + (k * AT_COLS + c) * OP + sl);
        float cm = at_m[0][c], cl = 0.f;
#pragma unroll
        for (int k = 1; k < AT_WAVES; k++) cm = fmaxf(cm, at_m[k][c]);
#pragma unroll
        for (int k = 0; k < AT_WAVES; k++) cl += at_l[k][c] * expf(at_m[k][c] - cm);
        if (p.splits > 1) {
            const int64_t row = ((int64_t)blockIdx.y * a.B + b) * a.Hk + g;
            const int64_t at = row * p.tiles * AT_COLS + c0 + c;
            *(at_f4*)(p.part_o + at * D + sl) = v;
            if (sl == 0) {
                p.part_ml[2 * at] = cm;
                p.part_ml[2 * at + 1] = cl;
            }
            continue;
        }
        const int s = (c0 + c) / p.G, hd = g * p.G + (c0 + c) - s * p.G;
        const at_f4 r = fine ? v / cl : v * (1.0f / cl);   // a rounding less where they are few
        at_store<PAIR, CAUSAL>(a, D, b, s, hd, sl, at_finish<D, KT, CAUSAL>(a, b, g, s, hd, sl, r, cm, cl));
    }
}

// Few columns (a decode step): the same split of keys over waves and
// workgroups, on the VALU. A launch is bound by reading K and V, and the MFMAs
// above would spend 32 columns' time on them: 4 sequences x 2047 keys, 2 heads
// per kv head, 20.3 us (8 of them MFMAs) against 15.1 here (4.4 TB/s); 16 x 4000
// keys run at 5.3 TB/s. Lane (i, h) holds
// half h of key i's K row and slots NT i .. of half of the tile's V rows, loaded
// as above; a score is summed over the two halves, the weights go through LDS
// to the lanes of the V rows. K and V of the next tile are loaded as soon as this
// one's registers are free.
template <int D, int C>
__global__ __launch_bounds__(64 * AT_WAVES, 2) void attn_vec_kernel(AttnParams p) {
    constexpr int NT = D / 32, KL = D / 8;
    typedef typename AtRaw<float, D>::v at_vt;
    __shared__ __attribute__((aligned(16))) float qs[C][D], ps[AT_WAVES][C][AT_KEYS], ob[AT_WAVES][C][D];
    __shared__ float at_m[AT_WAVES][C], at_l[AT_WAVES][C];
    const AttnArgs& a = p.a;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 31, h = lane >> 5;
    const int g = blockIdx.x % a.Hk, b = blockIdx.x / a.Hk, ncols = a.S * p.G;
    const int kt1 = min((int)(blockIdx.y + 1) * p.per_split, (a.T + AT_KEYS - 1) / AT_KEYS);
    const float* kb = (const float*)a.k + b * a.kv_b + g * a.kv_h;
    const float* vb = (const float*)a.v + b * a.kv_b + g * a.kv_h;
    at_f4 kr[KL];
    at_vt vr[16];
    auto load_k = [&](int kt) {   // rows past the last key re-read it
        const float* r = kb + (int64_t)min(kt * AT_KEYS + i, a.T - 1) * a.kv_t + 4 * h;
#pragma unroll
        for (int c = 0; c < KL; c++) kr[c] = *(const at_f4*)(r + 8 * c);
    };
    auto load_v = [&](int kt) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int t = min(kt * AT_KEYS + 8 * (e >> 2) + 4 * h + (e & 3), a.T - 1);
            vr[e] = *(const at_vt*)(vb + (int64_t)t * a.kv_t + NT * i);
        }
    };
    int kt = blockIdx.y * p.per_split + w;
    if (kt < kt1) {
        load_k(kt);
        load_v(kt);
    }
    for (int e = tid; e < C * (D / 4); e += 64 * AT_WAVES) {
        const int c = min(e / (D / 4), ncols - 1), sl = (e % (D / 4)) * 4, s = c / p.G, hd = g * p.G + c - s * p.G;
        *(at_f4*)&qs[e / (D / 4)][sl] = *(const at_f4*)(a.q + b * a.q_b + (int64_t)s * a.q_s + hd * D + sl);
    }
    __syncthreads();
    float m[C], l[C], o[C][NT];
#pragma unroll
    for (int c = 0; c < C; c++) {
        m[c] = a.m_seed;
        l[c] = 0.f;
#pragma unroll
        for (int n = 0; n < NT; n++) o[c][n] = 0.f;
    }
    for (; kt < kt1; kt += AT_WAVES) {
        const int t0 = kt * AT_KEYS;
        const bool live = t0 + i < a.T;
        // q stays in LDS: hoisted out of the loop it would fill the registers
        int qh = h;
        asm volatile("" : "+v"(qh));
        float s[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            at_f4 d[KL / 8];               // chains of 8 terms, added as a tree
#pragma unroll
            for (int k = 0; k < KL; k++) {
                const at_f4 qv = ((const at_f4*)&qs[c][8 * k])[qh];
                at_f4& dk = d[k / 8];
#pragma unroll
                for (int e = 0; e < 4; e++) dk[e] = k % 8 ? fmaf(kr[k][e], qv[e], dk[e]) : kr[k][e] * qv[e];
                if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // not all of q's reads at once
            }
            if (KL == 16) d[0] += d[KL / 8 - 1];
            s[c] = (d[0][0] + d[0][1]) + (d[0][2] + d[0][3]);
            asm volatile("" : "+v"(s[c]));   // formed here: sunk past the next loads, K would be held twice
        }
        if (kt + AT_WAVES < kt1) load_k(kt + AT_WAVES);
        if (t0 + AT_KEYS > a.T) {
            // a key past the last one: zero weight, and nothing inf or NaN in its row
#pragma unroll
            for (int e = 0; e < 16; e++)
                if (t0 + 8 * (e >> 2) + 4 * h + (e & 3) >= a.T)
#pragma unroll
                    for (int n = 0; n < NT; n++) vr[e][n] = 0.f;
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            const float v = (s[c] + __shfl_xor(s[c], 32, 64)) * a.scale;
            float mt = live ? v : a.m_seed;
            mt = fmaxf(mt, dpp<DPP_XOR1>(mt));
            mt = fmaxf(mt, dpp<DPP_XOR2>(mt));
            mt = fmaxf(mt, dpp<DPP_HMIRROR>(mt));
            mt = fmaxf(mt, dpp<DPP_MIRROR>(mt));
            mt = fmaxf(m[c], fmaxf(rlane(mt, 0), rlane(mt, 16)));
            const float pr = live ? expf(v - mt) : 0.f, corr = expf(m[c] - mt);
            l[c] = l[c] * corr + pr;
#pragma unroll
            for (int n = 0; n < NT; n++) o[c][n] *= corr;
            m[c] = mt;
            if (h == 0) ps[w][c][i] = pr;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                const at_f4 pr = *(const at_f4*)&ps[w][c][2 * e + 4 * h];
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int n = 0; n < NT; n++) o[c][n] = fmaf(pr[r], vr[e + r][n], o[c][n]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int n = 0; n < NT; n++) asm volatile("" : "+v"(o[c][n]));   // as above, for V
        if (kt + AT_WAVES < kt1) load_v(kt + AT_WAVES);
    }
#pragma unroll
    for (int c = 0; c < C; c++) {
        const float ls = wsum(l[c]) * 0.5f;   // every key's weight is in both halves
        if (lane == 0) {
            at_m[w][c] = m[c];
            at_l[w][c] = ls;
        }
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const float t = o[c][n] + __shfl_xor(o[c][n], 32, 64);
            if (h == 0) ob[w][c][NT * i + n] = t;
        }
    }
    __syncthreads();
    for (int e = tid; e < C * (D / 4); e += 64 * AT_WAVES) {
        const int c = e / (D / 4), sl = (e % (D / 4)) * 4;
        if (c >= ncols) continue;
        float cm = at_m[0][c], cl = 0.f;
#pragma unroll
        for (int k = 1; k < AT_WAVES; k++) cm = fmaxf(cm, at_m[k][c]);
        at_f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < AT_WAVES; k++) {
            const float f = expf(at_m[k][c] - cm);
            cl += at_l[k][c] * f;
            v += *(const at_f4*)&ob[k][c][sl] * f;
        }
        const int s = c / p.G;
        if (p.splits > 1) {
            const int64_t at = ((int64_t)blockIdx.y * a.B * a.Hk + blockIdx.x) * p.tiles * AT_COLS + c;
            *(at_f4*)(p.part_o + at * D + sl) = v;
            if (sl == 0) {
                p.part_ml[2 * at] = cm;
                p.part_ml[2 * at + 1] = cl;
            }
        } else {
            const int hd = g * p.G + c - s * p.G;
            at_store<false, false>(a, D, b, s, hd, sl, at_finish<D, float, false>(a, b, g, s, hd, sl, v / cl, cm, cl));
        }
    }
}

// One column per block: the key splits' (max, sum, O) merged. Thread group z of
// 256 / (D / 4) takes every such split, all loads of one in flight together (one
// thread per 4 slots walking the splits in turn took 8 us for 16 of them).
template <int D, bool PAIR, bool CAUSAL>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnParams p) {
    constexpr int TPC = D / 4, Z = 256 / TPC;
    __shared__ __attribute__((aligned(16))) float so[Z][D];
    __shared__ float sm[Z], sl_[Z];
    const AttnArgs& a = p.a;
    const int ncols = a.S * p.G;
    const int bg = blockIdx.x / ncols, c = blockIdx.x - bg * ncols, b = bg / a.Hk, g = bg - b * a.Hk;
    const int zg = threadIdx.x / TPC, sl = (threadIdx.x % TPC) * 4;
    const int64_t step = (int64_t)a.B * a.Hk * p.tiles * AT_COLS, at = (int64_t)bg * p.tiles * AT_COLS + c;
    float m = -FLT_MAX, l = 0.f;
    at_f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int z = zg; z < p.splits; z += Z) {
        const float zm = p.part_ml[2 * (at + z * step)], zl = p.part_ml[2 * (at + z * step) + 1];
        const at_f4 zo = *(const at_f4*)(p.part_o + (at + z * step) * D + sl);
        const float nm = fmaxf(m, zm), f = expf(m - nm), fz = expf(zm - nm);
        l = l * f + zl * fz;
        v = v * f + zo * fz;
        m = nm;
    }
    *(at_f4*)&so[zg][sl] = v;
    if (sl == 0) {
        sm[zg] = m;
        sl_[zg] = l;
    }
    __syncthreads();
    if (zg) return;
    const int nz = min(Z, p.splits);
    float mx = sm[0];
    for (int z = 1; z < nz; z++) mx = fmaxf(mx, sm[z]);
    l = 0.f;
    v = at_f4{0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < nz; z++) {
        const float f = expf(sm[z] - mx);
        l += sl_[z] * f;
        v += *(const at_f4*)&so[z][sl] * f;
    }
    const int s = c / p.G, hd = g * p.G + c - s * p.G;
    typedef typename std::conditional<PAIR, _Float16, float>::type KT;
    at_store<PAIR, CAUSAL>(a, D, b, s, hd, sl, at_finish<D, KT, CAUSAL>(a, b, g, s, hd, sl, v * (1.0f / l), mx, l));
}

bool attn_mfma_supported(const AttnArgs& a) {
    // causal: the decoder's prompt (head_dim 128, planes out); fp16 keys only there
    if (a.D != 128 && !(a.D == 64 && !a.causal)) return false;
    if (a.kv16 && !a.causal) return false;
    if (a.H % a.Hk || a.kv_t >= 1 << 25 || a.q_s % 4 || a.o_s % 4 || a.q_b % 4 || a.o_b % 4 || a.kv_t % 8 || a.kv_h % 8 || a.kv_b % 8)
        return false;
    return aligned16(a.q) && aligned16(a.k) && aligned16(a.v) && aligned16(a.out) && aligned16(a.planes);
}

template <int D, bool PAIR, bool CAUSAL>
static int attn_merge(const AttnParams& p, hipStream_t st) {
    if (p.splits == 1) return PIO_OK;
    const AttnArgs& a = p.a;
    attn_merge_kernel<D, PAIR, CAUSAL><<<(unsigned)((int64_t)a.B * a.Hk * a.S * p.G), 256, 0, st>>>(p);
    PIO_LAUNCHED();
    return PIO_OK;
}

template <int D, typename KT, bool CAUSAL>
static int attn_launch(const AttnParams& p, hipStream_t st) {
    const AttnArgs& a = p.a;
    const size_t lds = at_lds_bytes<D>();
    const dim3 grid((unsigned)((int64_t)p.tiles * a.B * a.Hk), p.splits);
    PIO_TRY((allow_lds<attn_mfma_kernel<D, KT, CAUSAL>>(lds)));
    attn_mfma_kernel<D, KT, CAUSAL><<<grid, 64 * AT_WAVES, lds, st>>>(p);
    PIO_LAUNCHED();
    return attn_merge<D, sizeof(KT) == 2, CAUSAL>(p, st);
}

template <int D>
static int attn_vec_launch(const AttnParams& p, hipStream_t st) {
    const AttnArgs& a = p.a;
    const dim3 grid(a.B * a.Hk, p.splits);
    const int cols = a.S * p.G;
    if (cols == 1) attn_vec_kernel<D, 1><<<grid, 64 * AT_WAVES, 0, st>>>(p);
    else if (cols == 2) attn_vec_kernel<D, 2><<<grid, 64 * AT_WAVES, 0, st>>>(p);
    else attn_vec_kernel<D, AT_VEC_COLS><<<grid, 64 * AT_WAVES, 0, st>>>(p);
    PIO_LAUNCHED();
    return attn_merge<D, false, false>(p, st);
}

int attn_mfma(const AttnArgs& a, hipStream_t st) {
    PIO_REQUIRE(a.B > 0 && a.S > 0 && a.T > 0 && a.Hk > 0 && (a.causal ? a.planes != nullptr : a.out != nullptr) &&
                    attn_mfma_supported(a),
                "attn_mfma: bad operands");
    AttnParams p{};
    p.a = a;
    p.G = a.H / a.Hk;
    const int64_t ncols = (int64_t)a.S * p.G;
    p.tiles = ceil_div(ncols, AT_COLS);
    const int64_t wgs = (int64_t)p.tiles * a.B * a.Hk;
    // Key splits while the workgroups stay within two per CU (what the
    // registers and LDS hold) and each keeps a tile for every wave.
    const int kt = ceil_div(a.T, AT_KEYS);
    int splits = (int)std::max<int64_t>(1, std::min<int64_t>(512 / std::max<int64_t>(wgs, 1), kt / AT_WAVES));
    p.per_split = ceil_div(ceil_div(kt, splits), AT_WAVES) * AT_WAVES;
    p.splits = ceil_div(kt, p.per_split);
    Scratch ws;
    if (p.splits > 1) {
        const size_t cols = (size_t)p.splits * wgs * AT_COLS;
        PIO_TRY(ws.get(cols * (a.D + 2) * sizeof(float), st));
        p.part_o = (float*)ws.ptr;
        p.part_ml = p.part_o + cols * a.D;
    }
    if (a.causal) return a.kv16 ? attn_launch<128, _Float16, true>(p, st) : attn_launch<128, float, true>(p, st);
    // measured at T = 1000, 8 kv heads: 8 columns 17.7 us here and 14.3 on the MFMAs
    if (ncols <= AT_VEC_COLS) return a.D == 128 ? attn_vec_launch<128>(p, st) : attn_vec_launch<64>(p, st);
    return a.D == 128 ? attn_launch<128, float, false>(p, st) : attn_launch<64, float, false>(p, st);
}

}  // namespace pio
