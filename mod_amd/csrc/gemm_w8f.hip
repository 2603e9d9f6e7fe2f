// W8 linear on the matrix cores for many activation rows (prefill, large M):
//   y[m,n] = s_w[n] * sum_k x[m,k] * float(W[n,k]) (+ bias[n]) (+ y[m,n])
// W int8 [N,K], x fp32 or fp16 [M,K], y fp32 or fp16 [M,N]. This is the same
// contract as the decode GEMV (gemv.hip), whose FMA kernels spend M fp32 FMAs
// per weight byte and re-stream W for every few rows. Here every weight byte
// is read once per launch from HBM, and the tiles are dealt to the XCDs so that
// one XCD's tiles share weight panels through its L2.
//
// Exactness. An int8 weight is exact in bf16 and in fp16. fp16 x is used as
// it is (v_mfma_f32_32x32x16_f16). fp32 x is split exactly into three bf16
// parts (wf_planes.hpp) and multiplied on v_mfma_f32_32x32x16_bf16. Every
// product of a part and a weight is exact in fp32, so, as in an fp32 GEMV, only
// the fp32 accumulation rounds (in another order).
//
// Two kernels. gemm_w8f_kernel takes x as it is (fp16, and smaller fp32
// products) and splits it on the way to LDS. gemm_w8p_kernel takes planes, x
// split beforehand: by the prompt's own kernels, which write their outputs so,
// or by a pass of its own for larger fp32 products.
//
// gemm_w8f_kernel: per K step of 64 elements each thread loads 16 x values and
// 16 weights of one row (registers, one step ahead), converts them and writes
// them to an LDS stage; rows are 128 B (64 two-byte elements) with the 16-byte
// chunks XOR-swizzled by row pair (chunk c of row r at c ^ ((r >> 1) & 7)), so
// the MFMA operand reads (16 consecutive rows per quarter wave, one chunk) are
// conflict-free. Two stages, one barrier per step. Tiles of 128 x 128 (each
// wave 2 x 2 MFMA tiles of 32 x 32, so each fragment read feeds two MFMAs)
// when they still give every CU a tile, else 64 x 64 (one MFMA tile per wave);
// when those leave CUs without two blocks, K is split and a reduce launch sums
// the fp32 partials in slice order.
#include "gemm_core.hpp"
#include "wf_planes.hpp"

#include <algorithm>
#include <type_traits>

namespace pio {

typedef __bf16 wf_bf8 __attribute__((ext_vector_type(8)));
typedef _Float16 wf_h8 __attribute__((ext_vector_type(8)));
typedef float wf_v16f __attribute__((ext_vector_type(16)));
typedef int wf_v4i __attribute__((ext_vector_type(4)));
typedef float wf_f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const wf_v4i wf_gv4i;
typedef __attribute__((address_space(1))) const wf_f4 wf_gf4;

constexpr int WF_BK = 64;
constexpr int WF_ROW = WF_BK * 2;   // LDS bytes per tile row of a step

enum { WF_STORE = 0, WF_RESID = 1, WF_PARTIAL = 2, WF_SWIGLU = 3 };   // RESID, SWIGLU: planes kernel

struct W8fParams {
    const void* x;
    const int8_t* w;
    const float* s_w;
    const float* bias;
    void* y;            // output, or the fp32 partials [splits][M][N] (WF_PARTIAL)
    int M, N, K;        // K: the whole reduction length
    int ks;             // K elements per split (a multiple of WF_BK)
    int m_tiles, n_tiles, per_xcd;
};

__device__ __forceinline__ int wf_swz(int r, int c) { return r * WF_ROW + ((c ^ ((r >> 1) & 7)) << 4); }

// 4 int8 weights (a dword) as 4 two-byte MFMA operands: bf16 for the fp32-x
// path (the high half of the exact fp32 value), fp16 otherwise.
template <int NL>
__device__ __forceinline__ void wf_widen4(int u, uint32_t& lo, uint32_t& hi) {
    float f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) f[i] = (float)(int8_t)(u >> (8 * i));
    if constexpr (NL == 3) {
        lo = __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u);
        hi = __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u);
    } else {
        lo = (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)f[0]) |
             (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)f[1]) << 16;
        hi = (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)f[2]) |
             (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)f[3]) << 16;
    }
}
template <int NL>
__device__ __forceinline__ void wf_widen(wf_v4i w, uint32_t (&o)[8]) {
#pragma unroll
    for (int d = 0; d < 4; d++) wf_widen4<NL>(w[d], o[2 * d], o[2 * d + 1]);
}

// One output: the unscaled partial of K slice blockIdx.y, or the scaled value
// (+ bias) stored or added to y.
template <typename YT, int EPI>
__device__ __forceinline__ void wf_put(void* y, int64_t ldy, int M, int N, int m, int n, float v, float sw,
                                       const float* bias, float bn) {
    if constexpr (EPI == WF_PARTIAL) {
        ((float*)y)[((int64_t)blockIdx.y * M + m) * N + n] = v;
    } else {
        v = v * sw;
        if (bias) v += bn;
        YT* yp = (YT*)y + (int64_t)m * ldy + n;
        if constexpr (EPI == WF_RESID) v += to_f32<YT>(*yp);
        *yp = from_f32<YT>(v);
    }
}

template <typename XT> struct WfXRegs;
template <> struct WfXRegs<float> { wf_f4 v[4]; };      // 16 fp32
template <> struct WfXRegs<_Float16> { wf_v4i v[2]; };  // 16 fp16

// Block tile BM x BN = 64 TM x 64 TN: 2 x 2 waves, each owning TM x TN MFMA
// tiles of 32 x 32 (a fragment read from LDS then feeds TN or TM MFMAs).
template <int NL, typename XT, typename YT, int EPI, int TM, int TN>
__global__ __launch_bounds__(256) void gemm_w8f_kernel(W8fParams p) {
    static_assert((NL == 3) == std::is_same<XT, float>::value, "three bf16 parts for fp32 x, one for fp16");
    static_assert(EPI == WF_STORE || EPI == WF_PARTIAL, "a residual is added by the planes kernel only");
    extern __shared__ __attribute__((aligned(16))) int8_t wf_lds[];
    constexpr int BM = 64 * TM, BN = 64 * TN;
    constexpr int XB = BM * WF_ROW;                    // one part's x tile
    constexpr int STAGE = NL * XB + BN * WF_ROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // block b runs on XCD b % 8: each XCD takes a contiguous run of tiles,
    // M-fastest, so consecutive tiles of an XCD share a weight panel
    const int b = blockIdx.x;
    const int t = (b & 7) * p.per_xcd + (b >> 3);
    if (t >= p.m_tiles * p.n_tiles) return;
    const int nt = t / p.m_tiles, mt = t - nt * p.m_tiles;
    const int m0 = mt * BM, n0 = nt * BN;
    const int64_t kb = (int64_t)blockIdx.y * p.ks;
    const int klen = (int)min((int64_t)p.ks, (int64_t)p.K - kb);
    const int nk = (klen + WF_BK - 1) / WF_BK;

    // the epilogue's scales and biases first (clamped: loaded with no branch)
    const int col = lane & 31, h = lane >> 5;
    float sw[TN], bn[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int nc = min(n0 + 32 * TN * wn + 32 * j + col, p.N - 1);
        sw[j] = EPI == WF_PARTIAL ? 0.f : p.s_w[nc];
        bn[j] = (EPI != WF_PARTIAL && p.bias) ? p.bias[nc] : 0.f;
    }

    // loads: thread -> rows r + 64 i of the tile, elements 16 q .. 16 q + 15 of the step
    const int r = tid >> 2, q = tid & 3;
    const XT* xsrc[TM];
    const int8_t* wsrc[TN];
#pragma unroll
    for (int i = 0; i < TM; i++) xsrc[i] = (const XT*)p.x + (int64_t)min(m0 + r + 64 * i, p.M - 1) * p.K + kb + 16 * q;
#pragma unroll
    for (int j = 0; j < TN; j++) wsrc[j] = p.w + (int64_t)min(n0 + r + 64 * j, p.N - 1) * p.K + kb + 16 * q;
    WfXRegs<XT> xr[TM];
    wf_v4i wr[TN];
    auto gload = [&](int kk) {
        // K % 16 == 0: a thread's 16 elements are all inside or all past the end
        const bool in = kk + 16 * q < klen;
        const int off = in ? kk : 0;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if constexpr (std::is_same<XT, float>::value) {
#pragma unroll
                for (int u = 0; u < 4; u++) xr[i].v[u] = *(wf_gf4*)(xsrc[i] + off + 4 * u);
                if (!in)
#pragma unroll
                    for (int u = 0; u < 4; u++) xr[i].v[u] = wf_f4{0.f, 0.f, 0.f, 0.f};
            } else {
#pragma unroll
                for (int u = 0; u < 2; u++) xr[i].v[u] = *(wf_gv4i*)(xsrc[i] + off + 8 * u);
                if (!in)
#pragma unroll
                    for (int u = 0; u < 2; u++) xr[i].v[u] = wf_v4i{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            wr[j] = *(wf_gv4i*)(wsrc[j] + off);
            if (!in) wr[j] = wf_v4i{0, 0, 0, 0};
        }
    };
    auto sstore = [&](int buf) {
        int8_t* st = wf_lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int c0 = wf_swz(r + 64 * i, 2 * q), c1 = wf_swz(r + 64 * i, 2 * q + 1);
            if constexpr (NL == 3) {
                int pt[3][8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    wf_split3_pair(xr[i].v[u >> 1][2 * (u & 1)], xr[i].v[u >> 1][2 * (u & 1) + 1], pt[0][u], pt[1][u],
                                   pt[2][u]);
#pragma unroll
                for (int L = 0; L < 3; L++) {
                    *(wf_v4i*)(st + L * XB + c0) = wf_v4i{pt[L][0], pt[L][1], pt[L][2], pt[L][3]};
                    *(wf_v4i*)(st + L * XB + c1) = wf_v4i{pt[L][4], pt[L][5], pt[L][6], pt[L][7]};
                }
            } else {
                *(wf_v4i*)(st + c0) = xr[i].v[0];
                *(wf_v4i*)(st + c1) = xr[i].v[1];
            }
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int c0 = wf_swz(r + 64 * j, 2 * q), c1 = wf_swz(r + 64 * j, 2 * q + 1);
            uint32_t o[8];
            wf_widen<NL>(wr[j], o);
            *(wf_v4i*)(st + NL * XB + c0) = wf_v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
            *(wf_v4i*)(st + NL * XB + c1) = wf_v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
        }
    };

    wf_v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
    gload(0);
    sstore(0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < nk) gload((kt + 1) * WF_BK);
        const int8_t* st = wf_lds + cur * STAGE;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int c = 2 * ks + h;   // elements 16 ks + 8 h .. + 8 of the step
            wf_v4i bw[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) bw[j] = *(const wf_v4i*)(st + NL * XB + wf_swz(32 * TN * wn + 32 * j + col, c));
            if constexpr (NL == 3) {
                // the low part first: the small products meet the smaller sums
#pragma unroll
                for (int L = 2; L >= 0; L--)
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const wf_v4i a = *(const wf_v4i*)(st + L * XB + wf_swz(32 * TM * wm + 32 * i + col, c));
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                __builtin_bit_cast(wf_bf8, a), __builtin_bit_cast(wf_bf8, bw[j]), acc[i][j], 0, 0, 0);
                    }
            } else {
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const wf_v4i a = *(const wf_v4i*)(st + wf_swz(32 * TM * wm + 32 * i + col, c));
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(wf_h8, a), __builtin_bit_cast(wf_h8, bw[j]), acc[i][j], 0, 0, 0);
                }
            }
        }
        if (kt + 1 < nk) sstore(cur ^ 1);
        __syncthreads();
    }

    // accumulator: element e of lane l is row 8 (e / 4) + 4 (l / 32) + e % 4 of
    // MFMA tile (i, j), column l % 32
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + 32 * TN * wn + 32 * j + col;
        if (n >= p.N) continue;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int m = m0 + 32 * TM * wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
                if (m >= p.M) continue;
                wf_put<YT, EPI>(p.y, p.N, p.M, p.N, m, n, acc[i][j][e], sw[j], p.bias, bn[j]);
            }
    }
}

// ---- planes ------------------------------------------------------------------
// The same linear on x split beforehand (wf_planes.hpp), so that the MFMA loop
// has no splitting in it: a step's time was the sum of its MFMA and its VALU
// cycles, with one and with two waves per SIMD, and splitting every x value once
// per 32 TN columns made the second as large as the first (48 MFMAs of a wave:
// 2.0 us split in the loop with every wait a drain, 1.5 us pipelined, 0.87 us
// from planes; 0.7 is the MFMAs alone).
// A wave loads its 32 rows' fragments straight from the planes into registers
// (1 KB contiguous per load, a step of 64 ahead; no other wave of the block
// wants them when WM = 4). The weights go through LDS, widened once per block:
// loaded two steps ahead, written one ahead, two stages, one barrier per step,
// placed before the step's last slice so that its MFMAs cover the next reads.
// Large product (2048, 12288, 4096): 789 -> 488 us with the split pass, 1.3 PFLOP/s
// of bf16 work where a library's bf16 GEMM reaches 1.2 on this card.
struct W8pParams {
    const int8_t* xp;     // planes of x [M][K]
    const int8_t* w;
    const float* s_w;
    const float* bias;
    void* y;
    int M, N, K, ks;
    int64_t ldy;
    int m_tiles, n_tiles, per_xcd;
};

// WF_SWIGLU (gate_up, w = [gate rows | up rows], N = 2 I): a 128-column tile is 64
// gate rows and the matching up rows, so that a wave holds g and u of the same
// outputs; silu(g) * u goes through the wave's part of the stages into the
// planes of act (y), a fragment part per store. It saves the round trip of [g|u]
// and a launch of 12 us per layer: 4 % of a 0.6B prompt of 1021 positions.
template <typename YT, int EPI, int WM, int TN>
__global__ __launch_bounds__(256, 2) void gemm_w8p_kernel(W8pParams p) {
    constexpr bool SWIGLU = EPI == WF_SWIGLU;
    static_assert(!SWIGLU || (WM == 4 && TN == 4), "a wave has the tile's 64 gate and 64 up columns");
    constexpr int NL = 3, WN = 4 / WM, BM = 32 * WM, BN = 32 * TN * WN, BK = 64, KS = 4;
    constexpr int WC = BN * BK / 16 / 256, STAGE = BN * WF_ROW;
    extern __shared__ __attribute__((aligned(16))) int8_t wf_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int b = blockIdx.x;
    const int t = (b & 7) * p.per_xcd + (b >> 3);   // tiles dealt to the XCDs as above
    if (t >= p.m_tiles * p.n_tiles) return;
    const int nt = t / p.m_tiles, mt = t - nt * p.m_tiles;
    const int I = p.N / 2, m0 = mt * BM, n0 = SWIGLU ? nt * (BN / 2) : nt * BN;
    const int kb = blockIdx.y * p.ks;
    const int klen = min(p.ks, p.K - kb), nk = (klen + BK - 1) / BK, slices = klen / 16;
    const int col = lane & 31, h = lane >> 5;
    float sw[TN], bn[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int nc = SWIGLU ? n0 + 32 * (j & 1) + (j >> 1) * I + col : min(n0 + 32 * TN * wn + 32 * j + col, p.N - 1);
        sw[j] = EPI == WF_PARTIAL ? 0.f : p.s_w[nc];
        bn[j] = (EPI != WF_PARTIAL && p.bias) ? p.bias[nc] : 0.f;
    }
    // fragments of the wave's row block (uniform base, lane offset); rows past M
    // are the last block's or its padding, their outputs are dropped
    const int mb = min((m0 >> 5) + wm, (p.M - 1) >> 5);
    const int8_t* xs = p.xp + ((int64_t)mb * (p.K / 16) + kb / 16) * WF_FRAG;
    const int xl = lane * 16;
    wf_v4i xr[KS][NL];
    auto load_x = [&](int kt, int ks) {
        const int8_t* f = xs + (int64_t)min(kt * KS + ks, slices - 1) * WF_FRAG;
#pragma unroll
        for (int L = 0; L < NL; L++) xr[ks][L] = *(wf_gv4i*)(f + 1024 * L + xl);
    };
    // weights: thread -> 16 bytes of rows r + 64 i
    const int8_t* wb = p.w + (int64_t)n0 * p.K + kb;
    const int wk = (tid & 3) * 16;
    int64_t wrow[WC];
#pragma unroll
    for (int i = 0; i < WC; i++)
        wrow[i] = (int64_t)(SWIGLU ? (tid >> 2) + i * I : min(n0 + (tid >> 2) + 64 * i, p.N - 1) - n0) * p.K;
    wf_v4i wr[2][WC];
    auto load_w = [&](int kt, int set) {
        const int k = kt * BK + wk, off = k < klen ? k : 0;   // past the slice: its MFMAs are skipped
#pragma unroll
        for (int i = 0; i < WC; i++) wr[set][i] = *(wf_gv4i*)(wb + wrow[i] + off);
    };
    auto put_w = [&](int buf, int set, int i) {
        int8_t* st = wf_lds + buf * STAGE;
        const int r = (tid >> 2) + 64 * i, q = tid & 3;
        uint32_t o[8];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            int u = wr[set][i][d];
            asm volatile("" : "+v"(u));   // the dword whole until here (else its bytes are kept apart)
            wf_widen4<NL>(u, o[2 * d], o[2 * d + 1]);
        }
        *(wf_v4i*)(st + wf_swz(r, 2 * q)) = wf_v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
        *(wf_v4i*)(st + wf_swz(r, 2 * q + 1)) = wf_v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
    };
    wf_v16f acc[TN];
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = 0.f;
    // Where the registers allow it the sums of 256 K values are added up apart:
    // a shorter chain of roundings (K = 1024: error 1.6e-7 against 3.1e-7)
    constexpr bool TWO = TN <= 2;
    wf_v16f sum[TWO ? TN : 1];
#pragma unroll
    for (int j = 0; j < (TWO ? TN : 1); j++)
#pragma unroll
        for (int e = 0; e < 16; e++) sum[j][e] = 0.f;
    auto flush = [&] {
        if constexpr (TWO)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    sum[j][e] += acc[j][e];
                    acc[j][e] = 0.f;
                }
    };
    wf_v4i bw[2][TN];
    auto read_w = [&](int buf, int ks) {
        const int8_t* st = wf_lds + buf * STAGE;
#pragma unroll
        for (int j = 0; j < TN; j++)
            bw[ks & 1][j] = *(const wf_v4i*)(st + wf_swz(32 * (TN * wn + j) + col, 2 * ks + h));
    };
    auto mma = [&](int ks) {
        // the low part first: the small products meet the smaller sums
#pragma unroll
        for (int L = NL - 1; L >= 0; L--)
#pragma unroll
            for (int j = 0; j < TN; j++)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(wf_bf8, xr[ks][L]),
                                                                 __builtin_bit_cast(wf_bf8, bw[ks & 1][j]), acc[j], 0, 0,
                                                                 0);
    };
    // LDS accesses done, then the workgroup barrier; the loads stay in flight
    auto lds_barrier = [&] { stage_barrier<63>(); };

    load_w(0, 0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) load_x(0, ks);
    load_w(min(1, nk - 1), 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < WC; i++) put_w(0, 0, i);
    load_w(min(2, nk - 1), 0);
    lds_barrier();
    read_w(0, 0);
    // step kt, stage buf = kt % 2. MORE: a next step exists; its x is loaded
    // into the registers this step frees, its weights (set buf ^ 1) are widened
    // into the other stage, and the set refilled with step kt + 3's (clamped:
    // loads under a branch would make every wait drain all of them).
    auto step = [&](int kt, int buf, auto more_) {
        constexpr bool MORE = decltype(more_)::value;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks < KS - 1) {
                read_w(buf, ks + 1);
            } else {
                lds_barrier();   // the other stage is written, this one read
                if (MORE) read_w(buf ^ 1, 0);
            }
            if (MORE || kt * KS + ks < slices) mma(ks);
            if (MORE) {
                load_x(kt + 1, ks);
#pragma unroll
                for (int i = 0; i < WC; i++)
                    if (i * 2 / WC == ks) put_w(buf ^ 1, buf ^ 1, i);   // slices 0 and 1
                if (ks == 2) load_w(min(kt + 3, nk - 1), buf ^ 1);
                // the reads, then one MFMA at a time with the rest behind it
                __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
#pragma unroll
                for (int i = 0; i < NL * TN; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 24 / TN, 0);
                    if (i >= TN) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kt = 0;
    for (; kt + 2 < nk; kt += 2) {
        step(kt, 0, std::true_type());
        step(kt + 1, 1, std::true_type());
        if (TWO && (kt & 2)) flush();
    }
    if (kt + 1 < nk) {
        step(kt, 0, std::true_type());
        step(kt + 1, 1, std::false_type());
    } else {
        step(kt, 0, std::false_type());
    }

    if constexpr (SWIGLU) {
        // the stages are free: the last step's barrier came after their last reads.
        // Row r of the wave: 64 floats, 16-byte chunk c at c ^ (r & 15).
        float* ht = (float*)wf_lds + wave * 32 * 64;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int r = 8 * (e >> 2) + 4 * h + (e & 3), c = 8 * j + (col >> 2);
                ht[r * 64 + ((c ^ (r & 15)) << 2) + (col & 3)] = wf_silu_mul(acc[j][e] * sw[j], acc[j + 2][e] * sw[j + 2]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own writes
        if (m0 + 32 * wm + col >= p.M) return;
#pragma unroll
        for (int f = 0; f < 4; f++) {
            const int c = 4 * f + 2 * h;
            const wf_f4 a = *(const wf_f4*)(ht + col * 64 + ((c ^ (col & 15)) << 2));
            const wf_f4 b = *(const wf_f4*)(ht + col * 64 + (((c + 1) ^ (col & 15)) << 2));
            int pt[3][4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                wf_split3_pair(u < 2 ? a[2 * u] : b[2 * u - 4], u < 2 ? a[2 * u + 1] : b[2 * u - 3], pt[0][u], pt[1][u], pt[2][u]);
            int8_t* d = (int8_t*)p.y + wf_plane_at(m0 + 32 * wm + col, n0 + 16 * f + 8 * h, I);
#pragma unroll
            for (int L = 0; L < 3; L++) *(wf_v4i*)(d + 1024 * L) = wf_v4i{pt[L][0], pt[L][1], pt[L][2], pt[L][3]};
        }
        return;
    }
    const bool inner = m0 + BM <= p.M && n0 + BN <= p.N;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + 32 * (TN * wn + j) + col;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int m = m0 + 32 * wm + 8 * (e >> 2) + 4 * h + (e & 3);
            if (inner || (m < p.M && n < p.N))
                wf_put<YT, EPI>(p.y, p.ldy, p.M, p.N, m, n, TWO ? sum[TWO ? j : 0][e] + acc[j][e] : acc[j][e], sw[j],
                                p.bias, bn[j]);
        }
    }
}

// Planes of x: a wave takes 8 rows x 8 groups of 8 values, so that its 16-byte
// writes of 8 rows make whole 128-byte lines.
__global__ __launch_bounds__(256) void wf_split_kernel(const float* __restrict__ x, int64_t ldx, int M, int K,
                                                       int8_t* __restrict__ xp) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m = blockIdx.y * 32 + 8 * w + (lane & 7), k = blockIdx.x * 64 + 8 * (lane >> 3);
    if (k >= K || m >= M) return;
    const float* src = x + (int64_t)m * ldx + k;
    const wf_f4 a = *(const wf_f4*)src, b = *(const wf_f4*)(src + 4);
    int pt[3][4];
#pragma unroll
    for (int u = 0; u < 4; u++)
        wf_split3_pair(u < 2 ? a[2 * u] : b[2 * u - 4], u < 2 ? a[2 * u + 1] : b[2 * u - 3], pt[0][u], pt[1][u], pt[2][u]);
    int8_t* d = xp + wf_plane_at(m, k, K);
#pragma unroll
    for (int L = 0; L < 3; L++) *(wf_v4i*)(d + 1024 * L) = wf_v4i{pt[L][0], pt[L][1], pt[L][2], pt[L][3]};
}

// y[m,n] = (sum over slices in order of part[z][m][n]) * s_w[n] (+ bias[n]).
template <typename YT>
__global__ __launch_bounds__(256) void gemm_w8f_reduce_kernel(const float* __restrict__ part, int splits, int M,
                                                              int N, const float* __restrict__ s_w,
                                                              const float* __restrict__ bias, YT* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, MN = (int64_t)M * N;
    if (i >= MN) return;
    const int n = (int)(i % N);
    const float sw = s_w[n], bn = (bias ? bias : s_w)[n];
    float acc = 0.f;
#pragma unroll 8
    for (int z = 0; z < splits; z++) acc += part[z * MN + i];   // unrolled: 8 slices' loads in flight
    float v = acc * sw;
    if (bias) v += bn;
    y[i] = from_f32<YT>(v);
}

// Slices of K for `tiles` output tiles: while the blocks stay within `blocks`
// and each keeps >= min_steps steps of bk.
static int wf_splits(int64_t tiles, int K, int bk, int blocks, int min_steps) {
    const int steps = ceil_div(K, bk);
    int splits = 1;
    while (tiles * splits * 2 <= blocks && steps / (splits * 2) >= min_steps) splits *= 2;
    return splits;
}

template <typename YT>
static int wf_reduce(const float* part, int splits, int M, int N, const float* s_w, const float* bias, YT* y,
                     hipStream_t st) {
    gemm_w8f_reduce_kernel<YT><<<(unsigned)ceil_div((int64_t)M * N, 256), 256, 0, st>>>(part, splits, M, N, s_w, bias,
                                                                                       y);
    PIO_LAUNCHED();
    return PIO_OK;
}

template <int NL, typename XT, typename YT, int EPI, int TM, int TN>
static int launch_w8f(const W8fParams& p, int splits, hipStream_t st) {
    constexpr size_t lds = 2 * (size_t)(NL * 64 * TM + 64 * TN) * WF_ROW;
    PIO_TRY((allow_lds<gemm_w8f_kernel<NL, XT, YT, EPI, TM, TN>>(lds)));
    gemm_w8f_kernel<NL, XT, YT, EPI, TM, TN><<<dim3(8 * p.per_xcd, splits), 256, lds, st>>>(p);
    PIO_LAUNCHED();
    return PIO_OK;
}

template <int NL, typename XT, typename YT, int TM, int TN>
static int run_w8f_tiles(W8fParams p, hipStream_t st) {
    p.m_tiles = ceil_div(p.M, 64 * TM);
    p.n_tiles = ceil_div(p.N, 64 * TN);
    const int tiles = p.m_tiles * p.n_tiles;
    p.per_xcd = ceil_div(tiles, 8);
    // K slices while the blocks stay within two per CU and each slice keeps
    // >= 4 steps (M = 127 linears: 11-15 % faster than with at most one block
    // per CU and 8 steps)
    int splits = wf_splits(tiles, p.K, WF_BK, 512, 4);
    p.ks = ceil_div(ceil_div(p.K, WF_BK), splits) * WF_BK;
    splits = ceil_div(p.K, p.ks);
    if (splits == 1) {
        p.ks = p.K;
        return launch_w8f<NL, XT, YT, WF_STORE, TM, TN>(p, 1, st);
    }
    YT* y = (YT*)p.y;
    Scratch ws;
    PIO_TRY(ws.get((size_t)splits * p.M * p.N * sizeof(float), st));
    p.y = ws.ptr;
    PIO_TRY((launch_w8f<NL, XT, YT, WF_PARTIAL, TM, TN>(p, splits, st)));
    return wf_reduce((const float*)ws.ptr, splits, p.M, p.N, p.s_w, p.bias, y, st);
}

template <typename YT, int EPI, int WM, int TN>
static int launch_w8p(const W8pParams& p, int splits, hipStream_t st) {
    constexpr size_t lds = 2 * (size_t)(32 * TN * (4 / WM)) * WF_ROW;
    PIO_TRY((allow_lds<gemm_w8p_kernel<YT, EPI, WM, TN>>(lds)));
    gemm_w8p_kernel<YT, EPI, WM, TN><<<dim3(8 * p.per_xcd, splits), 256, lds, st>>>(p);
    PIO_LAUNCHED();
    return PIO_OK;
}

// The planes GEMM on one tile shape. part != nullptr: K slices are left as
// unscaled partials in `ws` (the caller finishes them).
template <typename YT, bool RESID, int WM, int TN>
static int run_w8p_tiles(W8pParams p, int blocks, int min_steps, Scratch* ws, const float** part, int* splits_out, hipStream_t st) {
    p.m_tiles = ceil_div(p.M, 32 * WM);
    p.n_tiles = ceil_div(p.N, 32 * TN * (4 / WM));
    const int tiles = p.m_tiles * p.n_tiles;
    p.per_xcd = ceil_div(tiles, 8);
    const int steps = ceil_div(p.K, 64);
    // Few rows, more than 32 tiles: as many slices as fill the blocks, not a power
    // of two (96 tiles: 5 slices, 480 blocks, against 4 that give half the CUs two
    // blocks and half one: (13, 12288, 4096) 24.7 -> 22.6 us; 56 tiles: (32, 7168, 8192)
    // 27.7 -> 25.9; 48: (32, 6144, 4096) 18.4 -> 18.1; 40: 18.5 -> 18.4). Fewer tiles
    // have so many slices that the powers of two fill the CUs too, and each further
    // slice is another M x N of partials: (32, 2305, 12288), 19 tiles, 16 slices 24.2
    // us, 26 slices 26.0; 24 tiles 22.3 / 22.5.
    // Nor in 128 x 64 tiles whose slices a reduce launch adds: (200, 2560, 3072), 80
    // tiles, 2 slices 28.5 us, 3 slices 25.0.
    const bool fill = (WM == 1 && tiles > 32) || (WM == 4 && !part);
    int splits = fill ? std::max(1, std::min(blocks / tiles, steps / min_steps))
                      : wf_splits(tiles, p.K, 64, blocks, min_steps);
    p.ks = ceil_div(steps, splits) * 64;
    splits = ceil_div(p.K, p.ks);
    if (splits == 1) return launch_w8p<YT, RESID ? WF_RESID : WF_STORE, WM, TN>(p, 1, st);
    YT* y = (YT*)p.y;
    Scratch own;
    Scratch& w = part ? *ws : own;
    PIO_TRY(w.get((size_t)splits * p.M * p.N * sizeof(float), st));
    p.y = w.ptr;
    PIO_TRY((launch_w8p<YT, WF_PARTIAL, WM, TN>(p, splits, st)));
    if (part) {
        *part = (const float*)w.ptr;
        *splits_out = splits;
        return PIO_OK;
    }
    return wf_reduce((const float*)w.ptr, splits, p.M, p.N, p.s_w, p.bias, y, st);
}

// Whether the planes GEMM takes these sizes in 128 x 128 tiles (see run_w8p; such a
// plan never splits K). Up to 64 rows the narrower tiles are as fast or faster at
// any width, as half the wide tile's waves would repeat rows: (M, N, K) = (13,
// 24576, 4096) 73 us wide and 47 in 32 x 128 tiles, (32, 151936, 1024) 105 / 60, (33,
// 24576, 4096) 74 / 75, (64, 151936, 1024) 106 / 96 in 64 x 64; from 65 rows on the
// wide ones: (65, 24576, 4096) 75 / 103, (100, 20480, 1024) 25 / 28.
static bool w8p_wide(int M, int N) {
    return M > 64 && N >= 6144 && (int64_t)ceil_div(M, 128) * ceil_div(N, 128) >= 160;
}

template <typename YT, bool RESID>
static int run_w8p(const int8_t* xp, const int8_t* w, const float* s_w, const float* bias, YT* y, int64_t ldy, int M,
                   int N, int K, Scratch* ws, const float** part, int* splits, hipStream_t st) {
    W8pParams p{};
    p.xp = xp; p.w = w; p.s_w = s_w; p.bias = bias; p.y = y;
    p.M = M; p.N = N; p.K = K; p.ldy = ldy;
    // Wide outputs: 128 x 128 tiles once they occupy most CUs ((M, N, K) = (509,
    // 6144, 1024): 27 us with the split pass against 29 in 128 x 64 tiles, (256,
    // 12288, 4096): 72 against 83). Otherwise 128 x 64, whose sums are two-level,
    // with K slices up to one block per CU (two up to 256 rows), and for few rows
    // tiles of 64 x 64 and 32 x 128. A 0.6B prompt of 16 / 48 / 127 / 256 / 509 rows:
    // 1398 / 1558 / 1845 / 2427 / 3669 us against 1422 / 1590 / 2062 / 3532 / 7036
    // with fp32 activations split in the GEMM; 128 x 64 tiles alone 1720 / 1720 /
    // 1910 / 2438 / 3640.
    if (w8p_wide(M, N))
        return run_w8p_tiles<YT, RESID, 4, 4>(p, 256, 4, ws, part, splits, st);
    // A linear by itself (no part: its K slices cost a reduce launch) of 129 to 384
    // rows: 64 x 64 tiles where they take fewer rounds of the CUs than 128 x 64 ones,
    // a round of them counted as 0.7 of theirs ((300, 6144, 4096), 480 tiles against
    // 288: 65 us against 81; (160, 5003, 2064), 237 against 158: 25 / 32; not at (384,
    // 6144, 4096), 576 against 288: 95 / 86); K slices for one block per CU, two when
    // K is long ((230, 6144, 1024): 19 us, 27 with two; (160, 4096, 12288): 81, 79).
    if (!part && M > 128 && M <= 384) {
        const int tall = ceil_div(M, 128) * ceil_div(N, 64), small = ceil_div(M, 64) * ceil_div(N, 64);
        if (tall > 128 && 14 * ceil_div(small, 256) < 20 * ceil_div(tall, 256))
            return run_w8p_tiles<YT, RESID, 2, 1>(p, 256, 4, ws, part, splits, st);
        return run_w8p_tiles<YT, RESID, 4, 2>(p, K > 4096 && M <= 256 ? 512 : 256, 4, ws, part, splits, st);
    }
    if (M > 128) return run_w8p_tiles<YT, RESID, 4, 2>(p, M <= 256 ? 512 : 256, 4, ws, part, splits, st);
    if (M > 32) return run_w8p_tiles<YT, RESID, 2, 1>(p, 512, 4, ws, part, splits, st);
    return run_w8p_tiles<YT, RESID, 1, 1>(p, 512, 2, ws, part, splits, st);
}

// fp32 y on planes of x (wf_planes.hpp). When the plan splits K, only the
// slices' unscaled partials part[z][m][n] are produced (*part, *splits, in
// `ws`; y untouched) for the caller to finish; otherwise y is written (scaled,
// + bias, + y when resid) and *splits = 0.
int gemm_w8_planes(const int8_t* xp, const int8_t* w, const float* s_w, const float* bias, float* y, int64_t ldy, int M,
                   int N, int K, bool resid, Scratch& ws, const float** part, int* splits, hipStream_t st) {
    PIO_REQUIRE(xp && w && s_w && y && M > 0 && N > 0 && K > 0 && K % 16 == 0 && aligned16(xp) && aligned16(w),
                "gemm_w8_planes: bad operands");
    *part = nullptr;
    *splits = 0;
    return resid ? run_w8p<float, true>(xp, w, s_w, bias, y, ldy, M, N, K, &ws, part, splits, st)
                 : run_w8p<float, false>(xp, w, s_w, bias, y, ldy, M, N, K, &ws, part, splits, st);
}

// Whether the gate_up GEMM of M rows can form silu(g) * u in its epilogue
// (gemm_w8_planes_swiglu).
bool w8_planes_swiglu_fits(int M, int I) { return I % 64 == 0 && w8p_wide(M, 2 * I); }

// act = silu(g) * u as planes, [g|u] the linear of planes xp.
int gemm_w8_planes_swiglu(const int8_t* xp, const int8_t* w, const float* s_w, int8_t* act, int M, int I, int K,
                          hipStream_t st) {
    PIO_REQUIRE(xp && w && s_w && act && M > 0 && I > 0 && K > 0 && K % 16 == 0 && aligned16(xp) && aligned16(w) &&
                    aligned16(act) && w8_planes_swiglu_fits(M, I),
                "gemm_w8_planes_swiglu: bad operands");
    W8pParams p{};
    p.xp = xp; p.w = w; p.s_w = s_w; p.y = act;
    p.M = M; p.N = 2 * I; p.K = p.ks = K;
    p.m_tiles = ceil_div(M, 128);
    p.n_tiles = I / 64;
    p.per_xcd = ceil_div(p.m_tiles * p.n_tiles, 8);
    return launch_w8p<float, WF_SWIGLU, 4, 4>(p, 1, st);
}

template <typename XT, typename YT>
static int run_w8f(const XT* x, const int8_t* w, const float* s_w, const float* bias, YT* y, int M, int N, int K,
                   hipStream_t st) {
    constexpr int NL = std::is_same<XT, float>::value ? 3 : 1;
    if (K == 0) return wf_reduce<YT>(nullptr, 0, M, N, s_w, bias, y, st);
    if constexpr (NL == 3) {
        // The planes pay for their pass (a launch, 10 bytes per x value) once the
        // product is large enough, sooner when many columns share it. Measured,
        // this path against the other (us): (M, N, K) = (127, 4096, 1024) 16.3 /
        // 14.6, (127, 6144, 1024) 17.2 / 19.3, (509, 6144, 1024) 27 / 36, (1021,
        // 1024, 2048) 30 / 29, (1021, 1024, 3072) 37 / 41, (2048, 3072, 1024) 52 / 71,
        // (2048, 12288, 4096) 488 / 762; (40, 12288, 4096) 30 / 48, (64, 3072, 1024)
        // 12.9 / 11.1. Not for 129 to 256 rows of a small weight, which would need K
        // slices: (192, 4096, 1024) 19.9 / 19.0, (256, 2048, 2048) 19.9 / 16.4, but (192,
        // 3072, 2048) 24.6 / 26.9.
        const double mnk = (double)M * N * K;
        const bool sliced = M > 128 && M <= 256 && N <= 4096 && (int64_t)N * K <= 5000000;
        if (mnk >= (N >= 2048 && !sliced ? 0.6e9 : 3e9)) {
            // row chunks keep the planes within 64 MB
            const int rows = (int)std::max<int64_t>(128, ((64ll << 20) / (6ll * K)) & ~127ll);
            for (int m0 = 0; m0 < M; m0 += rows) {
                const int m = std::min(rows, M - m0);
                Scratch xs;
                PIO_TRY(xs.get(wf_planes_bytes(m, K), st));
                wf_split_kernel<<<dim3(ceil_div(K, 64), ceil_div(m, 32)), 256, 0, st>>>(x + (int64_t)m0 * K, K, m, K,
                                                                                      (int8_t*)xs.ptr);
                PIO_LAUNCHED();
                PIO_TRY((run_w8p<YT, false>((const int8_t*)xs.ptr, w, s_w, bias, y + (int64_t)m0 * N, N, m, N, K,
                                            nullptr, nullptr, nullptr, st)));
            }
            return PIO_OK;
        }
    }
    W8fParams p{};
    p.x = x; p.w = w; p.s_w = s_w; p.bias = bias; p.y = y;
    p.M = M; p.N = N; p.K = K;
    // 128 x 128 tiles (every fragment read feeds two MFMAs) when they still
    // give every CU a tile; 64 x 64 tiles (with K slices if needed) otherwise
    if ((int64_t)ceil_div(M, 128) * ceil_div(N, 128) >= 256) return run_w8f_tiles<NL, XT, YT, 2, 2>(p, st);
    return run_w8f_tiles<NL, XT, YT, 1, 1>(p, st);
}

// x [M, K], W [N, K], y [M, N], all contiguous.
int gemm_w8f(const void* x, int x_dtype, const int8_t* w, const float* s_w, const float* bias, void* y, int y_dtype,
             int M, int N, int K, hipStream_t st) {
    PIO_REQUIRE(x && w && s_w && y, "gemm_w8f: null pointer");
    PIO_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm_w8f: negative shape");
    PIO_REQUIRE(K % 16 == 0, "gemm_w8f: K=%d must be a multiple of 16", K);
    PIO_REQUIRE(aligned16(x) && aligned16(w), "gemm_w8f: x and W must be 16-byte aligned");
    PIO_REQUIRE(x_dtype == PIO_F32 || x_dtype == PIO_F16, "gemm_w8f: x must be fp32 or fp16");
    PIO_REQUIRE(y_dtype == PIO_F32 || y_dtype == PIO_F16, "gemm_w8f: y must be fp32 or fp16");
    if (M == 0 || N == 0) return PIO_OK;
    if (x_dtype == PIO_F32) {
        if (y_dtype == PIO_F32) return run_w8f((const float*)x, w, s_w, bias, (float*)y, M, N, K, st);
        return run_w8f((const float*)x, w, s_w, bias, (_Float16*)y, M, N, K, st);
    }
    if (y_dtype == PIO_F32) return run_w8f((const _Float16*)x, w, s_w, bias, (float*)y, M, N, K, st);
    return run_w8f((const _Float16*)x, w, s_w, bias, (_Float16*)y, M, N, K, st);
}

}  // namespace pio
