// Router: gate projection, row softmax, wave-level top-k, per-token-tile expert histogram.
//
// One workgroup routes a tile of TT tokens: 32, or 16 for layers with at most 16 experts (one thread per token and expert, 128
// or 256 threads: the sums are bound by LDS reads per compute unit, so such a layer spreads its tokens over twice as many
// workgroups) and for exact bf16 layers with more while tiles of 16 find a compute unit each.
//  phase 1  logits[t,e] = sum_k x[t,k]*Wg[e,k] (+bg[e]): one lane per (token, expert); x and Wg are
//           staged through LDS in chunks of 64..512 k.  EXACT mode adds the products one k at a time with
//           a separate multiply and add (this file is compiled with -ffp-contract=off), which is the
//           summation order of the reference's CPU dot (J/common/utils/MatrixOperation.java:1472-1478);
//           FAST mode uses fused multiply-adds (same order, one rounding per step).
//  phase 2  softmax as the reference's thread-per-row kernel (J/engine/gpu/SoftmaxKernel.cu:4-24, CPU twin
//           J/engine/gpu/SoftmaxKernel.java:69-87): max, e=(float)exp((double)(z-max)), sum in expert order,
//           divide -- the experts of a token live in the lanes of a wave (or of an 8/16/32-lane group),
//           the ordered sum is taken by one lane per token;
//           top-k: K rounds of a cross-lane (value,index) butterfly arg-max, "greater value, or equal
//           value and lower index" so ties go to the lowest expert; winners are masked out.
//  phase 3  LDS-atomic histogram of the selected experts, flushed as row `tile` of tile_counts[.,E].
// bf16 layers with more than 16 experts take phase 1 to the matrix cores: router_units_kernel with the same bits, in FAST mode
// router_mfma_kernel (both below).
// bf16 layers with at most 16 experts and at most one tile per compute unit take router_pipe_kernel: phase 1 is then as
// long as one chain of d dependent multiply-adds, and separate staging waves keep everything else out of the waves that
// run the chains (Mixtral shape: 4096 tokens 33 -> 29 us, 64 tokens 27 -> 22 us; of the 22, 11 are the chain itself at
// 6.25 clocks a term and 6.5 are launch, the first loads and phases 2 and 3).
#include "common.h"
#include <limits.h>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 rt_bf16x8;
typedef __attribute__((ext_vector_type(16))) float rt_f32x16;

#define ROUTER_EPT(EP) ((EP) >= 128 ? 4 : (EP) >= 32 ? 2 : 1)
// token tile and threads per workgroup for EP (padded) experts
#define ROUTER_TT(EP) ((EP) <= 16 ? 16 : 32)
#define ROUTER_NTHR(EP) ((EP) <= 8 ? 128 : 256)
// k per staged chunk for at most 16 experts: with 16-token tiles the sums of a 256-k chunk take less time than the
// next chunk's loads need to arrive, and the kernel is bound by one memory latency per chunk: 512-k chunks halve their
// number (Mixtral shape, 4096 tokens: 32-token tiles 42 us; 16-token tiles 54 us with 256-k chunks, 34 us with 512)
#define ROUTER_KC_SMALL 512
static bool router_on_mfma(const omega_moe *m) { return m->cfg.dtype == OMEGA_DTYPE_BF16 && m->cfg.E > 16; }
int router_tok_tile(const omega_moe *m, int T)
{
    if (m->cfg.E <= 16) return 16;
    // (matrix-core form: tiles of 16 tokens while they find a compute unit each)
    return router_on_mfma(m) && m->cfg.router_mode == OMEGA_ROUTER_EXACT && ceil_div(T, 16) <= m->ctx->num_cus ? 16 : 32;
}

// Phase 1 for the tokens t0.. of one workgroup: acc[x*NT + i] = logit of (token tg + i*TPP, expert e1 + x*EL), bias
// not yet added.  A thread owns EPT experts (2 from 128 experts on: each x value read from LDS then feeds two sums,
// which halves the LDS reads per multiply-add) and NT tokens.
// EP: experts padded to a power of two; KC: k per staged chunk (larger for few experts, where one chunk in
// flight per workgroup would otherwise leave the kernel waiting on memory latency).
// XBF: x and Wg are stored as bf16 (else fp32).  IO_FULL: rows are 16-byte aligned and d is a multiple of KC, so
// every load is a whole 16-byte vector; rows beyond T or E are redirected to the last valid row (their sums are
// never used), which keeps the loads free of branches - and with that really asynchronous: a load issued inside
// a divergent branch makes the compiler wait for all earlier ones first.  IO_VEC: rows are 16-byte aligned and whole 16-byte
// vectors long; vectors behind the row's end read its last one and count as zeros.  (Router launch, us, against
// element by element: 256 tokens x 128 columns, 8 experts 7.6 -> 5.4; 4096 x 1000 20.0 -> 14.7; bf16, 6000 x 1280 26.3 -> 13.9.)
enum { IO_ANY = 0, IO_VEC, IO_FULL };
template <int EP, int KC, bool EXACT, bool XBF, int IO>
__device__ __forceinline__ void router_sums(const void *__restrict__ x, const void *__restrict__ Wg, int T, int d, int E,
                                            int t0, float (*xs)[KC + 4], float (*ws)[KC + 4],
                                            float (&acc)[ROUTER_TT(EP) * EP / ROUTER_NTHR(EP)])
{
    constexpr int TOK_TILE = ROUTER_TT(EP), NTHR = ROUTER_NTHR(EP);
    constexpr int EPT = ROUTER_EPT(EP);           // experts per thread
    constexpr int EL = EP / EPT;                  // threads across the experts
    constexpr int NT = TOK_TILE * EL / NTHR;      // tokens per thread
    constexpr int TPP = NTHR / EL;                // tokens per pass
    static_assert(NT >= 1 && NT * NTHR == TOK_TILE * EL, "every thread owns whole (token, expert) sums");
    constexpr int TPR = NTHR / TOK_TILE;          // staging threads per token row (8 or 16)
    static_assert(TPR * TOK_TILE == NTHR && KC % (8 * TPR) == 0, "whole staging vectors per thread");
    const int tid = threadIdx.x;
    const int e1 = tid % EL, tg = tid / EL;
    // staging: every thread carries 8 consecutive k of one token and of WCH gate rows from global memory to LDS;
    // the next chunk is fetched into registers while the current one is being summed
    constexpr int XCH = KC / (8 * TPR);
    constexpr int WCH = EP * (KC / 8) / NTHR;
    static_assert(EP * (KC / 8) % NTHR == 0, "every thread stages the same number of gate vectors");
    const int x_tt = tid / TPR, x_ks = (tid % TPR) * 8;
    // raw staging registers: 8 k of bf16 = one uint4, 8 k of fp32 = two; conversion happens when they are
    // written to LDS, so the global loads stay in flight during the sums of the current chunk
    uint4 xr[XCH][2], wr[WCH][2];
    auto load8 = [&](const void *base, int row, int rows, int k, uint4 *out) {
        out[0] = make_uint4(0, 0, 0, 0);
        out[1] = make_uint4(0, 0, 0, 0);
        if (IO == IO_VEC) {
            const size_t row_off = (size_t)min(row, rows - 1) * d;
            constexpr int V = XBF ? 8 : 4;
#pragma unroll
            for (int h = 0; h < 8 / V; ++h) {
                const uint4 v = XBF ? *(const uint4 *)((const bf16_t *)base + row_off + min(k, d - V))
                                    : *(const uint4 *)((const float *)base + row_off + min(k + 4 * h, d - V));
                const bool in = k + 4 * h < d;
                out[h] = make_uint4(in ? v.x : 0, in ? v.y : 0, in ? v.z : 0, in ? v.w : 0);
            }
        } else if (IO == IO_FULL) {
            const size_t off = (size_t)min(row, rows - 1) * d + k;
            if (XBF) {
                out[0] = *(const uint4 *)((const bf16_t *)base + off);
            } else {
                out[0] = *(const uint4 *)((const float *)base + off);
                out[1] = *(const uint4 *)((const float *)base + off + 4);
            }
        } else if (row < rows) {  // unaligned or ragged rows: element by element, packed into the same form
            const size_t row_off = (size_t)row * d;
            uint32_t u[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                u[q] = 0;
                if (k + q < d)
                    u[q] = XBF ? (uint32_t)((const bf16_t *)base)[row_off + k + q]
                               : __float_as_uint(((const float *)base)[row_off + k + q]);
            }
            if (XBF) {
                out[0] = make_uint4(u[0] | (u[1] << 16), u[2] | (u[3] << 16), u[4] | (u[5] << 16), u[6] | (u[7] << 16));
            } else {
                out[0] = make_uint4(u[0], u[1], u[2], u[3]);
                out[1] = make_uint4(u[4], u[5], u[6], u[7]);
            }
        }
    };
    auto widen = [&](const uint4 *in, float *dst) {  // 8 floats to LDS
        float4 lo, hi;
        if (XBF) {
            lo = make_float4(__uint_as_float(in[0].x << 16), __uint_as_float(in[0].x & 0xffff0000u),
                             __uint_as_float(in[0].y << 16), __uint_as_float(in[0].y & 0xffff0000u));
            hi = make_float4(__uint_as_float(in[0].z << 16), __uint_as_float(in[0].z & 0xffff0000u),
                             __uint_as_float(in[0].w << 16), __uint_as_float(in[0].w & 0xffff0000u));
        } else {
            lo = make_float4(__uint_as_float(in[0].x), __uint_as_float(in[0].y), __uint_as_float(in[0].z), __uint_as_float(in[0].w));
            hi = make_float4(__uint_as_float(in[1].x), __uint_as_float(in[1].y), __uint_as_float(in[1].z), __uint_as_float(in[1].w));
        }
        *(float4 *)dst = lo;
        *(float4 *)(dst + 4) = hi;
    };
    auto fetch = [&](int k0) {
#pragma unroll
        for (int c = 0; c < XCH; ++c) load8(x, t0 + x_tt, T, k0 + x_ks + 8 * TPR * c, xr[c]);
#pragma unroll
        for (int c = 0; c < WCH; ++c) {
            const int idx = tid + c * NTHR;
            load8(Wg, idx / (KC / 8), E, k0 + (idx % (KC / 8)) * 8, wr[c]);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int c = 0; c < XCH; ++c) widen(xr[c], &xs[x_tt][x_ks + 8 * TPR * c]);
#pragma unroll
        for (int c = 0; c < WCH; ++c) {
            const int idx = tid + c * NTHR;
            widen(wr[c], &ws[idx / (KC / 8)][(idx % (KC / 8)) * 8]);
        }
    };

    // a wave whose lowest token is past the end of the batch has no sum to form (small batches, ragged last tile):
    // the sums are bound by LDS reads, which its silence leaves to the waves that have tokens
    const bool wave_live = t0 + (tid & ~63) / EL < T;
    fetch(0);
    for (int k0 = 0; k0 < d; k0 += KC) {
        const int kend = min(KC, d - k0);
        stash();
        __syncthreads();
        if (k0 + KC < d) fetch(k0 + KC);
        // the products are added one k at a time in index order: EXACT with a separate multiply and add,
        // FAST with a fused multiply-add (one rounding per step).  With bf16 operands the two are the same
        // arithmetic: a product of two 8-bit significands has 16 bits and is exact in fp32 (unless it falls below
        // 2^-134, far outside anything a layer holds), so the separate multiply rounds nothing and EXACT takes the
        // fused form too - bit for bit the sequential unfused sum, at one instruction per term.
#define ROUTER_K4(k4)                                                                  \
    do {                                                                               \
        float4 wv[EPT];                                                                \
        _Pragma("unroll") for (int x_ = 0; x_ < EPT; ++x_)                             \
            wv[x_] = *(const float4 *)&ws[e1 + x_ * EL][(k4) * 4];                     \
        _Pragma("unroll") for (int i = 0; i < NT; ++i)                                 \
        {                                                                              \
            const float4 xv = *(const float4 *)&xs[tg + i * TPP][(k4) * 4];            \
            _Pragma("unroll") for (int x_ = 0; x_ < EPT; ++x_)                         \
            {                                                                          \
                float &a_ = acc[x_ * NT + i];                                          \
                if (EXACT && !XBF) {                                                   \
                    float prod;                                                        \
                    prod = xv.x * wv[x_].x; a_ = a_ + prod;                            \
                    prod = xv.y * wv[x_].y; a_ = a_ + prod;                            \
                    prod = xv.z * wv[x_].z; a_ = a_ + prod;                            \
                    prod = xv.w * wv[x_].w; a_ = a_ + prod;                            \
                } else {                                                               \
                    a_ = fmaf(xv.x, wv[x_].x, a_);                                     \
                    a_ = fmaf(xv.y, wv[x_].y, a_);                                     \
                    a_ = fmaf(xv.z, wv[x_].z, a_);                                     \
                    a_ = fmaf(xv.w, wv[x_].w, a_);                                     \
                }                                                                      \
            }                                                                          \
        }                                                                              \
    } while (0)
        if (!wave_live) {
            // every token of this wave lies beyond T: it only stages and keeps the barriers
        } else if (IO == IO_FULL || kend == KC) {
            // whole chunk: no exit test inside, so the LDS reads of later steps are issued ahead of the sums
#pragma unroll(NT * EPT >= 8 ? 4 : 16)
            for (int k4 = 0; k4 < KC / 4; ++k4) ROUTER_K4(k4);
        } else {
            // last, partial chunk (zero-filled beyond d: a +0 product leaves every sum unchanged - none is ever -0), 32 k at a time
            for (int k32 = 0; k32 * 32 < kend; ++k32)
#pragma unroll
                for (int k4 = 0; k4 < 8; ++k4) ROUTER_K4(8 * k32 + k4);
        }
#undef ROUTER_K4
        __syncthreads();
    }
}

// Phases 2 and 3 for the tokens of one workgroup, from the logits in lg (all threads; lg and hist are complete and
// visible on entry; lg is overwritten).  LPT = NTHR / TOK_TILE lanes (8 or 16) share a token; lane j of them owns the
// experts j, j + LPT, ...  Softmax in the reference's order (J/engine/gpu/SoftmaxKernel.cu:4-24): the row maximum
// (any order gives the same value), e = (float)exp((double)(z - max)) written back to LDS, then ONE lane per token adds
// the E values in expert order - the reference's thread-per-row loop, run for all tokens of the tile side by side - and
// every lane divides.  Top-k: K rounds; a lane scans its own experts in ascending order with a strict comparison, the
// LPT lanes combine by a butterfly on (value, index) with "greater value, or equal value and lower index", so ties go
// to the lowest expert; the winner is masked out.  RELAXED (the matrix-core FAST path, tolerance mode) takes the
// exponentials in single precision.
// The value another lane of the token's 8 or 16 holds, in the lane's own pipeline (DPP) instead of through the LDS crossbar:
// step 1 and 2 pair the lanes of a quad, 4 the two quads of eight lanes and 8 the two eights of sixteen, each mirrored - after
// the steps before, the lanes that a mirror exchanges hold the same values, so a butterfly over steps 1, 2, 4 (, 8) leaves every
// lane with the result of all.  (Worth 1 us of a launch with 6 or 8 rounds.)
template <int STEP>
__device__ __forceinline__ int token_lane(int v)
{
    constexpr int ctrl = STEP == 1 ? 0xB1 : STEP == 2 ? 0x4E : STEP == 4 ? 0x141 : 0x140;  // quad_perm [1,0,3,2], [2,3,0,1]; row_half_mirror; row_mirror
    return __builtin_amdgcn_update_dpp(v, v, ctrl, 0xF, 0xF, true);
}
template <int STEP>
__device__ __forceinline__ float token_lane(float v)
{
    return __int_as_float(token_lane<STEP>(__float_as_int(v)));
}

template <int EP, bool RELAXED = false, int TOK_TILE = 32, int NTHR = 256>
__device__ __forceinline__ void router_select(float (*lg)[EP], int *hist, int t0, int tile, int T, int E, int K, int renorm,
                                              int32_t *__restrict__ ids, float *__restrict__ wout,
                                              int32_t *__restrict__ tile_counts, float *__restrict__ probs_out)
{
    constexpr int LPT = NTHR / TOK_TILE;            // lanes per token
    constexpr int VPL = (EP + LPT - 1) / LPT;       // experts per lane
    constexpr int KPL = (64 + LPT - 1) / LPT;       // slots per lane (K <= 64)
    static_assert(LPT == 8 || LPT == 16, "a token's lanes lie in one wave");
    const int tid = threadIdx.x;
    const int tt = tid / LPT, sub = tid % LPT;
    const int t = t0 + tt;
    const bool live = t < T;  // uniform over the LPT lanes that exchange data
    float p[VPL];
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < VPL; ++q) {
        const int e = sub + q * LPT;
        p[q] = (e < E && e < EP) ? lg[tt][e] : -INFINITY;
        mx = fmaxf(mx, p[q]);
    }
    mx = fmaxf(mx, token_lane<1>(mx));
    mx = fmaxf(mx, token_lane<2>(mx));
    mx = fmaxf(mx, token_lane<4>(mx));
    if (LPT == 16) mx = fmaxf(mx, token_lane<8>(mx));
#pragma unroll
    for (int q = 0; q < VPL; ++q) {
        const int e = sub + q * LPT;
        p[q] = (e < E && e < EP) ? (RELAXED ? __expf(p[q] - mx) : (float)exp((double)(p[q] - mx))) : 0.0f;
        if (e < EP) lg[tt][e] = p[q];
    }
    __syncthreads();
    float s = 0.0f;
    if (sub == 0 && live) {
        int e = 0;
        for (; e + 16 <= E; e += 16) {  // sixteen reads in flight; the additions stay in expert order
            float v[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) v[q] = lg[tt][e + q];
#pragma unroll
            for (int q = 0; q < 16; ++q) s = s + v[q];
        }
        for (; e < E; ++e) s = s + lg[tt][e];
    }
    s = __shfl(s, 0, LPT);
#pragma unroll
    for (int q = 0; q < VPL; ++q) {
        const int e = sub + q * LPT;
        p[q] = p[q] / s;
        if (probs_out != nullptr && live && e < E) probs_out[(size_t)t * E + e] = p[q];
        if (e >= E) p[q] = -1.0f;  // never selected: probabilities are >= 0
    }
    // lane `sub` keeps the winners of the rounds j = sub, sub + LPT, ...
    int myid[KPL];
    float myw[KPL];
#pragma unroll
    for (int u = 0; u < KPL; ++u) { myid[u] = 0; myw[u] = 0.0f; }
    float rs = 0.0f;  // sum of the selected weights in slot order, the same in all lanes of the token
    for (int j = 0; j < K; ++j) {
        float bv = p[0];
        int bi = sub;
#pragma unroll
        for (int q = 1; q < VPL; ++q)
            if (p[q] > bv) { bv = p[q]; bi = sub + q * LPT; }
        auto meet = [&](float ov, int oi) {
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        };
        meet(token_lane<1>(bv), token_lane<1>(bi));
        meet(token_lane<2>(bv), token_lane<2>(bi));
        meet(token_lane<4>(bv), token_lane<4>(bi));
        if (LPT == 16) meet(token_lane<8>(bv), token_lane<8>(bi));
        rs = rs + bv;
#pragma unroll
        for (int u = 0; u < KPL; ++u)
            if (j == sub + u * LPT) { myid[u] = bi; myw[u] = bv; }
#pragma unroll
        for (int q = 0; q < VPL; ++q)
            if (bi == sub + q * LPT) p[q] = -1.0f;
    }
#pragma unroll
    for (int u = 0; u < KPL; ++u) {
        const int j = sub + u * LPT;
        if (j < K && live) {
            ids[(size_t)t * K + j] = myid[u];
            wout[(size_t)t * K + j] = renorm ? myw[u] / rs : myw[u];
            atomicAdd(&hist[myid[u]], 1);
        }
    }
    __syncthreads();
    for (int e = tid; e < E; e += NTHR) tile_counts[(size_t)tile * E + e] = hist[e];
}

template <int EP, int KC, bool EXACT>
__global__ __launch_bounds__(ROUTER_NTHR(EP)) void router_kernel(const void *__restrict__ x, int dtype, const void *__restrict__ Wg,
                                                     const float *__restrict__ bg, int T, int d, int E, int K,
                                                     int renorm, int32_t *__restrict__ ids,
                                                     float *__restrict__ wout, int32_t *__restrict__ tile_counts,
                                                     float *__restrict__ logits_out, float *__restrict__ probs_out)
{
    constexpr int TOK_TILE = ROUTER_TT(EP), NTHR = ROUTER_NTHR(EP);
    constexpr int EPT = ROUTER_EPT(EP), EL = EP / EPT;  // phase 1: experts per thread, threads across the experts
    constexpr int NT = TOK_TILE * EL / NTHR;            // tokens per thread in phase 1
    constexpr int TPP = NTHR / EL;                      // tokens per pass
    constexpr int LDW = KC + 4;  // LDS row stride in floats: rows stay 16-byte aligned and bank-staggered
    __shared__ __attribute__((aligned(16))) float xs[TOK_TILE][LDW];
    __shared__ __attribute__((aligned(16))) float ws[EP][LDW];
    // up to 64 experts the logits take the place of the staged gate rows once phase 1 is over (its last step is a
    // barrier); measured a fifth faster at 64 experts and slightly slower at 128, which keep an array of their own
    constexpr bool LG_ALIAS = EP <= 64;
    static_assert(LDW >= TOK_TILE, "the gate staging area holds the logits");
    __shared__ float lg_own[LG_ALIAS ? 1 : TOK_TILE][EP];
    float(*lg)[EP] = LG_ALIAS ? (float(*)[EP]) & ws[0][0] : lg_own;
    __shared__ int hist[EP];

    const int tid = threadIdx.x;
    const int tile = blockIdx.x;
    const int t0 = tile * TOK_TILE;
    const int e1 = tid % EL, tg = tid / EL;
    if (tid < EP) hist[tid] = 0;

    float acc[NT * EPT];
#pragma unroll
    for (int i = 0; i < NT * EPT; ++i) acc[i] = 0.0f;

    const bool aligned = ((uintptr_t)x | (uintptr_t)Wg) % 16 == 0, full = aligned && d % KC == 0;
    if (EP <= 16 && dtype == OMEGA_DTYPE_BF16) {  // (bf16 layers with more experts run on the matrix cores; d is a multiple of 256)
        if (full) router_sums<EP, KC, EXACT, true, IO_FULL>(x, Wg, T, d, E, t0, xs, ws, acc);
        else if (aligned) router_sums<EP, KC, EXACT, true, IO_VEC>(x, Wg, T, d, E, t0, xs, ws, acc);
        else router_sums<EP, KC, EXACT, true, IO_ANY>(x, Wg, T, d, E, t0, xs, ws, acc);
    } else {
        if (full) router_sums<EP, KC, EXACT, false, IO_FULL>(x, Wg, T, d, E, t0, xs, ws, acc);
        else if (aligned && d % 4 == 0) router_sums<EP, KC, EXACT, false, IO_VEC>(x, Wg, T, d, E, t0, xs, ws, acc);
        else router_sums<EP, KC, EXACT, false, IO_ANY>(x, Wg, T, d, E, t0, xs, ws, acc);
    }
#pragma unroll
    for (int x_ = 0; x_ < EPT; ++x_) {
        const int e = e1 + x_ * EL;
        const float b = (bg != nullptr && e < E) ? bg[e] : 0.0f;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const float z = bg != nullptr ? acc[x_ * NT + i] + b : acc[x_ * NT + i];
            lg[tg + i * TPP][e] = z;
            const int t = t0 + tg + i * TPP;
            if (logits_out != nullptr && t < T && e < E) logits_out[(size_t)t * E + e] = z;
        }
    }
    __syncthreads();

    router_select<EP, false, TOK_TILE, NTHR>(lg, hist, t0, tile, T, E, K, renorm, ids, wout, tile_counts, probs_out);
}

// FAST mode of bf16 layers with 32 experts or more: the gate projection on the matrix cores.  x and Wg are bf16, so
// every product is exact in fp32 and only the order of the additions differs from the sequential sum (tolerance
// mode by definition).  One workgroup = 32 tokens x EP experts = EP/32 blocks of v_mfma_f32_32x32x16_bf16; its four
// waves split the k range (partial sums are added in a fixed order through LDS) or, from 128 experts on, the blocks.  Operand fragments come straight from memory (16 bytes per lane; the 64 bytes a lane pair
// needs of a row per 32 k are fetched by consecutive loads, so every line is read once): the kernel moves x once
// (Wg stays in the L2) and has almost no arithmetic, it lives on loads in flight.
template <int EP>
__global__ __launch_bounds__(256) void router_mfma_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ Wg,
                                                          const float *__restrict__ bg, int T, int d, int E, int K,
                                                          int renorm, int32_t *__restrict__ ids, float *__restrict__ wout,
                                                          int32_t *__restrict__ tile_counts, float *__restrict__ logits_out,
                                                          float *__restrict__ probs_out)
{
    constexpr int TOK_TILE = 32;                // only layers with more than 16 experts take this kernel
    constexpr int NB = EP / 32;                 // expert blocks
    // up to 64 experts every wave takes all blocks and a quarter of k; from 128 on the waves split the blocks (measured:
    // 64 experts 0.064 -> 0.058 ms with the k split at T = 8192, d = 2048; 128 experts 0.125 -> 0.157 ms at T = 16384)
    constexpr int KS = NB <= 2 ? 4 : 1;         // k splits
    constexpr int BPW = NB <= 2 ? NB : NB / 4;  // expert blocks per wave
    __shared__ float lg[TOK_TILE][EP];
    __shared__ float part[KS > 1 ? KS : 1][KS > 1 ? TOK_TILE : 1][KS > 1 ? EP : 1];
    __shared__ int hist[EP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.x, t0 = tile * TOK_TILE;
    if (tid < EP) hist[tid] = 0;
    const int l32 = lane & 31, kh = lane >> 5;
    const int b0 = KS > 1 ? 0 : wave * BPW;           // first expert block of this wave
    const int ks = KS > 1 ? wave : 0;
    const int klen = d / KS, kbeg = ks * klen;        // d is a multiple of 256
    const bf16_t *xrow = x + (size_t)min(t0 + l32, T - 1) * d + kh * 8;
    const bf16_t *wrow[BPW];
#pragma unroll
    for (int b = 0; b < BPW; ++b) wrow[b] = Wg + (size_t)min((b0 + b) * 32 + l32, E - 1) * d + kh * 8;
    rt_f32x16 acc[BPW];
#pragma unroll
    for (int b = 0; b < BPW; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = 0.0f;
    // 64 k per trip: 4 MFMA steps of 16 k; the fragments of the next trip are loaded while this one computes
    rt_bf16x8 xa[2][4], wb[2][BPW][4];
    auto fetch = [&](int buf, int k0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            xa[buf][q] = *(const rt_bf16x8 *)(xrow + k0 + q * 16);
#pragma unroll
            for (int b = 0; b < BPW; ++b) wb[buf][b][q] = *(const rt_bf16x8 *)(wrow[b] + k0 + q * 16);
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int b = 0; b < BPW; ++b)
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[buf][q], wb[buf][b][q], acc[b], 0, 0, 0);
    };
    const int kend = kbeg + klen;  // klen is a multiple of 64
    int k0 = kbeg;
    fetch(0, k0);
    for (; k0 + 128 <= kend; k0 += 128) {
        fetch(1, k0 + 64);
        compute(0);
        fetch(0, min(k0 + 128, kend - 64));  // (past the end: re-reads the last trip, never used)
        compute(1);
    }
    if (k0 < kend) compute(0);  // an odd number of trips: the last one sits in buffer 0
    // lane: expert column l32 of its block; register r -> token 8*(r/4) + 4*kh + r%4
#pragma unroll
    for (int b = 0; b < BPW; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int tt = 8 * (r >> 2) + 4 * kh + (r & 3), e = (b0 + b) * 32 + l32;
            if (KS > 1) part[ks][tt][e] = acc[b][r];
            else lg[tt][e] = acc[b][r];
        }
    __syncthreads();
    for (int i = tid; i < TOK_TILE * EP; i += 256) {
        const int tt = i / EP, e = i % EP;
        float z;
        if (KS > 1) {
            z = part[0][tt][e];
#pragma unroll
            for (int q = 1; q < KS; ++q) z = z + part[q][tt][e];
        } else {
            z = lg[tt][e];
        }
        if (bg != nullptr && e < E) z = z + bg[e];
        lg[tt][e] = z;
        if (logits_out != nullptr && t0 + tt < T && e < E) logits_out[(size_t)(t0 + tt) * E + e] = z;
    }
    __syncthreads();
    router_select<EP, true>(lg, hist, t0, tile, T, E, K, renorm, ids, wout, tile_counts, probs_out);
}

// Exact sums of bf16 layers with more than 16 experts on the matrix cores.  v_mfma_f32_16x16x4_f32 forms each element of
// its result as fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, c)))): a chain of them over k = 0..3, 4..7, ... is the
// sequential sum, term for term (checked bit for bit against fmaf, exponents from one end of the range to the other); the
// products of bf16 operands are exact in fp32, so it is also the unfused sum of the exact mode.  An instruction takes four k
// of 16 tokens x 16 experts where v_mfma_f32_16x16x1_4b_f32 takes one k of 16 x 64: the same rate per matrix core, but
// chains a quarter as long (d/4 instructions of 44 cycles; 32 where a SIMD has two chains), and four times as many of them.
// Bound: the chain while the tiles find a SIMD per unit (d = 2048: 512 x 44 cycles = 10 us), then the fp32 matrix rate
// (16384 tokens x 128 experts: 62 us).  A wave holds CE expert units x CT token units; the workgroup has TT tokens.  Operands: lane
// l supplies token (expert) l % 16 and k = 4 q + l / 16 of instruction q.  x passes through LDS as fp32, two buffers of RM_KC
// columns, every 16 columns stored [k % 4][k / 4] so that a lane's four instructions' worth is one 16-byte read; the gate
// comes from an fp32 image in that very order (router_pack_gate_kernel, made when the weights change), 1 KiB per wave and 16
// k straight from the L2, up to 16 such loads ahead.
// Router launch, us, one k per instruction -> four: 48 and 1500 tokens, d = 2048, 64 experts: 50 -> 18.5; 8192 tokens: 53 -> 34;
// 16384 tokens, 128 experts: 100 -> 88; 300 tokens, 128 experts: 58 -> 29.5; 8192 tokens, 200 experts: 164 -> 82; 4096 tokens,
// d = 1024, 32 experts: 26 -> 11.  The tolerance mode's kernel (router_mfma_kernel) is as fast up to 1500 tokens and faster
// behind (8192 tokens 20, 16384 tokens 67), where this one is bound by the fp32 matrix rate.
#define RM_KC 256
#define RM_LDW (RM_KC + 4)
typedef __attribute__((ext_vector_type(4))) float rt_f32x4;

// Wg [E,d] bf16 -> fp32 [unit of 16 experts][k / 16][lane][4]: lane l, value q = Wg[16 unit + l % 16][16 (k/16) + 4 q + l / 16]
__global__ __launch_bounds__(256) void router_pack_gate_kernel(const bf16_t *__restrict__ Wg, int E, int d, int units, float4 *__restrict__ img)
{
    const int KB = d >> 4;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < units * KB * 64; i += gridDim.x * 256) {
        const int l = i & 63, kb = (i >> 6) % KB, e = (i >> 6) / KB * 16 + (l & 15), k = 16 * kb + (l >> 4);
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (e < E) {
            const bf16_t *w = Wg + (size_t)e * d + k;
            v = make_float4(bf16_to_f32(w[0]), bf16_to_f32(w[4]), bf16_to_f32(w[8]), bf16_to_f32(w[12]));
        }
        img[i] = v;
    }
}

template <int EP, int TT, int NW, int CE, int CT>
__global__ __launch_bounds__(64 * NW) void router_units_kernel(const bf16_t *__restrict__ x, const float4 *__restrict__ img,
                                                               const float *__restrict__ bg, int T, int d, int E, int K, int renorm,
                                                               int32_t *__restrict__ ids, float *__restrict__ wout,
                                                               int32_t *__restrict__ tile_counts, float *__restrict__ logits_out,
                                                               float *__restrict__ probs_out)
{
    constexpr int NTHR = 64 * NW, EU = EP / 16, NWE = EU / CE;  // waves across the experts
    static_assert(NWE * (TT / 16 / CT) == NW, "every unit has one wave");
    constexpr int XV = TT * RM_KC / 8 / NTHR;                    // 16-byte pieces of x per thread and chunk
    static_assert(XV * NTHR * 8 == TT * RM_KC, "whole pieces per thread");
    constexpr int PD = CE > 2 ? 2 : 16 / CE, BPC = RM_KC / 16;         // gate loads in flight; 16-k blocks per chunk
    __shared__ __attribute__((aligned(16))) float xs[2][TT][RM_LDW];
    __shared__ int hist[EP];
    static_assert(EP <= RM_LDW, "the logits take the place of the staged rows");
    float(*lg)[EP] = (float(*)[EP]) & xs[0][0][0];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int tile = blockIdx.x, t0 = tile * TT;
    for (int i = tid; i < EP; i += NTHR) hist[i] = 0;
    const int u0 = (wave % NWE) * CE, tu0 = (wave / NWE) * CT;   // first expert unit, first token unit of this wave
    const int KB = d >> 4, nch = d / RM_KC;
    const bool live = 16 * u0 < E && t0 + 16 * tu0 < T;          // a wave without experts or tokens only stages
    const bool aligned = ((uintptr_t)x & 15) == 0;

    uint4 xr[XV];
    auto fetch = [&](int c) {
#pragma unroll
        for (int v = 0; v < XV; ++v) {
            const int i = tid + v * NTHR;
            const bf16_t *p = x + (size_t)min(t0 + i / (RM_KC / 8), T - 1) * d + c * RM_KC + (i % (RM_KC / 8)) * 8;
            if (aligned) xr[v] = *(const uint4 *)p;
            else xr[v] = make_uint4(p[0] | (uint32_t)p[1] << 16, p[2] | (uint32_t)p[3] << 16, p[4] | (uint32_t)p[5] << 16, p[6] | (uint32_t)p[7] << 16);
        }
    };
    auto stash = [&](int c) {
#pragma unroll
        for (int v = 0; v < XV; ++v) {
            const int i = tid + v * NTHR, k8 = i % (RM_KC / 8);
            float *o = &xs[c & 1][i / (RM_KC / 8)][(k8 >> 1) * 16 + (k8 & 1) * 2];  // k = 8 k8 + j: [j % 4][2 (k8 % 2) + j / 4]
            *(float2 *)(o + 0) = make_float2(__uint_as_float(xr[v].x << 16), __uint_as_float(xr[v].z << 16));
            *(float2 *)(o + 4) = make_float2(__uint_as_float(xr[v].x & 0xffff0000u), __uint_as_float(xr[v].z & 0xffff0000u));
            *(float2 *)(o + 8) = make_float2(__uint_as_float(xr[v].y << 16), __uint_as_float(xr[v].w << 16));
            *(float2 *)(o + 12) = make_float2(__uint_as_float(xr[v].y & 0xffff0000u), __uint_as_float(xr[v].w & 0xffff0000u));
        }
    };
    const float4 *wp[CE];
#pragma unroll
    for (int e = 0; e < CE; ++e) wp[e] = img + (size_t)min(u0 + e, (E - 1) >> 4) * KB * 64 + lane;
    float4 wb[PD][CE];
    rt_f32x4 acc[CT][CE];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int e = 0; e < CE; ++e)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][e][r] = 0.0f;

    fetch(0);
    if (live)
#pragma unroll
        for (int b = 0; b < PD; ++b)
#pragma unroll
            for (int e = 0; e < CE; ++e) wb[b][e] = wp[e][(size_t)b * 64];
    stash(0);
    for (int c = 0; c < nch; ++c) {
        __syncthreads();  // chunk c is staged, and chunk c - 1 summed
        if (c + 1 < nch) fetch(c + 1);
        if (live) {
            const float *xp = &xs[c & 1][16 * tu0 + l16][4 * lq];
#pragma unroll
            for (int b = 0; b < BPC; ++b) {
                float4 xa[CT], w[CE];
#pragma unroll
                for (int t = 0; t < CT; ++t) xa[t] = *(const float4 *)(xp + t * 16 * RM_LDW + b * 16);
#pragma unroll
                for (int e = 0; e < CE; ++e) {
                    w[e] = wb[b % PD][e];
                    wb[b % PD][e] = wp[e][(size_t)min(c * BPC + b + PD, KB - 1) * 64];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int t = 0; t < CT; ++t)
#pragma unroll
                        for (int e = 0; e < CE; ++e)
                            acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(((const float *)&xa[t])[q], ((const float *)&w[e])[q], acc[t][e], 0, 0, 0);
            }
        }
        if (c + 1 < nch) stash(c + 1);
    }
    __syncthreads();
    // lane: expert l16 of unit u0 + e; register r -> token 4 lq + r of unit tu0 + t
    if (live)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int e = 0; e < CE; ++e) {
                const int ex = 16 * (u0 + e) + l16;
                const float bias = bg != nullptr && ex < E ? bg[ex] : 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int tt = 16 * (tu0 + t) + 4 * lq + r;
                    const float z = bg != nullptr ? acc[t][e][r] + bias : acc[t][e][r];
                    lg[tt][ex] = z;
                    if (logits_out != nullptr && t0 + tt < T && ex < E) logits_out[(size_t)(t0 + tt) * E + ex] = z;
                }
            }
    __syncthreads();
    router_select<EP, false, TT, NTHR>(lg, hist, t0, tile, T, E, K, renorm, ids, wout, tile_counts, probs_out);
}

// Batches of at most one 16-token tile per compute unit, bf16, at most 16 experts (d is a multiple of 256: the
// last chunk may be half full; 90 tokens x 3328, 7 experts, on the kernel above 46 us, here 17; 777 x 2304, 16 experts 35 -> 16): the whole
// kernel is as long as ONE chain of d dependent multiply-adds (about 6 clocks a term on a SIMD that has no second wave
// to fill them), so everything else is taken out of the waves that run the chains.  The workgroup has two kinds of
// waves: 16*EP/64 sum waves, one lane per (token, expert), that only read LDS and add; and two staging waves that
// carry the NEXT 512-k chunk of x and Wg from memory to a second LDS buffer as fp32 while the current one is summed.
// One barrier per chunk, executed by every wave of both kinds (B_c: chunk c is staged, and chunk c-1 is summed - so
// its buffer may take chunk c+1).  The terms are the exact fp32 products of bf16 operands, added in k order by
// fused multiply-adds: the same bits as the separate multiply and add of the sequential sum, in either router mode.
#define RP_KC 512
#define RP_LDW (RP_KC + 4)
// SPLIT (more than 16 experts): `groups` workgroups per token tile take 16 experts each and leave the logits in logits_out, for
// router_select_kernel: where those find a compute unit each, a chain of the vector units' and a launch more are shorter than one
// of the matrix cores' in a workgroup that fetches the whole gate.  Router, us, matrix cores -> here: 1 token x 3328, 86 experts
// 38.6 -> 19.5; 2 x 3072, 26 experts 22.2 -> 16.3; 48 x 2048, 64 experts 18.2 -> 15.7; 109 x 3328, 83 experts 39 -> 21.5; 500 x 2048, 128 experts 27.7 ->
// 21.0; 1 x 2048, 250 experts 44 -> 17.7.
#define RP_STAGERS 128
template <int EP, bool SPLIT>
__global__ __launch_bounds__(16 * EP + RP_STAGERS) void router_pipe_kernel(
    const bf16_t *__restrict__ x, const bf16_t *__restrict__ Wg, const float *__restrict__ bg, int T, int d, int E_all, int K,
    int renorm, int32_t *__restrict__ ids, float *__restrict__ wout, int32_t *__restrict__ tile_counts,
    float *__restrict__ logits_out, float *__restrict__ probs_out, int groups, int tpw)
{
    constexpr int TT = 16, CT = 16 * EP, ST = RP_STAGERS, KC = RP_KC, LDW = RP_LDW;
    const int tile = SPLIT ? blockIdx.x / groups : blockIdx.x, e0 = SPLIT ? (blockIdx.x - tile * groups) * EP : 0;
    const int E = SPLIT ? min(EP, E_all - e0) : E_all;
    Wg += (size_t)e0 * d;
    if (bg != nullptr) bg += e0;
    extern __shared__ __attribute__((aligned(16))) float rp_smem[];
    float(*xs)[TT][LDW] = (float(*)[TT][LDW])rp_smem;                  // [2][TT][LDW]
    float(*ws)[EP][LDW] = (float(*)[EP][LDW])(rp_smem + 2 * TT * LDW);  // [2][EP][LDW]
    __shared__ float lg[TT][EP];
    __shared__ int hist[EP];
    const int tid = threadIdx.x, t0 = tile * (SPLIT ? tpw : TT);
    if (SPLIT) T = min(T, t0 + tpw);  // (tokens behind are another workgroup's)
    if (!SPLIT && tid < EP) hist[tid] = 0;
    const int nch = (d + KC - 1) / KC;  // (the last chunk of an odd multiple of 256 is half full)
    if (tid >= CT) {
        // staging wave: thread st carries 8 consecutive k (16 bytes of bf16) of one row per load
        const int st = tid - CT;
        constexpr int XCH = TT * (KC / 8) / ST, WCH = EP * (KC / 8) / ST;
        static_assert(TT * (KC / 8) % ST == 0 && EP * (KC / 8) % ST == 0, "whole vectors per staging thread");
        // (a second chunk of loads in flight gained nothing: the sum waves, bound by their LDS reads, set the pace)
        uint4 xr[XCH], wr[WCH];
        auto fetch = [&](int k0) {
#pragma unroll
            for (int c = 0; c < XCH; ++c) {
                const int idx = st + c * ST;
                xr[c] = *(const uint4 *)(x + (size_t)min(t0 + idx / (KC / 8), T - 1) * d + min(k0 + (idx % (KC / 8)) * 8, d - 8));
            }
#pragma unroll
            for (int c = 0; c < WCH; ++c) {
                const int idx = st + c * ST;
                wr[c] = *(const uint4 *)(Wg + (size_t)min(idx / (KC / 8), E - 1) * d + min(k0 + (idx % (KC / 8)) * 8, d - 8));
            }
        };
        auto widen = [&](const uint4 &v, float *dst) {
            *(float4 *)dst = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                                         __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
            *(float4 *)(dst + 4) = make_float4(__uint_as_float(v.z << 16), __uint_as_float(v.z & 0xffff0000u),
                                               __uint_as_float(v.w << 16), __uint_as_float(v.w & 0xffff0000u));
        };
        fetch(0);
        for (int c = 0; c < nch; ++c) {
            const int b = c & 1;
#pragma unroll
            for (int q = 0; q < XCH; ++q) {
                const int idx = st + q * ST;
                widen(xr[q], &xs[b][idx / (KC / 8)][(idx % (KC / 8)) * 8]);
            }
#pragma unroll
            for (int q = 0; q < WCH; ++q) {
                const int idx = st + q * ST;
                widen(wr[q], &ws[b][idx / (KC / 8)][(idx % (KC / 8)) * 8]);
            }
            if (c + 1 < nch) fetch((c + 1) * KC);
            __syncthreads();  // B_c
        }
    } else {
        const int e1 = tid % EP, tg = tid / EP;
        // a wave whose lowest token is past the end of the batch forms no sum; it keeps the barriers
        const bool wave_live = t0 + (tid & ~63) / EP < T;
        float a_ = 0.0f;
        for (int c = 0; c < nch; ++c) {
            __syncthreads();  // B_c
            if (!wave_live) continue;
            const float4 *wp = (const float4 *)&ws[c & 1][e1][0], *xp = (const float4 *)&xs[c & 1][tg][0];
            float4 wa[8], xa[8], wb[8], xb[8];
#define ROUTER_LD(W, X, g)                                    \
    _Pragma("unroll") for (int j = 0; j < 8; ++j)             \
    {                                                         \
        W[j] = wp[(g) * 8 + j];                               \
        X[j] = xp[(g) * 8 + j];                               \
    }
#define ROUTER_FM(W, X)                                       \
    _Pragma("unroll") for (int j = 0; j < 8; ++j)             \
    {                                                         \
        a_ = fmaf(X[j].x, W[j].x, a_);                        \
        a_ = fmaf(X[j].y, W[j].y, a_);                        \
        a_ = fmaf(X[j].z, W[j].z, a_);                        \
        a_ = fmaf(X[j].w, W[j].w, a_);                        \
    }
            // the LDS reads of the next 32 k are in flight while the terms of the current 32 are added (the fences
            // keep the reads where they are written: ahead of the other set's terms)
            auto sum = [&](auto groups) {  // of 32 k (the number is known at compile time: the loop unrolls)
                ROUTER_LD(wa, xa, 0)
#pragma unroll
                for (int g = 0; g < decltype(groups)::value; g += 2) {
                    __builtin_amdgcn_sched_barrier(0);
                    ROUTER_LD(wb, xb, g + 1)
                    __builtin_amdgcn_sched_barrier(0);
                    ROUTER_FM(wa, xa)
                    __builtin_amdgcn_sched_barrier(0);
                    if (g + 2 < decltype(groups)::value) {
                        ROUTER_LD(wa, xa, g + 2)
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    ROUTER_FM(wb, xb)
                }
            };
            if (d - c * KC >= KC) sum(std::integral_constant<int, KC / 32>());
            else sum(std::integral_constant<int, KC / 64>());
#undef ROUTER_LD
#undef ROUTER_FM
        }
        const float z = (bg != nullptr && e1 < E) ? a_ + bg[e1] : a_;
        if (!SPLIT) lg[tg][e1] = z;
        if ((SPLIT || logits_out != nullptr) && t0 + tg < T && e1 < E) logits_out[(size_t)(t0 + tg) * E_all + e0 + e1] = z;
    }
    if (SPLIT) return;
    __syncthreads();
    if (tid < CT) {
        router_select<EP, false, TT, CT>(lg, hist, t0, tile, T, E, K, renorm, ids, wout, tile_counts, probs_out);
    } else {
        __syncthreads();  // the staging waves keep the two barriers of the selection
        __syncthreads();
    }
}

// Selection from logits in memory, a workgroup per 16 tokens
template <int EP>
__global__ __launch_bounds__(256) void router_select_kernel(const float *__restrict__ logits, int T, int E, int K, int renorm,
                                                            int32_t *__restrict__ ids, float *__restrict__ wout,
                                                            int32_t *__restrict__ tile_counts, float *__restrict__ probs_out)
{
    __shared__ float lg[16][EP];
    __shared__ int hist[EP];
    const int tid = threadIdx.x, t0 = blockIdx.x * 16;
    for (int i = tid; i < EP; i += 256) hist[i] = 0;
    for (int i = tid; i < 16 * EP; i += 256) {
        const int tt = i / EP, e = i % EP;
        lg[tt][e] = e < E && t0 + tt < T ? logits[(size_t)(t0 + tt) * E + e] : 0.0f;
    }
    __syncthreads();
    router_select<EP, false, 16, 256>(lg, hist, t0, blockIdx.x, T, E, K, renorm, ids, wout, tile_counts, probs_out);
}

int router_pipe_smem_bytes(int EP) { return 2 * (16 + EP) * RP_LDW * (int)sizeof(float); }

hipError_t router_init(void)
{
    const struct { const void *f; int ep; } fns[] = {{(const void *)router_pipe_kernel<8, false>, 8}, {(const void *)router_pipe_kernel<16, false>, 16},
                                                     {(const void *)router_pipe_kernel<16, true>, 16}};
    for (const auto &k : fns) {
        hipError_t e = hipFuncSetAttribute(k.f, hipFuncAttributeMaxDynamicSharedMemorySize, router_pipe_smem_bytes(k.ep));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_router(const omega_moe *m, const void *x, int T, float *logits_out, float *probs_out, hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const int tiles = ceil_div(T, router_tok_tile(m, T));
    const int exact = c.router_mode == OMEGA_ROUTER_EXACT;
    const float *bg = c.has_gate_bias ? m->bg : nullptr;
    if (!exact && router_on_mfma(m) && ((uintptr_t)x % 16) == 0) {
#define ROUTER_MFMA_LAUNCH(EPV)                                                                                          \
    hipLaunchKernelGGL(router_mfma_kernel<EPV>, dim3(tiles), dim3(256), 0, s, (const bf16_t *)x, (const bf16_t *)m->Wg, bg, T, \
                       c.d, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, logits_out, probs_out)
        if (c.E <= 32) ROUTER_MFMA_LAUNCH(32);
        else if (c.E <= 64) ROUTER_MFMA_LAUNCH(64);
        else if (c.E <= 128) ROUTER_MFMA_LAUNCH(128);
        else ROUTER_MFMA_LAUNCH(256);
#undef ROUTER_MFMA_LAUNCH
        return hipGetLastError();
    }
    // (tokens per workgroup of the split form: the fewest that leave a workgroup a compute unit of its own, 4 are one wave of sums.
    // Rows have to be long enough to pay for the second launch, and the longer the fewer experts share a workgroup's chain on the matrix
    // cores.  One launch / two, us, around each line: 500 tokens x 1280, 20 experts 12.2 / 12.1, 640 x 1280 12.2 / 12.6, 1000 x 1536 13.9 / 13.7; 64
    // experts, 64 x 1280 12.8 / 12.7, 64 x 1536 14.6 / 13.4, 33 experts, 500 x 1536 14.0 / 14.4, 500 x 2048 16.9 / 16.4; 100 experts, 200 x 512 11.9 / 13.1,
    // 200 x 768 14.8 / 14.2, 500 x 768 14.9 / 15.6, 500 x 1024 17.5 / 16.5; 200 experts, 60 x 256 13.6 / 16.5, 60 x 512 18.2 / 16.0.)
    const int groups = ceil_div(c.E, 16);
    int tpw = 4;
    while (tpw < 16 && ceil_div(T, tpw) * groups > m->ctx->num_cus) tpw *= 2;
    const int split_d = c.E > 128 ? 512 : c.E > 64 ? (tpw < 16 ? 768 : 1024) : tpw == 16 ? INT_MAX : c.E > 32 ? (tpw < 8 ? 1536 : 2048) : (tpw < 8 ? 1280 : 1536);
    if (router_on_mfma(m) && (logits_out != nullptr || m->gate_logits != nullptr) && router_tok_tile(m, T) == 16 &&
        ceil_div(T, tpw) * groups <= m->ctx->num_cus && c.d >= split_d && (((uintptr_t)x | (uintptr_t)m->Wg) % 16) == 0) {
        float *lg = logits_out != nullptr ? logits_out : m->gate_logits;
        hipLaunchKernelGGL((router_pipe_kernel<16, true>), dim3(ceil_div(T, tpw) * groups), dim3(16 * 16 + RP_STAGERS), router_pipe_smem_bytes(16),
                           s, (const bf16_t *)x, (const bf16_t *)m->Wg, bg, T, c.d, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, lg,
                           (float *)nullptr, groups, tpw);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
#define ROUTER_SELECT(EPV) \
    hipLaunchKernelGGL(router_select_kernel<EPV>, dim3(tiles), dim3(256), 0, s, (const float *)lg, T, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, probs_out)
        if (c.E <= 32) ROUTER_SELECT(32);
        else if (c.E <= 64) ROUTER_SELECT(64);
        else if (c.E <= 128) ROUTER_SELECT(128);
        else ROUTER_SELECT(256);
#undef ROUTER_SELECT
        return hipGetLastError();
    }
    if (router_on_mfma(m)) {
        const int units = ceil_div(c.E, 16), tt = router_tok_tile(m, T);
        if (!m->gate_img_valid) {
            const int n = units * (c.d / 16) * 64;
            hipLaunchKernelGGL(router_pack_gate_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, (const bf16_t *)m->Wg, c.E, c.d, units,
                               (float4 *)m->gate_img);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            m->gate_img_valid = true;
        }
#define ROUTER_UNITS(EPV, TTV, NWV, CEV, CTV)                                                                            \
    hipLaunchKernelGGL((router_units_kernel<EPV, TTV, NWV, CEV, CTV>), dim3(tiles), dim3(64 * NWV), 0, s, (const bf16_t *)x, \
                       (const float4 *)m->gate_img, bg, T, c.d, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, logits_out, probs_out)
        if (c.E <= 32) { if (tt == 16) ROUTER_UNITS(32, 16, 2, 1, 1); else ROUTER_UNITS(32, 32, 4, 1, 1); }
        else if (c.E <= 64) { if (tt == 16) ROUTER_UNITS(64, 16, 4, 1, 1); else ROUTER_UNITS(64, 32, 4, 1, 2); }
        else if (c.E <= 128) { if (tt == 16) ROUTER_UNITS(128, 16, 4, 2, 1); else ROUTER_UNITS(128, 32, 8, 1, 2); }
        else { if (tt == 16) ROUTER_UNITS(256, 16, 4, 4, 1); else ROUTER_UNITS(256, 32, 8, 2, 2); }
#undef ROUTER_UNITS
        return hipGetLastError();
    }
    // at most 16 experts, bf16, at most one tile per compute unit: chains fed by staging waves (either mode: same bits)
    if (c.dtype == OMEGA_DTYPE_BF16 && c.E <= 16 && tiles <= m->ctx->num_cus &&
        (((uintptr_t)x | (uintptr_t)m->Wg) % 16) == 0) {
        if (c.E <= 8)
            hipLaunchKernelGGL((router_pipe_kernel<8, false>), dim3(tiles), dim3(16 * 8 + RP_STAGERS), router_pipe_smem_bytes(8), s,
                               (const bf16_t *)x, (const bf16_t *)m->Wg, bg, T, c.d, c.E, c.K, c.renorm, m->ids, m->w,
                               m->tile_counts, logits_out, probs_out, 1, 16);
        else
            hipLaunchKernelGGL((router_pipe_kernel<16, false>), dim3(tiles), dim3(16 * 16 + RP_STAGERS), router_pipe_smem_bytes(16), s,
                               (const bf16_t *)x, (const bf16_t *)m->Wg, bg, T, c.d, c.E, c.K, c.renorm, m->ids, m->w,
                               m->tile_counts, logits_out, probs_out, 1, 16);
        return hipGetLastError();
    }
#define ROUTER_LAUNCH(EPV, KCV)                                                                                    \
    do {                                                                                                           \
        if (exact)                                                                                                 \
            hipLaunchKernelGGL((router_kernel<EPV, KCV, true>), dim3(tiles), dim3(ROUTER_NTHR(EPV)), 0, s, x, c.dtype, m->Wg, bg, \
                               T, c.d, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, logits_out, probs_out);   \
        else                                                                                                       \
            hipLaunchKernelGGL((router_kernel<EPV, KCV, false>), dim3(tiles), dim3(ROUTER_NTHR(EPV)), 0, s, x, c.dtype, m->Wg,    \
                               bg, T, c.d, c.E, c.K, c.renorm, m->ids, m->w, m->tile_counts, logits_out,           \
                               probs_out);                                                                         \
    } while (0)
    if (c.E <= 8) ROUTER_LAUNCH(8, ROUTER_KC_SMALL);
    else if (c.E <= 16) ROUTER_LAUNCH(16, ROUTER_KC_SMALL);
    else if (c.E <= 32) ROUTER_LAUNCH(32, 128);
    else if (c.E <= 64) ROUTER_LAUNCH(64, 64);
    else if (c.E <= 128) ROUTER_LAUNCH(128, 64);
    else ROUTER_LAUNCH(256, 64);
#undef ROUTER_LAUNCH
    return hipGetLastError();
}
