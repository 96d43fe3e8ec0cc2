// Combine: out[t,:] = sum_j w[t,j] * y[row of pair t*K+j,:] in slot order, then + the shared experts' rows
// (rows are the physical rows the dispatch stage assigned; shared expert s owns rows first_tile[E+s]*bm + t).
// One to eight waves per token, each with a share of the columns; each lane owns 4 (fp32 out) or 8 (bf16 out) consecutive columns, read from the
// fp32 rows of y with 16-byte loads; products and sums are separate fp32 operations in slot order
// (this file is compiled with -ffp-contract=off), the weighted sum of add_mul_kernel
// (J/engine/gpu/BaseKernel.cu:228-241) generalised to K terms; shared rows are added as add_kernel
// (J/engine/ad/op/gpu/OPKernel.cu:359-366).  No atomics: every output element has one writer.
#include "common.h"
#include <algorithm>

// The slices of KU rows of y (SL below) added to what the lane holds of them, VEC columns from c0 on.  Lanes whose tile has fewer
// slices than others' read a row again and drop it: no branch keeps the loads from being in flight together.
template <int KU, int VEC>
__device__ __forceinline__ void add_slices(float4 (&v)[KU][VEC / 4], const int (&rows)[KU], int d, int c0, const float *__restrict__ y,
                                           const float *__restrict__ slabs, const int32_t *__restrict__ slab_tab)
{
    const int nct = d >> 8, ct = c0 >> 8;
    int ent[KU], most = 0;
#pragma unroll
    for (int u = 0; u < KU; ++u) ent[u] = slab_tab[(size_t)(rows[u] >> 5) * nct + ct];
#pragma unroll
    for (int u = 0; u < KU; ++u) most = max(most, (ent[u] >> 9) & 15);
    if (__ballot(most > 1) == 0) return;
    const bool more = __ballot(most > 5) != 0;
    constexpr int SB = KU < 2 ? KU : 2;  // rows whose slices are in flight together
#pragma unroll
    for (int u0 = 0; u0 < KU; u0 += SB) {
        for (int s0 = 1; s0 < (more ? 8 : 4); s0 += 4) {
            float4 w[SB][4][VEC / 4];  // slices s0 .. s0 + 3
#pragma unroll
            for (int u = 0; u < SB && u0 + u < KU; ++u) {
                const int e = ent[u0 + u], row = rows[u0 + u], ks = (e >> 9) & 15;
                const float *tile = slabs + (size_t)(e & 511) * 65536 + (size_t)((e >> 13) * 32 + (row & 31)) * 256 + (c0 & 255);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const float *p = s0 + s < ks ? tile + (size_t)(s0 + s) * 65536 : y + (size_t)row * d + c0;
#pragma unroll
                    for (int q = 0; q < VEC / 4; ++q) w[u][s][q] = ((const float4 *)p)[q];
                }
            }
#pragma unroll
            for (int u = 0; u < SB && u0 + u < KU; ++u) {
                const int ks = (ent[u0 + u] >> 9) & 15;
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (s0 + s < ks) {
#pragma unroll
                        for (int q = 0; q < VEC / 4; ++q) {
                            v[u0 + u][q].x = v[u0 + u][q].x + w[u][s][q].x;
                            v[u0 + u][q].y = v[u0 + u][q].y + w[u][s][q].y;
                            v[u0 + u][q].z = v[u0 + u][q].z + w[u][s][q].z;
                            v[u0 + u][q].w = v[u0 + u][q].w + w[u][s][q].w;
                        }
                    }
            }
        }
    }
}

// KU: slots (and shared experts behind them) whose rows are fetched together before any of them is used (all loads of a
// group are in flight at once).  Their number is exact up to eight: a row read twice costs what it weighs when y passes the cache
// by (9978 tokens, a routed and two shared rows each, four reads instead of three: pass 982 -> 998 us; groups of exact size 994 against 1005
// with the shared rows one after the other).  Rows, weights and the shared experts' places are asked for together, and a row costs no
// branch: 1500 tokens x 2048, 6 + 2 rows 17.3 -> 17.1 us (pass 361.5 -> 360.7), 48 tokens 3.06 -> 2.90, 3000 x 1024, 4 + 1 rows 11.7 -> 11.5.
// resid != nullptr (block form): the row of x is added to the fp32 sum before the output is rounded
// (Tensor_OP().add(mlp out, tmp1, tmp2), J/engine/nn/layer/llama/LlamaTransformerBlock.java:136).
// NT: the rows of y are read with non-temporal loads.  They are read exactly once; when y is larger than the last-level
// cache (256 MiB) letting them pass it by is worth 13 % (8192 tokens, 64 experts: 0.143 -> 0.125 ms; 16384 tokens, 128
// experts: 0.260 -> 0.225 ms), below that size nothing.
// SL: the batch's down product left k slices of some tiles in `slabs` (y_slabs) and `slab_tab` says which: entry [32-row block of
// the buffer][column tile] = first slice's place | slices << 9 | block within the tile << 13, 0 for a tile that is whole in y.
// They are added here, to the row of y and in slice order - the sums down_slab_reduce_kernel forms -, while the rows are in
// registers anyway: a launch and a round trip of y less.  (That kernel is left to what reads y itself: training, backward
// passes, omega_moe_get_workspace.)  Whole passes, reduce and combine / combine, us: 777 tokens x 4096 x 14336, 8 experts, top 2 (2
// slices of every tile) 630 / 624, 256 x 4096 x 7168 302 / 293, 4096 x 4096 x 14336 (4 slices of the last 64 tiles) 2208-2224 / 2210-2215.
// Rows in groups of four, two rows' slices in flight: 148 registers, three waves per SIMD; eight rows at a time, as
// without slices, and half of them in flight took 256, one wave, and lost where the table has few slices or none (the host knows bounds of
// the tiles only).  Combine, us, eight at a time / now: 1100 tokens x 4096, 8 experts of 4096, top 8 60.6 / 41.1 (pass 763 / 751, with the
// reduce launch 753); 300 x 2048, 64 experts, 6 + 2 rows, no slices 10.5 / 8.7; 200 x 1024, 6 + 2 rows, 6 slices of every tile 15.2 /
// 15.8 (one row's slices in flight 17.8, registers capped at 128 22.0); 4 rows: 300 x 2048 7.1 / 7.4, 200 x 1024 11.4 / 11.2, 1100 x 4096 26.8 / 25.4.
template <int VEC, bool BF16, int KU, bool NT, bool SL>
__global__ __launch_bounds__(256) void combine_kernel(const float *__restrict__ y, const int32_t *__restrict__ dst,
                                                      const float *__restrict__ w, int T, int K, int d, int Es,
                                                      const int32_t *__restrict__ tile_meta, int E, int bm,
                                                      const void *__restrict__ resid, void *__restrict__ out, int split,
                                                      const float *__restrict__ slabs, const int32_t *__restrict__ slab_tab, int dc)
{
    // `split` waves share a token, each taking dc consecutive columns, the last one what is left (more waves, more loads in
    // flight, when the batch has few tokens for the compute units there are)
    const int lane = threadIdx.x & 63;
    const int wv = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int t = wv / split, part = wv - t * split;
    if (t >= T) return;
    const int cend = min((part + 1) * dc, d);
    // lane j < K holds row index and weight of slot j, lane j < Es the row of shared expert j; handed out by lane reads
    // (bf16: without branches, the three loads travel together; fp32 batches, without shared experts for the most part, are
    // 0.1 of 23.4 us faster at 256 tokens x 128 without the third)
    const size_t slot = (size_t)t * K + min(lane, K - 1);
    const int myrow = dst[slot], shrow = BF16 || Es > 0 ? tile_meta[1 + E + min(lane, max(Es - 1, 0))] * bm + t : 0;
    const float myw = w[slot];
    const bool sliced = SL && tile_meta[E + Es + 9] > 0;  // (the host knows bounds of the number of tiles only)
    const int n = K + Es;
    // (lanes past the row's end work on column 0 and store nothing)
    for (int cb = part * dc; cb < cend; cb += 64 * VEC) {
        const bool on = cb + lane * VEC < cend;
        const int c0 = on ? cb + lane * VEC : 0;
        float acc[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = 0.0f;
        // the rows of the slots, then those of the shared experts, KU at a time
        for (int j0 = 0; j0 < n; j0 += KU) {
            float4 buf[KU][VEC / 4];
            int rows[KU];
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const int j = min(j0 + u, n - 1);  // (a last group with a row too few reads that of the last again)
                rows[u] = j < K ? __builtin_amdgcn_readlane(myrow, j) : __builtin_amdgcn_readlane(shrow, j - K);
                const float4 *src = (const float4 *)(y + (size_t)rows[u] * d + c0);
#pragma unroll
                for (int q = 0; q < VEC / 4; ++q) {
                    if (NT) {
                        typedef float v4f __attribute__((ext_vector_type(4)));
                        const v4f t4 = __builtin_nontemporal_load((const v4f *)(src + q));
                        buf[u][q] = make_float4(t4.x, t4.y, t4.z, t4.w);
                    } else {
                        buf[u][q] = src[q];
                    }
                }
            }
            if (SL && sliced) add_slices<KU, VEC>(buf, rows, d, c0, y, slabs, slab_tab);
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                // (a shared row's weight is one, and the product its value: a branch less per row)
                const float wj = j0 + u < K ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myw), j0 + u)) : 1.0f;
                if (j0 + u < n) {
#pragma unroll
                    for (int q = 0; q < VEC / 4; ++q) {
                        const float4 v4 = buf[u][q];
                        float term;
                        term = wj * v4.x; acc[q * 4 + 0] = acc[q * 4 + 0] + term;
                        term = wj * v4.y; acc[q * 4 + 1] = acc[q * 4 + 1] + term;
                        term = wj * v4.z; acc[q * 4 + 2] = acc[q * 4 + 2] + term;
                        term = wj * v4.w; acc[q * 4 + 3] = acc[q * 4 + 3] + term;
                    }
                }
            }
        }
        if (resid != nullptr) {
            if (BF16) {
                const uint4 u = *(const uint4 *)((const bf16_t *)resid + (size_t)t * d + c0);
                const uint32_t uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int v = 0; v < VEC / 2; ++v) {
                    acc[2 * v] = acc[2 * v] + __uint_as_float(uu[v] << 16);
                    acc[2 * v + 1] = acc[2 * v + 1] + __uint_as_float(uu[v] & 0xffff0000u);
                }
            } else {
                const float4 r4 = *(const float4 *)((const float *)resid + (size_t)t * d + c0);
                acc[0] = acc[0] + r4.x; acc[1] = acc[1] + r4.y; acc[2] = acc[2] + r4.z; acc[3] = acc[3] + r4.w;
            }
        }
        if (!on) continue;
        if (BF16) {
            uint32_t pk[VEC / 2];
#pragma unroll
            for (int v = 0; v < VEC / 2; ++v)
                pk[v] = (uint32_t)f32_to_bf16(acc[2 * v]) | ((uint32_t)f32_to_bf16(acc[2 * v + 1]) << 16);
            uint4 o = {pk[0], pk[1], pk[2], pk[3]};
            *(uint4 *)((bf16_t *)out + (size_t)t * d + c0) = o;
        } else {
            float4 o = {acc[0], acc[1], acc[2], acc[3]};
            *(float4 *)((float *)out + (size_t)t * d + c0) = o;
        }
    }
}

// Any d: scalar columns.
template <bool BF16>
__global__ __launch_bounds__(256) void combine_scalar_kernel(const float *__restrict__ y, const int32_t *__restrict__ dst,
                                                             const float *__restrict__ w, int T, int K, int d, int Es,
                                                             const int32_t *__restrict__ tile_meta, int E, int bm,
                                                             const void *__restrict__ resid, void *__restrict__ out)
{
    const int t = blockIdx.x;
    for (int c = threadIdx.x; c < d; c += 256) {
        float acc = 0.0f;
        for (int j = 0; j < K; ++j) {
            const float term = w[(size_t)t * K + j] * y[(size_t)dst[(size_t)t * K + j] * d + c];
            acc = acc + term;
        }
        for (int s = 0; s < Es; ++s) acc = acc + y[((size_t)tile_meta[1 + E + s] * bm + t) * d + c];
        if (resid != nullptr)
            acc = acc + (BF16 ? bf16_to_f32(((const bf16_t *)resid)[(size_t)t * d + c]) : ((const float *)resid)[(size_t)t * d + c]);
        if (BF16) ((bf16_t *)out)[(size_t)t * d + c] = f32_to_bf16(acc);
        else ((float *)out)[(size_t)t * d + c] = acc;
    }
}

hipError_t launch_combine(const omega_moe *m, int T, void *out, const void *resid, hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const bool bf = c.dtype == OMEGA_DTYPE_BF16;
    const int vec = bf ? 8 : 4;
    if (combine_by_vectors(m, out, resid)) {
        const bool nt = (size_t)T * (c.K + c.Es) * c.d * 4 > OMEGA_LLC_BYTES;
        // several waves per token, each with a share of the columns, until the launch has 256 waves per compute unit:
        // more loads in flight (4096 tokens x 4096 columns: 36.3 -> 30.6 us with 8 waves per token; 64 tokens:
        // 12.0 -> 6.9 us; 8192 tokens x 2048 columns x 8 rows: 122.6 -> 113.8 us with 4; 16384 tokens: 228 -> 210 us;
        // shares are whole trips of a wave, the last may be less: 90 tokens x 3328 columns, top 3, 7.3 -> 3.8 us with seven for one)
        const int trips = ceil_div(c.d, 64 * vec);
        int want = 1;
        while (want < 8 && (long long)T * want < 256LL * m->ctx->num_cus) want *= 2;
        const int dc = ceil_div(trips, std::min(want, trips)) * 64 * vec, split = ceil_div(c.d, dc);
        const bool sl = m->y_partial;
        const int n = c.K + c.Es, ku = ceil_div(n, ceil_div(n, sl ? 4 : 8));  // rows of a token in groups of one size, eight at most
        const int grid = ceil_div(T * split, 4);
#define COMBINE_LAUNCH(VECV, BFV, KUV, NTV, SLV)                                                                                       \
    hipLaunchKernelGGL((combine_kernel<VECV, BFV, KUV, NTV, SLV>), dim3(grid), dim3(256), 0, s, m->y, m->dstp, m->w, T, c.K, c.d, c.Es, \
                       m->tile_meta, c.E, m->bm, resid, out, split, m->y_slabs, m->slab_tab, dc)
#define COMBINE_SLOTS(VECV, BFV, NTV)                           \
    do {                                                         \
        switch (ku) {                                            \
        case 1: COMBINE_LAUNCH(VECV, BFV, 1, NTV, false); break; \
        case 2: COMBINE_LAUNCH(VECV, BFV, 2, NTV, false); break; \
        case 3: COMBINE_LAUNCH(VECV, BFV, 3, NTV, false); break; \
        case 4: COMBINE_LAUNCH(VECV, BFV, 4, NTV, false); break; \
        case 5: COMBINE_LAUNCH(VECV, BFV, 5, NTV, false); break; \
        case 6: COMBINE_LAUNCH(VECV, BFV, 6, NTV, false); break; \
        case 7: COMBINE_LAUNCH(VECV, BFV, 7, NTV, false); break; \
        default: COMBINE_LAUNCH(VECV, BFV, 8, NTV, false);       \
        }                                                        \
    } while (0)
#define COMBINE_SLICED(NTV)                              \
    do {                                                  \
        switch (ku) {                                     \
        case 1: COMBINE_LAUNCH(8, true, 1, NTV, true); break; \
        case 2: COMBINE_LAUNCH(8, true, 2, NTV, true); break; \
        case 3: COMBINE_LAUNCH(8, true, 3, NTV, true); break; \
        default: COMBINE_LAUNCH(8, true, 4, NTV, true);       \
        }                                                 \
    } while (0)
        if (sl && nt) COMBINE_SLICED(true);
        else if (sl) COMBINE_SLICED(false);
        else if (bf && nt) COMBINE_SLOTS(8, true, true);
        else if (bf) COMBINE_SLOTS(8, true, false);
        else if (nt) COMBINE_SLOTS(4, false, true);
        else COMBINE_SLOTS(4, false, false);
#undef COMBINE_SLICED
#undef COMBINE_SLOTS
#undef COMBINE_LAUNCH
    } else {
        if (bf)
            hipLaunchKernelGGL(combine_scalar_kernel<true>, dim3(T), dim3(256), 0, s, m->y, m->dstp, m->w, T, c.K, c.d,
                               c.Es, m->tile_meta, c.E, m->bm, resid, out);
        else
            hipLaunchKernelGGL(combine_scalar_kernel<false>, dim3(T), dim3(256), 0, s, m->y, m->dstp, m->w, T, c.K, c.d,
                               c.Es, m->tile_meta, c.E, m->bm, resid, out);
    }
    return hipGetLastError();
}
