// Expert products of bf16 layers for batches of a few tokens (decode): every expert that is used has one row tile of at most
// 16 * UM rows, and the products are as long as streaming its weights takes.
//   up    a[r,h] = silu(xg[r,:].W1g[h,:]) * (xg[r,:].W3g[h,:])   -> packed bf16
//   down  y[r,c] = a[r,:].W2g[c,:]                                -> fp32 rows
// (the products of experts_bf16.hip, J/engine/nn/layer/llama/LlamaMLPLayer.java:117-130.)
//
// Bound: HBM, 3 d H weights of two bytes per expert used.  The tile kernels keep five k steps of a 256-column item in flight
// per compute unit, in LDS, and a launch has few items: 6 experts of H = 768 are 36 for 256 compute units, 66 of d = 2048 are
// 2.06 rounds of 256-column items in the down product.  Here a workgroup takes 16 or 32 columns of W1 and of W3 (down: 32 or 64 of W2)
// of one expert, its waves share k, and each wave streams its blocks of the packed image straight into registers: a 1 KiB
// block is one MFMA fragment (16 rows x 32 k, lane l row l % 16, chunk l / 16), one coalesced 16-byte load per lane, past the
// last-level cache since nobody reads it again.  PF steps of loads are in flight per wave and 16 waves per compute unit.  The
// partial sums meet in LDS, added in wave order.  Rows come from x through the row -> token table, or from the packed copy.
// Forward pass, us, tile kernels -> here: 1 / 16 / 64 tokens, d = 4096, H = 14336, 8 experts, top 2: 144 -> 132, 482 -> 452, 470 -> 458
// (up product 6.6 TB/s of weights, 6.4 at 64 tokens); 16 / 48 tokens, d = 2048, H = 1408, 64 experts, top 6, 2 shared: 193 -> 163,
// 226 -> 209; 2 tokens, d = 3072, H = 768, 4 experts, 2 shared: 86 -> 48; 4 tokens, d = 1024, H = 1024, 64 experts, top 4: 53 -> 37.
#include "index_small.h"
#include "pack.h"
#include <algorithm>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 few_bf16x8;
typedef __attribute__((ext_vector_type(4))) float few_f32x4;
typedef const __attribute__((address_space(1))) unsigned char *few_ptr;           // global memory (a pointer put together from scalar
typedef const __attribute__((address_space(1))) few_bf16x8 *few_frag_ptr;          // registers does not say so by itself)

struct few_args {
    const unsigned char *x;     // up: token rows (null: the packed copy in A); with copy_wgs: what the copy is made from
    const unsigned char *A;     // packed rows: xg (up), a (down)
    const unsigned char *As;    // up: packed rows of the shared experts
    const unsigned char *B0, *B1;  // W1, W3; down: W2, unused
    unsigned char *a;           // up: output
    float *y;                   // down: output
    const omega_tile *tiles;
    const int32_t *tile_meta, *tokp, *dstp;
    index_args index;           // up: the launch makes the dispatch index itself from index.ids, the router's choices (or null: it is there)
    unsigned char *xg, *xs;     // up: the gathered copy, written by copy_wgs workgroups behind the products'; the one that leaves the index is the last
    int copy_wgs, T, K;
    int N, Kd;                  // output columns and k
};

// The dispatch index within the up launch.  A batch's pairs are so few that a workgroup finds its expert and rows from the router's choices in the
// time that reading them out of the index takes (three dependent loads), so nothing has to run in front of the product but the router;
// the index itself - what dispatch_rank_kernel leaves - is made by a workgroup of its own beside the products, the launch's last: the products'
// workgroups keep their XCDs, four that share the lines of a row group on XCDs 0-3 or 4-7 (moved on by one, two or three, 64 tokens x 4096 x 14336, 8
// experts, up product 278 -> 307, 327, 307 us).  Forward pass, us, with a launch for the index / without: 1 and 64 tokens x 4096 x 14336, 8 experts,
// top 2 132.1 -> 127.2, 454.5 -> 449; 48 tokens x 2048 x 1408, 64 experts, top 6, 2 shared 202 -> 195.6
#define FEW_BM 256         // rows of a tile: every expert that is used has one
struct few_shared {
    uint8_t flag[256];      // experts that have rows
    uint8_t id[INDEX_IN_UP_PAIRS];
    uint8_t tok[64];        // tokens of the workgroup's rows
};
struct few_used { unsigned long long m[4]; };  // the flags as bits, uniform

// The choices of all pairs, and who is chosen at all
__device__ __forceinline__ few_used few_choices(const few_args &p, few_shared &sh, int lane, int wave, int waves)
{
    const int P = p.T * p.K;
    if (wave == 0) ((uint32_t *)sh.flag)[lane] = 0u;
    __syncthreads();
    for (int i0 = 64 * wave; i0 < P; i0 += 64 * waves) {
        const int e = i0 + lane < P ? p.index.ids[i0 + lane] : 0;
        if (i0 + lane < P) {
            sh.id[i0 + lane] = (uint8_t)e;
            sh.flag[e] = 1;
        }
    }
    __syncthreads();
    few_used u;
#pragma unroll
    for (int q = 0; q < 4; ++q) u.m[q] = __ballot(sh.flag[64 * q + lane] != 0);
    return u;
}
// experts below e that have rows: e's row tile
__device__ __forceinline__ int few_tile(const few_used &us, int e)
{
    int n = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) n += __popcll(64 * q + 64 <= e ? us.m[q] : 64 * q < e ? us.m[q] & ((1ull << (e & 63)) - 1ull) : 0ull);
    return n;
}
// pairs before pair u (uniform over the wave) with its expert: its rank among that expert's rows
__device__ __forceinline__ int few_rank(const few_shared &sh, int u, int lane)
{
    const int e = sh.id[u];
    int n = 0;
    for (int c = 0; c < u; c += 64) n += __popcll(__ballot(c + lane < u && sh.id[c + lane] == e));
    return n;
}
// Row tile `mt` of the batch (the used experts in rising order, then the shared ones) and the tokens of its rows; every wave by itself
__device__ __forceinline__ omega_tile few_find(const few_args &p, few_shared &sh, const few_used &us, int mt, int n_used, int lane)
{
    omega_tile tl;
    tl.row0 = mt * FEW_BM;
    if (mt >= n_used) {
        tl.g = p.index.E + mt - n_used;
        tl.rows = p.T;
        tl.xrow0 = 0;
        return tl;
    }
    tl.xrow0 = -1;
    tl.g = 0;
    int k = mt;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = __popcll(us.m[q]);
        if (k >= 0 && k < c) tl.g = 64 * q + __ffsll(__ballot((us.m[q] >> lane & 1ull) && __popcll(us.m[q] & ((1ull << lane) - 1ull)) == k)) - 1;
        k -= c;
    }
    const int P = p.T * p.K;
    int n = 0;
    for (int c = 0; c < P; c += 64) {
        const bool mine = c + lane < P && sh.id[c + lane] == tl.g;
        const unsigned long long m = __ballot(mine);
        if (mine) sh.tok[n + __popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)((c + lane) / p.K);  // (each wave the same)
        n += __popcll(m);
    }
    tl.rows = n;
    return tl;
}
// Wave per row of the copy (a pair's row of xg, then the token rows of xs): what the dispatch launch does for larger batches,
// beside the products instead of in front of them
template <bool SELF>
__device__ __forceinline__ void few_copy(const few_args &p, const few_shared &sh, const few_used &us, int wg, int lane, int wave, int waves)
{
    const int KT = p.Kd >> 5, P = p.T * p.K, n = P + (p.xs != nullptr ? p.T : 0);
    for (int u = wg * waves + wave; u < n; u += waves * p.copy_wgs) {
        const int t = u < P ? u / p.K : u - P;
        const int row = u >= P ? t : SELF && p.index.ids != nullptr ? few_tile(us, sh.id[u]) * FEW_BM + few_rank(sh, u, lane) : p.dstp[u];
        const unsigned char *src = p.x + (size_t)t * p.Kd * 2;
        unsigned char *dst = u < P ? p.xg : p.xs;
        for (int c = lane; c < 4 * KT; c += 64) *(uint4 *)(dst + pk_chunk_off(row, c >> 2, c & 3, KT)) = *(const uint4 *)(src + (size_t)c * 16);
    }
}

// k steps in flight per wave: what 128 registers, four waves per SIMD, leave.  (Tiles of four units with four blocks have room for one step
// and spill three registers, one in the down product: stored once in front of the k loop and read once behind it.)
constexpr int few_depth(int U, int NB)
{
    const int d = (104 - 4 * U * NB) / (4 * (U + NB));
    return d > 8 * 2 / NB ? 8 * 2 / NB : d;
}

// The sums of n k steps for the fragments at A + a_off[u] + step * a_step and b[q] + b_off[q] + step * 8192 (bases uniform over the
// wave: they sit in scalar registers, and a load costs no address arithmetic in the lanes)
template <int U, int NB, int PF>
__device__ __forceinline__ void few_sums(few_ptr A, const uint32_t (&a_off)[U], uint32_t a_step, const few_ptr (&b)[NB],
                                         const uint32_t (&b_off)[NB], int n, few_f32x4 (&acc)[U][NB])
{
    few_bf16x8 fa[PF][U], fb[PF][NB];
    auto load = [&](int i, int s) {
        const uint32_t sb = (uint32_t)s * 8192u, sa = (uint32_t)s * a_step;
#pragma unroll
        for (int q = 0; q < NB; ++q) fb[i][q] = __builtin_nontemporal_load((few_frag_ptr)(b[q] + sb + b_off[q]));
#pragma unroll
        for (int u = 0; u < U; ++u) fa[i][u] = *(few_frag_ptr)(A + sa + a_off[u]);
    };
    auto mul = [&](int i) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < NB; ++q) acc[u][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[i][q], fa[i][u], acc[u][q], 0, 0, 0);
    };
    if (n <= 0) return;
#pragma unroll
    for (int i = 0; i < PF; ++i) {
        load(i, min(i, n - 1));
        __builtin_amdgcn_sched_barrier(0);
    }
    int s = 0;
    for (; s + 2 * PF <= n; s += PF) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            mul(i);
            load(i, s + PF + i);
            __builtin_amdgcn_sched_barrier(0);  // (in any other order the waits would be for all PF steps at a time)
        }
    }
    const int rest = n - s - PF;  // steps still to be asked for (below zero: some of those asked for are not there)
#pragma unroll
    for (int i = 0; i < PF; ++i) {
        if (s + i < n) mul(i);
        if (i < rest) load(i, s + PF + i);
    }
#pragma unroll
    for (int i = 0; i < PF; ++i)
        if (i < rest) mul(i);
}

// UM: units of 16 rows a tile may have; NW: waves per workgroup; NB: 16-row blocks of weights per step (up: half W1's, half W3's)
// (SELF: the up product makes the dispatch index)
template <bool UP, int UM, int NW, int NB, bool SELF>
__global__ __launch_bounds__(64 * NW, 4) void few_rows_kernel(few_args p)
{
    __shared__ few_f32x4 part[UM > 1 ? 2 : 1][NW][NB][64];
    __shared__ few_shared sh;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    constexpr int NC = UP ? NB / 2 : NB;  // 16-column blocks of the output per workgroup
    const int nc = p.N / (16 * NC);
    const bool self = SELF && p.index.ids != nullptr;  // (asked of the arguments in a SELF kernel too: known to be so, four units of rows spill 14 registers, not 3, and 64
    // tokens x 4096 x 14336, 8 experts, take 473 us, not 451)
    const int blk = blockIdx.x;
    int n_used = 0;
    few_used us = {};
    if (self) {
        us = few_choices(p, sh, lane, wave, NW);
#pragma unroll
        for (int q = 0; q < 4; ++q) n_used += __popcll(us.m[q]);
        if (blk == (int)gridDim.x - 1) {
            static_assert(sizeof(part) >= 3 * 256 * sizeof(int), "room for the index");
            small_index(p.index, sh.id, (int *)part, FEW_BM, 64 * NW);
            return;
        }
    }
    const int copy0 = (int)gridDim.x - (self ? 1 : 0) - p.copy_wgs;
    if (UP && blk >= copy0) {
        few_copy<SELF>(p, sh, us, blk - copy0, lane, wave, NW);
        return;
    }
    // the row tiles in falling order, which takes the shared experts - all T rows - first
    const int wt = blk / nc, n0 = (blk - wt * nc) * (16 * NC);
    const int mt = (self ? n_used + p.index.Es : p.tile_meta[0]) - 1 - wt;
    if (mt < 0) return;
    omega_tile tl = self ? few_find(p, sh, us, mt, n_used, lane) : p.tiles[mt];
    tl = {__builtin_amdgcn_readfirstlane(tl.g), __builtin_amdgcn_readfirstlane(tl.row0), __builtin_amdgcn_readfirstlane(tl.rows),
          __builtin_amdgcn_readfirstlane(tl.xrow0)};
    const int KT = p.Kd >> 5, units = (tl.rows + 15) >> 4;
    const int s0 = wave * KT / NW, n = (wave + 1) * KT / NW - s0;
    // uniform: k step s0 of the workgroup's 16-row blocks of the weights; lane: its chunk of a block (the swizzle depends on the
    // row through l16 and bit 4)
    auto uniform = [](const unsigned char *q) {
        const uint64_t v = (uint64_t)q;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return (few_ptr)(((uint64_t)hi << 32) | lo);
    };
    const size_t wblk = (((size_t)((tl.g * (p.N >> 7)) + (n0 >> 7)) * KT + s0) * 8 + ((n0 & 127) >> 4)) << 10;
    few_ptr b[NB];
    uint32_t b_off[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int c = q % NC;
        b[q] = uniform((q < NC ? p.B0 : p.B1) + wblk + c * 1024);
        b_off[q] = (uint32_t)(l16 * 64 + ((lq ^ pk_swz(((NC > 1 ? 16 * c : n0) & 16) | l16)) << 4));
    }
    const bool gather = UP && p.x != nullptr && p.A == nullptr;
    const bool own = UP && !gather && tl.xrow0 >= 0;  // a shared expert's rows of the packed copy xs
    const int prow0 = own ? tl.xrow0 : tl.row0;         // packed rows: a multiple of 256
    const uint32_t a_step = gather ? 64u : 8192u;
    const few_ptr A = uniform(gather ? p.x + (size_t)s0 * 64 : (own ? p.As : p.A) + ((size_t)(prow0 >> 7) * KT + s0) * 8192u);
    auto run = [&](auto uc) {
        constexpr int U = decltype(uc)::value, PF = few_depth(U, NB);
        uint32_t a_off[U];  // the lane's chunk of unit u's rows (rows past the tile's: its first)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = 16 * u + l16 < tl.rows ? 16 * u + l16 : 0;
            a_off[u] = gather ? (uint32_t)(tl.xrow0 >= 0 ? tl.xrow0 + r : self ? (int)sh.tok[r] : p.tokp[tl.row0 + r]) * (uint32_t)(p.Kd * 2) + lq * 16
                              : (uint32_t)((r >> 4) * 1024 + (r & 15) * 64 + ((lq ^ pk_swz(r)) << 4));
        }
        few_f32x4 acc[U][NB];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < NB; ++q) acc[u][q] = few_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        few_sums<U, NB, PF>(A, a_off, a_step, b, b_off, n, acc);
        // unit after unit the waves' sums meet in LDS (two buffers: one barrier per unit); a wave per column block adds them up in
        // wave order.  Lane: row l16 of the unit, columns 4 lq .. of the block
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int q = 0; q < NB; ++q) part[u & (UM > 1 ? 1 : 0)][wave][q][lane] = acc[u][q];
            __syncthreads();
            for (int c = (wave + NW - u % NW) % NW; c < NC; c += NW) {
                const few_f32x4(*pt)[NB][64] = part[u & (UM > 1 ? 1 : 0)];
                few_f32x4 v = pt[0][c][lane], h3 = v;
                if (UP) h3 = pt[0][NC + c < NB ? NC + c : 0][lane];
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    v += pt[w][c][lane];
                    if (UP) h3 += pt[w][NC + c < NB ? NC + c : 0][lane];
                }
                const int r = 16 * u + l16, col = n0 + 16 * c;
                if (r >= tl.rows) continue;
                if (UP) {
                    float a[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[i] = v[i] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[i])) * h3[i];  // as the tile kernels
                    const uint2 o = {(uint32_t)f32_to_bf16(a[0]) | (uint32_t)f32_to_bf16(a[1]) << 16,
                                     (uint32_t)f32_to_bf16(a[2]) | (uint32_t)f32_to_bf16(a[3]) << 16};
                    *(uint2 *)(p.a + pk_chunk_off(tl.row0 + r, col >> 5, ((col & 16) >> 3) + (lq >> 1), p.N >> 5) + (lq & 1) * 8) = o;
                } else {
                    *(few_f32x4 *)(p.y + (size_t)(tl.row0 + r) * p.N + col + 4 * lq) = v;
                }
            }
        }
    };
    if (UM == 1 || units == 1) run(std::integral_constant<int, 1>());
    else if (UM == 2 || units == 2) run(std::integral_constant<int, UM < 2 ? UM : 2>());
    else if (units == 3) run(std::integral_constant<int, UM < 3 ? UM : 3>());
    else run(std::integral_constant<int, UM>());
}

// which: 0 up - the rows come from x unless there is a gathered copy, and one is left beside if the layer keeps one -, 1 down
hipError_t launch_experts_few(const omega_moe *m, const void *x, int T, int which, hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const bool gather = !m->xg_valid, copy = gather && !m->gather_on_load;
    few_args p = {};
    p.tiles = m->tiles;
    p.tile_meta = m->tile_meta;
    p.tokp = m->tokp;
    p.dstp = m->dstp;
    p.T = T;
    p.K = c.K;
    const int tiles = (int)std::min((long long)m->G, (long long)T * c.K + c.Es);  // groups that can have rows: one tile each
    if (which == 0) {
        p.x = (const unsigned char *)x;
        p.A = gather ? nullptr : (const unsigned char *)m->xg;
        p.As = (const unsigned char *)m->xs;
        p.B0 = (const unsigned char *)m->W1;
        p.B1 = (const unsigned char *)m->W3;
        p.a = (unsigned char *)m->a;
        p.N = c.H;
        p.Kd = c.d;
        if (m->index_in_up) p.index = index_args_of(m, T);
        if (copy) {
            p.xg = (unsigned char *)m->xg;
            p.xs = (unsigned char *)m->xs;
            p.copy_wgs = std::min(ceil_div(T * (c.K + (c.Es > 0 ? 1 : 0)), 4), m->ctx->num_cus);
        }
#define FEW_LAUNCH(UPV, UMV, NWV, NBV)                                                                                              \
    do {                                                                                                                            \
        const dim3 grid(tiles * (p.N / (UPV ? 8 * NBV : 16 * NBV)) + (p.index.ids != nullptr ? 1 : 0) + p.copy_wgs);                 \
        if (UPV && p.index.ids != nullptr) hipLaunchKernelGGL((few_rows_kernel<UPV, UMV, NWV, NBV, UPV>), grid, dim3(64 * NWV), 0, s, p); \
        else hipLaunchKernelGGL((few_rows_kernel<UPV, UMV, NWV, NBV, false>), grid, dim3(64 * NWV), 0, s, p);                       \
    } while (0)
        // Four blocks of weights per step from 17 tokens on (two units of rows: 64 tokens x 4096 x 14336, 8 experts, up product 326 ->
        // 294 us), two below (1 token 71 against 73, 1 token x 3328 x 896, 86 experts 12.0 against 15.9).  Two waves where four would
        // have 8 k steps each or fewer, which is all start-up (64 tokens x 1024 x 768, 128 experts: pass 133 -> 128.5; d = 1536 169
        // against 173).
        const bool brief = c.d <= 1024;
        if (T <= 16) FEW_LAUNCH(true, 1, 4, 2);
        else if (T <= 32 && brief) FEW_LAUNCH(true, 2, 2, 4);
        else if (T <= 32) FEW_LAUNCH(true, 2, 4, 4);
        else if (brief) FEW_LAUNCH(true, 4, 2, 4);
        else FEW_LAUNCH(true, 4, 4, 4);
    } else {
        p.A = (const unsigned char *)m->a;
        p.B0 = (const unsigned char *)m->W2;
        p.y = m->y;
        p.N = c.d;
        p.Kd = c.H;
        // 64 columns per workgroup where that leaves one for every compute unit (3 tokens x 3328 x 13952, 9 experts: 126 -> 118 us;
        // 1 token x 4096 x 14336, 2 experts used, 128 workgroups: 40 -> 47, not taken)
        const bool wide = tiles * (c.d / 64) >= m->ctx->num_cus;
        if (T <= 16 && wide) FEW_LAUNCH(false, 1, 8, 4);
        else if (T <= 16) FEW_LAUNCH(false, 1, 8, 2);
        else if (T <= 32 && wide) FEW_LAUNCH(false, 2, 8, 4);
        else if (T <= 32) FEW_LAUNCH(false, 2, 8, 2);
        else if (wide) FEW_LAUNCH(false, 4, 8, 4);
        else FEW_LAUNCH(false, 4, 8, 2);
#undef FEW_LAUNCH
    }
    return hipGetLastError();
}
