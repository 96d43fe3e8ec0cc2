// What the two kernels of the fp32 products (experts_f32.hip, experts_f32_split.hip) share: arguments, the choices of a few pairs, the gathered copy, a
// tile on fp32 MFMAs, and which tiles go in parts.
#pragma once
#include "index_small.h"
#include <algorithm>
#include <type_traits>

struct f32_args {
    const float *A0, *A1;    // A operand; A1: F32_DXG second pair, F32_WG13 the second gradient's delta
    const float *Atok;       // shared groups: token rows instead of physical rows (or null)
    const int32_t *tokp;     // F32_UP: routed rows come from Atok through this row -> token table (or null: from A0) ...
    float *xg;               // ... and the launch's last `copy_wgs` workgroups leave the gathered rows here
    const int32_t *dstp;     // pair -> row
    index_args index;        // F32_UP, tiles of 32 rows: the launch makes the dispatch index itself (index.ids not null)
    int copy_wgs, K;
    const float *B0, *B1;    // weights (F32_UP, F32_RAW: W1 and W3; F32_DXG: second pair), F32_WG*: the layer input rows
    const float *Btok;       // F32_WG*: as Atok
    float *C, *H1, *H3;      // output; h1 / h3 (F32_UP: kept when not null; F32_RAW: written; F32_DA: read, then dh1 / dh3)
    const omega_tile *tiles;
    const int32_t *tile_meta, *counts;
    int N, Kd;               // row products: output columns and k; F32_WG*: columns and rows of one dW (k is the group's rows)
    int E, G, T, bm;
    wgrad_deal deal;         // F32_WG*: how the tiles go to the XCDs
    int slots, part_max, few;  // workgroups an XCD holds at a time; tiles of a last round, and of a launch without a whole one, that go in parts
};

#define F32_IS_WG(OP) ((OP) == F32_WG2 || (OP) == F32_WG13)
#define F32_PAIR(OP) ((OP) == F32_UP || (OP) == F32_RAW)

// The choices of a batch of few pairs in every wave's registers, for an up product that makes its own index
#define F32_SELF_CHUNKS (INDEX_IN_UP_PAIRS / 64)
template <int NC>
struct f32_choices {
    int id[NC];                // choice of pair 64 c + lane, -1 behind the last (every loop over the chunks is straight: its branches cost more than its sums)
    int first, tiles;          // first: lane e < E: the experts' first row tile; tiles: those of the routed experts
    int count;                 // lane e < E: pairs of expert e
    __device__ __forceinline__ void read(const f32_args &p, int lane)
    {
        const int P = p.T * p.K;
#pragma unroll
        for (int c = 0; c < NC; ++c) id[c] = p.index.ids[min(64 * c + lane, P - 1)];
#pragma unroll
        for (int c = 0; c < NC; ++c) id[c] = 64 * c + lane < P ? id[c] : -1;
        first = count = tiles = 0;
        for (int e = 0; e < p.E; ++e) {
            int n = 0;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                n += __popcll(__ballot(id[c] == e));
            first = lane == e ? tiles : first;
            count = lane == e ? n : count;
            tiles += (n + F32_TILE_M_SMALL - 1) / F32_TILE_M_SMALL;
        }
    }
    // row tile mt, and the tokens of its rows, to LDS; every wave by itself
    __device__ __forceinline__ omega_tile find(const f32_args &p, int mt, int lane, uint16_t *tok) const
    {
        omega_tile tl;
        tl.row0 = mt * F32_TILE_M_SMALL;
        if (mt >= tiles) {
            const int per = (p.T + F32_TILE_M_SMALL - 1) / F32_TILE_M_SMALL, s = (mt - tiles) / per;
            tl.g = p.E + s;
            tl.xrow0 = (mt - tiles - s * per) * F32_TILE_M_SMALL;
            tl.rows = min(F32_TILE_M_SMALL, p.T - tl.xrow0);
            return tl;
        }
        const int nt = (count + F32_TILE_M_SMALL - 1) / F32_TILE_M_SMALL;
        tl.g = __ffsll(__ballot(lane < p.E && first <= mt && mt < first + nt)) - 1;
        tl.xrow0 = -1;
        const int r0 = (mt - __builtin_amdgcn_readlane(first, tl.g)) * F32_TILE_M_SMALL;
        tl.rows = min(F32_TILE_M_SMALL, __builtin_amdgcn_readlane(count, tl.g) - r0);
        int n = -r0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const unsigned long long m = __ballot(id[c] == tl.g);
            const int rank = n + __popcll(m & ((1ull << lane) - 1ull));
            if (id[c] == tl.g && rank >= 0 && rank < F32_TILE_M_SMALL) tok[rank] = (uint16_t)((64 * c + lane) / p.K);
            n += __popcll(m);
        }
        return tl;
    }
    // The index, by the four waves of a workgroup, every fourth chunk of pairs each: what small_index leaves, from registers (its LDS
    // atomics and one wave's chain of ranks would outlast the products of such a batch)
    __device__ __forceinline__ void leave(const index_args &p, int lane, int wave) const
    {
        const int per = (p.T + F32_TILE_M_SMALL - 1) / F32_TILE_M_SMALL;
        int r[NC] = {}, row[NC] = {}, off = 0, at = 0;
        for (int e = 0; e < p.E; ++e) {
            const int row0 = __builtin_amdgcn_readlane(first, e) * F32_TILE_M_SMALL;
            int n = 0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const unsigned long long m = __ballot(id[c] == e);
                const int rank = n + __popcll(m & ((1ull << lane) - 1ull));
                r[c] = id[c] == e ? off + rank : r[c];
                row[c] = id[c] == e ? row0 + rank : row[c];
                n += __popcll(m);
            }
            at = lane == e ? off : at;
            off += n;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if ((c & 3) != wave || id[c] < 0) continue;
            const int i = 64 * c + lane, t = i / p.K;
            p.dst[i] = r[c];
            p.dstp[i] = row[c];
            p.src_row[r[c]] = t;
            p.tokp[row[c]] = t;
        }
        if (wave > 0) return;
        if (lane < p.E) {
            p.counts[lane] = count;
            p.offsets[lane] = at;
            p.tile_meta[1 + lane] = first;
            for (int q = 0; q < count; q += F32_TILE_M_SMALL)
                p.tiles[first + q / F32_TILE_M_SMALL] = {lane, first * F32_TILE_M_SMALL + q, min(F32_TILE_M_SMALL, count - q), -1};
        }
        for (int s = lane; s <= p.Es; s += 64) p.tile_meta[1 + p.E + s] = tiles + s * per;
        for (int q = lane; q < p.Es * per; q += 64) {
            const int s = q / per, x = (q - s * per) * F32_TILE_M_SMALL;
            p.tiles[tiles + q] = {p.E + s, (tiles + q) * F32_TILE_M_SMALL, min(F32_TILE_M_SMALL, p.T - x), x};
        }
        if (lane == 0) {
            p.offsets[p.E] = off;
            p.tile_meta[0] = tiles + p.Es * per;
        }
    }
    // row of pair u (uniform over the wave)
    __device__ __forceinline__ int row(const f32_args &p, int u, int lane) const
    {
        const int e = p.index.ids[u];
        int n = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            n += __popcll(__ballot(id[c] == e && 64 * c + lane < u));
        return __builtin_amdgcn_readlane(first, e) * F32_TILE_M_SMALL + n;
    }
};

// Gathered rows of a launch whose product workgroups fetch theirs from the tokens (a wave per token, the row read once and
// written to its K places): the backward pass reads them.  Beside the products instead of a launch in front of them.
// OWN: the places are found from the choices
template <bool VEC, bool OWN, class Choices>
__device__ __forceinline__ void copy_gathered(const f32_args &p, int wg, int lane, int wave, const Choices &own)
{
    const int d = p.Kd;
    for (int t = 4 * wg + wave; t < p.T; t += 4 * p.copy_wgs) {
        int row = 0;
        if constexpr (OWN) {
            for (int j = 0; j < p.K; ++j) {
                const int r = own.row(p, t * p.K + j, lane);
                row = lane == j ? r : row;
            }
        } else if (lane < p.K) row = p.dstp[(size_t)t * p.K + lane];
        const float *src = p.Atok + (size_t)t * d;
        for (int c0 = 0; c0 < d; c0 += VEC ? 256 : 64) {  // (every lane makes every trip: the cross-lane reads need them all)
            const int c = c0 + (VEC ? 4 : 1) * lane;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (c < d) {
                if (VEC) v = *(const float4 *)(src + c);
                else v.x = src[c];
            }
            for (int j = 0; j < p.K; ++j) {
                float *o = p.xg + (size_t)__shfl(row, j, 64) * d + c;
                if (c < d) {
                    if (VEC) *(float4 *)o = v;
                    else *o = v.x;
                }
            }
        }
    }
}

// matrix-core blocks of BS x BS: v_mfma_f32_32x32x2 (two k at a time, lane half = k) or v_mfma_f32_16x16x4 (four, lane
// quarter = k)
template <int BS> struct f32_block;
template <> struct f32_block<32> {
    typedef __attribute__((ext_vector_type(16))) float acc_t;
    static __device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
};
template <> struct f32_block<16> {
    typedef __attribute__((ext_vector_type(4))) float acc_t;
    static __device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

// LDS row stride in floats of an operand kept [row][FBK]: 16 consecutive rows start in 16 different groups of four banks
#define F32_LD_ROW (FBK + 4)
#define F32_FBK(TM) ((TM) == F32_TILE_M_SMALL ? 64 : 32)  // k places of a step
constexpr int f32_lds_floats(int tx, bool kmaj, int fbk) { return kmaj ? fbk * (tx + 4) : tx * (fbk + 4); }

// Pieces of one step of FBK k places that a thread carries: NV x 4 floats.  [row][k]: row r0 + (1024/FBK) u, 4 consecutive
// k; [k][column]: k place k0 + (1024/TX) u, 4 consecutive columns.
template <int TX, bool KMAJ, int FBK>
struct f32_piece {
    static constexpr int NV = TX * FBK / 1024;
    __device__ static __forceinline__ int x(int tid, int u) { return KMAJ ? 4 * (tid % (TX / 4)) : tid / (FBK / 4) + (1024 / FBK) * u; }
    __device__ static __forceinline__ int k(int tid, int u) { return KMAJ ? tid / (TX / 4) + (1024 / TX) * u : 4 * (tid % (FBK / 4)); }
    __device__ static __forceinline__ int lds(int tid, int u) { return KMAJ ? k(tid, u) * (TX + 4) + x(tid, u) : x(tid, u) * F32_LD_ROW + k(tid, u); }
};

// Piece u of a whole step: base = the step's first element (uniform), off = the thread's byte offset from it.  Without
// 16-byte loads the columns of a [k][column] piece are clamped one by one (ncols of them exist).
template <bool KMAJ, bool VEC>
__device__ __forceinline__ float4 fetch_piece(const float *base, uint32_t off, int x, int ncols)
{
    const float *q = (const float *)((const unsigned char *)base + off);
    if (VEC) return *(const float4 *)q;
    if (!KMAJ) return make_float4(q[0], q[1], q[2], q[3]);
    const int last = max(0, ncols - 1 - x);  // (q is the last column already where x lies past it)
    return make_float4(q[0], q[min(1, last)], q[min(2, last)], q[min(3, last)]);
}

// The last, partial step of kleft < FBK k places: those behind read as zero, addresses are clamped
template <int TX, bool KMAJ, int FBK>
__device__ __forceinline__ float4 fetch_partial(const float *base, uint32_t off, int tid, int u, int kleft, int ncols, int ld)
{
    float e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int k = f32_piece<TX, KMAJ, FBK>::k(tid, u) + (KMAJ ? 0 : q), kc = min(k, kleft - 1);
        const float *p = KMAJ ? base + (size_t)kc * ld + min(f32_piece<TX, KMAJ, FBK>::x(tid, u) + q, ncols - 1)
                              : (const float *)((const unsigned char *)base + off) - f32_piece<TX, KMAJ, FBK>::k(tid, u) + kc;
        const float w = *p;
        e[q] = k < kleft ? w : 0.0f;
    }
    return make_float4(e[0], e[1], e[2], e[3]);
}

// four k places of one block for this lane: LDS row / column x, places k .. k + 3
template <int TX, bool KMAJ, int FBK>
__device__ __forceinline__ float4 frag(const float *S, int x, int k)
{
    if (!KMAJ) return *(const float4 *)&S[x * F32_LD_ROW + k];
    return make_float4(S[k * (TX + 4) + x], S[(k + 1) * (TX + 4) + x], S[(k + 2) * (TX + 4) + x], S[(k + 3) * (TX + 4) + x]);
}

// a of h1 and h3; dh1 and dh3 of d(a)
__device__ __forceinline__ float f32_swiglu(float h1, float h3) { return (h1 / (1.0f + expf(-h1))) * h3; }
__device__ __forceinline__ void f32_swiglu_backward(float da, float h1, float h3, float &dh1, float &dh3)
{
    const float sg = 1.0f / (1.0f + expf(-h1));
    dh3 = da * (h1 * sg);
    dh1 = (da * h3) * sg * (1.0f + h1 * (1.0f - sg));
}

// One tile: row tile mt (tl) from its row r0 on (row products) or from row mt * TM of gradient matrix mat, and columns n0 ..; as and bs
// hold both operands of a row product twice.  (Weight gradients keep arrays of their own, and p is a copy: through pointers dW1 and dW3 of 4096 tokens x 1024
// x 3584, 8 experts, took 936 us instead of 915, in the tiles of 128 x 128 that such batches then had here.)
template <int OP, int TM, int TN, bool VEC>
__device__ __forceinline__ void f32_tile(const f32_args p, float *as, float *bs, int mt, const omega_tile tl, int r0, int n0, int mat, const uint16_t *tok = nullptr)
{
    constexpr bool WG = F32_IS_WG(OP), PAIR = F32_PAIR(OP);
    constexpr bool AK = WG, BK_ = WG || OP == F32_DA || OP == F32_DXG;  // operand contiguous across k
    constexpr int BS = TM == F32_TILE_M_SMALL ? 16 : 32, GK = 256 / BS, FBK = F32_FBK(TM);  // blocks; k places of a group
    static_assert(TM == 2 * BS, "a wave has one block of rows");
    constexpr int NB = TN / (2 * BS), NVA = TM * FBK / 1024, NVB = TN * FBK / 1024, NR = BS * BS / 64;
    typedef typename f32_block<BS>::acc_t acc_t;
    constexpr int CT = PAIR ? TN / 2 : TN;                             // output columns per tile
    constexpr int LA = f32_lds_floats(TM, AK, FBK), LB = f32_lds_floats(TN, BK_, FBK);
    __shared__ __attribute__((aligned(16))) float As[2][WG ? LA : 1];
    __shared__ __attribute__((aligned(16))) float Bs[2][WG ? LB : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lb = lane % BS, kh = lane / BS, wr = wave >> 1, wc = wave & 1;

    int g, rows, K1, row0 = 0, m0 = 0;
    const float *A0, *A1 = nullptr, *B0, *B1 = nullptr;
    bool fetch_rows = false;
    if (WG) {
        g = OP == F32_WG13 ? mat >> 1 : mat;
        const bool shared = g >= p.E;
        m0 = mt * TM;
        rows = min(TM, p.Kd - m0);
        K1 = shared ? p.T : p.counts[g];
        row0 = p.tile_meta[1 + g] * p.bm;
        const float *Ad = OP == F32_WG13 && (mat & 1) ? p.A1 : p.A0;
        A0 = shared && p.Atok ? p.Atok : Ad + (size_t)row0 * p.Kd;
        B0 = shared && p.Btok ? p.Btok : p.B0 + (size_t)row0 * p.N;
    } else {
        g = tl.g;
        rows = min(TM, tl.rows - r0);
        if (rows <= 0 || n0 >= p.N) return;  // (a part of a ragged tile)
        row0 = tl.row0 + r0;
        K1 = p.Kd;
        A0 = p.Atok && tl.xrow0 >= 0 ? p.Atok + (size_t)(tl.xrow0 + r0) * p.Kd : p.A0 + (size_t)row0 * p.Kd;
        fetch_rows = OP == F32_UP && p.tokp != nullptr && tl.xrow0 < 0;  // (up: through tokp, or tok)
        if (fetch_rows) A0 = p.Atok;
        if (OP == F32_DXG) A1 = p.A1 + (size_t)row0 * p.Kd;
        B0 = p.B0 + (size_t)g * p.N * p.Kd;
        if (PAIR || OP == F32_DXG) B1 = p.B1 + (size_t)g * p.N * p.Kd;
    }

    // Byte offsets of this thread's pieces from the step's first element (up: from W1's; the W3 columns add the distance).
    // Rows (columns) past the tile's edge repeat the last valid ones and are never stored.
    uint32_t oa[NVA], ob[NVB];
#pragma unroll
    for (int u = 0; u < NVA; ++u) {
        const int x = f32_piece<TM, AK, FBK>::x(tid, u), k = f32_piece<TM, AK, FBK>::k(tid, u);
        oa[u] = 4u * (AK ? (uint32_t)k * p.Kd + min(x, p.Kd - m0 - (VEC ? 4 : 1)) : (uint32_t)(!fetch_rows ? min(x, rows - 1) : tok != nullptr ? (int)tok[min(x, rows - 1)] : p.tokp[row0 + min(x, rows - 1)]) * K1 + k);
    }
#pragma unroll
    for (int u = 0; u < NVB; ++u) {
        const int x = f32_piece<TN, BK_, FBK>::x(tid, u), k = f32_piece<TN, BK_, FBK>::k(tid, u);
        ob[u] = 4u * (BK_ ? (uint32_t)k * p.N + min(x, p.N - n0 - (VEC ? 4 : 1)) : (uint32_t)min(PAIR && x >= CT ? x - CT : x, p.N - 1 - n0) * K1 + k);
    }

    // (first: F32_DXG's sum over the first pair.  One chain over both would carry 1.4 times the rounding error of two that are
    // added once: H = 3584, relative to float64, 1.57e-6 against 1.09e-6)
    acc_t acc[NB], first[OP == F32_DXG ? NB : 1];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            acc[n][r] = 0.0f;
            if (OP == F32_DXG) first[n][r] = 0.0f;
        }
    auto swap_first = [&]() {
        if constexpr (OP == F32_DXG) {
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const acc_t v = acc[n];
                acc[n] = first[n];
                first[n] = v;
            }
        }
    };

    // this wave's block: rows BS wr ..; columns: TN/2 wc + BS n (up: W1 columns BS wc, and the same of W3)
    const int xa = BS * wr + lb;
    int xb[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) xb[n] = (PAIR ? BS * wc + CT * n : (TN / 2) * wc + BS * n) + lb;

    const int S1 = K1 / FBK, steps = OP == F32_DXG ? 2 * S1 : S1;  // whole steps
    float4 va[NVA], vb[NVB];
    const float *a_at = AK ? A0 + m0 : A0, *b_at = BK_ ? B0 + n0 : B0 + (size_t)n0 * K1, *b3_at = PAIR ? B1 + (size_t)n0 * K1 : nullptr;
    auto fetch_a = [&](int u) { va[u] = fetch_piece<AK, VEC>(a_at, oa[u], f32_piece<TM, AK, FBK>::x(tid, u), p.Kd - m0); };
    auto fetch_b = [&](int u) {
        vb[u] = fetch_piece<BK_, VEC>(PAIR && u >= NVB / 2 ? b3_at : b_at, ob[u], f32_piece<TN, BK_, FBK>::x(tid, u), p.N - n0);
    };
    auto put_a = [&](int c, int u) { *(float4 *)&(WG ? As[c] : as + c * LA)[f32_piece<TM, AK, FBK>::lds(tid, u)] = va[u]; };
    auto put_b = [&](int c, int u) { *(float4 *)&(WG ? Bs[c] : bs + c * LB)[f32_piece<TN, BK_, FBK>::lds(tid, u)] = vb[u]; };
    // the load pointers move on to step s (which the next loads bring); behind the last one they stay
    auto advance = [&](int s) {
        if (s >= steps) return;
        a_at += AK ? (size_t)FBK * p.Kd : FBK;
        b_at += BK_ ? (size_t)FBK * p.N : FBK;
        if (PAIR) b3_at += FBK;
        if (OP == F32_DXG && s == S1) {
            a_at = A1;
            b_at = B1 + n0;
        }
    };
    // All steps for a wave whose block has rows (LIVE) or none.  One group = GK k of the step in buffer c: its MFMAs on the fragments
    // read during the group before, and spread between them (pinned, a quarter of the group at a time) the reads of the
    // next group's fragments and the group's share of the step's other work: group 0 writes the next step's pieces to the
    // other buffer, group 1 asks for those of the step behind it; the barrier lies in front of the last group, whose
    // fragment reads are the next step's first.  (Everything between two barriers of a step reads buffer c and writes
    // buffer 1 - c, except that last group's reads of 1 - c, which every wave has finished writing.)
    auto run = [&](auto live) {
        constexpr bool LIVE = decltype(live)::value;
        constexpr int NF = LIVE ? 1 + NB : 0;
        float4 fa[2], fb[2][NB];
        auto read = [&](int set, int c, int j, int r) {
            const int k = GK * j + 4 * kh;
            if (r == 0) fa[set] = frag<TM, AK, FBK>(WG ? As[c] : as + c * LA, xa, k);
            else if (r < NF) fb[set][r - 1 < NB ? r - 1 : 0] = frag<TN, BK_, FBK>(WG ? Bs[c] : bs + c * LB, xb[r - 1 < NB ? r - 1 : 0], k);
        };
        auto group = [&](auto cc, auto jj) {
            constexpr int c = decltype(cc)::value, j = decltype(jj)::value;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (NF > 0) read((j + 1) & 1, j == 3 ? 1 - c : c, (j + 1) & 3, q);
                if (j == 0) {
#pragma unroll
                    for (int u = q; u < NVA; u += 4) put_a(1 - c, u);
#pragma unroll
                    for (int u = q; u < NVB; u += 4) put_b(1 - c, u);
                } else if (j == 1) {
#pragma unroll
                    for (int u = q; u < NVA; u += 4) fetch_a(u);
#pragma unroll
                    for (int u = q; u < NVB; u += 4) fetch_b(u);
                }
#pragma unroll
                for (int n = 0; n < (LIVE ? NB : 0); ++n) acc[n] = f32_block<BS>::mfma(((const float *)&fa[j & 1])[q], ((const float *)&fb[j & 1][n])[q], acc[n]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto step = [&](auto cc, int s) {
            group(cc, std::integral_constant<int, 0>());
            advance(s + 2);
            group(cc, std::integral_constant<int, 1>());
            group(cc, std::integral_constant<int, 2>());
            __syncthreads();
            group(cc, std::integral_constant<int, 3>());
        };
        if (steps > 0) {
#pragma unroll
            for (int u = 0; u < NVA; ++u) { fetch_a(u); put_a(0, u); }
#pragma unroll
            for (int u = 0; u < NVB; ++u) { fetch_b(u); put_b(0, u); }
            advance(1);
#pragma unroll
            for (int u = 0; u < NVA; ++u) fetch_a(u);
#pragma unroll
            for (int u = 0; u < NVB; ++u) fetch_b(u);
            __syncthreads();
#pragma unroll
            for (int r = 0; r < NF; ++r) read(0, 0, 0, r);
            int s = 0;
            auto pairs = [&](int end) {
                for (; s + 1 < end; s += 2) {
                    step(std::integral_constant<int, 0>(), s);
                    step(std::integral_constant<int, 1>(), s + 1);
                }
            };
            pairs(S1);
            if (OP == F32_DXG) {  // the second pair's own sum starts at step S1
                if (S1 & 1) {
                    step(std::integral_constant<int, 0>(), s);
                    swap_first();
                    step(std::integral_constant<int, 1>(), s + 1);
                    s += 2;
                } else {
                    swap_first();
                }
                pairs(steps);
            } else if (s < steps) {
                step(std::integral_constant<int, 0>(), s);
            }
        }
        // what is left of k (of both pairs; without whole steps both sums are still zero)
        const int kleft = K1 - S1 * FBK;
        for (int seg = 0; kleft > 0 && seg < (OP == F32_DXG ? 2 : 1); ++seg) {
            if (OP == F32_DXG) swap_first();  // to the first sum, and back
            const float *at = (seg ? A1 : A0) + (AK ? (size_t)S1 * FBK * p.Kd + m0 : S1 * FBK);
            const float *bt = (OP == F32_DXG && seg ? B1 : B0) + (BK_ ? (size_t)S1 * FBK * p.N + n0 : (size_t)n0 * K1 + S1 * FBK);
            const float *b3 = PAIR ? B1 + (size_t)n0 * K1 + S1 * FBK : bt;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < NVA; ++u) { va[u] = fetch_partial<TM, AK, FBK>(at, oa[u], tid, u, kleft, p.Kd - m0, p.Kd); put_a(0, u); }
#pragma unroll
            for (int u = 0; u < NVB; ++u) {
                vb[u] = fetch_partial<TN, BK_, FBK>(PAIR && u >= NVB / 2 ? b3 : bt, ob[u], tid, u, kleft, p.N - n0, p.N);
                put_b(0, u);
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int r = 0; r < NF; ++r) read(0, 0, j, r);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int n = 0; n < (LIVE ? NB : 0); ++n) acc[n] = f32_block<BS>::mfma(((const float *)&fa[0])[q], ((const float *)&fb[0][n])[q], acc[n]);
            }
        }
    };
    if (rows > BS * wr) run(std::true_type());
    else run(std::false_type());

    // lane: column lb of a block; register r -> row 8*(r/4) + 4*kh + r%4
    float *C = p.C;
    if (OP == F32_WG2) C += (size_t)g * p.N * p.Kd;
    if (OP == F32_WG13) C += (size_t)mat * p.N * p.Kd;
#pragma unroll
    for (int n = 0; n < (PAIR ? 1 : NB); ++n) {
        const int col = n0 + xb[n], rbase = BS * wr + 4 * kh;
        if (col >= p.N) continue;
        const size_t o = (size_t)(WG ? m0 : row0) * p.N + col;
        float h1[NR], h3[NR];
        if (OP == F32_DA) {  // all of the block's h1 and h3 are asked for before any is used (clamped rows: no branches)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const size_t at = o + (size_t)min(rbase + 8 * (r >> 2) + (r & 3), rows - 1) * p.N;
                h1[r] = p.H1[at];
                h3[r] = p.H3[at];
            }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int row = rbase + 8 * (r >> 2) + (r & 3);
            if (row >= rows) continue;
            const size_t at = o + (size_t)row * p.N;
            const float v = OP == F32_DXG ? first[OP == F32_DXG ? n : 0][r] + acc[n][r] : acc[n][r];
            if (PAIR) {
                const float u = acc[NB - 1][r];
                if (OP == F32_UP) C[at] = f32_swiglu(v, u);
                if (OP == F32_RAW || p.H1 != nullptr) {
                    p.H1[at] = v;
                    p.H3[at] = u;
                }
            } else if (OP == F32_DA) {
                f32_swiglu_backward(v, h1[r], h3[r], p.H1[at], p.H3[at]);
            } else {
                C[at] = v;
            }
        }
    }
}

// Whether the j-th workgroup of an XCD with `per` tiles has a tile (part = -1) or one of the PARTS parts of one: tile of the XCD, `per` or more: none
template <int PARTS>
__device__ __forceinline__ int f32_part(const f32_args &p, int per, int j, int &part)
{
    const int rest = per % p.slots;
    part = -1;
    if (PARTS == 1 || rest > (per < p.slots ? p.few : p.part_max) || j < per - rest) return j;
    part = (j - (per - rest)) % PARTS;
    return per - rest + (j - (per - rest)) / PARTS;
}
// workgroups of a row product with up to `tiles` tiles; p.slots, p.part_max and p.few set
static inline unsigned f32_grid(const f32_args &p, size_t tiles, int parts)
{
    const size_t per = (tiles + 7) / 8, cut = std::min(per, (size_t)std::max(p.few, per >= (size_t)p.slots ? p.part_max : 0));
    return (unsigned)(8 * (per + cut * (parts - 1)));
}

#define SP_TERMS_MIN 4  // sums of fewer terms are not split
hipError_t launch_product_f32_split(const f32_args &p, int op, bool vec, int max_tiles, hipStream_t s);  // experts_f32_split.hip
