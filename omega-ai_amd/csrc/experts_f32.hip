// Grouped products of fp32 layers on the matrix cores (v_mfma_f32_32x32x2_f32, fp32 operands and accumulators): the
// expert SwiGLU of the forward pass and every product of the backward pass.
//   up     a[r,h] = silu(xg[r,:].W1g[h,:]) * (xg[r,:].W3g[h,:])     silu(v) = v/(1+exp(-v))
//   down   y[r,c] = a[r,:].W2g[c,:]
//   da     d(a)[r,h] = dy[r,:].W2g[:,h], and from it dh1, dh3 (SwiGLU backward in the epilogue)
//   dxg    dxg[r,c] = dh1[r,:].W1g[:,c] + dh3[r,:].W3g[:,c]
//   wgrad  dW2g = dy^T a, dW1g = dh1^T xg, dW3g = dh3^T xg over the rows of group g
// (J/engine/nn/layer/llama/LlamaMLPLayer.java:117-130,139-158; silu J/engine/nn/layer/active/gpu/activeFunction.cu:172-190;
//  product J/engine/ad/op/gpu/OPKernel.cu:1103-1110; y = x W^T with W [out,in], J/engine/nn/layer/FullyLayer.java:181,235,
//  diffW = delta^T input, diff = delta W, FullyLayer.java:292-334; the reference's product is a cuBLAS sgemm on the tensor
//  cores, J/engine/gpu/GPUOP.java:395,405-417.)
// Row tiles come from the tile list written by the dispatch stage: a tile never straddles two experts.
//
// Bound: fp32 MFMA, 157.3 TFLOP/s (256 FLOP per clock and compute unit; 154 measured with nothing else going on).  One
// workgroup = four waves = one tile of TM rows x TN MFMA columns, 128 x 128, 64 x 64 (up: 64 x 128) or, for small batches, 32 x 32 (up: 32 x 64;
// half of the columns are W1's, half W3's, so a wave holds h1 and h3 of the same elements; weight gradients: 64 x 64).  A wave has TM/2 x TN/2 of it
// as 32 x 32 blocks; its row blocks alternate with the other row half's, so a ragged tile leaves both the same work.  At
// 128 x 128 a step of 32 k is 64 MFMAs of 64 cycles per wave against 32 KiB of operands, 8 bytes per clock and compute unit.
// A wave of such a step left to the compiler's order (barrier, LDS writes, loads, fragment reads, MFMAs) loses 2000 cycles
// next to its 4096, and a second workgroup on the compute unit does not hide them: both run in step (MFMA busy 0.74 - 0.80,
// whatever the number of buffers, workgroups or wave priorities).  So the order of a step is pinned: the fragments of the
// next 8 k are read, the next step's pieces written to the other LDS buffer and the pieces of the step behind it asked for
// between the MFMAs, a few at a time, and the one barrier of a step stands in front of MFMAs whose operands are in registers
// (up product, ragged tiles and the last round included: MFMA busy 0.80 and 125 TFLOP/s at k = 1024, 0.82 and 124 at k =
// 8192).  No vector instruction but the address sums of the loads is spent per step.
// The down and the input-gradient product, which have the fewest column tiles, take tiles of 128 x 64 (N = 1024, 8192
// rows: 0.65 -> 0.55 and 1.26 -> 1.10 ms: 544 tiles of 128 x 128 leave the third round of two per compute unit nearly empty;
// 0.49 and 0.99 since a nearly empty last round goes in parts).
// A small batch leaves compute units idle and is as long as the chain of one wave: its tiles are 32 x 32 of four waves with
// one block of v_mfma_f32_16x16x4 each (the same rate, four k in 32 cycles instead of two in 64) and steps of 64 k, so a wave's
// chain is a quarter of that of the 64 x 64 tiles they replace.  Forward pass of 8 experts, top 2, us: 256 tokens x 128 x 256
// 33 -> 26, 1 token x 1024 x 3584 109 -> 56, 256 tokens 206 -> 164; forward + backward of 64 tokens x 256 x 1024 137 -> 101.
// An operand whose rows are contiguous in k (x, W of y = x W^T) is kept [row][k] in LDS and read 16 bytes (4 k) per lane; one
// that is contiguous across k (W of delta W, both operands of delta^T input) is kept [k][column] and read one float per
// lane.  Both hand lane half (quarter) h the k places 4h .. 4h+3 of every 8 (16), so the two kinds combine freely.
// Any width and alignment: VEC takes 16-byte loads, otherwise elements are loaded one by one.  Addresses past an edge
// are clamped to the last valid element instead of branched over (a load in a divergent branch waits for those before
// it); what they bring meets a zero (k past the end) or is never stored.
//
// T = 4096, d = 1024, H = 3584, E = 8, K = 2 (8192 rows), ms, before (64 x 64 tiles for the forward products, FMA kernels
// for the others) and now: up 1.14 -> 0.96 (125 TFLOP/s), down 0.63 -> 0.49 (124), h1 and h3 again 1.91 -> 0.97, d(a) 1.08 -> 0.58,
// dxg 3.00 -> 0.99, dW2 0.99 -> 0.48, dW1 and dW3 2.01 -> 0.94.
#include "common.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

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

struct f32_args {
    const float *A0, *A1;    // A operand; A1: F32_DXG second pair, F32_WG13 the second gradient's delta
    const float *Atok;       // shared groups: token rows instead of physical rows (or null)
    const int32_t *tokp;     // F32_UP: routed rows come from Atok through this row -> token table (or null: from A0) ...
    float *xg;               // ... and the launch's last `copy_wgs` workgroups leave the gathered rows here
    const int32_t *dstp;     // pair -> row
    int copy_wgs, K;
    const float *B0, *B1;    // weights (F32_UP, F32_RAW: W1 and W3; F32_DXG: second pair), F32_WG*: the layer input rows
    const float *Btok;       // F32_WG*: as Atok
    float *C, *H1, *H3;      // output; h1 / h3 (F32_UP: kept when not null; F32_RAW: written; F32_DA: read, then dh1 / dh3)
    const omega_tile *tiles;
    const int32_t *tile_meta, *counts;
    int N, Kd;               // row products: output columns and k; F32_WG*: columns and rows of one dW (k is the group's rows)
    int E, G, T, bm;
    wgrad_deal deal;         // F32_WG*: how the tiles go to the XCDs
    int slots, part_max;     // workgroups an XCD holds at a time; tiles of a last round that go in parts
};

#define F32_IS_WG(OP) ((OP) == F32_WG2 || (OP) == F32_WG13)
#define F32_PAIR(OP) ((OP) == F32_UP || (OP) == F32_RAW)
// parts of 32 rows x 32 output columns that a row product's tile of 128 or 64 rows may be cut into (the input gradient's of 64 rows
// without 16-byte loads is left whole: the second body alone made its tiles slower, 38 -> 41 us at 2180 x 290 x 225)
#define F32_PARTS(OP, TM, TN, VEC) (F32_IS_WG(OP) || (TM) == F32_TILE_M_SMALL || ((OP) == F32_DXG && (TM) == F32_TILE_M_MID && !(VEC)) ? 1 : (TM) / 32 * ((TN) / (F32_PAIR(OP) ? 64 : 32)))

// Gathered rows of a launch whose product workgroups fetch theirs from the tokens (a wave per token, the row read once and
// written to its K places): the backward pass reads them.  Beside the products instead of a launch in front of them.
template <bool VEC>
__device__ __forceinline__ void copy_gathered(const f32_args &p, int wg, int lane, int wave)
{
    const int d = p.Kd;
    for (int t = 4 * wg + wave; t < p.T; t += 4 * p.copy_wgs) {
        const int row = lane < p.K ? p.dstp[(size_t)t * p.K + lane] : 0;
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

// One tile: row tile mt from its row r0 on (row products) or from row mt * TM of gradient matrix mat, and columns n0 ..; as and bs
// hold both operands of a row product twice.  (Weight gradients keep arrays of their own: read through pointers dW1 and dW3 of 4096
// tokens x 1024 x 3584, 8 experts, took 936 us instead of 915.  For the same reason p is a copy.)
template <int OP, int TM, int TN, bool VEC>
__device__ __forceinline__ void f32_tile(const f32_args p, float *as, float *bs, int mt, int r0, int n0, int mat)
{
    constexpr bool WG = F32_IS_WG(OP), PAIR = F32_PAIR(OP);
    constexpr bool AK = WG, BK_ = WG || OP == F32_DA || OP == F32_DXG;  // operand contiguous across k
    constexpr int BS = TM == F32_TILE_M_SMALL ? 16 : 32, GK = 256 / BS, FBK = F32_FBK(TM);  // blocks; k places of a group
    constexpr int MB = TM / (2 * BS), NB = TN / (2 * BS), NVA = TM * FBK / 1024, NVB = TN * FBK / 1024, NR = BS * BS / 64;
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
        const omega_tile tl = p.tiles[mt];
        g = tl.g;
        rows = min(TM, tl.rows - r0);
        if (rows <= 0 || n0 >= p.N) return;  // (a part of a ragged tile)
        row0 = tl.row0 + r0;
        K1 = p.Kd;
        A0 = p.Atok && tl.xrow0 >= 0 ? p.Atok + (size_t)(tl.xrow0 + r0) * p.Kd : p.A0 + (size_t)row0 * p.Kd;
        fetch_rows = OP == F32_UP && p.tokp != nullptr && tl.xrow0 < 0;
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
        oa[u] = 4u * (AK ? (uint32_t)k * p.Kd + min(x, p.Kd - m0 - (VEC ? 4 : 1)) : (uint32_t)(fetch_rows ? p.tokp[row0 + min(x, rows - 1)] : min(x, rows - 1)) * K1 + k);
    }
#pragma unroll
    for (int u = 0; u < NVB; ++u) {
        const int x = f32_piece<TN, BK_, FBK>::x(tid, u), k = f32_piece<TN, BK_, FBK>::k(tid, u);
        ob[u] = 4u * (BK_ ? (uint32_t)k * p.N + min(x, p.N - n0 - (VEC ? 4 : 1)) : (uint32_t)min(PAIR && x >= CT ? x - CT : x, p.N - 1 - n0) * K1 + k);
    }

    // (first: F32_DXG's sum over the first pair.  One chain over both would carry 1.4 times the rounding error of two that are
    // added once: H = 3584, relative to float64, 1.57e-6 against 1.09e-6)
    acc_t acc[MB][NB], first[OP == F32_DXG ? MB : 1][OP == F32_DXG ? NB : 1];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                acc[i][n][r] = 0.0f;
                if (OP == F32_DXG) first[i][n][r] = 0.0f;
            }
    auto swap_first = [&]() {
        if constexpr (OP == F32_DXG) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    const acc_t v = acc[i][n];
                    acc[i][n] = first[i][n];
                    first[i][n] = v;
                }
        }
    };

    // this wave's row blocks: rows BS (2 i + wr) ..; columns: TN/2 wc + BS n (up: W1 columns BS wc, and the same of W3)
    const int live = max(0, min(MB, ((rows + BS - 1) / BS + 1 - wr) / 2));
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
    // All steps for a wave with MBL live row blocks.  One group = GK k of the step in buffer c: its MFMAs on the fragments
    // read during the group before, and spread between them (pinned, a quarter of the group at a time) the reads of the
    // next group's fragments and the group's share of the step's other work: group 0 writes the next step's pieces to the
    // other buffer, group 1 asks for those of the step behind it; the barrier lies in front of the last group, whose
    // fragment reads are the next step's first.  (Everything between two barriers of a step reads buffer c and writes
    // buffer 1 - c, except that last group's reads of 1 - c, which every wave has finished writing.)
    auto run = [&](auto mbl) {
        constexpr int MBL = decltype(mbl)::value, NF = MBL > 0 ? MBL + NB : 0;
        float4 fa[2][MBL > 0 ? MBL : 1], fb[2][NB];
        auto read = [&](int set, int c, int j, int r) {
            const int k = GK * j + 4 * kh;
            if (r < MBL) fa[set][r < MBL ? r : 0] = frag<TM, AK, FBK>(WG ? As[c] : as + c * LA, xa + 2 * BS * r, k);
            else if (r < NF) fb[set][r - MBL < NB ? r - MBL : 0] = frag<TN, BK_, FBK>(WG ? Bs[c] : bs + c * LB, xb[r - MBL < NB ? r - MBL : 0], k);
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
                for (int i = 0; i < MBL; ++i)
#pragma unroll
                    for (int n = 0; n < NB; ++n)
                        acc[i][n] = f32_block<BS>::mfma(((const float *)&fa[j & 1][i])[q], ((const float *)&fb[j & 1][n])[q], acc[i][n]);
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
                    for (int i = 0; i < MBL; ++i)
#pragma unroll
                        for (int n = 0; n < NB; ++n)
                            acc[i][n] = f32_block<BS>::mfma(((const float *)&fa[0][i])[q], ((const float *)&fb[0][n])[q], acc[i][n]);
            }
        }
    };
    if (live == MB) run(std::integral_constant<int, MB>());
    else if (MB > 1 && live == 1) run(std::integral_constant<int, 1>());
    else run(std::integral_constant<int, 0>());

    // lane: column lb of a block; register r -> row 8*(r/4) + 4*kh + r%4
    float *C = p.C;
    if (OP == F32_WG2) C += (size_t)g * p.N * p.Kd;
    if (OP == F32_WG13) C += (size_t)mat * p.N * p.Kd;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if (i >= live) continue;
#pragma unroll
        for (int n = 0; n < (PAIR ? 1 : NB); ++n) {
            const int col = n0 + xb[n], rbase = BS * (2 * i + wr) + 4 * kh;
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
                const float v = OP == F32_DXG ? first[OP == F32_DXG ? i : 0][OP == F32_DXG ? n : 0][r] + acc[i][n][r] : acc[i][n][r];
                if (PAIR) {
                    const float u = acc[i][NB - 1][r];
                    if (OP == F32_UP) C[at] = (v / (1.0f + expf(-v))) * u;
                    if (OP == F32_RAW || p.H1 != nullptr) {
                        p.H1[at] = v;
                        p.H3[at] = u;
                    }
                } else if (OP == F32_DA) {
                    const float sg = 1.0f / (1.0f + expf(-h1[r]));
                    p.H3[at] = v * (h1[r] * sg);
                    p.H1[at] = (v * h3[r]) * sg * (1.0f + h1[r] * (1.0f - sg));
                } else {
                    C[at] = v;
                }
            }
        }
    }
}

template <int OP, int TM, int TN, bool VEC>
__global__ __launch_bounds__(256, 2) void f32_product_kernel(f32_args p)
{
    constexpr bool WG = F32_IS_WG(OP), PAIR = F32_PAIR(OP), PARTS = F32_PARTS(OP, TM, TN, VEC) > 1;
    constexpr int CT = PAIR ? TN / 2 : TN;                             // output columns per tile
    constexpr bool BK_ = WG || OP == F32_DA || OP == F32_DXG;
    constexpr int PN = PAIR ? 64 : 32;                                 // MFMA columns of a part
    constexpr int LA = f32_lds_floats(TM, WG, F32_FBK(TM)), LB = f32_lds_floats(TN, BK_, F32_FBK(TM));
    // A part works in the room of its tile.  The input gradient's of 128 rows, whose B is wider in a part than in the tile, keeps both
    // operands in one array, behind one another from its start on: 54272 bytes, three workgroups per compute unit, where 55296 would
    // leave two (backward pass, us: 4096 tokens x 1024 x 3584, 8 experts 2982 / 2972, 3333 x 333 x 1111, 6 experts 755-761 / 750).
    constexpr int LAP = f32_lds_floats(32, WG, F32_FBK(32)), LBP = f32_lds_floats(PN, BK_, F32_FBK(32));
    constexpr bool ONE = OP == F32_DXG && TM == F32_TILE_M;
    static_assert(!PARTS || (ONE ? LAP + LBP <= LA + LB : LAP <= LA), "a part's operands fit");
    __shared__ __attribute__((aligned(16))) float as[WG ? 1 : ONE ? 2 * (LA + LB) : 2 * LA], bs[WG || ONE ? 1 : 2 * (PARTS && LBP > LB ? LBP : LB)];
    if (OP == F32_UP && (int)blockIdx.x >= (int)gridDim.x - p.copy_wgs) {
        copy_gathered<VEC>(p, blockIdx.x - (gridDim.x - p.copy_wgs), threadIdx.x & 63, threadIdx.x >> 6);
        return;
    }

    // Tile of this workgroup.  Consecutive workgroups go round the eight XCDs.  Row products: XCD x takes the x-th eighth of the tiles, and
    // within it up to 8 row tiles walk the column tiles together, so that its workgroups share operand rows in its L2.  Weight
    // gradients, whose length is the expert's rows: every XCD takes an eighth of every matrix (wgrad_tile).
    const int NT = (p.N + CT - 1) / CT;
    const int MT = WG ? (p.Kd + TM - 1) / TM : p.tile_meta[0];  // row tiles (of one gradient matrix)
    const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
    int t, mat = 0, part = -1;
    if (WG) {
        t = wgrad_tile(p.deal, x, j, &mat);
        if (t < 0) return;
        for (; p.deal.together > 1 && t >= MT * NT; t -= MT * NT) ++mat;
    } else {
        // Where at least one whole round of p.slots workgroups is followed by a last one of a quarter or less of it (p.part_max), that
        // last round's tiles go in parts of 32 rows x 32 columns: the workgroups that would idle share what one would work on.  us in
        // tiles / parts, tiles of 128 rows: down product of 8192 rows, k = 3584, N = 1024 (two rounds and 12 of 64 tiles) 540 / 486,
        // dxg 1090 / 986; of 64 rows: up product of 4024 tokens x 928 x 252, 12 experts, top 2 (one round and 1) 93 / 74, down product of
        // 2036 x 680 x 1980, 3 experts, top 3 (one round and 4 of 128) 173 / 152.  Parts cost more per element than a tile: k = 1536,
        // N = 1024, 128 rows, rounds + rest: 1 + 16 143 / 132, 1 + 24 145 / 149, 1 + 32 149 / 165, 2 + 8 236 / 210, 2 + 24 238 / 247; forward
        // passes with 64 rows and up's rest at 3/8 63.0 / 65.4, at 1/2 141 / 149.
        const int total = MT * NT, per = (total + 7) >> 3, rest = per % p.slots;
        int i = j;
        if (PARTS && rest <= p.part_max && per >= p.slots && j >= per - rest) {
            part = (j - (per - rest)) % F32_PARTS(OP, TM, TN, VEC);
            i = per - rest + (j - (per - rest)) / F32_PARTS(OP, TM, TN, VEC);
        }
        t = x * per + i;
        if (i >= per || t >= total) return;
    }
    const int rb = t / (8 * NT), nrb = min(8, MT - 8 * rb), ti = t - rb * 8 * NT;
    const int mt = 8 * rb + ti % nrb, n0 = (ti / nrb) * CT;

    if constexpr (PARTS) {
        if (part >= 0) {
            f32_tile<OP, 32, PN, VEC>(p, as, ONE ? as + 2 * LAP : bs, mt, 32 * (part % (TM / 32)), n0 + 32 * (part / (TM / 32)), mat);
            return;
        }
    }
    f32_tile<OP, TM, TN, VEC>(p, as, ONE ? as + 2 * LA : bs, mt, 0, n0, mat);
}

// The largest row-tile height that a batch of up to T tokens takes: with fewer than 128 rows per expert always 32 (160 shapes of
// 1 to 4096 tokens, d = 64 .. 1024, H = 64 .. 3584, 2 to 16 experts: tiles of 64 took 0.97 to 1.90 times as long)
int experts_f32_tile_m_max(const omega_moe *m, int T)
{
    return (long long)T * m->cfg.K >= 128LL * m->cfg.E ? F32_TILE_M : F32_TILE_M_SMALL;
}

// From there on the height whose forward products are the shortest by this estimate.  A tile takes its k places in whole steps, a
// fixed number more and, for a last partial step, `rest` more, at a rate that falls a little with its size (`a`: time per
// column of k); a product takes rounds of one tile per compute unit, its last, partial round `part` of one and that share of the
// rest, or `cut` of its share where it goes in parts (f32_product_kernel), all of them `least` rounds or more; an expert has `pad` tiles
// more than its rows.  The numbers are fitted to 720 forward passes of the range above at all three heights, of which the estimate takes
// the best or one within 5 % (14 within 13 %; 0.4 % in the mean).  The fit to the kernels without parts charged a nearly empty last round four
// or five tenths of one: 0.8 % in the mean, 36 passes more than 5 % off, one of them 44 %.  Within 2 % the tallest is taken, for the backward
// pass: 4096 tokens x 1024 x 3584, 8 experts, top 2 at 64 / 128 rows forward 1526 / 1523, step of training 5255 / 5091; over 160 steps the estimate
// is 0.5 % off in the mean, the earlier one 0.8.  Forward pass, us, at 32 / 64 / 128 rows: 2073 tokens x 296 x 264, 4 experts, top 3 72 / 65 / 95,
// 1001 x 124 x 1676, 6 experts, top 5 and 2 shared 190 / 136 / 152, 3496 x 120 x 452, 9 experts, top 7 189 / 146 / 139, 2048 x 1024 x 1024, 16 experts,
// top 2 283 / 284 / 367.
int experts_f32_tile_m(const omega_moe *m, int T)
{
    if (experts_f32_tile_m_max(m, T) == F32_TILE_M_SMALL) return F32_TILE_M_SMALL;
    const omega_moe_config &c = m->cfg;
    static const struct { int bm, step, cols; double a, more, rest, pad, least, part, cut; } form[] = {
        {F32_TILE_M_SMALL, 64, 32, 1.0, 104, 74, 0.925, 1.26, 0.216, 1.0},
        {F32_TILE_M_MID, 32, 64, 4.0, 60, 43, 0.57, 0.79, 0.395, 1.65},
        {F32_TILE_M, 32, 64, 7.2, 65, 39, 0.8, 0.9, 0.865, 2.1}};
    int best = F32_TILE_M_SMALL;
    double least_time = 0.0;
    for (const auto &f : form) {
        const double tiles_m = (double)T * c.K / f.bm + f.pad * c.E + (double)c.Es * ceil_div(T, f.bm);
        auto product = [&](int k, int n, int slots) {  // (workgroups of a compute unit: a round of f32_product_kernel)
            const double all = tiles_m * ceil_div(n, f.cols) / m->ctx->num_cus, whole = std::floor(all), full = std::floor(all / slots) * slots;
            double rounds = all < f.least ? f.least : whole + (all > whole ? f.part + (1.0 - f.part) * (all - whole) : 0.0);
            if (f.bm != F32_TILE_M_SMALL && full > 0.0 && all - full <= 0.25 * slots) rounds = std::min(rounds, full + f.cut * (all - full));
            return rounds * (ceil_div(k, f.step) * f.step + f.more + (k % f.step != 0 ? f.rest : 0.0));
        };
        // (the up product's tiles hold two columns of weights for each of their own)
        const double time = f.a * (product(c.d, c.H, 2) + 0.58 * product(c.H, c.d, f.bm == F32_TILE_M_MID ? 4 : 2));
        if (f.bm == F32_TILE_M_SMALL || time < (f.bm == F32_TILE_M ? 1.02 : 1.0) * least_time) {
            best = f.bm;
            least_time = time;
        }
    }
    return best;
}

template <int OP, int TM, int TN>
static hipError_t f32_launch(f32_args p, bool vec, int max_tiles, hipStream_t s)
{
    constexpr int CT = F32_PAIR(OP) ? TN / 2 : TN;
    const size_t tiles = (size_t)ceil_div(p.N, CT) * (F32_IS_WG(OP) ? (size_t)ceil_div(p.Kd, TM) * p.G * (OP == F32_WG13 ? 2 : 1) : max_tiles);
    // (what LDS holds of the workgroups of tiles of 128 and 64 rows; a third one of the input gradient's comes and goes between the others:
    // with rounds of three 2972 -> 3088 and 795 -> 868 us at 4096 tokens x 1024 x 3584, 8 experts and x 512 x 1536, 4 experts)
    p.slots *= TM == F32_TILE_M || F32_PAIR(OP) ? 2 : 4;
    p.part_max = p.slots / 4;
    const size_t parts = F32_PARTS(OP, TM, TN, vec) > 1 && (tiles + 7) / 8 >= (size_t)p.slots ? (size_t)8 * p.part_max * (F32_PARTS(OP, TM, TN, vec) - 1) : 0;
    if (F32_IS_WG(OP)) p.deal = wgrad_deal_of(ceil_div(p.N, CT) * ceil_div(p.Kd, TM), p.G * (OP == F32_WG13 ? 2 : 1));
    // (weight gradients: whole groups of matrices and one of what is left over, each to eight XCDs)
    const unsigned grid = (unsigned)(F32_IS_WG(OP) ? (tiles + 7) / 8 * 8 + (p.deal.rest > 0 ? 8 : 0) : (tiles + 7) / 8 * 8 + parts) + p.copy_wgs;
    if (vec) hipLaunchKernelGGL((f32_product_kernel<OP, TM, TN, true>), dim3(grid), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((f32_product_kernel<OP, TM, TN, false>), dim3(grid), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_product_f32(const omega_moe *m, int op, const float *x, const float *dout, int T, hipStream_t s, bool gather, bool keep)
{
    const omega_moe_config &c = m->cfg;
    f32_args p = {};
    p.tiles = m->tiles;
    p.tile_meta = m->tile_meta;
    p.counts = m->counts;
    p.E = c.E;
    p.G = m->G;
    p.T = T;
    p.bm = m->bm;
    p.slots = m->ctx->num_cus / 8;  // (f32_launch: times the workgroups of a compute unit)
    const float *W1 = (const float *)m->W1, *W3 = (const float *)m->W3, *W2 = (const float *)m->W2;
    switch (op) {
        case F32_UP:
        case F32_RAW:
            p.A0 = (const float *)m->xg; p.Atok = x; p.B0 = W1; p.B1 = W3; p.N = c.H; p.Kd = c.d;
            p.C = (float *)m->a;
            if (gather) {
                p.tokp = m->tokp; p.dstp = m->dstp; p.xg = (float *)m->xg; p.K = c.K;
                // (a token per wave until there are four workgroups per compute unit: a wave with several waits for each in
                // turn behind the last product; 4096 tokens x 64 x 64, 64 experts, top 6, forward pass: 48.0 -> 46.4 us)
                p.copy_wgs = std::min(ceil_div(T, 4), 4 * m->ctx->num_cus);
            }
            if (op == F32_RAW || keep) { p.H1 = m->bw_h1; p.H3 = m->bw_h3; }
            break;
        case F32_DOWN:
            p.A0 = (const float *)m->a; p.B0 = W2; p.C = m->y; p.N = c.d; p.Kd = c.H;
            break;
        case F32_DA:
            p.A0 = m->bw_dy; p.Atok = dout; p.B0 = W2; p.H1 = m->bw_h1; p.H3 = m->bw_h3; p.N = c.H; p.Kd = c.d;
            break;
        case F32_DXG:
            p.A0 = m->bw_h1; p.A1 = m->bw_h3; p.B0 = W1; p.B1 = W3; p.C = m->bw_dxg; p.N = c.d; p.Kd = c.H;
            break;
        case F32_WG2:
            p.A0 = m->bw_dy; p.Atok = dout; p.B0 = (const float *)m->a; p.C = m->dW2; p.N = c.H; p.Kd = c.d;
            break;
        case F32_WG13:
            p.A0 = m->bw_h1; p.A1 = m->bw_h3; p.B0 = (const float *)m->xg; p.Btok = x; p.C = m->dW13; p.N = c.d; p.Kd = c.H;
            break;
        default: return hipErrorInvalidValue;
    }
    // 16-byte loads, where every row of either operand starts on 16 bytes: the rows of the layer's buffers and weights are d or
    // H floats long, those of the caller (x or dout, where the product reads it) need their buffer aligned as well.  Up and down
    // read rows of one width only.   (Forward pass
    // of 4096 tokens, 8 experts, top 2, us, both widths asked of every product and now: d = 1024, H = 2731 1238 -> 1214; d = 512, H = 1001 305 -> 299.)
    const bool d4 = c.d % 4 == 0, H4 = c.H % 4 == 0;
    const bool vec = (op == F32_DOWN || d4) && (op == F32_UP || op == F32_RAW || H4) && (((uintptr_t)p.Atok | (uintptr_t)p.Btok) % 16) == 0;
    // weight gradients, whose tiles do not depend on the row tiles: of 128 x 128 from 128 rows per expert on, once the down product
    // would have such a tile for every compute unit
    const long long rows = (long long)T * c.K;
    const bool wide = rows >= 128LL * c.E && rows / 128 * ceil_div(c.d, 128) >= m->ctx->num_cus;
#define F32_ROWS(OP, TN_BIG, TN_MID, TN_SMALL)                                                 \
    (m->bm == F32_TILE_M ? f32_launch<OP, F32_TILE_M, TN_BIG>(p, vec, m->max_m_tiles, s)       \
     : m->bm == F32_TILE_M_MID ? f32_launch<OP, F32_TILE_M_MID, TN_MID>(p, vec, m->max_m_tiles, s) \
                               : f32_launch<OP, F32_TILE_M_SMALL, TN_SMALL>(p, vec, m->max_m_tiles, s))
    switch (op) {
        case F32_UP: return F32_ROWS(F32_UP, 128, 128, 64);
        case F32_RAW: return F32_ROWS(F32_RAW, 128, 128, 64);
        case F32_DOWN: return F32_ROWS(F32_DOWN, 64, 64, 32);
        case F32_DA: return F32_ROWS(F32_DA, 128, 64, 32);
        case F32_DXG: return F32_ROWS(F32_DXG, 64, 64, 32);
        case F32_WG2: return wide ? f32_launch<F32_WG2, 128, 128>(p, vec, 0, s) : f32_launch<F32_WG2, 64, 64>(p, vec, 0, s);
        default: return wide ? f32_launch<F32_WG13, 128, 128>(p, vec, 0, s) : f32_launch<F32_WG13, 64, 64>(p, vec, 0, s);
    }
#undef F32_ROWS
}
