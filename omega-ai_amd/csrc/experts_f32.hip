// Grouped products of fp32 layers on the matrix cores, fp32 operands and accumulators: the expert SwiGLU of the forward pass and every
// product of the backward pass, for batches whose tiles are few or small.  The others run on experts_f32_split.hip, in tiles of 128 x 128
// or 64 x 128 on the bf16 matrix cores; experts_f32_tile_m and launch_product_f32 say which.
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
// Bound: fp32 MFMA, 157.3 TFLOP/s (256 FLOP per clock and compute unit; 154 measured with nothing else going on), and for small batches the
// chain of one wave.  One workgroup = four waves = one tile: 64 x 64 (v_mfma_f32_32x32x2, steps of 32 k; down, d(a), input gradient, weight gradients) or
// 32 x 32 (up: 32 x 64, half of the columns W1's, half W3's, so a wave holds h1 and h3 of the same elements; four waves with one block of
// v_mfma_f32_16x16x4 each - the same rate, four k in 32 cycles instead of two in 64 - and steps of 64 k, so a wave's chain is a quarter of that
// of 64 x 64).  Forward pass of 8 experts, top 2, us, 64 x 64 -> 32 x 32: 256 tokens x 128 x 256 33 -> 26, 1 token x 1024 x 3584 109 -> 56, 256
// tokens 206 -> 164; forward + backward of 64 tokens x 256 x 1024 137 -> 101.
// A step left to the compiler's order (barrier, LDS writes, loads, fragment reads, MFMAs) loses half of its MFMA time again, and a second
// workgroup on the compute unit does not hide it: both run in step.  So the order of a step is pinned: the fragments of the next 8 k are
// read, the next step's pieces written to the other LDS buffer and the pieces of the step behind it asked for between the MFMAs, a few at
// a time, and the one barrier of a step stands in front of MFMAs whose operands are in registers.  No vector instruction but the address
// sums of the loads is spent per step.
// An operand whose rows are contiguous in k (x, W of y = x W^T) is kept [row][k] in LDS and read 16 bytes (4 k) per lane; one
// that is contiguous across k (W of delta W, both operands of delta^T input) is kept [k][column] and read one float per
// lane.  Both hand lane half (quarter) h the k places 4h .. 4h+3 of every 8 (16), so the two kinds combine freely.
// Any width and alignment: VEC takes 16-byte loads, otherwise elements are loaded one by one.  Addresses past an edge
// are clamped to the last valid element instead of branched over (a load in a divergent branch waits for those before
// it); what they bring meets a zero (k past the end) or is never stored.
#include "f32_product.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

// parts of 32 rows x 32 columns that a row product's tile of 64 rows may be cut into (up products here have tiles of 32)
#define F32_PARTS(OP, TM, TN) (F32_IS_WG(OP) || (TM) == F32_TILE_M_SMALL ? 1 : (TM) / 32 * ((TN) / 32))

// The up product of a few pairs finds its rows from the router's choices and leaves the dispatch index, made by the launch's last workgroup, to the
// launches behind: a launch less in front of it.  First column of this workgroup's tile (tl, tokens of its rows in tok), or -1: nothing to do.
// Forward pass of 256 tokens x 128 x 256, 8 experts, top 2: 23.5 -> 19.8 us (with loops over the chunks that branch 22.8, with the index made in LDS by
// small_index 21.9).
template <int NC, bool VEC>
__device__ __forceinline__ int f32_self(const f32_args &p, uint16_t *tok, omega_tile &tl)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), last = gridDim.x - 1;
    f32_choices<NC> ch;
    ch.read(p, lane);
    if ((int)blockIdx.x >= last - p.copy_wgs) {
        if ((int)blockIdx.x == last) ch.leave(p.index, lane, wave);
        else copy_gathered<VEC, true>(p, blockIdx.x - (last - p.copy_wgs), lane, wave, ch);
        return -1;
    }
    // (the tile as f32_product_kernel finds it)
    const int NT = (p.N + 31) / 32, MT = ch.tiles + (p.G - p.E) * ((p.T + F32_TILE_M_SMALL - 1) / F32_TILE_M_SMALL), total = MT * NT, per = (total + 7) >> 3;
    const int i = blockIdx.x >> 3, t = (blockIdx.x & 7) * per + i;
    if (i >= per || t >= total) return -1;
    const int rb = t / (8 * NT), nrb = min(8, MT - 8 * rb), ti = t - rb * 8 * NT;
    tl = ch.find(p, 8 * rb + ti % nrb, lane, tok);
    return (ti / nrb) * 32;
}

// SELF: the launch makes the dispatch index (a kernel of its own: in one with the others its registers, 105 for 84, and its scalar spills cost them up
// to 6 %: forward pass, us, 2373 tokens x 142 x 88, 5 experts, top 1 30.7 -> 29.1, 566 x 192 x 109, 10 experts, top 3, one shared 30.5 -> 29.0)
template <int OP, int TM, int TN, bool VEC, bool SELF>
__global__ __launch_bounds__(256, 2) void f32_product_kernel(f32_args p)
{
    constexpr bool WG = F32_IS_WG(OP), PAIR = F32_PAIR(OP), PARTS = F32_PARTS(OP, TM, TN) > 1;
    constexpr int CT = PAIR ? TN / 2 : TN;                             // output columns per tile
    constexpr bool BK_ = WG || OP == F32_DA || OP == F32_DXG;
    constexpr int LA = f32_lds_floats(TM, WG, F32_FBK(TM)), LB = f32_lds_floats(TN, BK_, F32_FBK(TM));
    // (a part works in the room of its tile)
    constexpr int LAP = f32_lds_floats(32, WG, F32_FBK(32)), LBP = f32_lds_floats(32, BK_, F32_FBK(32));
    static_assert(!PARTS || LAP <= LA, "a part's operands fit");
    __shared__ __attribute__((aligned(16))) float as[WG ? 1 : 2 * LA], bs[WG ? 1 : 2 * (PARTS && LBP > LB ? LBP : LB)];
    if constexpr (SELF) {
        __shared__ uint16_t tok[F32_TILE_M_SMALL];
        omega_tile tl;
        const int P = p.T * p.K;
        const int chunks = INDEX_IN_UP_CHUNKS_F32(P);
        const int n0 = chunks == 4 ? f32_self<4, VEC>(p, tok, tl) : chunks == 8 ? f32_self<8, VEC>(p, tok, tl) : f32_self<F32_SELF_CHUNKS, VEC>(p, tok, tl);
        if (n0 >= 0) f32_tile<OP, TM, TN, VEC>(p, as, bs, 0, tl, 0, n0, 0, tok);
        return;
    }
    if (OP == F32_UP && (int)blockIdx.x >= (int)gridDim.x - p.copy_wgs) {
        copy_gathered<VEC, false>(p, blockIdx.x - (gridDim.x - p.copy_wgs), threadIdx.x & 63, threadIdx.x >> 6, 0);
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
        // tiles / parts: down product of 2036 x 680 x 1980, 3 experts, top 3 (one round and 4 of 128) 173 / 152; forward passes of such tiles
        // with a rest of 3/8 63.0 / 65.4, of 1/2 141 / 149.
        // Without a whole round all tiles do, up to three for four compute units (p.few).
        const int total = MT * NT, per = (total + 7) >> 3, i = f32_part<F32_PARTS(OP, TM, TN)>(p, per, j, part);
        t = x * per + i;
        if (i >= per || t >= total) return;
    }
    const int rb = t / (8 * NT), nrb = min(8, MT - 8 * rb), ti = t - rb * 8 * NT;
    const int mt = 8 * rb + ti % nrb, n0 = (ti / nrb) * CT;

    if constexpr (PARTS) {
        if (part >= 0) {
            f32_tile<OP, 32, 32, VEC>(p, as, bs, mt, p.tiles[mt], 32 * (part % (TM / 32)), n0 + 32 * (part / (TM / 32)), mat);
            return;
        }
    }
    f32_tile<OP, TM, TN, VEC>(p, as, bs, mt, WG ? omega_tile{} : p.tiles[mt], 0, n0, mat);
}

// The largest row-tile height that a batch of up to T tokens takes: with fewer than 128 rows per expert always 32 (160 shapes of
// 1 to 4096 tokens, d = 64 .. 1024, H = 64 .. 3584, 2 to 16 experts: tiles of 64 took 0.97 to 1.90 times as long)
int experts_f32_tile_m_max(const omega_moe *m, int T)
{
    return (long long)T * m->cfg.K >= 128LL * m->cfg.E ? F32_TILE_M : F32_TILE_M_SMALL;
}

// From there on the height whose forward products are the shortest by this estimate.  A product starts in `base`; a tile takes its k
// places in whole steps, a fixed number more and, for a last partial step, `rest` more, at `a` ns per k; a product takes rounds of
// one tile per compute unit, its last, partial round `part` of one and that share of the rest, or `cut` of its share where it goes in
// parts (up to `few` of the workgroups that are there at a time), all of them `least` rounds or more; an expert has `pad` tiles more than its
// rows.  A product that goes in parts altogether takes `parts` times what tiles of 32 rows do.  Of two heights within 2 % the lower one is taken.  The
// numbers are fitted to the stage times of 900 forward passes (64 to 8192 tokens, d = 64 .. 1024, H = 64 .. 3584, 1 to 24 experts) at all three heights; of
// these passes the estimate takes the best or one within 5 % (40 are further off, one 23 %; 0.6 % in the mean), of the passes with a backward
// pass behind them 22 are further off (one 18 %; 0.5 %).  (The earlier fit, to kernels that looked at no factors: 77 and 66, one 29 %.)  Forward products, us, at 32 /
// 64 / 128 rows: 622 tokens x 130 x 420, one expert 13.9 / 22.2 / 46.9, 1982 x 512 x 1144, 4 experts, top 1 85.9 / 69.2 / 113.7, 2842 x 65 x 922, 4 experts, top 4
// 114 / 85 / 102, 1376 x 223 x 3135, 15 experts, top 6 455 / 351 / 378, 4096 x 1024 x 3584, 8 experts, top 2 1690 / 1420 / 1000.
int experts_f32_tile_m(const omega_moe *m, int T)
{
    const omega_moe_config &c = m->cfg;
    if (experts_f32_tile_m_max(m, T) == F32_TILE_M_SMALL || c.d < SP_TERMS_MIN || c.H < SP_TERMS_MIN) return F32_TILE_M_SMALL;
    struct product { int step, cols, slots; double a, more, rest, pad, least, part, cut, few, base, parts; };
    static const struct { int bm; product up, down; } form[] = {
        {F32_TILE_M_SMALL, {64, 32, 2, 8.35, 92.6, 58.9, 0.462, 0.97, 1.1, 1, 0, 3.62, 1}, {64, 32, 2, 4.81, 42, 63.6, 0.459, 1.02, 1.04, 1, 0, 3.21, 1}},
        {F32_TILE_M_MID, {32, 64, 3, 23.1, 58.4, 30.2, 0.483, 1.01, 0.596, 1.48, 0.375, 6.48, 1}, {32, 64, 4, 18.5, 26.4, 21.9, 0.402, 0.326, 0.782, 2.65, 0.25, 3.18, 1.02}},
        {F32_TILE_M, {32, 64, 2, 40.5, 78.8, 38.4, 0.465, 1.06, 0.412, 1.56, 0.375, 7.52, 1.09}, {32, 128, 2, 45.4, 25.8, 21.4, 0.659, 1.07, 0.439, 1.36, 0.375, 7.31, 1.24}}};
    int best = F32_TILE_M_SMALL;
    double least_time = 0.0;
    for (const auto &f : form) {
        auto rounds_of = [&](const product &q, int bm, int n) {
            return ((double)T * c.K / bm + q.pad * c.E + (double)c.Es * ceil_div(T, bm)) * ceil_div(n, q.cols) / m->ctx->num_cus;
        };
        auto time = [&](product q, const product &parts, int k, int n) {
            double all = rounds_of(q, f.bm, n);
            const double slower = all <= 0.75 ? q.parts : 1.0;
            if (all <= 0.75) all = rounds_of(q = parts, F32_TILE_M_SMALL, n);  // (f32_part)
            const double whole = std::floor(all), full = std::floor(all / q.slots) * q.slots;
            double rounds = all < q.least ? q.least : whole + (all > whole ? q.part + (1.0 - q.part) * (all - whole) : 0.0);
            if (full > 0.0 && all - full <= q.few * q.slots) rounds = std::min(rounds, full + q.cut * (all - full));
            return slower * (q.base + 1e-3 * q.a * rounds * (ceil_div(k, q.step) * q.step + q.more + (k % q.step != 0 ? q.rest : 0.0)));
        };
        const double t = time(f.up, form[0].up, c.d, c.H) + time(f.down, form[0].down, c.H, c.d);
        if (f.bm == F32_TILE_M_SMALL || 1.02 * t < least_time) {
            best = f.bm;
            least_time = t;
        }
    }
    return best;
}

template <int OP, int TM, int TN>
static hipError_t f32_launch(f32_args p, bool vec, int max_tiles, hipStream_t s)
{
    constexpr int CT = F32_PAIR(OP) ? TN / 2 : TN;
    const size_t tiles = (size_t)ceil_div(p.N, CT) * (F32_IS_WG(OP) ? (size_t)ceil_div(p.Kd, TM) * p.G * (OP == F32_WG13 ? 2 : 1) : max_tiles);
    p.slots *= 4;  // (what LDS holds of the workgroups of tiles of 64 rows)
    p.part_max = p.slots / 4;
    if (F32_IS_WG(OP)) p.deal = wgrad_deal_of(ceil_div(p.N, CT) * ceil_div(p.Kd, TM), p.G * (OP == F32_WG13 ? 2 : 1));
    // (weight gradients: whole groups of matrices and one of what is left over, each to eight XCDs)
    const unsigned grid = (F32_IS_WG(OP) ? (unsigned)((tiles + 7) / 8 * 8 + (p.deal.rest > 0 ? 8 : 0)) : f32_grid(p, tiles, F32_PARTS(OP, TM, TN))) + p.copy_wgs + (p.index.ids != nullptr ? 1 : 0);
    auto launch = [&](auto self) {
        if (vec) hipLaunchKernelGGL((f32_product_kernel<OP, TM, TN, true, decltype(self)::value>), dim3(grid), dim3(256), 0, s, p);
        else hipLaunchKernelGGL((f32_product_kernel<OP, TM, TN, false, decltype(self)::value>), dim3(grid), dim3(256), 0, s, p);
        return hipGetLastError();
    };
    if constexpr (OP == F32_UP && TM == F32_TILE_M_SMALL)
        if (p.index.ids != nullptr) return launch(std::true_type());
    return launch(std::false_type());
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
    p.slots = m->ctx->num_cus / 8;  // (the launchers: times the workgroups of a compute unit)
    p.few = p.slots * 3 / 4;
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
            if (op == F32_UP && gather && m->index_in_up) p.index = index_args_of(m, T);
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
    // Row products: tiles of 128 rows are split ones, those of 64 where they read H columns of weights (the others have fewer columns
    // and a longer k).  Up product of 64 rows, split / fp32 MFMAs in 64 x 128: from one tile per compute unit on 0.60 - 0.97, below, where most
    // launches go in parts of 32 x 32, 1.03 - 1.14.
    // d(a) of 64 rows: tiles of 64 x 128 from three for two compute units on, for a short k from six for one, else 64 x 64 on fp32 MFMAs.  Backward pass, split / fp32, by
    // tiles of 64 x 128 per compute unit, means of 10 to 30 shapes: 0.2 - 0.5 1.01 - 1.04, 0.75 - 1 1.06, 1 - 1.5 1.03, from 1.5 on with d >= 256 0.99 - 0.96, with
    // d < 256 1.5 - 6 1.01, beyond 0.99.  (1240 tokens x 624 x 352, 4 experts, top 2, the launch alone 29.8 / 20.9.)
    const double da_tiles = (double)m->max_m_tiles * ceil_div(c.H, 128) / m->ctx->num_cus;
    const bool mid = m->bm == F32_TILE_M_MID && (op == F32_UP || op == F32_RAW || (op == F32_DA && da_tiles >= (c.d < 256 ? 6.0 : 1.5)));
    if (op == F32_WG2 || op == F32_WG13 ? f32_wgrad_wide(m, T, op == F32_WG13 ? 2 * m->G : m->G) : m->bm == F32_TILE_M || mid)
        return launch_product_f32_split(p, op, vec, m->max_m_tiles, s);
#define F32_ROWS(OP)                                                                           \
    (m->bm == F32_TILE_M_MID ? f32_launch<OP, F32_TILE_M_MID, 64>(p, vec, m->max_m_tiles, s) \
                             : f32_launch<OP, F32_TILE_M_SMALL, 32>(p, vec, m->max_m_tiles, s))
    switch (op) {
        case F32_UP: return f32_launch<F32_UP, F32_TILE_M_SMALL, 64>(p, vec, m->max_m_tiles, s);
        case F32_RAW: return f32_launch<F32_RAW, F32_TILE_M_SMALL, 64>(p, vec, m->max_m_tiles, s);
        case F32_DOWN: return F32_ROWS(F32_DOWN);
        case F32_DA: return F32_ROWS(F32_DA);
        case F32_DXG: return F32_ROWS(F32_DXG);
        case F32_WG2: return f32_launch<F32_WG2, 64, 64>(p, vec, 0, s);
        default: return f32_launch<F32_WG13, 64, 64>(p, vec, 0, s);
    }
#undef F32_ROWS
}
