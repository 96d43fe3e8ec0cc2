// Grouped products of fp32 layers on the bf16 matrix cores: the products of experts_f32.hip for batches with enough rows to fill tiles of
// 128 x 128 (or 64 x 128), fp32 operands and fp32 results.
//
// Every operand is split into three bf16 parts, each the rounding of what the parts before it leave: h + m + l = x exactly (24 bits in three times
// 8, unless l falls below the bf16 denormals, |x| < 2^-110).  A product of two numbers is the six partial products hh, hm, mh, mm, hl and
// lh - what is left out, ml, lm and ll, is at most 2^-24.01 of it (|m| <= 2^-8, |l| <= 2^-17) -, each exact in fp32, and v_mfma_f32_16x16x32_bf16 adds 32 of one kind to an fp32 sum.  hh has a
// sum of its own, the five small ones another, and the two are added once: a sum of K terms is rounded K / 32 times where a chain of
// fp32 fused multiply-adds is rounded K times.  Error against float64, 2-norm, chain -> here: normal factors, K = 32 1.0e-7 -> 3.9e-8, 256 2.9e-7 ->
// 9.1e-8, 1024 5.7e-7 -> 1.9e-7, 3584 1.06e-6 -> 3.7e-7; positive ones, 3584 9.1e-7 -> 3.3e-7 (with one sum for all six parts 9.2e-7 and 5.7e-7).
// A wave whose sums are infinite, no numbers or below 2^-100 - partial products round to multiples of 2^-149, as denormal factors and results do on
// these matrix cores, and 2^20 of them are then below 2^-27 of the sum - computes its part of the tile again on fp32 MFMAs.  A factor below 2^-110
// other than zero, whose last part would need bits below those of a bf16 denormal, loses up to 2^-134 of itself: where there is one, a tile's sums are held to
// 2^-106 of the largest factor times the number of terms, so that what is lost is below 2^-26 of them.
// The look at every factor is one v_min3_f32 for two of them; from a wave's first step with a zero on - a second copy of its loop, which costs every launch less
// than the branch in the first one - small ones are told from zeros.  Batches with zeros in every eighth row 1 % longer.  Where there is a tiny one the largest is found by fetching all of them once more (input gradient below 700 -> 950 us), and a launch all of whose waves compute again takes 2.7 times as
// long (dW1 and dW3 below 675 -> 1810: a unit in 64 that is saturated, h1 = -64, for every token).
//
// Bound: bf16 MFMA at a sixth of its rate, 417 TFLOP/s nominal, 240 under the power cap where fp32 MFMA has 154.  One workgroup = four waves of 64 rows
// x 64 columns (64 x 128 tiles: 64 x 32), two (three) workgroups per compute unit, one writing its parts to LDS while the other multiplies:
// 96 MFMAs, 176 vector instructions for the split, 24 fragment reads and 24 writes per wave and step of 32 k.  What a workgroup waits for in
// between leaves the matrix cores busy half of the time at 1.9 - 2.0 GHz.  Tried on the way (up product of 8192 rows, d = 1024, H = 3584, us): eight
// waves of 64 x 32 in one workgroup, two LDS buffers, the split between the MFMAs 745; the order of that pinned 727 - 740; four waves as here, 64-bit
// addresses per unit in registers, which spilled 917; as here 660.  Wave priorities, loads two steps ahead: no gain.
// T = 4096, d = 1024, H = 3584, E = 8, K = 2 (8192 rows), us, fp32 MFMAs -> here: up 1018 -> 660, down 515 -> 340, d(a) 604 -> 436, dxg 1040 -> 720, dW2
// 494 -> 352, dW1 and dW3 980 -> 678.
#include "f32_product.h"
#include "pack.h"
#include <algorithm>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 sp_bf16x8;
typedef __attribute__((ext_vector_type(4))) float sp_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t sp_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t sp_u32x2;

__device__ __forceinline__ uint32_t sp_pack(float lo, float hi)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {lo, hi};
    const bf16x2 r = __builtin_convertvector(v, bf16x2);
    return *(const uint32_t *)&r;
}

// two floats as three bf16 parts each
__device__ __forceinline__ void sp_split(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l)
{
    h = sp_pack(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    m = sp_pack(ra, rb);
    l = sp_pack(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}

// smallest magnitude so far (no number: left out)
__device__ __forceinline__ void sp_least(float &least, float a, float b)
{
    asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(least) : "v"(a), "v"(b));
}

// A thread's unit of one step: U = 4 k places of a row of an operand contiguous in k (a line of a row per 8 lanes), 8 of a column of one
// contiguous across k (64 columns per wave).  base = the step's first element (uniform), off = the unit's byte offset from it, ld = the
// distance of two k places
template <bool KMAJ> constexpr int sp_unit = KMAJ ? 8 : 4;
template <bool KMAJ, bool VEC>
__device__ __forceinline__ void sp_fetch(float (&v)[sp_unit<KMAJ>], const float *base, uint32_t off, int ld)
{
    asm volatile("" : "+v"(off));  // (widened here: a scalar base and 32 bits per lane, not a 64-bit address per unit)
    if constexpr (KMAJ) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *(const float *)((const unsigned char *)(base + (size_t)i * ld) + off);
    } else {
        const float *q = (const float *)((const unsigned char *)base + off);
        if (VEC) {
            const float4 a = *(const float4 *)q;
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = q[i];
        }
    }
}

// The last, partial step of kleft < 32 k places: those behind read as zero, addresses are clamped (k = the unit's first place)
template <bool KMAJ>
__device__ __forceinline__ void sp_fetch_partial(float (&v)[sp_unit<KMAJ>], const float *base, uint32_t off, int k, int kleft, int ld)
{
#pragma unroll
    for (int i = 0; i < sp_unit<KMAJ>; ++i) {
        const int kc = min(k + i, kleft - 1) - k;  // relative to the unit's first place
        const float *q = (const float *)((const unsigned char *)base + off);
        const float w = KMAJ ? q[(ptrdiff_t)kc * ld] : q[kc];
        v[i] = k + i < kleft ? w : 0.0f;
    }
}

// places k .. k + 3 of a row or column (ld: distance of two places of a column), zero from K1 on
template <bool KMAJ, bool VEC>
__device__ __forceinline__ void sp_four(float (&v)[4], const float *x, int k, int K1, int ld)
{
    if constexpr (!KMAJ && VEC) {  // (K1 % 4 == 0)
        const float4 q = *(const float4 *)(x + min(k, K1 - 4));
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = x[(size_t)min(k + i, K1 - 1) * (KMAJ ? ld : 1)];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (k + i >= K1) v[i] = 0.0f;
}

// Chunk swizzle of the planes (rows of 64 bytes).  LDS serves a ds_read_b128 in four passes of 16 lanes - 0-3, 12-15 and 20-27; 4-11, 16-19 and
// 28-31; the same of the upper half - over 64 banks: a fragment's pass takes rows 0-3 and 12-15 of one chunk and 4-11 of its neighbour, and rows r,
// r + 12 (chunk c), r + 4 and r + 8 (c ^ 1), which share four places, are kept apart by 0, 3, 2, 1 (4.7 cycles a read; 8 with pk_swz)
__device__ __forceinline__ int sp_swz(int row) { return ((row >> 2) & 1) | (((row >> 1) ^ (row >> 2)) & 2); }

// parts of 32 rows x 32 output columns that a row product's tile may be cut into (on fp32 MFMAs, f32_tile)
#define SP_PARTS(OP, TM, CT) (F32_IS_WG(OP) ? 1 : (TM) / 32 * ((CT) / 32))
// waves per SIMD, that is workgroups per compute unit, that the registers leave room for
#define SP_WAVES(NB) ((NB) == 2 ? 3 : 2)
#define SP_FACTOR_MIN 0x1p-110f
#define SP_SUM_MIN 0x1p-100f
// One tile of 64 WR rows x 16 NB WC MFMA columns (up: half of them W1's, half W3's): WR x WC = 4 waves of 4 x NB blocks of 16 x 16.
template <int OP, int WR, int WC, int NB, bool VEC>
__global__ __launch_bounds__(256, SP_WAVES(NB)) void f32_split_kernel(f32_args p)
{
    constexpr bool WG = F32_IS_WG(OP), PAIR = F32_PAIR(OP);
    constexpr bool AK = WG, BKM = WG || OP == F32_DA || OP == F32_DXG;  // operand contiguous across k
    constexpr int TM = 64 * WR, TN = 16 * NB * WC, THR = 256, NUA = 32 * TM / (sp_unit<AK> * THR), NUB = 32 * TN / (sp_unit<BKM> * THR), CT = PAIR ? TN / 2 : TN;
    constexpr int PA = 64 * TM, PB = 64 * TN;  // bytes of a plane of A, of B
    static_assert(WR * WC == 4, "four waves");
    extern __shared__ __attribute__((aligned(1024))) unsigned char sp_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4, wr = wave / WC, wc = wave % WC;
    if (OP == F32_UP && (int)blockIdx.x >= (int)gridDim.x - p.copy_wgs) {
        copy_gathered<VEC, false>(p, blockIdx.x - (gridDim.x - p.copy_wgs), lane, wave, 0);
        return;
    }
    const int NT = (p.N + CT - 1) / CT;
    const int MT = WG ? (p.Kd + TM - 1) / TM : p.tile_meta[0];
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    int t, mat = 0, part = -1;
    if (WG) {
        t = wgrad_tile(p.deal, xcd, j, &mat);
        if (t < 0) return;
        for (; p.deal.together > 1 && t >= MT * NT; t -= MT * NT) ++mat;
    } else {
        // Tiles of a last round of up to 3/8 of what an XCD holds (p.part_max) go in parts: alone on its compute unit a workgroup takes 0.6 of
        // what two take together, a part on fp32 MFMAs a thirteenth of that.  us, in tiles / parts: down product of 8192 rows, k = 3584, N = 1024
        // (one round of 64 and 4) 450 / 323, dxg 954 / 714; a limit of 5/8 was no better.  So do all tiles of a launch with up to three for four
        // compute units (p.few): a product of few columns does not hold the other one's tile height back.  Tiles of 128 against 32 rows, 900 shapes: up
        // to 0.1 tiles per unit 3.0 - 6.8 times as long, 0.5 to 0.6 1.0 - 1.4, 0.6 to 0.8 0.9 - 1.2, 0.8 to 1 0.7 - 1.1.
        const int total = MT * NT, per = (total + 7) >> 3, i = f32_part<SP_PARTS(OP, TM, CT)>(p, per, j, part);
        t = xcd * per + i;
        if (i >= per || t >= total) return;
    }
    const int rb = t / (8 * NT), nrb = min(8, MT - 8 * rb), ti = t - rb * 8 * NT;
    const int mt = 8 * rb + ti % nrb, n0 = (ti / nrb) * CT;
    if constexpr (!WG) {
        if (part >= 0) {
            constexpr int PN = PAIR ? 64 : 32, LAP = f32_lds_floats(32, false, F32_FBK(32));
            f32_tile<OP, 32, PN, VEC>(p, (float *)sp_lds, (float *)sp_lds + 2 * LAP, mt, p.tiles[mt], 32 * (part % (TM / 32)), n0 + 32 * (part / (TM / 32)), mat);
            return;
        }
    }

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
        A0 = (shared && p.Atok ? p.Atok : Ad + (size_t)row0 * p.Kd) + m0;
        B0 = (shared && p.Btok ? p.Btok : p.B0 + (size_t)row0 * p.N) + n0;
    } else {
        const omega_tile tl = p.tiles[mt];
        g = tl.g;
        rows = tl.rows;
        row0 = tl.row0;
        K1 = p.Kd;
        A0 = p.Atok && tl.xrow0 >= 0 ? p.Atok + (size_t)tl.xrow0 * p.Kd : p.A0 + (size_t)row0 * p.Kd;
        fetch_rows = OP == F32_UP && p.tokp != nullptr && tl.xrow0 < 0;
        if (fetch_rows) A0 = p.Atok;
        if (OP == F32_DXG) A1 = p.A1 + (size_t)row0 * p.Kd;
        const size_t wo = (size_t)g * p.N * p.Kd + (BKM ? (size_t)n0 : (size_t)n0 * K1);
        B0 = p.B0 + wo;
        if (PAIR || OP == F32_DXG) B1 = p.B1 + wo;
    }

    // This thread's units: byte offsets from the step's first element (up: the W3 columns from W3's) and places in a plane.  Rows
    // (columns) past the tile's edge repeat the last valid one and are never stored.
    constexpr int UA = sp_unit<AK>, UB = sp_unit<BKM>;
    auto unit_x = [&](bool kmaj, int tx, int u) { return kmaj ? (tid + THR * u) % tx : (tid + THR * u) >> 3; };
    auto unit_k = [&](bool kmaj, int tx, int u) { return kmaj ? (tid + THR * u) / tx * 8 : (tid & 7) * 4; };
    // (K-contiguous units of a thread lie THR / 8 rows apart, at the same place of their rows)
    constexpr uint32_t ROWS = THR / 8 * 64;
    auto place = [&](int x, int k) { return (uint32_t)(x * 64 + (((k >> 3) ^ sp_swz(x)) << 4) + (k & 4) * 2); };
    uint32_t oa[NUA], ob[NUB], la[AK ? NUA : 1], lb[BKM ? NUB : 1];
#pragma unroll
    for (int u = 0; u < NUA; ++u) {
        const int x = unit_x(AK, TM, u), k = unit_k(AK, TM, u);
        oa[u] = 4u * (AK ? (uint32_t)k * p.Kd + min(x, rows - 1) : (uint32_t)(fetch_rows ? p.tokp[row0 + min(x, rows - 1)] : min(x, rows - 1)) * K1 + k);
        if (AK || u == 0) la[AK ? u : 0] = place(x, k);
    }
#pragma unroll
    for (int u = 0; u < NUB; ++u) {
        const int x = unit_x(BKM, TN, u), k = unit_k(BKM, TN, u);
        ob[u] = 4u * (BKM ? (uint32_t)k * p.N + min(x, p.N - 1 - n0) : (uint32_t)min(PAIR && x >= CT ? x - CT : x, p.N - 1 - n0) * K1 + k);
        if (BKM || u == 0) lb[BKM ? u : 0] = 3 * PA + place(x, k);
    }
    auto of_w3 = [](int u) { return PAIR && THR / 8 * u >= CT; };

    // (weight gradients of a few rows: of one product the sum of its six parts is rounded several times.  Largest error against float64, chain / here, of
    // one term 5.96e-8 / 1.03e-7 of it, of four 1.9e-7 / 1.6e-7)
    const bool few = WG && K1 < SP_TERMS_MIN;
    const int S1 = few ? 0 : K1 / 32, steps = OP == F32_DXG ? 2 * S1 : S1;
    const float *a_at = A0, *b_at = B0, *b3_at = B1;
    float va[NUA][UA], vb[NUB][UB];
    auto fetch = [&]() {
#pragma unroll
        for (int u = 0; u < NUA; ++u) sp_fetch<AK, VEC>(va[u], a_at, oa[u], p.Kd);
#pragma unroll
        for (int u = 0; u < NUB; ++u) sp_fetch<BKM, VEC>(vb[u], of_w3(u) ? b3_at : b_at, ob[u], p.N);
    };
    auto advance = [&](int s) {  // to step s; behind the last one they stay
        if (s >= steps) return;
        a_at += AK ? (size_t)32 * p.Kd : 32;
        b_at += BKM ? (size_t)32 * p.N : 32;
        if (PAIR) b3_at += 32;
        if (OP == F32_DXG && s == S1) {
            a_at = A1;
            b_at = B1;
        }
    };
    const int kleft = few ? 0 : K1 - S1 * 32;
    auto fetch_rest = [&](int seg) {  // the places behind the whole steps
        const float *at = (seg ? A1 : A0) + (AK ? (size_t)S1 * 32 * p.Kd : S1 * 32);
        const float *bt = (OP == F32_DXG && seg ? B1 : B0) + (BKM ? (size_t)S1 * 32 * p.N : S1 * 32);
        const float *b3t = PAIR ? B1 + S1 * 32 : bt;
#pragma unroll
        for (int u = 0; u < NUA; ++u) sp_fetch_partial<AK>(va[u], at, oa[u], unit_k(AK, TM, u), kleft, p.Kd);
#pragma unroll
        for (int u = 0; u < NUB; ++u) sp_fetch_partial<BKM>(vb[u], of_w3(u) ? b3t : bt, ob[u], unit_k(BKM, TN, u), kleft, p.N);
    };
    // Splitting: pair q of the thread's places (A's units, then B's) into w, which goes to LDS with the last pair of a unit
    constexpr int QA = NUA * UA / 2, QB = NUB * UB / 2;
    struct parts { uint32_t h[4], m[4], l[4]; };
    auto store = [&](unsigned char *at, const uint32_t (&v)[4], bool eight) {
        if (eight) *(sp_u32x4 *)at = sp_u32x4{v[0], v[1], v[2], v[3]};
        else *(sp_u32x2 *)at = sp_u32x2{v[0], v[1]};
    };
    auto split = [&](parts &w, int q) {
        const bool a = q < QA;
        const int U = a ? UA : UB, qq = a ? q : q - QA, u = qq / (U / 2), i = qq % (U / 2);
        const float *v = a ? va[a ? u : 0] : vb[a ? 0 : u];
        sp_split(v[2 * i], v[2 * i + 1], w.h[i], w.m[i], w.l[i]);
        if (i < U / 2 - 1) return;
        unsigned char *at = sp_lds + (a ? AK ? la[a && AK ? u : 0] : la[0] + u * ROWS : BKM ? lb[!a && BKM ? u : 0] : lb[0] + u * ROWS);
        store(at, w.h, U == 8);
        store(at + (a ? PA : PB), w.m, U == 8);
        store(at + 2 * (a ? PA : PB), w.l, U == 8);
    };

    float least = 1.0f;               // smallest magnitude among this lane's factors of the steps before the first with a small one ...
    int small_step = -1;              // ... and that step
    uint32_t smallest = 0xffffffffu;  // of its factors other than zero, from there on: the bits but the sign, less one (zeros wrap)
    auto note_small = [&]() {
#pragma unroll
        for (int u = 0; u < NUA; ++u)
#pragma unroll
            for (int i = 0; i < UA; ++i) smallest = min(smallest, (__float_as_uint(va[u][i]) << 1) - 1u);
#pragma unroll
        for (int u = 0; u < NUB; ++u)
#pragma unroll
            for (int i = 0; i < UB; ++i) smallest = min(smallest, (__float_as_uint(vb[u][i]) << 1) - 1u);
    };

    // row units of 16: unit WR i + wr; columns: block n of the wave
    const int live = max(0, min(4, ((rows + 15) / 16 + WR - 1 - wr) / WR));
    const int xu = 16 * wr + l16;
    const uint32_t ra = (uint32_t)(xu * 64 + ((lq ^ sp_swz(xu)) << 4));  // (the swizzle goes by the row within its 16)
    int xb[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) xb[n] = (PAIR ? 8 * NB * wc + 16 * (n % (NB / 2)) + CT * (n / (NB / 2)) : 16 * NB * wc + 16 * n) + l16;
    const uint32_t rb0 = (uint32_t)(3 * PA + xb[0] * 64 + ((lq ^ sp_swz(xb[0])) << 4));
    sp_f32x4 acc[4][NB], low[4][NB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[i][n] = low[i][n] = sp_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // All steps for a wave with MBL live row units.  A step: the places in registers are split into the planes, the next step's are asked for, a barrier - the
    // planes are whole -, the products, row unit by row unit, 6 NB MFMAs each with the next unit's fragments read before them, and a barrier: the planes,
    // of which there is one set, have been read and may be written again.
    auto run = [&](auto mbl) {
        constexpr int MBL = decltype(mbl)::value;
        sp_bf16x8 fa[2][3], fb[NB][3];
        auto read_a = [&](int i) {
            if (i >= MBL) return;
#pragma unroll
            for (int q = 0; q < 3; ++q) fa[i & 1][q] = *(const sp_bf16x8 *)(sp_lds + q * PA + ra + i * WR * 1024);
        };
        auto read_b = [&](int n) {
            if (MBL == 0) return;
#pragma unroll
            for (int q = 0; q < 3; ++q) fb[n][q] = *(const sp_bf16x8 *)(sp_lds + q * PB + rb0 + (xb[n] - xb[0]) * 64);
        };
        // MFMA m of the six of a block: the smallest parts first, so that what they sum to is not rounded to the whole sum's last place
        auto mul = [&](int i, int n, int m) {
            constexpr int pa[6] = {2, 0, 0, 1, 1, 0}, pb[6] = {0, 0, 2, 1, 0, 1};
            if (i >= MBL) return;
            sp_f32x4 &d = m == 1 ? acc[i][n] : low[i][n];
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i & 1][pa[m]], fb[n][pb[m]], d, 0, 0, 0);
        };
        auto stage = [&](auto careful) {
            parts w;
            float now = 1.0f, &low_end = decltype(careful)::value ? now : least;
#pragma unroll
            for (int q = 0; q < QA + QB; ++q) {
                const int qq = q < QA ? q : q - QA;
                if (q < QA) sp_least(low_end, va[qq / (UA / 2)][2 * (qq % (UA / 2))], va[qq / (UA / 2)][2 * (qq % (UA / 2)) + 1]);
                else sp_least(low_end, vb[qq / (UB / 2)][2 * (qq % (UB / 2))], vb[qq / (UB / 2)][2 * (qq % (UB / 2)) + 1]);
                split(w, q);
            }
            if (decltype(careful)::value && __any(now < SP_FACTOR_MIN)) note_small();
        };
        auto multiply = [&]() {
            read_a(0);
#pragma unroll
            for (int n = 0; n < NB; ++n) read_b(n);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                read_a(i + 1 < 4 ? i + 1 : 4);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < 6; ++m)
#pragma unroll
                    for (int n = 0; n < NB; ++n) mul(i, n, m);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // from step s on; not careful: up to the first one with a zero or less than SP_FACTOR_MIN
        auto steps_from = [&](auto careful, int s) {
            for (bool small = false; s < steps && !small; ++s) {
                stage(careful);
                advance(s + 1);
                fetch();
                if (!decltype(careful)::value) small = __any(least < SP_FACTOR_MIN);
                __syncthreads();
                multiply();
                __syncthreads();
            }
            return s;
        };
        if (steps > 0) {
            fetch();
            const int s = steps_from(std::false_type(), 0);
            if (__any(least < SP_FACTOR_MIN)) {
                small_step = s - 1;
                steps_from(std::true_type(), s);
            }
        }
        for (int seg = 0; kleft > 0 && seg < (OP == F32_DXG ? 2 : 1); ++seg) {
            fetch_rest(seg);
            stage(std::true_type());
            __syncthreads();
            multiply();
            __syncthreads();
        }
    };
    switch (live) {
        case 4: run(std::integral_constant<int, 4>()); break;
        case 3: run(std::integral_constant<int, 3>()); break;
        case 2: run(std::integral_constant<int, 2>()); break;
        case 1: run(std::integral_constant<int, 1>()); break;
        default: run(std::integral_constant<int, 0>()); break;
    }

    // What the three parts cannot carry: sums that are infinite or no number (an infinite h times a part that is zero, and what rounds to an
    // infinite h), or so small that what factors and partial products have lost counts.  Their wave computes its part of the tile again: fragments
    // straight from memory, 16 k places at a time.
    float limit = SP_SUM_MIN;
    auto words = [&](int at, uint32_t v) {  // one of each wave (every wave's last reads of the planes are behind it)
        if (lane == 0) ((uint32_t *)sp_lds)[at + wave] = v;
        __syncthreads();
        return *(const sp_u32x4 *)(sp_lds + 4 * at);
    };
    if (small_step >= 0) {  // (its factors were on their way out when it was seen)
        const int s = OP == F32_DXG && small_step >= S1 ? small_step - S1 : small_step;
        a_at = (s != small_step ? A1 : A0) + (AK ? (size_t)32 * s * p.Kd : 32 * s);
        b_at = (s != small_step ? B1 : B0) + (BKM ? (size_t)32 * s * p.N : 32 * s);
        b3_at = PAIR ? B1 + 32 * s : nullptr;
        fetch();
        note_small();
    }
    const sp_u32x4 w = words(0, __any(smallest < 2u * __float_as_uint(SP_FACTOR_MIN) - 1u));
    const bool tiny = __builtin_amdgcn_readfirstlane(w[0] | w[1] | w[2] | w[3]) != 0;
    if (tiny) {  // the largest factor, from all of them once more
        float most = 0.0f;
        auto all = [&]() {
#pragma unroll
            for (int u = 0; u < NUA; ++u)
#pragma unroll
                for (int i = 0; i < UA; ++i) most = fmaxf(most, fabsf(va[u][i]));
#pragma unroll
            for (int u = 0; u < NUB; ++u)
#pragma unroll
                for (int i = 0; i < UB; ++i) most = fmaxf(most, fabsf(vb[u][i]));
        };
        a_at = A0;
        b_at = B0;
        b3_at = B1;
        for (int s = 0; s < steps; ++s) {
            fetch();
            advance(s + 1);
            all();
        }
        for (int seg = 0; kleft > 0 && seg < (OP == F32_DXG ? 2 : 1); ++seg) {
            fetch_rest(seg);
            all();
        }
#pragma unroll
        for (int q = 1; q < 64; q <<= 1) most = fmaxf(most, __shfl_xor(most, q, 64));
        const sp_u32x4 m = words(4, __float_as_uint(most));
        limit = fmaxf(limit, __uint_as_float(max(max(m[0], m[1]), max(m[2], m[3]))) * K1 * 0x1p-106f);
    }
    // (infinities and no numbers show in the sum of all, the smallest one other than zero in its bits; units behind the tile's rows are zero)
    float all = 0.0f;
    uint32_t low_end = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            acc[i][n] += low[i][n];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                all += acc[i][n][r];
                low_end = min(low_end, (__float_as_uint(acc[i][n][r]) << 1) - 1u);
            }
        }
    bool odd = few || !(fabsf(all) < INFINITY) || low_end < 2u * __float_as_uint(limit) - 1u;
    if (tiny) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) odd |= i < live && acc[i][n][r] == 0.0f;
    }
    if (__any(odd && live > 0)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[i][n] = sp_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int seg = 0; seg < (OP == F32_DXG ? 2 : 1); ++seg) {
            const float *A = seg ? A1 : A0, *B = OP == F32_DXG && seg ? B1 : B0;
            if (seg) {  // (the second pair's own sum, as in f32_tile)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        low[i][n] = acc[i][n];
                        acc[i][n] = sp_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
            size_t xa[4], xo[NB];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int x = min(16 * (WR * i + wr) + l16, rows - 1);
                xa[i] = AK ? (size_t)x : (size_t)(fetch_rows ? p.tokp[row0 + x] : x) * K1;
            }
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const int x = min(PAIR && n >= NB / 2 ? xb[n] - CT : xb[n], p.N - 1 - n0);
                xo[n] = BKM ? (size_t)x : (size_t)x * K1;
            }
            for (int k0 = 0; k0 < K1; k0 += 16) {  // (lane quarter q: places 4 q .. 4 q + 3 of 16)
                const int k = k0 + 4 * lq;
                float a[4][4], b[NB][4];
#pragma unroll
                for (int n = 0; n < NB; ++n) sp_four<BKM, VEC>(b[n], (PAIR && n >= NB / 2 ? B1 : B) + xo[n], k, K1, p.N);
#pragma unroll
                for (int i = 0; i < 4; ++i) sp_four<AK, VEC>(a[i], A + xa[i], k, K1, p.Kd);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int n = 0; n < NB; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][u], b[n][u], acc[i][n], 0, 0, 0);
            }
            if (seg) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int n = 0; n < NB; ++n) acc[i][n] += low[i][n];
            }
        }
    }

    // lane: column l16 of a block; register r -> row 4 lq + r
    float *C = p.C;
    if (OP == F32_WG2) C += (size_t)g * p.N * p.Kd;
    if (OP == F32_WG13) C += (size_t)mat * p.N * p.Kd;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= live) continue;
#pragma unroll
        for (int n = 0; n < (PAIR ? NB / 2 : NB); ++n) {
            const int col = n0 + xb[n], rbase = 16 * (WR * i + wr) + 4 * lq;
            if (col >= p.N) continue;
            const size_t o = (size_t)(WG ? m0 : row0) * p.N + col;
            float h1[4], h3[4];
            if (OP == F32_DA) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const size_t at = o + (size_t)min(rbase + r, rows - 1) * p.N;
                    h1[r] = p.H1[at];
                    h3[r] = p.H3[at];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = rbase + r;
                if (row >= rows) continue;
                const size_t at = o + (size_t)row * p.N;
                const float v = acc[i][n][r];
                if (PAIR) {
                    const float u = acc[i][PAIR ? n + NB / 2 : 0][r];
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
}

template <int OP, int WR, int WC, int NB>
static hipError_t sp_launch(f32_args p, bool vec, int max_tiles, hipStream_t s)
{
    constexpr bool WG = F32_IS_WG(OP), BKM = WG || OP == F32_DA || OP == F32_DXG;
    constexpr int TM = 64 * WR, TN = 16 * NB * WC, CT = F32_PAIR(OP) ? TN / 2 : TN;
    // (a part keeps both operands twice, as floats)
    constexpr int PART = 8 * (f32_lds_floats(32, false, F32_FBK(32)) + f32_lds_floats(F32_PAIR(OP) ? 64 : 32, BKM, F32_FBK(32)));
    constexpr int LDS = std::max(3 * 64 * (TM + TN), WG ? 0 : PART);
    const int mats = OP == F32_WG13 ? 2 * p.G : p.G;
    const size_t tiles = (size_t)ceil_div(p.N, CT) * (WG ? (size_t)ceil_div(p.Kd, TM) * mats : max_tiles);
    if (WG) p.deal = wgrad_deal_of(ceil_div(p.N, CT) * ceil_div(p.Kd, TM), mats);
    p.slots *= SP_WAVES(NB);
    p.part_max = p.slots * 3 / 8;
    const unsigned grid = (WG ? (unsigned)((tiles + 7) / 8 * 8 + (p.deal.rest > 0 ? 8 : 0)) : f32_grid(p, tiles, SP_PARTS(OP, TM, CT))) + p.copy_wgs;
    // (weight gradients load element by element in any case)
    if (WG || vec) hipLaunchKernelGGL((f32_split_kernel<OP, WR, WC, NB, true>), dim3(grid), dim3(256), LDS, s, p);
    else if constexpr (!WG) hipLaunchKernelGGL((f32_split_kernel<OP, WR, WC, NB, false>), dim3(grid), dim3(256), LDS, s, p);
    return hipGetLastError();
}

hipError_t launch_product_f32_split(const f32_args &p, int op, bool vec, int max_tiles, hipStream_t s)
{
#define SP_ROWS(OP) (p.bm == F32_TILE_M ? sp_launch<OP, 2, 2, 4>(p, vec, max_tiles, s) : sp_launch<OP, 1, 4, 2>(p, vec, max_tiles, s))
    switch (op) {
        case F32_UP: return SP_ROWS(F32_UP);
        case F32_RAW: return SP_ROWS(F32_RAW);
        case F32_DOWN: return sp_launch<F32_DOWN, 2, 2, 4>(p, vec, max_tiles, s);
        case F32_DA: return SP_ROWS(F32_DA);
        case F32_DXG: return sp_launch<F32_DXG, 2, 2, 4>(p, vec, max_tiles, s);
        case F32_WG2: return sp_launch<F32_WG2, 2, 2, 4>(p, vec, max_tiles, s);
        default: return sp_launch<F32_WG13, 2, 2, 4>(p, vec, max_tiles, s);
    }
#undef SP_ROWS
}
