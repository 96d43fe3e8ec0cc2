// The dispatch index of a batch of few pairs - what dispatch_rank_kernel (dispatch.hip) leaves - by one workgroup within another launch.
#pragma once
#include "common.h"

struct index_args {
    const int32_t *ids;
    int32_t *counts, *offsets, *dst, *dstp, *src_row, *tokp, *tile_meta;
    omega_tile *tiles;
    int T, K, E, Es;
};
static inline index_args index_args_of(const omega_moe *m, int T)
{
    return {m->ids, m->counts, m->offsets, m->dst, m->dstp, m->src_row, m->tokp, m->tile_meta, m->tiles, T, m->cfg.K, m->cfg.E, m->cfg.Es};
}

// id: the choices of all pairs; s: 3 x 256 ints; both LDS.  bm: rows of a row tile.
__device__ __forceinline__ void small_index(const index_args &p, const uint8_t *id, int *s, int bm, int nthr)
{
    const int P = p.T * p.K, tid = threadIdx.x, lane = tid & 63;
    int *run = s, *off = s + 256, *first = s + 512;
    for (int e = tid; e < p.E; e += nthr) run[e] = 0;
    __syncthreads();
    for (int i = tid; i < P; i += nthr) atomicAdd(&run[id[i]], 1);
    __syncthreads();
    if (tid >= 64) return;
    // exclusive scans of the counts and of their tiles, four experts per lane; run[e] becomes the rows of e that have their place
    int c[4], sum = 0, sumt = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int e = 4 * lane + i;
        c[i] = e < p.E ? run[e] : 0;
        sum += c[i];
        sumt += (c[i] + bm - 1) / bm;
    }
    int incl = sum, inclt = sumt;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const int o = __shfl_up(incl, m, 64), ot = __shfl_up(inclt, m, 64);
        if (lane >= m) { incl += o; inclt += ot; }
    }
    const int tiles = __builtin_amdgcn_readlane(inclt, 63), per_shared = (p.T + bm - 1) / bm;
    int at = incl - sum, mt = inclt - sumt;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int e = 4 * lane + i;
        if (e >= p.E) continue;
        p.counts[e] = c[i];
        p.offsets[e] = at;
        p.tile_meta[1 + e] = mt;
        for (int r = 0; r < c[i]; r += bm) p.tiles[mt + r / bm] = {e, mt * bm + r, min(bm, c[i] - r), -1};
        run[e] = 0;
        off[e] = at;
        first[e] = mt;
        at += c[i];
        mt += (c[i] + bm - 1) / bm;
    }
    for (int g = lane; g <= p.Es; g += 64) {
        const int m0 = tiles + g * per_shared;
        p.tile_meta[1 + p.E + g] = m0;
        for (int r = 0; g < p.Es && r < p.T; r += bm) p.tiles[m0 + r / bm] = {p.E + g, m0 * bm + r, min(bm, p.T - r), r};
    }
    if (lane == 0) {
        p.offsets[p.E] = P;
        p.tile_meta[0] = tiles + p.Es * per_shared;
    }
    // Stable ranks, 64 pairs at a time: the lanes with one expert find each other by one ballot per bit of its number, run[e] moves on by their
    // number.  (This wave's chain ends the launch.  With a ballot per expert of the 64 pairs, forward pass of 26 tokens x 1024 x 384, 172 experts, top 38 153
    // us, 130 with a launch for the index.)
    const int bits = 32 - __clz(p.E - 1 | 1);
    for (int c0 = 0; c0 < P; c0 += 64) {
        const int i = c0 + lane;
        const bool valid = i < P;
        const int e = valid ? id[i] : -1;
        unsigned long long mine = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const unsigned long long m = __ballot(e >> b & 1);
            mine &= e >> b & 1 ? m : ~m;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const unsigned long long below = mine & ((1ull << lane) - 1ull);
        if (valid) {
            const int rank = run[e] + __popcll(below), r = off[e] + rank, prow = first[e] * bm + rank, t = i / p.K;
            p.dst[i] = r;
            p.dstp[i] = prow;
            p.src_row[r] = t;
            p.tokp[prow] = t;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (valid && below == 0) run[e] += __popcll(mine);
    }
}
