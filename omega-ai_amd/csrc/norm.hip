// RMSNorm in front of the layer (block form): rms[t] = sqrtf(sum_k x[t,k]^2 / d + 1e-6f), h[t,k] = (x[t,k] / rms[t]) * w[k],
// with the sum taken exactly as rmsnorm_forward_kernel2 takes it
// (J/engine/nn/layer/normalization/gpu/RMSKernel.cu:185-223): 32 lanes per row, lane l adds x[i]*x[i] for
// i = l, l+32, ... in index order with one fused multiply-add per step, then an xor butterfly (16, 8, 4, 2, 1) over
// the 32 partial sums.  h is written once, in the layer's storage type (rounded to bf16 in bf16 layers), and is what
// the router and the gather read; the residual x is added back by the combine kernel.
//
// One workgroup = 8 rows x 32 lanes.  The rows come in with 16-byte loads, pass through LDS as fp32 and are read
// back lane-strided (32 consecutive floats per row and step: no bank conflicts); chunks of NORM_DC columns keep the
// order of every lane's additions (chunk boundaries are multiples of 32).  The second pass re-reads the rows (they
// are still in L2) and writes h with 16-byte stores.
// This file is compiled with -ffp-contract=off; the only fused operation is the explicit fmaf.
#include "common.h"
#include <algorithm>

#define NORM_ROWS 8
#define NORM_DC 2048  // columns per staged chunk: 8 rows x 2048 x 4 B = 64 KiB of LDS

// h == nullptr: statistics only
template <bool XBF>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const void *__restrict__ x, const float *__restrict__ gamma, int T,
                                                      int d, float *__restrict__ rms, void *__restrict__ h)
{
    __shared__ float rms_s[NORM_ROWS];
    __shared__ __attribute__((aligned(16))) float xs[NORM_ROWS][NORM_DC];
    const int tid = threadIdx.x;
    const int r = tid >> 5, l = tid & 31;
    const int t0 = blockIdx.x * NORM_ROWS;
    const bool vec_ok = (d % 8 == 0) && ((uintptr_t)x % 16 == 0);
    float s = 0.0f;
    for (int c0 = 0; c0 < d; c0 += NORM_DC) {
        const int cw = min(NORM_DC, d - c0);  // columns of this chunk
        // stage: 8 consecutive columns per thread and pass
        for (int i = tid * 8; i < NORM_ROWS * NORM_DC; i += 256 * 8) {
            const int rr = i / NORM_DC, cc = i % NORM_DC;
            const int t = t0 + rr;
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = 0.0f;
            if (t < T && cc < cw) {
                const size_t off = (size_t)t * d + c0 + cc;
                if (vec_ok && cc + 8 <= cw) {
                    if (XBF) {
                        const uint4 u = *(const uint4 *)((const bf16_t *)x + off);
                        v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
                        v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
                        v[4] = __uint_as_float(u.z << 16); v[5] = __uint_as_float(u.z & 0xffff0000u);
                        v[6] = __uint_as_float(u.w << 16); v[7] = __uint_as_float(u.w & 0xffff0000u);
                    } else {
                        const float4 a = *(const float4 *)((const float *)x + off);
                        const float4 b = *(const float4 *)((const float *)x + off + 4);
                        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
                        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        if (cc + q < cw)
                            v[q] = XBF ? bf16_to_f32(((const bf16_t *)x)[off + q]) : ((const float *)x)[off + q];
                }
            }
            *(float4 *)&xs[rr][cc] = make_float4(v[0], v[1], v[2], v[3]);
            *(float4 *)&xs[rr][cc + 4] = make_float4(v[4], v[5], v[6], v[7]);
        }
        __syncthreads();
        // columns beyond the row are zero: fmaf(0, 0, s) leaves s unchanged
        const int steps = (cw + 31) / 32;
#pragma unroll 8
        for (int j = 0; j < steps; ++j) {
            const float v = xs[r][l + 32 * j];
            s = fmaf(v, v, s);
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) s = s + __shfl_xor(s, m, 32);
    const int t = t0 + r;
    const float my = sqrtf(s / (float)d + 1e-6f);
    if (l == 0) {
        rms_s[r] = my;
        if (t < T) rms[t] = my;
    }
    if (h == nullptr) return;
    __syncthreads();
    // second pass: 8 consecutive columns per thread and step
    const int per_row = (d + 7) / 8;
    for (int i = tid; i < NORM_ROWS * per_row; i += 256) {
        const int rr = i / per_row, cc = (i % per_row) * 8;
        const int tt = t0 + rr;
        if (tt >= T) continue;
        const float rv = rms_s[rr];
        const size_t off = (size_t)tt * d + cc;
        float v[8], g[8];
        const bool full = vec_ok && ((uintptr_t)h % 16 == 0) && ((uintptr_t)gamma % 16 == 0) && cc + 8 <= d;
        if (full) {
            const float4 g0 = *(const float4 *)(gamma + cc), g1 = *(const float4 *)(gamma + cc + 4);
            g[0] = g0.x; g[1] = g0.y; g[2] = g0.z; g[3] = g0.w; g[4] = g1.x; g[5] = g1.y; g[6] = g1.z; g[7] = g1.w;
            if (XBF) {
                const uint4 u = *(const uint4 *)((const bf16_t *)x + off);
                v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
                v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
                v[4] = __uint_as_float(u.z << 16); v[5] = __uint_as_float(u.z & 0xffff0000u);
                v[6] = __uint_as_float(u.w << 16); v[7] = __uint_as_float(u.w & 0xffff0000u);
            } else {
                const float4 a = *(const float4 *)((const float *)x + off), b = *(const float4 *)((const float *)x + off + 4);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = norm_apply<XBF>(v[q], rv, g[q]);
            if (XBF) {
                uint4 o;
                o.x = (__float_as_uint(v[0]) >> 16) | (__float_as_uint(v[1]) & 0xffff0000u);
                o.y = (__float_as_uint(v[2]) >> 16) | (__float_as_uint(v[3]) & 0xffff0000u);
                o.z = (__float_as_uint(v[4]) >> 16) | (__float_as_uint(v[5]) & 0xffff0000u);
                o.w = (__float_as_uint(v[6]) >> 16) | (__float_as_uint(v[7]) & 0xffff0000u);
                *(uint4 *)((bf16_t *)h + off) = o;
            } else {
                *(float4 *)((float *)h + off) = make_float4(v[0], v[1], v[2], v[3]);
                *(float4 *)((float *)h + off + 4) = make_float4(v[4], v[5], v[6], v[7]);
            }
        } else {
            for (int q = 0; q < 8 && cc + q < d; ++q) {
                const float xv = XBF ? bf16_to_f32(((const bf16_t *)x)[off + q]) : ((const float *)x)[off + q];
                const float hv = norm_apply<XBF>(xv, rv, gamma[cc + q]);
                if (XBF) ((bf16_t *)h)[off + q] = f32_to_bf16(hv);
                else ((float *)h)[off + q] = hv;
            }
        }
    }
}

// Rows of whole 16-byte pieces (d % 8 == 0, aligned): R rows per workgroup of 256 threads, NV pieces of 8 columns per thread,
// all asked for at once and kept in registers from the statistics to the normalised store, so the launch is one memory
// latency, the 32-lane sums (which read the staged fp32 values in their order) and the divisions.  Bound: the bytes of x and h;
// the chunked kernel above exposed a latency per piece: 777 rows of 4096 columns 28 -> 14 us, 3000 of 2048 17 -> 11 us.
template <bool XBF>
__device__ __forceinline__ void load_piece(const void *__restrict__ p, size_t off, float (&v)[8])
{
    if (XBF) {
        const uint4 u = *(const uint4 *)((const bf16_t *)p + off);
        v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
        v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
        v[4] = __uint_as_float(u.z << 16); v[5] = __uint_as_float(u.z & 0xffff0000u);
        v[6] = __uint_as_float(u.w << 16); v[7] = __uint_as_float(u.w & 0xffff0000u);
    } else {
        *(float4 *)&v[0] = *(const float4 *)((const float *)p + off);
        *(float4 *)&v[4] = *(const float4 *)((const float *)p + off + 4);
    }
}
// eight values, already rounded to the storage type where it is bf16
template <bool XBF>
__device__ __forceinline__ void store_piece(void *__restrict__ p, size_t off, const float (&v)[8])
{
    if (XBF) {
        uint4 o;
        o.x = (__float_as_uint(v[0]) >> 16) | (__float_as_uint(v[1]) & 0xffff0000u);
        o.y = (__float_as_uint(v[2]) >> 16) | (__float_as_uint(v[3]) & 0xffff0000u);
        o.z = (__float_as_uint(v[4]) >> 16) | (__float_as_uint(v[5]) & 0xffff0000u);
        o.w = (__float_as_uint(v[6]) >> 16) | (__float_as_uint(v[7]) & 0xffff0000u);
        *(uint4 *)((bf16_t *)p + off) = o;
    } else {
        *(float4 *)((float *)p + off) = make_float4(v[0], v[1], v[2], v[3]);
        *(float4 *)((float *)p + off + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
}
// sum of 32 lanes as the reference's warp reduction takes it
__device__ __forceinline__ float warp32_sum(float s)
{
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) s = s + __shfl_xor(s, m, 32);
    return s;
}

template <bool XBF, int R, int NV>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const void *__restrict__ x, const float *__restrict__ gamma, int T, int d,
                                                           float *__restrict__ rms, void *__restrict__ h)
{
    extern __shared__ __attribute__((aligned(16))) float xs[];  // [R][d]
    __shared__ float rms_s[R];
    const int tid = threadIdx.x, t0 = blockIdx.x * R, ppr = d >> 3, np = R * ppr;  // pieces per row, of the workgroup
    float v[NV][8];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = min(tid + 256 * u, np - 1), rr = i / ppr;
        load_piece<XBF>(x, (size_t)min(t0 + rr, T - 1) * d + (i - rr * ppr) * 8, v[u]);
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = min(tid + 256 * u, np - 1);
        *(float4 *)&xs[i * 8] = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
        *(float4 *)&xs[i * 8 + 4] = make_float4(v[u][4], v[u][5], v[u][6], v[u][7]);
    }
    __syncthreads();
    if (tid < 32 * R) {
        const int r = tid >> 5, l = tid & 31;
        const float *row = xs + (size_t)r * d;
        float s = 0.0f;
        int i = l;
        for (; i + 32 * 15 < d; i += 32 * 16) {  // sixteen reads in flight, added in column order
            float q[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) q[j] = row[i + 32 * j];
#pragma unroll
            for (int j = 0; j < 16; ++j) s = fmaf(q[j], q[j], s);
        }
        for (; i < d; i += 32) s = fmaf(row[i], row[i], s);
        s = warp32_sum(s);
        if (l == 0) {
            rms_s[r] = sqrtf(s / (float)d + 1e-6f);
            if (t0 + r < T) rms[t0 + r] = rms_s[r];
        }
    }
    if (h == nullptr) return;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = tid + 256 * u, rr = min(i, np - 1) / ppr, cc = (min(i, np - 1) - rr * ppr) * 8;
        float g[8], o[8];
        *(float4 *)&g[0] = *(const float4 *)(gamma + cc);
        *(float4 *)&g[4] = *(const float4 *)(gamma + cc + 4);
        const float rv = rms_s[rr];
#pragma unroll
        for (int q = 0; q < 8; ++q) o[q] = norm_apply<XBF>(v[u][q], rv, g[q]);
        if (i < np && t0 + rr < T) store_piece<XBF>(h, (size_t)(t0 + rr) * d + cc, o);
    }
}

// rows per workgroup of the row kernels (forward and backward): two, or one where two rows do not fit their registers
// and LDS; 0: the chunked kernels (d % 8 != 0, unaligned rows, or rows that are too long)
static int norm_rows_per_wg(int d, uintptr_t addresses)
{
    if (d % 8 != 0 || addresses % 16 != 0) return 0;
    return 2 * d <= 8192 ? 2 : d <= 8192 ? 1 : 0;
}

hipError_t launch_rmsnorm(const omega_moe *m, const void *x, int T, void *h, hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const int grid = ceil_div(T, NORM_ROWS);
    const int R = norm_rows_per_wg(c.d, (uintptr_t)x | (uintptr_t)h | (uintptr_t)m->gamma);
    if (R > 0) {
        const int nv = ceil_div(R * c.d, 2048);
#define RMS_ROWS(BF, RV, NVV)                                                                                            \
    hipLaunchKernelGGL((rmsnorm_rows_kernel<BF, RV, NVV>), dim3(ceil_div(T, RV)), dim3(256), RV * c.d * sizeof(float), s, x, m->gamma, T, \
                       c.d, m->rms, h)
#define RMS_ROWS_T(BF)                                                                                                   \
    do {                                                                                                                 \
        if (R == 1) RMS_ROWS(BF, 1, 4);                                                                                  \
        else if (nv <= 1) RMS_ROWS(BF, 2, 1);                                                                            \
        else if (nv <= 2) RMS_ROWS(BF, 2, 2);                                                                            \
        else RMS_ROWS(BF, 2, 4);                                                                                         \
    } while (0)
        if (c.dtype == OMEGA_DTYPE_BF16) RMS_ROWS_T(true);
        else RMS_ROWS_T(false);
#undef RMS_ROWS_T
#undef RMS_ROWS
        return hipGetLastError();
    }
    if (c.dtype == OMEGA_DTYPE_BF16)
        hipLaunchKernelGGL(rmsnorm_kernel<true>, dim3(grid), dim3(256), 0, s, x, m->gamma, T, c.d, m->rms, h);
    else
        hipLaunchKernelGGL(rmsnorm_kernel<false>, dim3(grid), dim3(256), 0, s, x, m->gamma, T, c.d, m->rms, h);
    return hipGetLastError();
}

// ---- backward of the pre-norm (block form) ----
// rmsnorm_backward_kernel2 (J/engine/nn/layer/normalization/gpu/RMSKernel.cu:226-277): per row, with the forward's rms,
//   drms = sum_i x[i]*dh[i]*w[i] (lane l adds i = l, l+32, ... in order: product x*dh, then one fused multiply-add with w;
//          xor butterfly over the 32 lanes) * (-1 / (rms^3 * C))
//   dx[i] = dh[i]*w[i]/rms + drms*x[i]   (+ resid[i]: the gradient that bypasses the norm, Tensor_OP().add(norm2.diff, delta),
//          J/engine/nn/layer/llama/LlamaTransformerBlock.java:157-158), rounded once in bf16 layers
// 8 rows x 32 lanes per workgroup, rows read straight from memory (this kernel moves 4 rows of T x d once).
template <bool XBF>
__global__ __launch_bounds__(256) void rmsnorm_backward_kernel(const void *__restrict__ x, const void *__restrict__ dh,
                                                               const float *__restrict__ gamma, const float *__restrict__ rms,
                                                               const void *__restrict__ resid, int T, int d, void *__restrict__ dx)
{
    const int r = threadIdx.x >> 5, l = threadIdx.x & 31;
    const int t = blockIdx.x * NORM_ROWS + r;
    if (t >= T) return;  // whole 32-lane groups leave together; the shuffles below stay within a group
    const size_t base = (size_t)t * d;
    auto ld = [&](const void *p, int i) {
        return XBF ? bf16_to_f32(((const bf16_t *)p)[base + i]) : ((const float *)p)[base + i];
    };
    float s = 0.0f;
    for (int i = l; i < d; i += 32) {
        const float pr = ld(x, i) * ld(dh, i);
        s = fmaf(pr, gamma[i], s);
    }
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) s = s + __shfl_xor(s, m, 32);
    const float rv = rms[t];
    const float drms = s * (-1.0f / (rv * rv * rv * (float)d));
    for (int i = l; i < d; i += 32) {
        const float a = ld(dh, i) * gamma[i];
        const float q = a / rv;
        float v = fmaf(drms, ld(x, i), q);
        if (resid != nullptr) v = v + ld(resid, i);
        if (XBF) ((bf16_t *)dx)[base + i] = f32_to_bf16(v);
        else ((float *)dx)[base + i] = v;
    }
}

// The same for rows of whole 16-byte pieces: laid out as rmsnorm_rows_kernel.  The pieces of x and dh stay in registers; the
// products x*dh pass through LDS to the 32 lanes that add them.  Bound: the bytes of x, dh, resid and dx (3000 rows of 2048
// bf16 columns: 90 -> 16 us).
template <bool XBF, int R, int NV>
__global__ __launch_bounds__(256) void rmsnorm_backward_rows_kernel(const void *__restrict__ x, const void *__restrict__ dh,
                                                                    const float *__restrict__ gamma, const float *__restrict__ rms,
                                                                    const void *__restrict__ resid, int T, int d, void *__restrict__ dx)
{
    extern __shared__ __attribute__((aligned(16))) float ps[];  // [R][d]
    __shared__ float rms_s[R], drms_s[R];
    const int tid = threadIdx.x, t0 = blockIdx.x * R, ppr = d >> 3, np = R * ppr;
    float xv[NV][8], gv[NV][8];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = min(tid + 256 * u, np - 1), rr = i / ppr;
        const size_t off = (size_t)min(t0 + rr, T - 1) * d + (i - rr * ppr) * 8;
        load_piece<XBF>(x, off, xv[u]);
        load_piece<XBF>(dh, off, gv[u]);
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = min(tid + 256 * u, np - 1);
        float p[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] = xv[u][q] * gv[u][q];
        *(float4 *)&ps[i * 8] = make_float4(p[0], p[1], p[2], p[3]);
        *(float4 *)&ps[i * 8 + 4] = make_float4(p[4], p[5], p[6], p[7]);
    }
    __syncthreads();
    if (tid < 32 * R) {
        const int r = tid >> 5, l = tid & 31;
        const float *row = ps + (size_t)r * d;
        float s = 0.0f;
        int i = l;
        for (; i + 32 * 7 < d; i += 32 * 8) {
            float q[8], w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) { q[j] = row[i + 32 * j]; w[j] = gamma[i + 32 * j]; }
#pragma unroll
            for (int j = 0; j < 8; ++j) s = fmaf(q[j], w[j], s);
        }
        for (; i < d; i += 32) s = fmaf(row[i], gamma[i], s);
        s = warp32_sum(s);
        if (l == 0) {
            const float rv = rms[min(t0 + r, T - 1)];
            rms_s[r] = rv;
            drms_s[r] = s * (-1.0f / (rv * rv * rv * (float)d));
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = tid + 256 * u, rr = min(i, np - 1) / ppr, cc = (min(i, np - 1) - rr * ppr) * 8;
        const size_t off = (size_t)min(t0 + rr, T - 1) * d + cc;
        float w[8], o[8], rs[8];
        *(float4 *)&w[0] = *(const float4 *)(gamma + cc);
        *(float4 *)&w[4] = *(const float4 *)(gamma + cc + 4);
        if (resid != nullptr) load_piece<XBF>(resid, off, rs);
        const float rv = rms_s[rr], drms = drms_s[rr];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float a = gv[u][q] * w[q];
            const float b = a / rv;
            float v = fmaf(drms, xv[u][q], b);
            if (resid != nullptr) v = v + rs[q];
            o[q] = XBF ? bf16_to_f32(f32_to_bf16(v)) : v;
        }
        if (i < np && t0 + rr < T) store_piece<XBF>(dx, off, o);
    }
}

// dgamma[c] = sum_t (x[t,c]/rms[t]) * dh[t,c]: partial sums over slices of the rows (fixed order, no atomics; the
// reference accumulates with atomicAdd in no defined order), then their sum.  A thread owns NC adjacent columns, several rows
// of loads in flight (3000 rows of 2048 columns, both launches: 40 -> 17 us).
template <bool XBF, int NC>
__global__ __launch_bounds__(64) void rmsnorm_dgamma_partial_kernel(const void *__restrict__ x, const void *__restrict__ dh,
                                                                    const float *__restrict__ rms, int T, int d, int tslice,
                                                                    float *__restrict__ part)
{
    const int c = (blockIdx.x * 64 + threadIdx.x) * NC;
    if (c >= d) return;
    const int t0 = blockIdx.y * tslice, t1 = min(T, t0 + tslice);
    float acc[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) acc[q] = 0.0f;
    constexpr int U = NC > 1 ? 4 : 8;
    for (int tb = t0; tb < t1; tb += U) {
        float xv[U][NC], gv[U][NC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t o = (size_t)min(tb + u, t1 - 1) * d + c;
            if constexpr (NC == 8) {
                load_piece<XBF>(x, o, xv[u]);
                load_piece<XBF>(dh, o, gv[u]);
            } else {
                xv[u][0] = XBF ? bf16_to_f32(((const bf16_t *)x)[o]) : ((const float *)x)[o];
                gv[u][0] = XBF ? bf16_to_f32(((const bf16_t *)dh)[o]) : ((const float *)dh)[o];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (tb + u >= t1) break;
            const float rv = rms[tb + u];
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const float n = xv[u][q] / rv;
                const float pr = n * gv[u][q];
                acc[q] = acc[q] + pr;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) part[(size_t)blockIdx.y * d + c + q] = acc[q];
}

// dx = resid + rmsnorm backward of dh; dgamma into m->dgamma (partials in m->bw_gpart)
hipError_t launch_rmsnorm_backward(const omega_moe *m, const void *x, const void *dh, const void *resid, int T, void *dx,
                                   hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const bool bf = c.dtype == OMEGA_DTYPE_BF16;
    const int R = norm_rows_per_wg(c.d, (uintptr_t)x | (uintptr_t)dh | (uintptr_t)resid | (uintptr_t)dx | (uintptr_t)m->gamma);
    if (R > 0) {
        const int nv = ceil_div(R * c.d, 2048);
#define RMSB_ROWS(BF, RV, NVV)                                                                                           \
    hipLaunchKernelGGL((rmsnorm_backward_rows_kernel<BF, RV, NVV>), dim3(ceil_div(T, RV)), dim3(256), RV * c.d * sizeof(float), s, x, dh, \
                       m->gamma, m->rms, resid, T, c.d, dx)
#define RMSB_ROWS_T(BF)                                                                                                  \
    do {                                                                                                                 \
        if (R == 1) RMSB_ROWS(BF, 1, 4);                                                                                 \
        else if (nv <= 1) RMSB_ROWS(BF, 2, 1);                                                                           \
        else if (nv <= 2) RMSB_ROWS(BF, 2, 2);                                                                           \
        else RMSB_ROWS(BF, 2, 4);                                                                                        \
    } while (0)
        if (bf) RMSB_ROWS_T(true);
        else RMSB_ROWS_T(false);
#undef RMSB_ROWS_T
#undef RMSB_ROWS
    } else {
        const int grid = ceil_div(T, NORM_ROWS);
        if (bf) hipLaunchKernelGGL(rmsnorm_backward_kernel<true>, dim3(grid), dim3(256), 0, s, x, dh, m->gamma, m->rms, resid, T, c.d, dx);
        else hipLaunchKernelGGL(rmsnorm_backward_kernel<false>, dim3(grid), dim3(256), 0, s, x, dh, m->gamma, m->rms, resid, T, c.d, dx);
    }
    // slices of the rows: as many as the partial sums have room for, each of 16 rows or more
    const int tslice = std::max(16, ceil_div(T, bw_norm_slices(m))), nsl = ceil_div(T, tslice);
    const bool wide = R > 0;
    const dim3 pg(ceil_div(c.d, wide ? 512 : 64), nsl);
    if (bf && wide) hipLaunchKernelGGL((rmsnorm_dgamma_partial_kernel<true, 8>), pg, dim3(64), 0, s, x, dh, m->rms, T, c.d, tslice, m->bw_gpart);
    else if (bf) hipLaunchKernelGGL((rmsnorm_dgamma_partial_kernel<true, 1>), pg, dim3(64), 0, s, x, dh, m->rms, T, c.d, tslice, m->bw_gpart);
    else if (wide) hipLaunchKernelGGL((rmsnorm_dgamma_partial_kernel<false, 8>), pg, dim3(64), 0, s, x, dh, m->rms, T, c.d, tslice, m->bw_gpart);
    else hipLaunchKernelGGL((rmsnorm_dgamma_partial_kernel<false, 1>), pg, dim3(64), 0, s, x, dh, m->rms, T, c.d, tslice, m->bw_gpart);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_part_sums(m->bw_gpart, nsl, (size_t)c.d, m->dgamma, s);
}
