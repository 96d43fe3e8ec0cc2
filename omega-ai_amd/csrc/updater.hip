// AdamW step of the layer's parameters: the Updater branch of FullyLayer.update
// (J/engine/nn/layer/FullyLayer.java:569-590 -> AdamW.update, J/engine/updater/AdamW.java:69-92 ->
// AdamWKernel.updateW / updateB, J/engine/updater/gpu/AdamWKernel.java:177-195,380-399 -> adamw_kernel,
// J/engine/updater/gpu/updater.cu:31-52).  Built without contraction: every operation below rounds once, where it is
// written, so the result is the same bits as the same formula on any IEEE machine.
#include "common.h"
#include "pack.h"

// lerp(start, end, weight) = fma(weight, end, fma(-weight, start, start)) (updater.cu:31-33); the decay term and the
// final step are written as the fused operations the source's expression shape offers to the CUDA compiler
__device__ __forceinline__ float adamw_elem(float w, float g, float &m, float &v, const omega_adamw &p)
{
    m = fmaf(p.beta1, m, fmaf(-p.beta1, g, g));
    const float g2 = g * g;
    v = fmaf(p.beta2, v, fmaf(-p.beta2, g2, g2));
    const float mh = m / p.b1c, vh = v / p.b2c;
    const float t = fmaf(p.wd, w, mh / (sqrtf(vh) + p.eps));
    return fmaf(-p.lr, t, w);
}

// fp32 tensors: group blockIdx.y of `n` elements at w + y*wstride, its gradient and moments at + y*gstride
__global__ __launch_bounds__(256) void adamw_f32_kernel(float *__restrict__ w, size_t wstride, const float *__restrict__ grad,
                                                        float *__restrict__ mw, float *__restrict__ vw, size_t gstride, size_t n,
                                                        omega_adamw p)
{
    w += blockIdx.y * wstride;
    grad += blockIdx.y * gstride;
    mw += blockIdx.y * gstride;
    vw += blockIdx.y * gstride;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float m = mw[i], v = vw[i];
        w[i] = adamw_elem(w[i], grad[i], m, v, p);
        mw[i] = m;
        vw[i] = v;
    }
}

// bf16 expert weights: the step is taken on the fp32 master, the packed bf16 image is re-rounded from it, and with it the
// transposed image that the next backward pass reads (T = true: it is there).  A workgroup takes 32 rows x 128 columns of expert
// blockIdx.y: rows of 512 bytes of the four fp32 arrays, sixteen 16-byte loads in flight per thread; the bf16 tile goes through
// LDS and out as whole 1 KiB blocks of either image (of the transposed one the 8 blocks of one k step of a row group: 8 KiB in
// a row).  Bound: the 30 bytes per weight (32 with the transposed image, whose pass over the weights is saved: 4 bytes), which pass
// the last-level cache by.  A thread per four columns, then this form (with the transposed image and the
// blocks of 64 x 64 that made it in launches of their own): 3 x 49 million weights 3 x 269 + 3 x 37 -> 3 x 283 us, 1.41 billion 9.2 + 1.0 ->
// 8.3 ms (5.4 TB/s).  The blocks have to start on cache lines: 32 bytes off the earlier form took 11.6 ms instead of 9.8.
typedef __attribute__((ext_vector_type(4))) float adamw_f32x4;
template <bool T>
__global__ __launch_bounds__(256) void adamw_packed_kernel(float *__restrict__ master, const float *__restrict__ grad,
                                                           float *__restrict__ mw, float *__restrict__ vw, size_t stride,
                                                           unsigned char *__restrict__ packed, size_t pstride, int K,
                                                           unsigned char *__restrict__ tr, size_t tstride, int KTt, int kt0, omega_adamw p)
{
    constexpr int LDB = 136;  // LDS row of 128 columns: rows stay on 16 bytes and start 4 banks apart
    __shared__ __attribute__((aligned(16))) bf16_t tile[32][LDB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, KT = K >> 5, nct = K >> 7;
    const int rt = blockIdx.x / nct, r0 = 32 * rt, c0 = 128 * (blockIdx.x - rt * nct);
    const size_t at = (size_t)blockIdx.y * stride + (size_t)(r0 + (tid >> 5)) * K + c0 + 4 * (tid & 31);
    adamw_f32x4 wv[4], mv[4], vv[4], gv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const size_t o = at + (size_t)(8 * i) * K;
        wv[i] = __builtin_nontemporal_load((const adamw_f32x4 *)(master + o));
        mv[i] = __builtin_nontemporal_load((const adamw_f32x4 *)(mw + o));
        vv[i] = __builtin_nontemporal_load((const adamw_f32x4 *)(vw + o));
        gv[i] = __builtin_nontemporal_load((const adamw_f32x4 *)(grad + o));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const size_t o = at + (size_t)(8 * i) * K;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float mq = mv[i][q], vq = vv[i][q];
            wv[i][q] = adamw_elem(wv[i][q], gv[i][q], mq, vq, p);
            mv[i][q] = mq;
            vv[i][q] = vq;
        }
        __builtin_nontemporal_store(wv[i], (adamw_f32x4 *)(master + o));
        __builtin_nontemporal_store(mv[i], (adamw_f32x4 *)(mw + o));
        __builtin_nontemporal_store(vv[i], (adamw_f32x4 *)(vw + o));
        const uint2 u = {(uint32_t)f32_to_bf16(wv[i][0]) | ((uint32_t)f32_to_bf16(wv[i][1]) << 16),
                         (uint32_t)f32_to_bf16(wv[i][2]) | ((uint32_t)f32_to_bf16(wv[i][3]) << 16)};
        *(uint2 *)&tile[8 * i + (tid >> 5)][4 * (tid & 31)] = u;
    }
    __syncthreads();
    // lane: row lane / 4 of a block, chunk lane % 4 as stored
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int blk = 2 * wave + i, rb = blk >> 2, kb = blk & 3;  // block of 16 rows, k step
        const int row = r0 + 16 * rb + (lane >> 2), c = (lane & 3) ^ pk_swz(row);
        *(uint4 *)(packed + (size_t)blockIdx.y * pstride + pk_chunk_off(row, (c0 >> 5) + kb, c, KT)) = *(const uint4 *)&tile[16 * rb + (lane >> 2)][32 * kb + 8 * c];
    }
    if (T) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int col = 16 * (2 * wave + i) + (lane >> 2), c = (lane & 3) ^ pk_swz(c0 + col);  // 8 rows of a column
            uint32_t u[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) u[q] = (uint32_t)tile[8 * c + 2 * q][col] | (uint32_t)tile[8 * c + 2 * q + 1][col] << 16;
            *(uint4 *)(tr + (size_t)blockIdx.y * tstride + pk_chunk_off(c0 + col, kt0 + rt, c, KTt)) = make_uint4(u[0], u[1], u[2], u[3]);
        }
    }
}

// the bf16 gate weight: row-major
__global__ __launch_bounds__(256) void adamw_rows_bf16_kernel(float *__restrict__ master, const float *__restrict__ grad,
                                                              float *__restrict__ mw, float *__restrict__ vw,
                                                              bf16_t *__restrict__ w, size_t n, omega_adamw p)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float m = mw[i], v = vw[i];
        const float nw = adamw_elem(master[i], grad[i], m, v, p);
        master[i] = nw;
        mw[i] = m;
        vw[i] = v;
        w[i] = f32_to_bf16(nw);
    }
}

static inline unsigned grid_for(size_t n, unsigned cap)
{
    const size_t b = (n + 255) / 256;
    return (unsigned)(b < cap ? (b ? b : 1) : cap);
}

// mw, vw (and master for bf16 layers) are laid out like the gradient block
hipError_t launch_update_adamw(const omega_moe *m, float *master, float *mw, float *vw, const omega_adamw &p, hipStream_t s)
{
    const omega_moe_config &c = m->cfg;
    const size_t HD = (size_t)c.H * c.d, nWg = (size_t)c.E * c.d;
    const size_t o_g = m->dWg - m->grads, o_bg = m->dbg - m->grads, o_gm = m->dgamma - m->grads, o13 = m->dW13 - m->grads, o2 = m->dW2 - m->grads;
    const bool bf = c.dtype == OMEGA_DTYPE_BF16;
    if (bf)
        hipLaunchKernelGGL(adamw_rows_bf16_kernel, dim3(grid_for(nWg, 1024)), dim3(256), 0, s, master + o_g, (const float *)m->dWg,
                           mw + o_g, vw + o_g, (bf16_t *)m->Wg, nWg, p);
    else
        hipLaunchKernelGGL(adamw_f32_kernel, dim3(grid_for(nWg, 1024)), dim3(256), 0, s, (float *)m->Wg, (size_t)0,
                           (const float *)m->dWg, mw + o_g, vw + o_g, (size_t)0, nWg, p);
    if (c.has_gate_bias)
        hipLaunchKernelGGL(adamw_f32_kernel, dim3(grid_for(c.E, 1024)), dim3(256), 0, s, m->bg, (size_t)0, (const float *)m->dbg,
                           mw + o_bg, vw + o_bg, (size_t)0, (size_t)c.E, p);
    if (m->gamma_set)
        hipLaunchKernelGGL(adamw_f32_kernel, dim3(grid_for(c.d, 1024)), dim3(256), 0, s, m->gamma, (size_t)0,
                           (const float *)m->dgamma, mw + o_gm, vw + o_gm, (size_t)0, (size_t)c.d, p);
    if (bf) {
        // (widths are multiples of 256 and 128; the images of m->W2T: [H,d] per expert, of m->W13T: [d, H | H])
        auto step = [&](size_t o, size_t stride, void *w, int R, int K, void *tr, size_t tstride, int KTt, int kt0) {
            const dim3 grid((unsigned)(R / 32) * (K / 128), m->G);
            if (m->W2T && m->W13T)
                hipLaunchKernelGGL(adamw_packed_kernel<true>, grid, dim3(256), 0, s, master + o, (const float *)m->grads + o, mw + o, vw + o, stride,
                                   (unsigned char *)w, HD * 2, K, (unsigned char *)tr, tstride, KTt, kt0, p);
            else
                hipLaunchKernelGGL(adamw_packed_kernel<false>, grid, dim3(256), 0, s, master + o, (const float *)m->grads + o, mw + o, vw + o, stride,
                                   (unsigned char *)w, HD * 2, K, (unsigned char *)nullptr, (size_t)0, 0, 0, p);
        };
        step(o13, 2 * HD, m->W1, c.H, c.d, m->W13T, 4 * HD, 2 * c.H / 32, 0);
        step(o13 + HD, 2 * HD, m->W3, c.H, c.d, m->W13T, 4 * HD, 2 * c.H / 32, c.H / 32);
        step(o2, HD, m->W2, c.d, c.H, m->W2T, 2 * HD, c.d / 32, 0);
    } else {
        const dim3 grid(grid_for(HD, 512), m->G);
        hipLaunchKernelGGL(adamw_f32_kernel, grid, dim3(256), 0, s, (float *)m->W1, HD, (const float *)m->dW13, mw + o13,
                           vw + o13, 2 * HD, HD, p);
        hipLaunchKernelGGL(adamw_f32_kernel, grid, dim3(256), 0, s, (float *)m->W3, HD, (const float *)m->dW13 + HD,
                           mw + o13 + HD, vw + o13 + HD, 2 * HD, HD, p);
        hipLaunchKernelGGL(adamw_f32_kernel, grid, dim3(256), 0, s, (float *)m->W2, HD, (const float *)m->dW2, mw + o2, vw + o2,
                           HD, HD, p);
    }
    return hipGetLastError();
}
