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

// bf16 expert weights: the step is taken on the fp32 master, the packed bf16 image is re-rounded from it.  A thread takes four
// adjacent columns of a row of expert blockIdx.y, so that every load and store of a wave is one contiguous kilobyte (master,
// gradient and moments share one layout; the image gets 8 bytes of a 16-byte chunk).  Bound: the 30 bytes per weight, which
// pass the last-level cache by.  Two 16-byte halves of a chunk per thread and 64-bit indices -> now: 49 million weights 347
// -> 269 us (5.5 TB/s), 470 million 3633 -> 3246 us (4.3 TB/s).  All of it with the blocks on cache lines: 64 bytes off the
// line the new form took 293 us, 32 bytes off 3850.
typedef __attribute__((ext_vector_type(4))) float adamw_f32x4;
__global__ __launch_bounds__(256) void adamw_packed_kernel(float *__restrict__ master, const float *__restrict__ grad,
                                                           float *__restrict__ mw, float *__restrict__ vw, size_t stride,
                                                           unsigned char *__restrict__ packed, size_t pstride, int R, int K,
                                                           omega_adamw p)
{
    const int g = blockIdx.y, KT = K >> 5;
    const uint32_t nq = K >> 2, n = (uint32_t)R * nq;  // (an expert of 2^34 weights and its moments would not fit the memory)
    adamw_f32x4 *w4 = (adamw_f32x4 *)(master + (size_t)g * stride), *m4 = (adamw_f32x4 *)(mw + (size_t)g * stride), *v4 = (adamw_f32x4 *)(vw + (size_t)g * stride);
    const adamw_f32x4 *g4 = (const adamw_f32x4 *)(grad + (size_t)g * stride);
    unsigned char *pg = packed + (size_t)g * pstride;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const uint32_t r = i / nq, c4 = i % nq;
        adamw_f32x4 wv = __builtin_nontemporal_load(w4 + i), mv = __builtin_nontemporal_load(m4 + i), vv = __builtin_nontemporal_load(v4 + i);
        const adamw_f32x4 gv = __builtin_nontemporal_load(g4 + i);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float mq = mv[q], vq = vv[q];
            wv[q] = adamw_elem(wv[q], gv[q], mq, vq, p);
            mv[q] = mq;
            vv[q] = vq;
        }
        __builtin_nontemporal_store(wv, w4 + i);
        __builtin_nontemporal_store(mv, m4 + i);
        __builtin_nontemporal_store(vv, v4 + i);
        uint2 u;
        u.x = (uint32_t)f32_to_bf16(wv[0]) | ((uint32_t)f32_to_bf16(wv[1]) << 16);
        u.y = (uint32_t)f32_to_bf16(wv[2]) | ((uint32_t)f32_to_bf16(wv[3]) << 16);
        *(uint2 *)(pg + pk_chunk_off(r, c4 >> 3, (c4 >> 1) & 3, KT) + (c4 & 1) * 8) = u;
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
        const dim3 grid(512, m->G);
        hipLaunchKernelGGL(adamw_packed_kernel, grid, dim3(256), 0, s, master + o13, (const float *)m->dW13, mw + o13, vw + o13,
                           2 * HD, (unsigned char *)m->W1, HD * 2, c.H, c.d, p);
        hipLaunchKernelGGL(adamw_packed_kernel, grid, dim3(256), 0, s, master + o13 + HD, (const float *)m->dW13 + HD,
                           mw + o13 + HD, vw + o13 + HD, 2 * HD, (unsigned char *)m->W3, HD * 2, c.H, c.d, p);
        hipLaunchKernelGGL(adamw_packed_kernel, grid, dim3(256), 0, s, master + o2, (const float *)m->dW2, mw + o2, vw + o2, HD,
                           (unsigned char *)m->W2, HD * 2, c.d, c.H, p);
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
