// Stand-ins for the HIP runtime calls and the kernel launchers that api.hip makes, so that its host logic - workspaces, which
// stage may follow which, what is kept for whom - runs on a machine without a GPU.  Memory is host memory, launches are
// lines of a log, and the allocation that a test names runs out of memory.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include "common.h"

static std::map<void *, size_t> g_live;
static std::map<void *, int> g_device;  // blocks of another device than 0
static size_t g_bytes;
static int g_fail_in;  // > 0: the allocation with this number from now on fails
static hipError_t g_last = hipSuccess;
static std::string g_fail_launch;  // the next launch of this name fails
static float g_clock;  // advanced by every launch: what the events read
static std::string g_log;

static hipError_t line(const char *fmt, ...)
{
    char buf[160];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (g_fail_launch == buf) {
        g_fail_launch.clear();
        return hipErrorLaunchFailure;
    }
    g_log += buf;
    g_log += '\n';
    g_clock += 1.0f;
    return hipGetLastError();  // as behind a real launch: an error that nobody fetched shows up here
}

extern "C" {

void host_fail_allocation(int n) { g_fail_in = n; }
void host_fail_launch(const char *name) { g_fail_launch = name; }
int host_wgrad_tile(int n, int mats, int x, int j)  // of all matrices, one after the other
{
    int mat = 0;
    const int t = wgrad_tile(wgrad_deal_of(n, mats), x, j, &mat);
    return t < 0 ? -1 : mat * n + t;
}
void host_move_to_device(void *p, int device) { g_device[p] = device; }
size_t host_live_bytes(void) { return g_bytes; }
int host_live_count(void) { return (int)g_live.size(); }
const char *host_take_log(void)
{
    static std::string taken;
    taken.swap(g_log);
    g_log.clear();
    return taken.c_str();
}

hipError_t hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (g_fail_in > 0 && --g_fail_in == 0) return g_last = hipErrorOutOfMemory;
    *p = aligned_alloc(256, (n + 256) / 256 * 256);  // (as the device's allocations are aligned)
    memset(*p, 0, n);
    g_live[*p] = n;
    g_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    auto it = g_live.find(p);
    if (it == g_live.end()) abort();  // freed twice, or never allocated
    g_bytes -= it->second;
    g_live.erase(it);
    g_device.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { memset(p, v, n); return hipSuccess; }
// the allocation that p points into
static std::map<void *, size_t>::iterator live_at(const void *p)
{
    auto it = g_live.upper_bound((void *)p);
    if (it == g_live.begin() || (char *)p >= (char *)(--it)->first + it->second) return g_live.end();
    return it;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t)
{
    auto it = live_at(d);
    if (it != g_live.end() && (char *)d + n > (char *)it->first + it->second) return g_last = hipErrorInvalidValue;
    g_log += kind == hipMemcpyDeviceToDevice ? "copy\n" : "";
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    auto it = live_at(p);
    if (it == g_live.end()) return g_last = hipErrorInvalidValue;
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeDevice;
    a->device = g_device.count(it->first) ? g_device[it->first] : 0;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t p)
{
    auto it = live_at(p);
    if (it == g_live.end()) return g_last = hipErrorInvalidValue;
    *base = it->first;
    *size = it->second;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { hipError_t e = g_last; g_last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)calloc(1, sizeof(float)); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { *(float *)e = g_clock; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { *ms = *(float *)b - *(float *)a; return hipSuccess; }

}  // extern "C"

hipError_t router_init(void) { return hipSuccess; }
hipError_t experts_bf16_init(void) { return hipSuccess; }
int router_tok_tile(const omega_moe *m, int) { return m->cfg.E <= 16 ? 16 : 32; }
int experts_bf16_tile_m(const omega_moe *, int) { return 256; }
int experts_f32_tile_m_max(const omega_moe *, int T) { return T >= 1024 ? F32_TILE_M : F32_TILE_M_SMALL; }
int experts_f32_tile_m(const omega_moe *, int T) { return T >= 1024 ? F32_TILE_M : F32_TILE_M_SMALL; }  // (a rule of the same kind)

hipError_t launch_fill_normal(void *, uint64_t, uint64_t, uint64_t, double, uint64_t, int, hipStream_t) { return line("fill"); }
hipError_t launch_convert(void *, int, const void *, int, uint64_t, hipStream_t) { return line("convert"); }
hipError_t launch_rmsnorm(const omega_moe *, const void *, int, void *, hipStream_t) { return line("rmsnorm"); }
hipError_t launch_rmsnorm_backward(const omega_moe *, const void *, const void *, const void *, int, void *, hipStream_t) { return line("rmsnorm_backward"); }
hipError_t launch_router(const omega_moe *, const void *, int, float *, float *probs, hipStream_t) { return line("router probs=%d", probs != nullptr); }
hipError_t launch_dispatch_index(const omega_moe *, int, int, hipStream_t, const void *) { return line("index"); }
hipError_t launch_dispatch_gather(const omega_moe *, const void *, int, hipStream_t) { return line("gather"); }
hipError_t launch_product_f32(const omega_moe *m, int op, const float *, const float *, int, hipStream_t, bool gather, bool keep)
{
    if (keep && (!m->bw_h1 || !m->bw_h3)) return line("product_f32 without room for h1 and h3");
    return line("product_f32 op=%d gather=%d keep=%d", op, gather, keep);
}
hipError_t launch_experts_bf16(const omega_moe *m, const void *, int, int which, hipStream_t, bool keep)
{
    if (keep && (!m->bw_h1 || !m->bw_h3)) return line("experts_bf16 without room for h1 and h3");
    return line("experts_bf16 which=%d keep=%d", which, keep);
}
hipError_t launch_down_slab_reduce(const omega_moe *, float *, hipStream_t) { return line("slab_reduce"); }
hipError_t launch_combine(const omega_moe *, int, void *, const void *, hipStream_t) { return line("combine"); }
hipError_t launch_backward_f32(omega_moe *m, const void *, const void *, int, void *, hipStream_t)
{
    const bool kept = m->rec_valid;
    m->rec_valid = false;  // (as the real one: the d(a) product overwrites what was kept)
    return line("backward_f32 kept=%d", kept);
}
hipError_t launch_backward_bf16(const omega_moe *m, const void *, const void *, int, void *, hipStream_t)
{
    if (!m->bw_zero_state || !m->W2T || !m->W13T) return line("backward_bf16 without its buffers");
    return line("backward_bf16 kept=%d", m->rec_valid);
}
hipError_t launch_transpose_images(const void *, int, int, void *dst, int, int, int, size_t, size_t, hipStream_t)
{
    return line(dst ? "transpose" : "transpose into nothing");
}
hipError_t launch_update_bf16(const omega_moe *, float *, float, int, hipStream_t) { return line("update"); }
hipError_t launch_update_adamw(const omega_moe *m, float *master, float *mw, float *vw, const omega_adamw &, hipStream_t)
{
    const size_t o13 = m->dW13 - m->grads;
    uintptr_t at = (uintptr_t)m->dW13 | (uintptr_t)(mw + o13) | (uintptr_t)(vw + o13);
    if (master) at |= (uintptr_t)(master + o13);
    uintptr_t block = (uintptr_t)m->grads | (uintptr_t)mw | (uintptr_t)vw | (uintptr_t)master;
    return line("adamw block %d experts %d", (int)(block % 16), (int)(at % 128));
}
hipError_t launch_zero_f32(float *, size_t, hipStream_t) { return line("zero"); }
hipError_t launch_axpy_f32(float *, const float *, float, size_t, hipStream_t) { return line("axpy"); }
hipError_t launch_axpy_groups_f32(float *, size_t, const float *, size_t, float, size_t, int, hipStream_t) { return line("axpy"); }
hipError_t launch_sumsq_f32(const float *, size_t, double *, hipStream_t) { return line("sumsq"); }
hipError_t launch_scale_f32(float *, float, size_t, hipStream_t) { return line("scale"); }
hipError_t launch_pack_rows(void *, const void *, int, int, hipStream_t) { return line("pack"); }
hipError_t launch_unpack_rows(void *, const void *, int, int, hipStream_t) { return line("unpack"); }
hipError_t launch_param_read(void *, const void *, int R, int, size_t, hipEvent_t, hipStream_t) { return line(R > 0 ? "param_read of a packed image" : "param_read"); }
