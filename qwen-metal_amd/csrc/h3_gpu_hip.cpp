/* h3_gpu over HIP: device, one stream, hipModule-loaded gfx950 kernels,
 * hipMalloc'd tensors, and the host-side launch/validation of every DiT
 * dispatch. The reference's Metal runtime is h3_gpu.m; the conventions
 * (int return, error string, begin/submit chain, stats) follow
 * h3_gpu.h:7-112 of the reference. Every launch checks operand sizes on the
 * host first, so a bad call fails with an error string instead of faulting
 * the device. */
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

#include <string>

#include "../../include/h3_gpu.h"
#include "../../include/qwen_gpu_ext.h"
#include <algorithm>

#include "qw_kernel_args.h"
#include "qw_static_scratch.h"

enum {
    K_LN_MOD, K_RMS_ONE, K_QK_NORM_ROPE, K_GATE, K_ACT, K_SWIGLU, K_CAST,
    K_REORDER, K_FILL, K_QUANT, K_DEQUANT, K_COPY2D, K_ATTN,
    /* GEMM kernels in QW_EPI_* order (store, gelu, gate, qknorm, swiglu) */
    K_GEMM_BF16_STORE_Q, K_GEMM_BF16_GELU_Q, K_GEMM_BF16_GATE_Q, K_GEMM_BF16_QKN_Q, K_GEMM_BF16_SWIGLU_Q,
    K_WIDEN, K_LN_MOD_WIDE, K_EULER, K_LORA,
    K_GEMV_BF16_STORE, K_GEMV_BF16_GELU, K_GEMV_I8_STORE, K_GEMV_I8_GELU, K_ZERO,
    K_GEMM_W8_STORE_Q, K_GEMM_W8_GELU_Q, K_GEMM_W8_GATE_Q, K_GEMM_W8_QKN_Q, K_GEMM_W8_SWIGLU_Q,
    K_GEMM_BF16_STORE_MIX, K_GEMM_BF16_GELU_MIX, K_GEMM_BF16_GATE_MIX, K_GEMM_BF16_QKN_MIX, K_GEMM_BF16_SWIGLU_MIX,
    /* narrow tiles of 64, 128, 192 and 256 rows, each in the same order */
    K_GEMM_N1, K_GEMM_N1_LAST = K_GEMM_N1 + 4, K_GEMM_N2, K_GEMM_N2_LAST = K_GEMM_N2 + 4,
    K_GEMM_N3, K_GEMM_N3_LAST = K_GEMM_N3 + 4, K_GEMM_N4, K_GEMM_N4_LAST = K_GEMM_N4 + 4,
    K_ATTN_W4, K_ATTN_SPLIT, K_ATTN_W4_SPLIT, K_COND_L1, K_COND_L2, K_COND_MOD,
    /* with K_LN_MOD: width up to 4096 and 3072, without shift and with */
    K_LN_MOD_SHIFT, K_LN_MOD_3072, K_LN_MOD_3072_SHIFT,
    K_COUNT
};
static const char *k_names[K_COUNT] = {
    "qw_layer_norm_mod_bf16", "qw_rms_norm_one_bf16", "qw_qk_norm_rope_bf16",
    "qw_gate_bf16", "qw_act_bf16", "qw_swiglu_bf16", "qw_cast_f32_bf16",
    "qw_modulation_reorder_bf16", "qw_fill_normal_bf16", "qw_quantize_int8_rows",
    "qw_dequant_int8_f32", "qw_copy2d", "qw_attention_bf16",
    "qw_gemm_bf16_store_q", "qw_gemm_bf16_gelu_q", "qw_gemm_bf16_gate_q", "qw_gemm_bf16_qkn_q", "qw_gemm_bf16_swiglu_q",
    "qw_widen_i8_bf16",
    "qw_layer_norm_mod_wide_bf16", "qw_cfg_euler_f32", "qw_lora_fuse_bf16",
    "qw_gemv_bf16_store", "qw_gemv_bf16_gelu", "qw_gemv_i8_store", "qw_gemv_i8_gelu",
    "qw_zero_u32",
    "qw_gemm_w8_store_q", "qw_gemm_w8_gelu_q", "qw_gemm_w8_gate_q", "qw_gemm_w8_qkn_q", "qw_gemm_w8_swiglu_q",
    "qw_gemm_bf16_store_mix", "qw_gemm_bf16_gelu_mix", "qw_gemm_bf16_gate_mix",
    "qw_gemm_bf16_qkn_mix", "qw_gemm_bf16_swiglu_mix",
    "qw_gemm_bf16_store_n1", "qw_gemm_bf16_gelu_n1", "qw_gemm_bf16_gate_n1", "qw_gemm_bf16_qkn_n1", "qw_gemm_bf16_swiglu_n1",
    "qw_gemm_bf16_store_n2", "qw_gemm_bf16_gelu_n2", "qw_gemm_bf16_gate_n2", "qw_gemm_bf16_qkn_n2", "qw_gemm_bf16_swiglu_n2",
    "qw_gemm_bf16_store_n3", "qw_gemm_bf16_gelu_n3", "qw_gemm_bf16_gate_n3", "qw_gemm_bf16_qkn_n3", "qw_gemm_bf16_swiglu_n3",
    "qw_gemm_bf16_store_n4", "qw_gemm_bf16_gelu_n4", "qw_gemm_bf16_gate_n4", "qw_gemm_bf16_qkn_n4", "qw_gemm_bf16_swiglu_n4",
    "qw_attention_w4_bf16", "qw_attention_split_bf16", "qw_attention_w4_split_bf16",
    "qw_cond_l1", "qw_cond_l2", "qw_cond_mod", "qw_layer_norm_mod_shift_bf16",
    "qw_layer_norm_mod_3072_bf16", "qw_layer_norm_mod_3072_shift_bf16"};

/* How int8 linears of more than 8 rows run (QW_INT8_ROUTE, a measurement
 * switch): AUTO (the default) widens the weight to a bf16 copy by a pass and
 * runs the bf16 kernels, or runs the int8 kernels that widen each W tile once
 * per workgroup in LDS, whichever w8_faster expects to be faster; WIDEN and
 * W8 force one route wherever it can run. */
enum { QW_INT8_AUTO = 0, QW_INT8_WIDEN = 1, QW_INT8_W8 = 2 };

#define QW_SPAN_MAX 4096

struct h3_gpu {
    int device;
    hipStream_t stream;
    hipModule_t module;
    hipFunction_t fn[K_COUNT];
    char error[1024];
    h3_gpu_stats stats;
    hipEvent_t timer0, timer1;
    hipEvent_t chain0, chain1;
    int chain_open;
    std::string label;
    void *scratch;
    size_t scratch_bytes;
    uint32_t attn_threads;  /* attention workgroup size, 64 per 32-query wave */
    uint32_t attn4_threads; /* the same for the small launches' kernel */
    int attn_small; /* launches of fewer 256-query blocks than CUs on the 4-wave kernel (QW_ATTN_W4=0: off) */
    int int8_route; /* QW_INT8_* : how int8 linears of many rows run */
    int mixed;      /* 192- and 224-row tiles allowed (QW_GEMM_T224=0 turns them off, for measurement) */
    uint32_t split_min_steps, split_force; /* measurement: QW_SPLIT_MIN_STEPS, QW_SPLIT_FORCE */
    int workspaces; /* split partials and widened copies allowed (QW_WORKSPACES=0: as if none could be had) */
    int narrow;     /* narrow tiles allowed (QW_GEMM_HALF_SMALL=0: off) */
    /* qw_gpu_last_route: the launches of the last linear or attention call */
    struct { int kid; uint32_t split, half, from, h1, rows1, h2, rows2; } route[4];
    int route_n;
    /* qw_gpu_span_*: event pairs recorded on the stream, read after a sync */
    hipEvent_t *span_ev;
    int *span_tag;
    int span_n, span_open;
    void *widen; /* bf16 copy of the int8 weight of the linear in flight */
    size_t widen_bytes;
    uint32_t cus;      /* compute units */
    float *sk_part;    /* split-tile partials: 256 x 256 fp32 each */
    uint32_t *sk_flag; /* split piece counters (QW_FLAGS a CU), 0 between launches */
    /* this device's copy of the static workspace (qw_static_scratch.hip):
     * partials, then QW_STATIC_FLAGS counters */
    unsigned char *static_scratch;
};

struct h3_gpu_tensor {
    h3_gpu *gpu;
    unsigned char *ptr;
    size_t elements;
    h3_gpu_dtype dtype;
    int owns;
};

static size_t dtype_size(h3_gpu_dtype d) {
    return d == H3_GPU_BF16 ? 2 : d == H3_GPU_I8 ? 1 : 4;
}

static int fail(h3_gpu *g, const char *fmt, ...) {
    if (g) {
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(g->error, sizeof(g->error), fmt, ap);
        va_end(ap);
    }
    return 0;
}

static void set_err(char *error, size_t n, const char *fmt, ...) {
    if (!error || !n) return;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error, n, fmt, ap);
    va_end(ap);
}

static double now_s() {
    timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return ts.tv_sec + ts.tv_nsec * 1e-9;
}

/* ---------------------------------------------------------------------- */
/* context                                                                */

extern "C" h3_gpu *h3_gpu_create(const char *code_object_path, char *error,
                                 size_t error_size) {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) {
        set_err(error, error_size, "no HIP device available");
        return NULL;
    }
    const char *dev_env = getenv("QW_HIP_DEVICE");
    int device = dev_env && *dev_env ? atoi(dev_env) : 0;
    if (device < 0 || device >= count) {
        set_err(error, error_size, "QW_HIP_DEVICE=%d out of range (%d devices)", device, count);
        return NULL;
    }
    if (hipSetDevice(device) != hipSuccess) {
        set_err(error, error_size, "hipSetDevice(%d) failed", device);
        return NULL;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
        set_err(error, error_size, "hipGetDeviceProperties failed");
        return NULL;
    }
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        set_err(error, error_size, "device %d is %s; this code object is gfx950 only",
                device, prop.gcnArchName);
        return NULL;
    }
    std::string path;
    if (code_object_path && *code_object_path) {
        path = code_object_path;
    } else {
        Dl_info info;
        if (!dladdr((void *)&h3_gpu_create, &info) || !info.dli_fname) {
            set_err(error, error_size, "cannot locate libqwen_dit_hip.so");
            return NULL;
        }
        path = info.dli_fname;
        size_t slash = path.rfind('/');
        path = (slash == std::string::npos ? std::string(".") : path.substr(0, slash)) +
               "/qwen_kernels.hsaco";
    }
    h3_gpu *g = new h3_gpu();
    memset(g->error, 0, sizeof(g->error));
    memset(&g->stats, 0, sizeof(g->stats));
    g->device = device;
    g->chain_open = 0;
    g->scratch = NULL;
    g->scratch_bytes = 0;
    g->widen = NULL;
    g->widen_bytes = 0;
    g->route_n = 0;
    g->span_ev = NULL;
    g->span_tag = NULL;
    g->span_n = 0;
    g->span_open = 0;
    g->int8_route = QW_INT8_AUTO;
    if (const char *r = getenv("QW_INT8_ROUTE")) {
        if (!strcmp(r, "w8")) g->int8_route = QW_INT8_W8;
        else if (!strcmp(r, "widen")) g->int8_route = QW_INT8_WIDEN;
    }
    g->mixed = 1;
    if (const char *r = getenv("QW_GEMM_T224")) g->mixed = atoi(r) != 0;
    g->split_min_steps = 32;
    if (const char *r = getenv("QW_SPLIT_MIN_STEPS")) g->split_min_steps = (uint32_t)atoi(r);
    g->split_force = 0;
    if (const char *r = getenv("QW_SPLIT_FORCE")) g->split_force = (uint32_t)atoi(r);
    g->workspaces = 1;
    if (const char *r = getenv("QW_WORKSPACES")) g->workspaces = atoi(r) != 0;
    g->narrow = 1;
    if (const char *r = getenv("QW_GEMM_HALF_SMALL")) g->narrow = atoi(r) != 0;
    g->cus = 0;
    g->sk_part = NULL;
    g->sk_flag = NULL;
    g->static_scratch = NULL;
    hipError_t e = hipModuleLoad(&g->module, path.c_str());
    if (e != hipSuccess) {
        set_err(error, error_size, "hipModuleLoad(%s): %s", path.c_str(), hipGetErrorString(e));
        delete g;
        return NULL;
    }
    for (int k = 0; k < K_COUNT; k++) {
        e = hipModuleGetFunction(&g->fn[k], g->module, k_names[k]);
        if (e != hipSuccess) {
            set_err(error, error_size, "kernel %s missing from %s", k_names[k], path.c_str());
            hipModuleUnload(g->module);
            delete g;
            return NULL;
        }
    }
    /* The attention kernels' workgroups (their launch bounds) set the query
     * blocks: one 64-lane wave per 32 queries. */
    for (int w = 0; w < 2; w++) {
        const int kid = w ? K_ATTN_W4 : K_ATTN;
        int attn_threads = 0;
        e = hipFuncGetAttribute(&attn_threads, HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK, g->fn[kid]);
        if (e != hipSuccess || attn_threads < 64 || attn_threads > 1024 || attn_threads % 64) {
            set_err(error, error_size, "%s: bad workgroup bound %d", k_names[kid], attn_threads);
            hipModuleUnload(g->module);
            delete g;
            return NULL;
        }
        (w ? g->attn4_threads : g->attn_threads) = (uint32_t)attn_threads;
    }
    g->attn_small = 1;
    if (const char *r = getenv("QW_ATTN_W4")) g->attn_small = atoi(r) != 0;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device) != hipSuccess ||
        cus <= 0) {
        set_err(error, error_size, "compute unit count unavailable");
        hipModuleUnload(g->module);
        delete g;
        return NULL;
    }
    g->cus = (uint32_t)cus;
    {
        /* once per device, with the device current: the address of its
         * copy of the no-allocation entry points' static workspace */
        void *ss = NULL;
        char se[256] = {0};
        if (qw_static_scratch_address(device, &ss, se, sizeof(se)) != 0) {
            set_err(error, error_size, "%s", se);
            hipModuleUnload(g->module);
            delete g;
            return NULL;
        }
        g->static_scratch = (unsigned char *)ss;
    }
    if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&g->timer0) != hipSuccess || hipEventCreate(&g->timer1) != hipSuccess ||
        hipEventCreate(&g->chain0) != hipSuccess || hipEventCreate(&g->chain1) != hipSuccess) {
        set_err(error, error_size, "stream/event creation failed");
        hipModuleUnload(g->module);
        delete g;
        return NULL;
    }
    return g;
}

extern "C" void h3_gpu_free(h3_gpu *g) {
    if (!g) return;
    hipSetDevice(g->device);
    hipStreamSynchronize(g->stream);
    if (g->scratch) hipFree(g->scratch);
    if (g->widen) hipFree(g->widen);
    if (g->sk_part) hipFree(g->sk_part);
    if (g->sk_flag) hipFree(g->sk_flag);
    if (g->span_ev) {
        for (int i = 0; i < 2 * QW_SPAN_MAX; i++) hipEventDestroy(g->span_ev[i]);
        free(g->span_ev);
        free(g->span_tag);
    }
    hipEventDestroy(g->timer0);
    hipEventDestroy(g->timer1);
    hipEventDestroy(g->chain0);
    hipEventDestroy(g->chain1);
    hipStreamDestroy(g->stream);
    hipModuleUnload(g->module);
    delete g;
}

extern "C" const char *h3_gpu_error(const h3_gpu *g) { return g ? g->error : "no gpu"; }

extern "C" int h3_gpu_get_stats(const h3_gpu *g, h3_gpu_stats *s) {
    if (!g || !s) return 0;
    *s = g->stats;
    return 1;
}

extern "C" void h3_gpu_profile_set_label(h3_gpu *g, const char *label) {
    if (g) g->label = label ? label : "";
}

extern "C" void h3_gpu_profile_mark(h3_gpu *g, const char *phase) {
    if (!g || !getenv("H3_PROFILE")) return;
    hipStreamSynchronize(g->stream);
    fprintf(stderr, "[h3-profile] %s %s: dispatches=%llu submissions=%llu live=%.1f MB\n",
            g->label.c_str(), phase ? phase : "", (unsigned long long)g->stats.direct_dispatches,
            (unsigned long long)g->stats.submissions, g->stats.live_bytes / 1e6);
}

extern "C" int h3_gpu_begin(h3_gpu *g) {
    if (!g) return 0;
    if (!g->chain_open) {
        hipEventRecord(g->chain0, g->stream);
        g->chain_open = 1;
    }
    return 1;
}

extern "C" int h3_gpu_continue(h3_gpu *g) {
    /* HIP streams are already asynchronous and ordered: nothing to commit. */
    return g ? 1 : 0;
}

extern "C" int h3_gpu_submit(h3_gpu *g) {
    if (!g) return 0;
    double t0 = now_s();
    if (g->chain_open) hipEventRecord(g->chain1, g->stream);
    hipError_t e = hipStreamSynchronize(g->stream);
    g->stats.command_wait_seconds += now_s() - t0;
    g->stats.submissions++;
    if (e == hipSuccess) e = hipGetLastError();
    if (g->chain_open) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, g->chain0, g->chain1) == hipSuccess)
            g->stats.gpu_seconds += ms * 1e-3;
        g->chain_open = 0;
    }
    if (e != hipSuccess) return fail(g, "submit: %s", hipGetErrorString(e));
    return 1;
}

extern "C" int h3_gpu_timer_begin(h3_gpu *g) {
    if (!g) return 0;
    return hipEventRecord(g->timer0, g->stream) == hipSuccess ? 1
                                                            : fail(g, "timer_begin failed");
}

extern "C" double h3_gpu_timer_end(h3_gpu *g) {
    if (!g) return -1.0;
    if (hipEventRecord(g->timer1, g->stream) != hipSuccess) return -1.0;
    if (hipEventSynchronize(g->timer1) != hipSuccess) return -1.0;
    float ms = 0;
    if (hipEventElapsedTime(&ms, g->timer0, g->timer1) != hipSuccess) return -1.0;
    return ms;
}

/* Spans: a begin and an end event recorded on the stream around a piece of
 * work, no synchronisation; qw_gpu_span_collect waits for the last one and
 * returns every span's device time. Up to QW_SPAN_MAX spans between
 * collects; events are created on the first span. */
extern "C" int qw_gpu_span_begin(h3_gpu *g, int tag) {
    if (!g) return 0;
    if (g->span_open) return fail(g, "span_begin: a span is already open");
    if (!g->span_ev) {
        g->span_ev = (hipEvent_t *)calloc(2 * QW_SPAN_MAX, sizeof(hipEvent_t));
        g->span_tag = (int *)calloc(QW_SPAN_MAX, sizeof(int));
        if (!g->span_ev || !g->span_tag) return fail(g, "span_begin: out of host memory");
        for (int i = 0; i < 2 * QW_SPAN_MAX; i++)
            if (hipEventCreate(&g->span_ev[i]) != hipSuccess) {
                for (int j = 0; j < i; j++) hipEventDestroy(g->span_ev[j]);
                free(g->span_ev);
                free(g->span_tag);
                g->span_ev = NULL;
                g->span_tag = NULL;
                return fail(g, "span_begin: event creation failed");
            }
    }
    if (g->span_n >= QW_SPAN_MAX) return fail(g, "span_begin: more than %d spans", QW_SPAN_MAX);
    g->span_tag[g->span_n] = tag;
    if (hipEventRecord(g->span_ev[2 * g->span_n], g->stream) != hipSuccess)
        return fail(g, "span_begin: event record failed");
    g->span_open = 1;
    return 1;
}

extern "C" int qw_gpu_span_end(h3_gpu *g) {
    if (!g) return 0;
    if (!g->span_open) return fail(g, "span_end: no open span");
    if (hipEventRecord(g->span_ev[2 * g->span_n + 1], g->stream) != hipSuccess)
        return fail(g, "span_end: event record failed");
    g->span_open = 0;
    g->span_n++;
    return 1;
}

extern "C" int qw_gpu_span_collect(h3_gpu *g, int *tags, double *ms, int max) {
    if (!g) return -1;
    if (g->span_open) {
        fail(g, "span_collect: a span is still open");
        return -1;
    }
    const int n = g->span_n < max ? g->span_n : max;
    if (g->span_n && hipEventSynchronize(g->span_ev[2 * g->span_n - 1]) != hipSuccess) {
        fail(g, "span_collect: event wait failed");
        return -1;
    }
    for (int i = 0; i < n; i++) {
        float t = 0;
        if (hipEventElapsedTime(&t, g->span_ev[2 * i], g->span_ev[2 * i + 1]) != hipSuccess) {
            fail(g, "span_collect: elapsed time unavailable");
            return -1;
        }
        if (tags) tags[i] = g->span_tag[i];
        if (ms) ms[i] = t;
    }
    g->span_n = 0;
    return n;
}

/* ---------------------------------------------------------------------- */
/* tensors                                                                */

static h3_gpu_tensor *tensor_new(h3_gpu *g, size_t elements, h3_gpu_dtype d) {
    if (!g) return NULL;
    size_t bytes = elements * dtype_size(d);
    if (bytes == 0) bytes = 16;
    bytes = (bytes + 255) & ~(size_t)255;
    void *p = NULL;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {
        fail(g, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
        return NULL;
    }
    if (hipMemsetAsync(p, 0, bytes, g->stream) != hipSuccess ||
        hipStreamSynchronize(g->stream) != hipSuccess) {
        hipFree(p);
        fail(g, "tensor zero-fill failed");
        return NULL;
    }
    h3_gpu_tensor *t = new h3_gpu_tensor{g, (unsigned char *)p, elements, d, 1};
    g->stats.allocated_bytes += bytes;
    g->stats.live_bytes += bytes;
    g->stats.tensor_allocations++;
    if (g->stats.live_bytes > g->stats.peak_live_bytes) g->stats.peak_live_bytes = g->stats.live_bytes;
    return t;
}

extern "C" h3_gpu_tensor *h3_gpu_tensor_new_f32(h3_gpu *g, size_t n) { return tensor_new(g, n, H3_GPU_F32); }
extern "C" h3_gpu_tensor *h3_gpu_tensor_new_bf16(h3_gpu *g, size_t n) { return tensor_new(g, n, H3_GPU_BF16); }
extern "C" h3_gpu_tensor *h3_gpu_tensor_new_i8(h3_gpu *g, size_t n) { return tensor_new(g, n, H3_GPU_I8); }
extern "C" h3_gpu_tensor *h3_gpu_tensor_new_u32(h3_gpu *g, size_t n) { return tensor_new(g, n, H3_GPU_U32); }

static int copy_in(h3_gpu_tensor *t, size_t off_bytes, const void *src, size_t bytes) {
    h3_gpu *g = t->gpu;
    if (off_bytes + bytes > t->elements * dtype_size(t->dtype))
        return fail(g, "tensor write out of range (%zu + %zu > %zu bytes)", off_bytes, bytes,
                    t->elements * dtype_size(t->dtype));
    if (!bytes) return 1;
    hipError_t e = hipMemcpyAsync(t->ptr + off_bytes, src, bytes, hipMemcpyHostToDevice, g->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g->stream);
    return e == hipSuccess ? 1 : fail(g, "tensor write: %s", hipGetErrorString(e));
}

static int copy_out(const h3_gpu_tensor *t, size_t off_bytes, void *dst, size_t bytes) {
    h3_gpu *g = t->gpu;
    if (off_bytes + bytes > t->elements * dtype_size(t->dtype))
        return fail(g, "tensor read out of range");
    if (!bytes) return 1;
    hipError_t e = hipMemcpyAsync(dst, t->ptr + off_bytes, bytes, hipMemcpyDeviceToHost, g->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g->stream);
    return e == hipSuccess ? 1 : fail(g, "tensor read: %s", hipGetErrorString(e));
}

static h3_gpu_tensor *tensor_from(h3_gpu *g, const void *v, size_t n, h3_gpu_dtype d) {
    h3_gpu_tensor *t = tensor_new(g, n, d);
    if (t && v && !copy_in(t, 0, v, n * dtype_size(d))) {
        h3_gpu_tensor_free(t);
        return NULL;
    }
    return t;
}

extern "C" h3_gpu_tensor *h3_gpu_tensor_from_f32(h3_gpu *g, const float *v, size_t n) {
    return tensor_from(g, v, n, H3_GPU_F32);
}
extern "C" h3_gpu_tensor *h3_gpu_tensor_from_bf16(h3_gpu *g, const uint16_t *v, size_t n) {
    return tensor_from(g, v, n, H3_GPU_BF16);
}
extern "C" h3_gpu_tensor *h3_gpu_tensor_from_u32(h3_gpu *g, const uint32_t *v, size_t n) {
    return tensor_from(g, v, n, H3_GPU_U32);
}

extern "C" h3_gpu_tensor *h3_gpu_tensor_view(const h3_gpu_tensor *base, size_t offset,
                                             size_t elements) {
    if (!base) return NULL;
    if (offset + elements > base->elements) {
        fail(base->gpu, "view [%zu, +%zu) outside tensor of %zu", offset, elements,
             base->elements);
        return NULL;
    }
    return new h3_gpu_tensor{base->gpu, base->ptr + offset * dtype_size(base->dtype), elements,
                             base->dtype, 0};
}

extern "C" void h3_gpu_tensor_free(h3_gpu_tensor *t) {
    if (!t) return;
    if (t->owns) {
        h3_gpu *g = t->gpu;
        /* the stream may still reference the buffer */
        hipStreamSynchronize(g->stream);
        size_t bytes = (t->elements * dtype_size(t->dtype) + 255) & ~(size_t)255;
        if (!bytes) bytes = 256;
        g->stats.live_bytes -= bytes < g->stats.live_bytes ? bytes : g->stats.live_bytes;
        hipFree(t->ptr);
    }
    delete t;
}

extern "C" size_t h3_gpu_tensor_elements(const h3_gpu_tensor *t) { return t ? t->elements : 0; }
extern "C" h3_gpu_dtype h3_gpu_tensor_dtype(const h3_gpu_tensor *t) { return t ? t->dtype : H3_GPU_F32; }
extern "C" void *h3_gpu_tensor_device_ptr(const h3_gpu_tensor *t) { return t ? t->ptr : NULL; }

#define REQ_DT(t, d, what)                                                           \
    do {                                                                             \
        if (!(t)) return fail(g, "%s: missing tensor", what);                        \
        if ((t)->dtype != (d)) return fail(g, "%s: wrong dtype", what);              \
    } while (0)

extern "C" int h3_gpu_tensor_read_f32(const h3_gpu_tensor *t, float *v, size_t n) {
    if (!t || t->dtype != H3_GPU_F32) return t ? fail(t->gpu, "read_f32: dtype") : 0;
    return copy_out(t, 0, v, n * 4);
}
extern "C" int h3_gpu_tensor_read_f32_range(const h3_gpu_tensor *t, size_t off, float *v, size_t n) {
    if (!t || t->dtype != H3_GPU_F32) return t ? fail(t->gpu, "read_f32: dtype") : 0;
    return copy_out(t, off * 4, v, n * 4);
}
extern "C" int h3_gpu_tensor_read_bf16(const h3_gpu_tensor *t, uint16_t *v, size_t n) {
    if (!t || t->dtype != H3_GPU_BF16) return t ? fail(t->gpu, "read_bf16: dtype") : 0;
    return copy_out(t, 0, v, n * 2);
}
extern "C" int h3_gpu_tensor_write_f32(h3_gpu_tensor *t, const float *v, size_t n) {
    if (!t || t->dtype != H3_GPU_F32) return t ? fail(t->gpu, "write_f32: dtype") : 0;
    return copy_in(t, 0, v, n * 4);
}
extern "C" int h3_gpu_tensor_write_f32_range(h3_gpu_tensor *t, size_t off, const float *v, size_t n) {
    if (!t || t->dtype != H3_GPU_F32) return t ? fail(t->gpu, "write_f32: dtype") : 0;
    return copy_in(t, off * 4, v, n * 4);
}
extern "C" int h3_gpu_tensor_write_bf16(h3_gpu_tensor *t, const uint16_t *v, size_t n) {
    if (!t || t->dtype != H3_GPU_BF16) return t ? fail(t->gpu, "write_bf16: dtype") : 0;
    return copy_in(t, 0, v, n * 2);
}
extern "C" int h3_gpu_tensor_write_bf16_range(h3_gpu_tensor *t, size_t off, const uint16_t *v,
                                              size_t n) {
    if (!t || t->dtype != H3_GPU_BF16) return t ? fail(t->gpu, "write_bf16: dtype") : 0;
    return copy_in(t, off * 2, v, n * 2);
}
extern "C" int h3_gpu_tensor_read_bytes(const h3_gpu_tensor *t, void *b, size_t n) {
    return t ? copy_out(t, 0, b, n) : 0;
}
extern "C" int h3_gpu_tensor_write_bytes(h3_gpu_tensor *t, const void *b, size_t n) {
    return t ? copy_in(t, 0, b, n) : 0;
}

/* ---------------------------------------------------------------------- */
/* launches                                                               */

template <class T>
static int launch(h3_gpu *g, int kid, dim3 grid, dim3 block, const T &args) {
    if (grid.x == 0 || grid.y == 0 || grid.z == 0) return 1; /* empty problem */
    void *params[] = {(void *)&args};
    hipError_t e = hipModuleLaunchKernel(g->fn[kid], grid.x, grid.y, grid.z, block.x, block.y,
                                         block.z, 0, g->stream, params, NULL);
    if (e != hipSuccess) return fail(g, "launch %s: %s", k_names[kid], hipGetErrorString(e));
    g->stats.direct_dispatches++;
    return 1;
}

/* launch(), kept for qw_gpu_last_route: split: pieces a tile or block is cut
 * into, half: half tiles, from: first row */
template <typename T>
static int launch_step(h3_gpu *g, int kid, dim3 grid, dim3 block, const T &args, uint32_t split,
                       uint32_t half = 0, uint32_t from = 0) {
    if (g->route_n < 4) g->route[g->route_n++] = {kid, split, half, from, 0, 0, 0, 0};
    return launch(g, kid, grid, block, args);
}

extern "C" int qw_gpu_last_route(const h3_gpu *g, char *text, size_t size) {
    if (!g || !text || !size) return -1;
    size_t n = 0;
    text[0] = '\0';
    for (int i = 0; i < g->route_n && n < size; i++) {
        const auto &r = g->route[i];
        n += snprintf(text + n, size - n, "%s%s", i ? " " : "", k_names[r.kid]);
        if (r.split > 1 && n < size) n += snprintf(text + n, size - n, ":split=%u", r.split);
        if (r.half && n < size) n += snprintf(text + n, size - n, ":half=%u", r.half);
        if (r.from && n < size) n += snprintf(text + n, size - n, ":from=%u", r.from);
        if (r.h1 && n < size)
            n += snprintf(text + n, size - n, ":%ux%u+%ux%u", r.rows1, 32 * r.h1, r.rows2, 32 * r.h2);
    }
    return g->route_n;
}

static bool fits(const h3_gpu_tensor *t, size_t offset, size_t elements) {
    return t && offset + elements <= t->elements;
}

static bool apart(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return x + a_bytes <= y || y + b_bytes <= x;
}

static uint32_t blocks_for(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }

static int ln_mod(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                  const h3_gpu_tensor *mod, const h3_gpu_tensor *row_map, uint32_t rows,
                  uint32_t width, uint32_t slots, uint32_t scale_slot, int32_t shift_slot,
                  float eps) {
    REQ_DT(out, H3_GPU_BF16, "layer_norm_mod out");
    REQ_DT(in, H3_GPU_BF16, "layer_norm_mod in");
    REQ_DT(mod, H3_GPU_BF16, "layer_norm_mod modulation");
    REQ_DT(row_map, H3_GPU_U32, "layer_norm_mod row_map");
    if (width % 8 || width / 8 > 1024 || width == 0)
        return fail(g, "layer_norm_mod: width %u must be a multiple of 8, <= 8192", width);
    if (scale_slot >= slots || (shift_slot >= 0 && (uint32_t)shift_slot >= slots))
        return fail(g, "layer_norm_mod: slot out of range");
    if (!fits(out, 0, (size_t)rows * width) || !fits(in, 0, (size_t)rows * width) ||
        !fits(row_map, 0, rows))
        return fail(g, "layer_norm_mod: tensor too small");
    /* every row_map entry must address a modulation row: checked on host */
    uint32_t mod_rows = (uint32_t)(mod->elements / ((size_t)slots * width));
    if (mod_rows == 0) return fail(g, "layer_norm_mod: modulation too small");
    qw_ln_mod_args a = {(uint16_t *)out->ptr, (const uint16_t *)in->ptr,
                        (const uint16_t *)mod->ptr, (const uint32_t *)row_map->ptr,
                        rows, width, slots, scale_slot, shift_slot, eps};
    if (width <= 4096)
        return launch(g, shift_slot >= 0 ? (width <= 3072 ? K_LN_MOD_3072_SHIFT : K_LN_MOD_SHIFT)
                                         : (width <= 3072 ? K_LN_MOD_3072 : K_LN_MOD),
                      dim3((rows + 3) / 4), dim3(256), a);
    return launch(g, K_LN_MOD_WIDE, dim3(rows), dim3((width / 8 + 63) / 64 * 64), a);
}

extern "C" int qw_gpu_layer_norm_mod_bf16(h3_gpu *g, h3_gpu_tensor *out,
                                          const h3_gpu_tensor *in,
                                          const h3_gpu_tensor *mod,
                                          const h3_gpu_tensor *row_map, uint32_t rows,
                                          uint32_t width, uint32_t slots, uint32_t scale_slot,
                                          float eps) {
    return ln_mod(g, out, in, mod, row_map, rows, width, slots, scale_slot, -1, eps);
}

extern "C" int qw_gpu_layer_norm_mod_shift_bf16(h3_gpu *g, h3_gpu_tensor *out,
                                                const h3_gpu_tensor *in,
                                                const h3_gpu_tensor *mod,
                                                const h3_gpu_tensor *row_map, uint32_t rows,
                                                uint32_t width, uint32_t slots,
                                                uint32_t scale_slot, int32_t shift_slot,
                                                float eps) {
    return ln_mod(g, out, in, mod, row_map, rows, width, slots, scale_slot, shift_slot, eps);
}

extern "C" int qw_gpu_rms_norm_one_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                        const h3_gpu_tensor *w, uint32_t rows, uint32_t width,
                                        float eps) {
    REQ_DT(out, H3_GPU_BF16, "rms_norm_one out");
    REQ_DT(in, H3_GPU_BF16, "rms_norm_one in");
    REQ_DT(w, H3_GPU_BF16, "rms_norm_one weight");
    if (width % 8 || width / 8 > 1024 || width == 0)
        return fail(g, "rms_norm_one: width %u must be a multiple of 8, <= 8192", width);
    if (!fits(out, 0, (size_t)rows * width) || !fits(in, 0, (size_t)rows * width) ||
        !fits(w, 0, width))
        return fail(g, "rms_norm_one: tensor too small");
    qw_rms_one_args a = {(uint16_t *)out->ptr, (const uint16_t *)in->ptr,
                         (const uint16_t *)w->ptr, rows, width, eps};
    return launch(g, K_RMS_ONE, dim3(rows), dim3((width / 8 + 63) / 64 * 64), a);
}

static int act(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in, uint64_t n, int kind) {
    REQ_DT(out, H3_GPU_BF16, "activation out");
    REQ_DT(in, H3_GPU_BF16, "activation in");
    if (!fits(out, 0, n) || !fits(in, 0, n)) return fail(g, "activation: tensor too small");
    qw_act_args a = {(uint16_t *)out->ptr, (const uint16_t *)in->ptr, n, kind};
    return launch(g, K_ACT, dim3(blocks_for(n, 256)), dim3(256), a);
}

extern "C" int h3_gpu_silu_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                uint32_t n) {
    return act(g, out, in, n, QW_ACT_SILU);
}
extern "C" int h3_gpu_gelu_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                uint32_t n, int approximate) {
    if (!approximate) return fail(g, "gelu: only the tanh approximation is on the DiT path");
    return act(g, out, in, n, QW_ACT_GELU_TANH);
}
extern "C" int qw_gpu_tanh_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                uint32_t n) {
    return act(g, out, in, n, QW_ACT_TANH);
}

extern "C" int qw_gpu_swiglu_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *fc1,
                                  uint32_t rows, uint32_t width) {
    REQ_DT(out, H3_GPU_BF16, "swiglu out");
    REQ_DT(fc1, H3_GPU_BF16, "swiglu fc1");
    if (!fits(out, 0, (size_t)rows * width) || !fits(fc1, 0, (size_t)rows * width * 2))
        return fail(g, "swiglu: tensor too small");
    qw_swiglu_args a = {(uint16_t *)out->ptr, (const uint16_t *)fc1->ptr, rows, width};
    return launch(g, K_SWIGLU, dim3(blocks_for((uint64_t)rows * width, 256)), dim3(256), a);
}

extern "C" int h3_gpu_cast_f32_to_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                       uint32_t n) {
    REQ_DT(out, H3_GPU_BF16, "cast out");
    REQ_DT(in, H3_GPU_F32, "cast in");
    if (!fits(out, 0, n) || !fits(in, 0, n)) return fail(g, "cast: tensor too small");
    qw_cast_args a = {(uint16_t *)out->ptr, (const float *)in->ptr, n};
    return launch(g, K_CAST, dim3(blocks_for(n, 256)), dim3(256), a);
}

extern "C" int qw_gpu_cfg_euler_f32(h3_gpu *g, h3_gpu_tensor *x, const h3_gpu_tensor *pos,
                                    size_t pos_offset, const h3_gpu_tensor *neg,
                                    size_t neg_offset, size_t count, float dt, float cfg) {
    if (!g) return 0;
    REQ_DT(x, H3_GPU_F32, "euler sample");
    REQ_DT(pos, H3_GPU_BF16, "euler prediction");
    if (neg) REQ_DT(neg, H3_GPU_BF16, "euler unconditional prediction");
    if (!fits(x, 0, count) || !fits(pos, pos_offset, count) ||
        (neg && !fits(neg, neg_offset, count)))
        return fail(g, "euler: tensor too small");
    qw_euler_args a = {(float *)x->ptr, (const uint16_t *)pos->ptr + pos_offset,
                       neg ? (const uint16_t *)neg->ptr + neg_offset : NULL, count, dt, cfg};
    return launch(g, K_EULER, dim3(blocks_for(count, 256)), dim3(256), a);
}

extern "C" int qw_gpu_lora_fuse_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *base,
                                     uint32_t rows, uint32_t cols, const qw_lora_term_desc *terms,
                                     uint32_t nterms) {
    if (!g) return 0;
    REQ_DT(out, H3_GPU_BF16, "lora out");
    REQ_DT(base, H3_GPU_BF16, "lora base");
    if (!fits(out, 0, (size_t)rows * cols) || !fits(base, 0, (size_t)rows * cols))
        return fail(g, "lora: tensors smaller than %u x %u", rows, cols);
    if (nterms > QW_LORA_MAX_TERMS) return fail(g, "lora: %u terms (max %d)", nterms, QW_LORA_MAX_TERMS);
    qw_lora_args a;
    memset(&a, 0, sizeof(a));
    a.out = (uint16_t *)out->ptr;
    a.base = (const uint16_t *)base->ptr;
    a.rows = rows;
    a.cols = cols;
    a.nterms = nterms;
    for (uint32_t t = 0; t < nterms; t++) {
        const qw_lora_term_desc *d = &terms[t];
        REQ_DT(d->a, H3_GPU_BF16, "lora A");
        REQ_DT(d->b, H3_GPU_BF16, "lora B");
        if (!d->rank || d->rank > QW_LORA_MAX_RANK)
            return fail(g, "lora: rank %u outside [1, %d]", d->rank, QW_LORA_MAX_RANK);
        if ((uint64_t)d->row0 + d->rows > rows) return fail(g, "lora: term rows outside the weight");
        if (!fits(d->a, 0, (size_t)d->rank * cols) || !fits(d->b, 0, (size_t)d->rows * d->rank))
            return fail(g, "lora: A or B smaller than its shape");
        a.terms[t] = qw_lora_term{(const uint16_t *)d->a->ptr, (const uint16_t *)d->b->ptr, d->row0,
                                  d->rows, d->rank, d->scale};
    }
    return launch(g, K_LORA, dim3((cols + 63) / 64, (rows + 63) / 64), dim3(256), a);
}

extern "C" int h3_gpu_gate_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *res,
                                const h3_gpu_tensor *branch, const h3_gpu_tensor *mod,
                                const h3_gpu_tensor *row_map, uint32_t rows, uint32_t width,
                                uint32_t slots, uint32_t gate_slot) {
    REQ_DT(out, H3_GPU_BF16, "gate out");
    REQ_DT(res, H3_GPU_BF16, "gate residual");
    REQ_DT(branch, H3_GPU_BF16, "gate branch");
    REQ_DT(mod, H3_GPU_BF16, "gate modulation");
    REQ_DT(row_map, H3_GPU_U32, "gate row_map");
    size_t n = (size_t)rows * width;
    if (width % 8) return fail(g, "gate: width must be a multiple of 8");
    if (gate_slot >= slots) return fail(g, "gate: slot out of range");
    if (!fits(out, 0, n) || !fits(res, 0, n) || !fits(branch, 0, n) || !fits(row_map, 0, rows) ||
        mod->elements < (size_t)slots * width)
        return fail(g, "gate: tensor too small");
    qw_gate_args a = {(uint16_t *)out->ptr, (const uint16_t *)res->ptr,
                      (const uint16_t *)branch->ptr, (const uint16_t *)mod->ptr,
                      (const uint32_t *)row_map->ptr, rows, width, slots, gate_slot};
    return launch(g, K_GATE, dim3(blocks_for(n / 8, 256)), dim3(256), a);
}

extern "C" int qw_gpu_qk_norm_rope_bf16(h3_gpu *g, h3_gpu_tensor *qk, uint32_t rows,
                                        uint32_t heads, uint32_t ld, uint32_t k_offset,
                                        const h3_gpu_tensor *norm_q, const h3_gpu_tensor *norm_k,
                                        const h3_gpu_tensor *rope_cos,
                                        const h3_gpu_tensor *rope_sin, uint32_t rope_rows,
                                        float eps) {
    REQ_DT(qk, H3_GPU_BF16, "qk_norm_rope qk");
    int do_norm = norm_q || norm_k;
    int do_rope = rope_cos || rope_sin;
    if (do_norm) {
        REQ_DT(norm_q, H3_GPU_BF16, "qk_norm_rope norm_q");
        REQ_DT(norm_k, H3_GPU_BF16, "qk_norm_rope norm_k");
        if (norm_q->elements < 128 || norm_k->elements < 128)
            return fail(g, "qk_norm_rope: norm weights need 128 elements");
    }
    if (do_rope) {
        REQ_DT(rope_cos, H3_GPU_F32, "qk_norm_rope cos");
        REQ_DT(rope_sin, H3_GPU_F32, "qk_norm_rope sin");
        if (!rope_rows || !fits(rope_cos, 0, (size_t)rope_rows * 64) ||
            !fits(rope_sin, 0, (size_t)rope_rows * 64))
            return fail(g, "qk_norm_rope: rope tables too small");
    }
    if (((uintptr_t)qk->ptr | (do_rope ? (uintptr_t)rope_cos->ptr | (uintptr_t)rope_sin->ptr : 0) |
         (do_norm ? (uintptr_t)norm_q->ptr | (uintptr_t)norm_k->ptr : 0)) % 16)
        return fail(g, "qk_norm_rope: tensors must be 16-byte aligned");
    if (ld % 8 || k_offset % 8 || k_offset + (size_t)heads * 128 > ld ||
        (size_t)heads * 128 > ld || (rows && !fits(qk, 0, (size_t)(rows - 1) * ld + k_offset + heads * 128)))
        return fail(g, "qk_norm_rope: bad geometry");
    qw_qk_norm_rope_args a = {(uint16_t *)qk->ptr,
                              do_norm ? (const uint16_t *)norm_q->ptr : NULL,
                              do_norm ? (const uint16_t *)norm_k->ptr : NULL,
                              do_rope ? (const float *)rope_cos->ptr : NULL,
                              do_rope ? (const float *)rope_sin->ptr : NULL,
                              rows, heads, ld, k_offset, do_rope ? rope_rows : 1,
                              do_norm, do_rope, eps};
    uint64_t items = (uint64_t)rows * heads * 2;
    return launch(g, K_QK_NORM_ROPE, dim3(blocks_for(items, 16)), dim3(256), a);
}

extern "C" int h3_gpu_head_rms_norm_bf16(h3_gpu *g, h3_gpu_tensor *t, const h3_gpu_tensor *w,
                                         uint32_t seq, uint32_t heads, uint32_t head_dim,
                                         float eps) {
    if (head_dim != 128) return fail(g, "head_rms_norm: head_dim must be 128");
    REQ_DT(t, H3_GPU_BF16, "head_rms_norm tensor");
    REQ_DT(w, H3_GPU_BF16, "head_rms_norm weight");
    if (heads % 2) return fail(g, "head_rms_norm: heads must be even");
    /* The fused kernel's "q" half covers heads [0, heads/2) and its "k" half
     * heads [heads/2, heads) of the same row, both with this weight. */
    return qw_gpu_qk_norm_rope_bf16(g, t, seq, heads / 2, heads * 128, (heads / 2) * 128, w, w,
                                    NULL, NULL, 0, eps);
}

extern "C" int qw_gpu_qk_rope_bf16(h3_gpu *g, h3_gpu_tensor *qo, h3_gpu_tensor *ko,
                                   const h3_gpu_tensor *qi, const h3_gpu_tensor *ki,
                                   const h3_gpu_tensor *cos_t, const h3_gpu_tensor *sin_t,
                                   uint32_t seq, uint32_t heads, uint32_t head_dim) {
    if (head_dim != 128) return fail(g, "qk_rope: head_dim must be 128");
    if (qo != qi || ko != ki) return fail(g, "qk_rope: only in-place operation is supported");
    REQ_DT(qo, H3_GPU_BF16, "qk_rope q");
    REQ_DT(ko, H3_GPU_BF16, "qk_rope k");
    size_t n = (size_t)seq * heads * 128;
    if (!fits(qo, 0, n) || !fits(ko, 0, n)) return fail(g, "qk_rope: tensor too small");
    if (heads % 2) return fail(g, "qk_rope: heads must be even");
    /* one rotation-only pass per tensor (head halves as in head_rms_norm) */
    for (int pass = 0; pass < 2; pass++) {
        h3_gpu_tensor *t = pass ? ko : qo;
        if (!qw_gpu_qk_norm_rope_bf16(g, t, seq, heads / 2, heads * 128, (heads / 2) * 128, NULL,
                                      NULL, cos_t, sin_t, seq, 0.0f))
            return 0;
    }
    return 1;
}

extern "C" int qw_gpu_modulation_reorder_bf16(h3_gpu *g, h3_gpu_tensor *out,
                                              const h3_gpu_tensor *raw, uint32_t mod_rows,
                                              uint32_t hidden, int shift_variant) {
    REQ_DT(out, H3_GPU_BF16, "reorder out");
    REQ_DT(raw, H3_GPU_BF16, "reorder raw");
    size_t n = (size_t)mod_rows * hidden * (shift_variant ? 6 : 4);
    if (!fits(out, 0, n) || !fits(raw, 0, n)) return fail(g, "reorder: tensor too small");
    if (out->ptr == raw->ptr) return fail(g, "reorder: output must not alias the input");
    qw_reorder_args a = {(uint16_t *)out->ptr, (const uint16_t *)raw->ptr, mod_rows, hidden,
                         shift_variant};
    return launch(g, K_REORDER, dim3(blocks_for((uint64_t)mod_rows * hidden, 256)), dim3(256), a);
}

extern "C" int qw_gpu_conditioning_bf16(h3_gpu *g, const qw_conditioning_desc *d) {
    if (!g || !d) return 0;
    const uint32_t H = d->hidden, rows = d->rows, S = d->shift_variant ? 6 : 4;
    const uint32_t nout = d->shift_variant ? 2 * H : H;
    if (!rows || rows > 2) return fail(g, "conditioning: rows must be 1 or 2");
    if (!H || H % 8 || (uint64_t)S * H * H >= (1ull << 32))
        return fail(g, "conditioning: hidden %u must be a multiple of 8", H);
    const struct { const h3_gpu_tensor *t; size_t n; h3_gpu_dtype type; int optional; } need[] = {
        {d->features, (size_t)rows * 256, H3_GPU_F32, 0},  {d->l1, (size_t)H * 256, H3_GPU_BF16, 0},
        {d->l2, (size_t)H * H, H3_GPU_BF16, 0},            {d->mod, (size_t)S * H * H, H3_GPU_BF16, 0},
        {d->norm_out, (size_t)nout * H, H3_GPU_BF16, 0},   {d->l1_bias, H, H3_GPU_BF16, 1},
        {d->l2_bias, H, H3_GPU_BF16, 1},                   {d->mod_bias, (size_t)S * H, H3_GPU_BF16, 1},
        {d->norm_out_bias, nout, H3_GPU_BF16, 1},          {d->wide, (size_t)rows * H, H3_GPU_BF16, 0},
        {d->silu, (size_t)rows * H, H3_GPU_BF16, 0},       {d->temb, (size_t)rows * H, H3_GPU_BF16, 0},
        {d->modulation, (size_t)rows * S * H, H3_GPU_BF16, 0},
        {d->norm_out_scale, (size_t)rows * nout, H3_GPU_BF16, 0}};
    for (const auto &x : need) {
        if (!x.t && x.optional) continue;
        if (!x.t || x.t->dtype != x.type) return fail(g, "conditioning: missing tensor or wrong dtype");
        if (!fits(x.t, 0, x.n)) return fail(g, "conditioning: tensor too small");
    }
    /* within a launch, workgroups read and write in any order */
    const size_t R = (size_t)rows * 2;
    const struct { const h3_gpu_tensor *a; size_t an; const h3_gpu_tensor *b; size_t bn; } clear[] = {
        {d->features, (size_t)rows * 256 * 4, d->wide, R * H}, {d->wide, R * H, d->temb, R * H},
        {d->wide, R * H, d->silu, R * H},                      {d->temb, R * H, d->silu, R * H},
        {d->silu, R * H, d->modulation, R * S * H},            {d->silu, R * H, d->norm_out_scale, R * nout}};
    for (const auto &c : clear)
        if (!apart(c.a->ptr, c.an, c.b->ptr, c.bn))
            return fail(g, "conditioning: a stage's output overlaps its input or its other output");
    /* the operands that are read 16 bytes at a time */
    for (const h3_gpu_tensor *t : {d->l1, d->l2, d->mod, d->norm_out,
                                   (const h3_gpu_tensor *)d->wide, (const h3_gpu_tensor *)d->silu})
        if ((uintptr_t)t->ptr % 16) return fail(g, "conditioning: tensors must be 16-byte aligned");
    auto bias = [](const h3_gpu_tensor *t) { return t ? (const uint16_t *)t->ptr : NULL; };
    auto grid = [](uint32_t n) { return dim3((n + 7) / 8); }; /* 4 waves of 2 columns */
    qw_cond_args a;
    memset(&a, 0, sizeof(a));
    a.rows = rows;
    a.hidden = H;
    a.shift_variant = d->shift_variant;
    a.in = d->features->ptr;
    a.w = (const uint16_t *)d->l1->ptr;
    a.bias = bias(d->l1_bias);
    a.out = (uint16_t *)d->wide->ptr;
    a.k = 256;
    a.n = H;
    if (!launch(g, K_COND_L1, grid(H), dim3(256), a)) return 0;
    a.in = d->wide->ptr;
    a.w = (const uint16_t *)d->l2->ptr;
    a.bias = bias(d->l2_bias);
    a.out = (uint16_t *)d->temb->ptr;
    a.out2 = (uint16_t *)d->silu->ptr;
    a.k = H;
    if (!launch(g, K_COND_L2, grid(H), dim3(256), a)) return 0;
    a.in = d->silu->ptr;
    a.w = (const uint16_t *)d->mod->ptr;
    a.bias = bias(d->mod_bias);
    a.out = (uint16_t *)d->modulation->ptr;
    a.n = S * H;
    a.w2 = (const uint16_t *)d->norm_out->ptr;
    a.bias2 = bias(d->norm_out_bias);
    a.out2 = (uint16_t *)d->norm_out_scale->ptr;
    a.n2 = nout;
    if (!apart(a.out, R * a.n, a.out2, R * a.n2)) {
        /* one over the other: the modulation stands, as from separate linears */
        qw_cond_args first = a;
        first.n = 0;
        if (!launch(g, K_COND_MOD, grid(nout), dim3(256), first)) return 0;
        a.n2 = 0;
    }
    return launch(g, K_COND_MOD, grid(a.n + a.n2), dim3(256), a);
}

extern "C" int qw_gpu_fill_normal_bf16(h3_gpu *g, h3_gpu_tensor *t, size_t off, size_t count,
                                       uint64_t seed, uint64_t stream, float std, float offset) {
    REQ_DT(t, H3_GPU_BF16, "fill tensor");
    if (!fits(t, off, count)) return fail(g, "fill: range outside tensor");
    qw_fill_args a = {(uint16_t *)t->ptr + off, count, seed, stream, std, offset};
    return launch(g, K_FILL, dim3(blocks_for(count, 256)), dim3(256), a);
}

extern "C" int h3_gpu_quantize_weight_int8(h3_gpu *g, h3_gpu_tensor *out, h3_gpu_tensor *scales,
                                           const h3_gpu_tensor *in, uint32_t rows,
                                           uint32_t cols) {
    REQ_DT(out, H3_GPU_I8, "quantize out");
    REQ_DT(scales, H3_GPU_F32, "quantize scales");
    REQ_DT(in, H3_GPU_BF16, "quantize in");
    size_t n = (size_t)rows * cols;
    if (!fits(out, 0, n) || !fits(in, 0, n) || !fits(scales, 0, rows))
        return fail(g, "quantize: tensor too small");
    qw_quant_args a = {(int8_t *)out->ptr, (float *)scales->ptr, (const uint16_t *)in->ptr, rows,
                       cols};
    return launch(g, K_QUANT, dim3(rows), dim3(256), a);
}

extern "C" int qw_gpu_dequant_int8_f32(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                                       const h3_gpu_tensor *scales, uint32_t rows,
                                       uint32_t cols) {
    REQ_DT(out, H3_GPU_F32, "dequant out");
    REQ_DT(q, H3_GPU_I8, "dequant q");
    REQ_DT(scales, H3_GPU_F32, "dequant scales");
    size_t n = (size_t)rows * cols;
    if (!fits(out, 0, n) || !fits(q, 0, n) || !fits(scales, 0, rows))
        return fail(g, "dequant: tensor too small");
    qw_dequant_args a = {(float *)out->ptr, (const int8_t *)q->ptr, (const float *)scales->ptr,
                         rows, cols};
    return launch(g, K_DEQUANT, dim3(blocks_for(n, 256)), dim3(256), a);
}

extern "C" int qw_gpu_copy_rows(h3_gpu *g, h3_gpu_tensor *dst, size_t doff, uint32_t dstride,
                                const h3_gpu_tensor *src, size_t soff, uint32_t sstride,
                                uint32_t rows, uint32_t row_elems) {
    if (!dst || !src || dst->dtype != src->dtype) return fail(g, "copy_rows: dtype mismatch");
    size_t es = dtype_size(dst->dtype);
    if (!rows || !row_elems) return 1;
    if ((row_elems * es) % 4 || (doff * es) % 4 || (soff * es) % 4 || (dstride * es) % 4 ||
        (sstride * es) % 4)
        return fail(g, "copy_rows: rows must be 4-byte aligned");
    if (!fits(dst, doff, (size_t)(rows - 1) * dstride + row_elems) ||
        !fits(src, soff, (size_t)(rows - 1) * sstride + row_elems))
        return fail(g, "copy_rows: range outside tensor");
    qw_copy2d_args a = {dst->ptr + doff * es, src->ptr + soff * es, rows, row_elems * es,
                        dstride * es, sstride * es};
    uint64_t words = (uint64_t)rows * row_elems * es / 4;
    g->stats.blit_copies++;
    return launch(g, K_COPY2D, dim3(blocks_for(words, 256)), dim3(256), a);
}

extern "C" int h3_gpu_copy_bf16(h3_gpu *g, h3_gpu_tensor *dst, size_t doff,
                                const h3_gpu_tensor *src, size_t soff, size_t n) {
    REQ_DT(dst, H3_GPU_BF16, "copy dst");
    REQ_DT(src, H3_GPU_BF16, "copy src");
    if (!fits(dst, doff, n) || !fits(src, soff, n)) return fail(g, "copy: range outside tensor");
    if (!n) return 1;
    hipError_t e = hipMemcpyAsync(dst->ptr + doff * 2, src->ptr + soff * 2, n * 2,
                                  hipMemcpyDeviceToDevice, g->stream);
    g->stats.blit_copies++;
    return e == hipSuccess ? 1 : fail(g, "copy: %s", hipGetErrorString(e));
}

/* ---- GEMM ---------------------------------------------------------------- */

static int widen_launch(h3_gpu *g, uint16_t *out, const int8_t *in, size_t n) {
    qw_widen_args wa;
    wa.out = out;
    wa.in = in;
    wa.count = n;
    unsigned blocks = (unsigned)std::min<size_t>((n / 8 + 255) / 256, 65536);
    return launch(g, K_WIDEN, dim3(blocks ? blocks : 1), dim3(256), wa);
}

extern "C" int qw_gpu_widen_int8_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                                      size_t count) {
    if (!g) return 0;
    REQ_DT(out, H3_GPU_BF16, "widen out");
    REQ_DT(q, H3_GPU_I8, "widen in");
    if (count % 16) return fail(g, "widen: count %zu is not a multiple of 16", count);
    if (!fits(out, 0, count) || !fits(q, 0, count)) return fail(g, "widen: tensor too small");
    if (!count) return 1;
    return widen_launch(g, (uint16_t *)out->ptr, (const int8_t *)q->ptr, count);
}


/* Split tiles. A grid of one workgroup per 256 x 256 tile runs in waves of
 * `cus` tiles; when the last wave is partly filled (R = tiles % cus tiles,
 * all of them when there is no full wave), each of its tiles can instead be
 * cut into s k-ranges: R s pieces taking ceil(R s / cus) waves of 1/s the
 * length. s minimises that tail time plus 0.02 (s - 1) for writing and
 * re-reading the fp32 partials, and is used only when that beats 0.9 of the
 * whole-tile tail (M = 8704, K = 12288, N = 3072, residual-gate epilogue:
 * 152 tail tiles in 3 pieces 557-588 us against 573-644 us for the
 * whole-tile walk, same boxes; 2, 4 or 5 pieces 595-660 us). Pieces stay at least 32 k-steps (2048 k) long: shorter
 * pieces lost more to their partials than they gained (K = 3072 linears
 * measured slower when split, K = 12288 ones faster). And
 * R s <= QW_SPLIT_MAX_PIECES * cus bounds the partial workspace. */
#define QW_SPLIT_MAX_PIECES 2
static uint32_t split_choice(h3_gpu *g, uint32_t tiles, uint32_t ksteps,
                             uint64_t max_pieces = (uint64_t)QW_SPLIT_MAX_PIECES * 1024u) {
    const uint32_t G = g->cus, R = tiles % G;
    if (R == 0) return 1; /* every wave is full: nothing to split */
    if (g->split_force > 1 && (uint64_t)R * g->split_force <= (uint64_t)QW_SPLIT_MAX_PIECES * G &&
        (uint64_t)R * g->split_force <= max_pieces && ksteps >= g->split_force)
        return g->split_force;
    uint32_t best = 1;
    double best_t = 0.9;
    for (uint32_t s = 2; s <= 8; s++) {
        if ((uint64_t)R * s > (uint64_t)QW_SPLIT_MAX_PIECES * G || (uint64_t)R * s > max_pieces ||
            ksteps < g->split_min_steps * s)
            break;
        const double t = (double)((R * s + G - 1) / G) / s + 0.02 * (s - 1);
        if (t < best_t) {
            best_t = t;
            best = s;
        }
    }
    return best;
}

/* Time models of a linear on bf16 W, in microseconds, that pick its tiles.
 *
 * Wide (gemm_q.h): a round of 256-row tiles takes 1.3 us a k-step (64 k) and
 * 12 us for prologue and epilogue (measured at M = 1152-8704: 75-88 us a
 * round at K = 3072, 92-102 at 4096, 274 at 12288); a partly filled last
 * round the length of split_choice's pieces and 8 + 0.055 R s^2 us for their
 * partial sums (M = 4119 against 4096, K = 4096: 59, 65 and 79 us for 16, 48
 * and 96 tail tiles in 2; K = 12288: 79 us for 16 in 6, 138 for 60 in 4), or
 * 0.6 of a round on half tiles. Mixed heights instead fill `n` rounds with T
 * tile rows, as few of the taller as cover the rows; each CU's tiles, tallest
 * first, in proportion to their heights. h1 = 0: 256-row tiles. */
struct wide_plan {
    double us;
    uint32_t h1, h2, rows1, rows2;
};
/* 256-row tiles in rounds of `round` us; half: the share of a round that a
 * last one on half tiles takes */
static double wide_us(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t ksteps, double round,
                      double half) {
    const uint32_t C = g->cus, tiles = (rows + 255) / 256 * ((cols + 255) / 256);
    const uint32_t R = tiles % C, s = split_choice(g, tiles, ksteps);
    const double us = (double)(tiles / C) * round;
    if (s > 1) return us + (double)((R * s + C - 1) / C) / s * round + 8.0 + 0.055 * R * s * s;
    return us + (!R ? 0.0 : tiles > C && 2 * R <= C ? half * round : round);
}
static wide_plan plan_wide(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t ksteps) {
    const uint32_t C = g->cus, tn = (cols + 255) / 256;
    const double step = 1.3 * ksteps, fix = 12.0;
    wide_plan p = {wide_us(g, rows, cols, ksteps, step + fix, 0.6), 0, 0, 0, 0};
    if (!g->mixed || C % 8) return p;
    const uint32_t m32 = (rows + 31) / 32;
    double best = 0.98 * p.us;
    const uint32_t n0 = std::max(1u, (uint32_t)((uint64_t)m32 * tn / 8 / C));
    for (uint32_t n = n0; n <= n0 + 2; n++) {
        const uint32_t T = (uint32_t)((uint64_t)n * C / tn);
        for (uint32_t h = 7; h >= 6; h--) { /* r1 rows of h + 1, r2 of h */
            if (!T || (uint64_t)T * (h + 1) < m32) continue;
            const uint32_t low = T * h;
            const uint32_t r1 = m32 > low ? m32 - low : 0;
            const uint32_t r2 = m32 > r1 * (h + 1) ? (m32 - r1 * (h + 1) + h - 1) / h : 0;
            const uint32_t all = ((r1 + r2) * tn + C - 1) / C, tall = (r1 * tn + C - 1) / C;
            const double us = tall * (step * (h + 1) / 8 + fix) + (all - tall) * (step * h / 8 + fix);
            if (us < best) {
                best = us;
                p = {us, h + 1, h, r1, r2};
            }
        }
    }
    return p;
}

/* Narrow (gemm_s.h), tiles of 64 mb rows x 128 columns in s k-range pieces:
 * a k-step of a tile takes 0.30, 0.39, 0.56, 0.70 us (mb = 1-4), times 0.85
 * to 1.2 from an idle to a full chip and 1.35 to 1 from K = 8192 on (an A
 * panel no longer stays in L2 beside the weights), a round 5 us more, and s
 * pieces 0.5 + s (0.5 + 0.45 mb) us for the partial sums. Fitted to M =
 * 23-1152 at K = 3072, 4096 and 12288 within 15% (M = 320: 26, 14, 37, 42 us
 * for QKV, out, up and down, against 45, 33, 46 and 62 on the 128 x 256 tiles
 * that these replace; M = 100, K = 4096: 13 against 31). The weights cannot
 * come faster than 5 TB/s. The times are of calls repeated on the same
 * weights, which a 256 MB cache holds; in a model each layer's come from HBM,
 * and the short linears take up to 1.4 times as long (out projection, M =
 * 1152: 32.9 us in the loop of layers, 23.9 alone). Returns the least time
 * and its mb and s. */
static double narrow_us(const h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t ksteps,
                        uint32_t max_s, uint32_t *mb_out, uint32_t *s_out) {
    static const double step_us[4] = {0.30, 0.39, 0.56, 0.70}, long_k[4] = {1.35, 1.3, 1.15, 1.0};
    const uint32_t C = g->cus, tn = (cols + 127) / 128;
    const double hbm_us = (double)cols * ksteps * 128 / 5e6;
    double best = 1e30;
    for (uint32_t mb = 1; mb <= 4; mb++) {
        const uint32_t R = (rows + 64 * mb - 1) / (64 * mb) * tn;
        for (uint32_t s = 1; s <= max_s; s++) {
            /* pieces of at least 4 k-steps, all in one round, a counter each */
            if (s > 1 && ((uint64_t)R * s > C || ksteps < 4 * s)) break;
            const double rounds = (double)(((uint64_t)R * s + C - 1) / C);
            if (rounds > 2) break; /* not fitted, and the wide tiles' ground */
            const double fill = std::min(1.0, (double)R * s / C);
            double t = rounds * ((ksteps + s - 1) / s * step_us[mb - 1] * (0.85 + 0.35 * fill) *
                                     (ksteps >= 128 ? long_k[mb - 1] : 1.0) + 5.0);
            if (s > 1) t += 0.5 + s * (0.5 + 0.45 * mb);
            t = std::max(t, hbm_us + 3.0);
            if (t < best) {
                best = t;
                *mb_out = mb;
                *s_out = s;
            }
        }
    }
    return best;
}

/* Whether workspaces may be made now: not while the stream is being captured
 * into a graph, nor where they are switched off. */
static int can_allocate(h3_gpu *g) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return g->workspaces && hipStreamIsCapturing(g->stream, &st) == hipSuccess &&
           st == hipStreamCaptureStatusNone;
}

/* Partial sums and piece counters of split tiles (and of split attention
 * blocks), from the first one on. 0 where there are none and none can be had:
 * the launch then runs whole. */
#define QW_FLAGS 4
static int split_workspace(h3_gpu *g) {
    if (g->sk_part) return 1;
    if (!can_allocate(g)) return 0;
    hipStreamSynchronize(g->stream);
    const size_t n = (size_t)QW_SPLIT_MAX_PIECES * g->cus * 256 * 256 * 4;
    const size_t flags = (size_t)g->cus * QW_FLAGS * 4;
    if (hipMalloc((void **)&g->sk_part, n) == hipSuccess) {
        if (hipMalloc((void **)&g->sk_flag, flags) == hipSuccess &&
            hipMemsetAsync(g->sk_flag, 0, flags, g->stream) == hipSuccess) {
            g->stats.allocated_bytes += n + flags;
            return 1;
        }
        if (g->sk_flag) hipFree(g->sk_flag);
        hipFree(g->sk_part);
    }
    (void)hipGetLastError(); /* seen to here */
    g->sk_part = NULL;
    g->sk_flag = NULL;
    return 0;
}

/* How the rows of a linear on bf16 W run: the first `wide` of them (a
 * multiple of 256 when the rest are not none) on wide tiles, the rest on
 * narrow ones. A last tile row of few rows costs a whole round of wide tiles
 * wherever it opens one (M = 4119, K = 4096, N = 4096: 161 us against 102
 * for M = 4096), and one or two us per column of narrow tiles. */
struct linear_plan {
    uint32_t wide, mb, s;
    wide_plan w; /* how the first run */
    double us;
};
static linear_plan plan_linear(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t ksteps,
                               uint32_t max_s) {
    linear_plan p = {rows, 0, 1, plan_wide(g, rows, cols, ksteps), 0.0};
    p.us = p.w.us;
    if (!g->narrow) return p;
    uint32_t mb, s;
    const double all = narrow_us(g, rows, cols, ksteps, max_s, &mb, &s);
    if (all < 0.98 * p.us) p = {0, mb, s, p.w, all};
    /* the last, ragged tile row on narrow tiles, or up to three more with it */
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t rem = rows % 256 + 256 * j;
        if (!rem || rows < rem + 256) continue;
        const wide_plan w = plan_wide(g, rows - rem, cols, ksteps);
        const double t = w.us + narrow_us(g, rem, cols, ksteps, max_s, &mb, &s);
        if (t < 0.97 * p.us) p = {rows - rem, mb, s, w, t};
    }
    return p;
}

/* Whether an int8 linear is faster on the "_w8" kernels, which widen inside
 * (256-row tiles whose round takes 1.45 us a k-step and 7 us, no half tiles),
 * than as a pass that widens its weight (3 bytes an element at 6.2 TB/s, 2.5
 * us more) and the bf16 kernels of plan p. Fewer than 512 rows that no narrow
 * tiles suit, and long K on whole tiles of 256 rows, run there in any case;
 * else the times decide, at K from 3072 (where the bf16 tiles' are fitted) or
 * within a round of tiles.
 *
 * Against the faster of the two, at 430 shapes of 16 to 8704 rows with weights
 * that are in no cache, the choice costs 0.2% on average at K >= 3072 and 1.4%
 * over all. Where the sides meet, us (pass / _w8): 24576 x 4096 at 200 rows
 * 122 / 76, at 700 208 / 156, at 1752 293 / 294, at 4119 629 / 680; 12288 x
 * 4096 at 700 rows 88 / 88, at 1152 113 / 101, at 1400 137 / 155; 3072 x
 * 12288 at 64 rows 40 / 77, at 1400 130 / 121, at 3000 196 / 237, at 8704 499
 * / 549; 3072 x 3072 at 16 to 8704 rows 21-125 / 63-149. */
static bool w8_faster(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t ksteps,
                      const linear_plan &p, bool low_tiles) {
    if (!p.mb && (rows < 512 || (ksteps >= 128 && !low_tiles))) return true;
    const uint64_t tiles = (uint64_t)((rows + 255) / 256) * ((cols + 255) / 256);
    if (ksteps < 48 && tiles > g->cus) return false;
    const double pass = 2.5 + 192.0 * cols * ksteps / 6.2e6;
    return wide_us(g, rows, cols, ksteps, 1.45 * ksteps + 7.0, 1.0) < 0.94 * (pass + p.us);
}

/* the widened copy of an int8 weight, grown to `bytes`; 0 where it cannot be
 * (the "_w8" kernels need none) */
static int widen_workspace(h3_gpu *g, size_t bytes) {
    if (g->widen_bytes >= bytes) return 1;
    if (!can_allocate(g)) return 0;
    hipStreamSynchronize(g->stream);
    if (g->widen) hipFree(g->widen);
    g->widen = NULL;
    g->widen_bytes = 0;
    if (hipMalloc(&g->widen, bytes) != hipSuccess) {
        (void)hipGetLastError(); /* seen to here */
        g->widen = NULL;
        return 0;
    }
    g->widen_bytes = bytes;
    g->stats.allocated_bytes += bytes; /* runtime workspaces count too */
    return 1;
}

/* no_alloc: the workspace-free form behind qw_gpu_linear_static (int8
 * weights always widen inside the GEMM; split-tile partials and counters live
 * in the static workspace, as far as it holds them) */
/* kv: outputs of their own for the k and v thirds (QKNORM), or NULL */
struct kv_out {
    uint16_t *k, *v;
    uint32_t ld;
    size_t bytes;
};
static int linear_impl(h3_gpu *g, const qw_linear_desc *d, int no_alloc,
                       const kv_out *kv = NULL) {
    if (!g || !d) return 0;
    REQ_DT(d->out, H3_GPU_BF16, "linear out");
    REQ_DT(d->in, H3_GPU_BF16, "linear in");
    if (!d->weight) return fail(g, "linear: missing weight");
    const int int8 = d->weight->dtype == H3_GPU_I8;
    if (!int8 && d->weight->dtype != H3_GPU_BF16) return fail(g, "linear: weight dtype");
    if (d->rows == 0 || d->cols == 0) return 1;
    if (d->k == 0 || d->k % 64) return fail(g, "linear: k=%u must be a positive multiple of 64", d->k);
    if (d->lda % 8 || d->in_offset % 8 || d->lda < d->k)
        return fail(g, "linear: input rows must be 16-byte aligned (lda %u, offset %zu)", d->lda,
                    d->in_offset);
    const int glu = d->epilogue == QW_EPI_SWIGLU; /* cols = 2 F, output [rows, F] */
    const uint32_t out_cols = glu ? d->cols / 2 : d->cols;
    if (d->ldc < out_cols) return fail(g, "linear: ldc < cols");
    if (out_cols % 8 || (glu && d->cols % 16) || d->ldc % 4 || d->out_offset % 4)
        return fail(g, "linear: cols (%u) must be a multiple of 8 and output rows 8-byte aligned",
                    d->cols);
    if (!fits(d->in, d->in_offset, (size_t)(d->rows - 1) * d->lda + d->k))
        return fail(g, "linear: input too small");
    if (!fits(d->out, d->out_offset, (size_t)(d->rows - 1) * d->ldc + out_cols))
        return fail(g, "linear: output too small");
    if (!fits(d->weight, 0, (size_t)d->cols * d->k)) return fail(g, "linear: weight too small");
    if ((uint64_t)d->cols * d->k >= (1ull << 32) || (uint64_t)d->rows * d->lda >= (1ull << 32))
        return fail(g, "linear: operand exceeds 32-bit element offsets");
    if (int8 || d->wscale) {
        REQ_DT(d->wscale, H3_GPU_F32, "linear scales");
        if (!fits(d->wscale, 0, d->cols)) return fail(g, "linear: scales too small");
    }
    if (d->bias) {
        REQ_DT(d->bias, H3_GPU_BF16, "linear bias");
        if (!fits(d->bias, 0, d->cols)) return fail(g, "linear: bias too small");
    }
    const uint16_t *gate = NULL;
    const uint32_t *row_map = NULL;
    uint32_t gate_stride = 0;
    if (d->epilogue == QW_LINEAR_GATE) {
        REQ_DT(d->modulation, H3_GPU_BF16, "linear gate modulation");
        REQ_DT(d->row_map, H3_GPU_U32, "linear gate row_map");
        if (d->gate_slot >= d->slots) return fail(g, "linear: gate slot out of range");
        if (!fits(d->row_map, 0, d->rows)) return fail(g, "linear: row_map too small");
        gate_stride = d->slots * d->cols;
        if (d->modulation->elements < gate_stride) return fail(g, "linear: modulation too small");
        gate = (const uint16_t *)d->modulation->ptr + (size_t)d->gate_slot * d->cols;
        row_map = (const uint32_t *)d->row_map->ptr;
    } else if (d->epilogue == QW_LINEAR_QKNORM) {
        REQ_DT(d->norm_q, H3_GPU_BF16, "linear qk norm_q");
        REQ_DT(d->norm_k, H3_GPU_BF16, "linear qk norm_k");
        REQ_DT(d->rope_cos, H3_GPU_F32, "linear qk rope cos");
        REQ_DT(d->rope_sin, H3_GPU_F32, "linear qk rope sin");
        if (d->cols % 384 || d->out_offset || d->ldc % 8)
            return fail(g, "linear qk: cols must be q|k|v heads of 128, output at offset 0");
        if (d->norm_q->elements < 128 || d->norm_k->elements < 128 || !d->rope_rows ||
            !fits(d->rope_cos, 0, (size_t)d->rope_rows * 64) ||
            !fits(d->rope_sin, 0, (size_t)d->rope_rows * 64))
            return fail(g, "linear qk: norm weights or rope tables too small");
        if (((uintptr_t)d->norm_q->ptr | (uintptr_t)d->norm_k->ptr | (uintptr_t)d->rope_cos->ptr |
             (uintptr_t)d->rope_sin->ptr | (uintptr_t)d->out->ptr) % 16)
            return fail(g, "linear qk: tensors must be 16-byte aligned");
    } else if (d->epilogue != QW_LINEAR_STORE && d->epilogue != QW_LINEAR_GELU && !glu) {
        return fail(g, "linear: unknown epilogue %d", d->epilogue);
    }
    if (d->epilogue == QW_LINEAR_QKNORM && d->rope_rows < 128) {
        /* the fused epilogue wraps a 128-row block's RoPE table rows with one
         * subtraction, which needs a table of at least 128 rows; a shorter
         * one runs the plain linear, then the standalone norm + RoPE
         * (bit-identical to the fused epilogue) */
        qw_linear_desc plain = *d;
        plain.epilogue = QW_LINEAR_STORE;
        if (!linear_impl(g, &plain, no_alloc)) return 0;
        return qw_gpu_qk_norm_rope_bf16(g, d->out, d->rows, d->cols / 384, d->ldc, d->cols / 3,
                                        d->norm_q, d->norm_k, d->rope_cos, d->rope_sin,
                                        d->rope_rows, d->eps);
    }
    /* at most 8 rows, plain or GELU epilogue: one wave per 2 output columns
     * streams the weight once */
    if (d->rows <= 8 &&
        (d->epilogue == QW_LINEAR_STORE || d->epilogue == QW_LINEAR_GELU)) {
        qw_gemm_args a;
        memset(&a, 0, sizeof(a));
        a.a = (const uint16_t *)d->in->ptr + d->in_offset;
        a.w = d->weight->ptr;
        a.wscale = d->wscale ? (const float *)d->wscale->ptr : NULL;
        a.bias = d->bias ? (const uint16_t *)d->bias->ptr : NULL;
        a.out = (uint16_t *)d->out->ptr + d->out_offset;
        a.m = d->rows;
        a.n = d->cols;
        a.k = d->k;
        a.lda = d->lda;
        a.ldc = d->ldc;
        const int kid = (int8 ? K_GEMV_I8_STORE : K_GEMV_BF16_STORE) +
                        (d->epilogue == QW_LINEAR_GELU ? 1 : 0);
        const uint32_t waves = (d->cols + 1) / 2; /* 2 columns per wave */
        g->route_n = 0;
        return launch_step(g, kid, dim3((waves + 3) / 4), dim3(256), a, 1);
    }
    /* int8 weights: the "_w8" kernels widen each int8 W tile once per
     * workgroup into the bf16 W stage in LDS (no copy through HBM, half the
     * weight bytes; 1.5 VALU instructions per weight per workgroup), or one
     * bandwidth-bound pass widens the weight to a bf16 copy for the bf16
     * kernels. Both give the same bits where the sums' pieces are the same
     * (the per-row scale multiplies the finished fp32 sums). */
    const linear_plan wide_all = {d->rows, 0, 1, plan_wide(g, d->rows, d->cols, d->k / 64), 0.0};
    linear_plan plan = no_alloc || (int8 && g->int8_route == QW_INT8_W8)
                           ? wide_all : plan_linear(g, d->rows, d->cols, d->k / 64, 8);
    const size_t weights = (size_t)d->cols * d->k;
    g->route_n = 0;
    const int widen = int8 && !no_alloc && g->int8_route != QW_INT8_W8 &&
                      (g->int8_route == QW_INT8_WIDEN ||
                       !w8_faster(g, d->rows, d->cols, d->k / 64, plan, wide_all.w.h1)) &&
                      weights * 2 < (1ull << 31) /* a buffer's range */ &&
                      widen_workspace(g, weights * 2);
    if (int8 && !widen) plan = wide_all;
    if (plan.s > 1 && !split_workspace(g))
        plan = plan_linear(g, d->rows, d->cols, d->k / 64, 1);
    const void *wptr = d->weight->ptr;
    if (widen) {
        if (!widen_launch(g, (uint16_t *)g->widen, (const int8_t *)d->weight->ptr, weights)) return 0;
        wptr = g->widen;
    }
    qw_gemm_args a;
    a.a = (const uint16_t *)d->in->ptr + d->in_offset;
    a.w = wptr;
    a.wscale = d->wscale ? (const float *)d->wscale->ptr : NULL;
    a.bias = d->bias ? (const uint16_t *)d->bias->ptr : NULL;
    a.out = (uint16_t *)d->out->ptr + d->out_offset;
    a.gate = gate;
    a.row_map = row_map;
    a.m = d->rows;
    a.n = d->cols;
    a.k = d->k;
    a.lda = d->lda;
    a.ldc = d->ldc;
    a.gate_row_stride = gate_stride;
    {
        const uint64_t ab = ((uint64_t)(d->rows - 1) * d->lda + d->k) * 2;
        const uint64_t wb = (uint64_t)d->cols * d->k * (int8 && !widen ? 1 : 2);
        const uint64_t ob = ((uint64_t)(d->rows - 1) * d->ldc + out_cols) * 2;
        if (ab >= (1ull << 31) || wb >= (1ull << 31) || ob >= (1ull << 31))
            return fail(g, "linear: operand exceeds 2 GiB buffer range");
        a.a_bytes = (uint32_t)ab;
        a.w_bytes = (uint32_t)wb;
        a.out_bytes = (uint32_t)ob;
    }
    const int qkn = d->epilogue == QW_LINEAR_QKNORM;
    /* the 4-wave kernels (one wave per SIMD, 128 x 128 per wave). Same box,
     * alternating, M = 8704, us, against the 8-wave 16x16x32 kernels they
     * replaced (two waves per SIMD, 64 x 128 per wave): QKV 447 / 458, out
     * 149 / 155, up (GELU) 537 / 554, down 598 / 623. */
    const int kid = (int8 && !widen ? K_GEMM_W8_STORE_Q : K_GEMM_BF16_STORE_Q) + d->epilogue;
    const unsigned threads = 256, bm = 256, bn = 256;
    a.norm_q = qkn ? (const uint16_t *)d->norm_q->ptr : NULL;
    a.norm_k = qkn ? (const uint16_t *)d->norm_k->ptr : NULL;
    a.rope_cos = qkn ? (const float *)d->rope_cos->ptr : NULL;
    a.rope_sin = qkn ? (const float *)d->rope_sin->ptr : NULL;
    a.rope_rows = qkn ? d->rope_rows : 1;
    a.qk_cols = qkn ? d->cols / 3 * 2 : 0;
    a.eps = qkn ? d->eps : 0.0f;
    a.out_k = kv ? kv->k : NULL;
    a.out_v = kv ? kv->v : NULL;
    a.ld_kv = kv ? kv->ld : 0;
    a.kv_bytes = kv ? (uint32_t)kv->bytes : 0;
    a.half_from = 0;
    a.half_count = 0;
    a.m_base = 0;
    a.mix_h1 = a.mix_h2 = a.mix_rows1 = a.mix_rows2 = a.mix_dealt = 0;
    a.sk_part = NULL;
    a.sk_flag = NULL;
    if (plan.mb) { /* the rows past plan.wide on narrow tiles */
        qw_gemm_args n = a;
        n.m_base = plan.wide;
        n.tiles_m = (d->rows - plan.wide + 64 * plan.mb - 1) / (64 * plan.mb);
        n.tiles_n = (d->cols + 127) / 128;
        n.dp_tiles = 0;
        n.split = plan.s;
        const uint64_t np = (uint64_t)n.tiles_m * n.tiles_n * plan.s;
        if (np >= (1ull << 31)) return fail(g, "linear: grid too large");
        if (plan.s > 1) {
            /* narrow_us keeps the pieces within a round: checked, so that a
             * change to it fails loudly */
            if (np > g->cus) return fail(g, "linear: internal error: %llu pieces", (unsigned long long)np);
            n.sk_part = g->sk_part;
            n.sk_flag = g->sk_flag;
        }
        static const int first[4] = {K_GEMM_N1, K_GEMM_N2, K_GEMM_N3, K_GEMM_N4};
        if (!launch_step(g, first[plan.mb - 1] + d->epilogue, dim3((uint32_t)np), dim3(threads), n,
                         plan.s, 0, plan.wide))
            return 0;
        if (!plan.wide) return 1;
        a.m = plan.wide;
    }
    const uint32_t rows = plan.wide; /* on wide tiles */
    a.tiles_m = (rows + bm - 1) / bm;
    a.tiles_n = (d->cols + bn - 1) / bn;
    const uint32_t tiles = a.tiles_m * a.tiles_n;
    a.dp_tiles = tiles;
    a.split = 1;
    uint32_t grid = tiles;
    const int mix = !(int8 && !widen) && plan.w.h1;
    if (no_alloc) {
        const uint32_t s = split_choice(g, tiles, d->k / 64, QW_STATIC_PARTS);
        if (s > 1) {
            const uint32_t R = tiles % g->cus;
            const size_t need = (size_t)R * s * QW_STATIC_PART_BYTES;
            /* split_choice caps R s at QW_STATIC_PARTS and R < cus: an
             * internal invariant, checked so a change to either fails loudly */
            if (need > (size_t)QW_STATIC_PARTS * QW_STATIC_PART_BYTES || R > QW_STATIC_FLAGS)
                return fail(g, "linear_static: internal error: %u split pieces over the static "
                               "workspace's %u", R * s, QW_STATIC_PARTS);
            uint32_t *flags = (uint32_t *)(g->static_scratch +
                                           (size_t)QW_STATIC_PARTS * QW_STATIC_PART_BYTES);
            /* the counters must start at zero: a previous call leaves them
             * zero, but one that did not complete might not */
            qw_zero_args za;
            za.p = flags;
            za.count = R;
            if (!launch(g, K_ZERO, dim3(blocks_for(R, 256)), dim3(256), za)) return 0;
            a.dp_tiles = tiles - R;
            a.split = s;
            a.sk_part = (float *)g->static_scratch;
            a.sk_flag = flags;
            grid = a.dp_tiles + R * s;
        }
    } else {
        /* where mixed heights fill the rounds they also beat split tiles
         * (down projection shape, bf16 W, M = 8704: 500 us on 224-row tiles
         * against 568 with 256-row tiles and a 3-piece tail) */
        const uint32_t s = mix ? 1u : split_choice(g, tiles, d->k / 64);
        if (s > 1 && split_workspace(g)) {
            const uint32_t R = tiles % g->cus;
            /* the workspace holds QW_SPLIT_MAX_PIECES * cus partials and
             * cus counters; split_choice keeps within both */
            if ((uint64_t)R * s > (uint64_t)QW_SPLIT_MAX_PIECES * g->cus || R > g->cus)
                return fail(g, "linear: %u x %u split pieces exceed the partial workspace", R, s);
            a.dp_tiles = tiles - R;
            a.split = s;
            a.sk_part = g->sk_part;
            a.sk_flag = g->sk_flag;
            grid = a.dp_tiles + R * s;
        }
    }
    /* bf16-weight kernels without split tiles: one workgroup per CU walks
     * the tiles, so a tile's output stores drain under the next tile's first
     * loads (up 521 -> 514 us, QKV 365 -> 359 us against one workgroup per
     * tile) */
    if (a.split == 1 && mix) {
        a.mix_h1 = plan.w.h1;
        a.mix_h2 = plan.w.h2;
        a.mix_rows1 = plan.w.rows1;
        a.mix_rows2 = plan.w.rows2;
        /* few tile columns: an XCD's share of the ids as they are dealt (one
         * row of each group of 4, every second column) spans no more panels
         * than a range of tiles does, and at long K their slices stay in step
         * better. M = 8704 and 12000, us, range / dealt: 12 columns, K = 12288
         * 497 / 483 and 748 / 718, K = 8192 306 / 303 and 453 / 432, K = 4096
         * 159 / 160 and 234 / 225; 16 columns level within 1.5%; 20 columns
         * 783 / 797 and 1106 / 1070; 24 columns 998 / 1033 and 1424 / 1326,
         * but 484 / 542 at M = 4119 (int8); 32 columns 1269 / 1314; 36 columns
         * 1459 / 1473 and 1968 / 2043, 3% either way at other row counts. So
         * the line is at 16 columns, up to where no shape measured loses. */
        a.mix_dealt = a.tiles_n <= 16 && d->k >= 8192;
        const uint32_t n = (a.mix_rows1 + a.mix_rows2) * a.tiles_n;
        if (!launch_step(g, K_GEMM_BF16_STORE_MIX + d->epilogue, dim3(n < g->cus ? n : g->cus),
                         dim3(threads), a, 1))
            return 0;
        auto &r = g->route[g->route_n - 1];
        r.h1 = a.mix_h1, r.rows1 = a.mix_rows1, r.h2 = a.mix_h2, r.rows2 = a.mix_rows2;
        return 1;
    }
    if (a.split == 1 && grid > g->cus && g->cus % 8 == 0) {
        grid = g->cus;
        /* a last wave of at most half the CUs' tiles runs as twice as many
         * half tiles (bf16 W kernels): up projection at M = 8704, 96 tail
         * tiles of 1632, 577-580 us against 511 us for the 1536 tiles of
         * M = 8192 */
        const uint32_t R = tiles % g->cus;
        if (R && 2 * R <= g->cus && !(int8 && !widen)) {
            a.half_from = tiles - R;
            a.half_count = 2 * R;
        }
    }
    return launch_step(g, kid, dim3(grid), dim3(threads), a, a.split, a.half_count);
}

static int check_epilogue(h3_gpu *g, const qw_linear_desc *d) {
    if (d && (d->epilogue < QW_LINEAR_STORE || d->epilogue > QW_LINEAR_QKNORM))
        return fail(g, "linear: unknown epilogue %d", d->epilogue);
    return 1;
}

extern "C" int qw_gpu_linear(h3_gpu *g, const qw_linear_desc *d) {
    return check_epilogue(g, d) ? linear_impl(g, d, 0) : 0;
}

/* Where the fused epilogue does not run (a RoPE table of fewer than 128
 * rows), the k and v thirds are copied out of the projection. */
extern "C" int qw_gpu_copy_rows(h3_gpu *g, h3_gpu_tensor *dst, size_t doff, uint32_t dstride,
                                const h3_gpu_tensor *src, size_t soff, uint32_t sstride,
                                uint32_t rows, uint32_t row_elems);
extern "C" int qw_gpu_qkv_linear(h3_gpu *g, const qw_linear_desc *d, h3_gpu_tensor *k,
                                 h3_gpu_tensor *v, size_t kv_offset) {
    if (!g || !d) return 0;
    if (d->epilogue != QW_LINEAR_QKNORM) return fail(g, "qkv_linear: epilogue must be QKNORM");
    REQ_DT(k, H3_GPU_BF16, "qkv_linear k");
    REQ_DT(v, H3_GPU_BF16, "qkv_linear v");
    const uint32_t H = d->cols / 3;
    const size_t n = (size_t)d->rows * H;
    if (!fits(k, kv_offset, n) || !fits(v, kv_offset, n))
        return fail(g, "qkv_linear: k or v too small");
    if (d->rows == 0 || d->cols == 0) return 1;
    /* The epilogue stores k and v 16 bytes at a time, in workgroups that run
     * in any order beside those that read in and write out; the copies below
     * would take less, but what is accepted does not depend on the table. */
    const uintptr_t kp = (uintptr_t)k->ptr + kv_offset * 2, vp = (uintptr_t)v->ptr + kv_offset * 2;
    if ((kp | vp) % 16) return fail(g, "qkv_linear: k and v must be 16-byte aligned");
    auto clear_of = [&](uintptr_t p, const h3_gpu_tensor *t, size_t off, size_t elements) {
        return !t || apart((const void *)p, n * 2, t->ptr + off * 2, elements * 2);
    };
    const size_t in_n = (size_t)(d->rows - 1) * d->lda + d->k;
    const size_t out_n = (size_t)(d->rows - 1) * d->ldc + d->cols;
    for (uintptr_t p : {kp, vp})
        if (!clear_of(p, d->in, d->in_offset, in_n) || !clear_of(p, d->out, d->out_offset, out_n))
            return fail(g, "qkv_linear: k or v overlaps the input or the output");
    if (!clear_of(kp, v, kv_offset, n)) return fail(g, "qkv_linear: k and v overlap");
    if (d->rope_rows < 128 || n * 2 >= (1ull << 31))
        return linear_impl(g, d, 0) &&
               qw_gpu_copy_rows(g, k, kv_offset, H, d->out, H, d->ldc, d->rows, H) &&
               qw_gpu_copy_rows(g, v, kv_offset, H, d->out, 2 * (size_t)H, d->ldc, d->rows, H);
    const kv_out kv = {(uint16_t *)k->ptr + kv_offset, (uint16_t *)v->ptr + kv_offset, H, n * 2};
    return linear_impl(g, d, 0, &kv);
}

/* The tile kernels from 9 rows on, and for an output that the separate pass
 * cannot write (strided, or at an offset); else at most 8 rows keep the
 * streaming linear and that pass, in the runtime's scratch buffer. */
static void *scratch(h3_gpu *g, size_t bytes);
extern "C" int qw_gpu_linear_swiglu(h3_gpu *g, const qw_linear_desc *d) {
    if (!g || !d) return 0;
    if (!check_epilogue(g, d)) return 0;
    if (d->epilogue != QW_LINEAR_STORE) return fail(g, "linear_swiglu: epilogue must be STORE");
    if (d->rows && d->in && d->out && d->in->dtype == H3_GPU_BF16 && d->out->dtype == H3_GPU_BF16 &&
        !apart(d->in->ptr + d->in_offset * 2, ((size_t)(d->rows - 1) * d->lda + d->k) * 2,
               d->out->ptr + d->out_offset * 2, ((size_t)(d->rows - 1) * d->ldc + d->cols / 2) * 2))
        return fail(g, "linear_swiglu: the output overlaps the input");
    qw_linear_desc t = *d;
    if (d->rows > 8 || d->cols % 16 || d->ldc != d->cols / 2 || d->out_offset) {
        t.epilogue = QW_EPI_SWIGLU;
        return linear_impl(g, &t, 0);
    }
    if (!d->rows || !d->cols) return 1;
    const size_t wide = (size_t)d->rows * d->cols;
    void *s = scratch(g, wide * 2);
    if (!s) return fail(g, "linear_swiglu: scratch allocation failed");
    h3_gpu_tensor tw = {g, (unsigned char *)s, wide, H3_GPU_BF16, 0};
    t.out = &tw;
    t.ldc = d->cols;
    return linear_impl(g, &t, 0) && qw_gpu_swiglu_bf16(g, d->out, &tw, d->rows, d->cols / 2);
}

extern "C" int qw_gpu_linear_static(h3_gpu *g, const qw_linear_desc *d) {
    if (!g) return 0;
    if (!g->static_scratch) return fail(g, "linear_static: no static workspace");
    if (!check_epilogue(g, d)) return 0;
    /* every context on this device shares the workspace: this call's
     * kernels wait for the last call that used it, from any stream */
    hipError_t e = (hipError_t)qw_static_scratch_acquire(g->device, g->stream);
    if (e != hipSuccess) return fail(g, "linear_static: ordering: %s", hipGetErrorString(e));
    const int ok = linear_impl(g, d, 1);
    e = (hipError_t)qw_static_scratch_release(g->device, g->stream);
    if (e != hipSuccess) return fail(g, "linear_static: ordering: %s", hipGetErrorString(e));
    return ok;
}

static qw_linear_desc plain_linear(h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                   const h3_gpu_tensor *w, const h3_gpu_tensor *bias,
                                   uint32_t rows, uint32_t k, uint32_t n) {
    qw_linear_desc d;
    memset(&d, 0, sizeof(d));
    d.out = out;
    d.ldc = n;
    d.in = in;
    d.lda = k;
    d.weight = w;
    d.bias = bias;
    d.rows = rows;
    d.k = k;
    d.cols = n;
    d.epilogue = QW_LINEAR_STORE;
    return d;
}

extern "C" int h3_gpu_linear_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                                  const h3_gpu_tensor *w, const h3_gpu_tensor *bias,
                                  uint32_t rows, uint32_t k, uint32_t n) {
    if (!w || w->dtype != H3_GPU_BF16) return fail(g, "linear_bf16: weight must be bf16");
    qw_linear_desc d = plain_linear(out, in, w, bias, rows, k, n);
    return qw_gpu_linear(g, &d);
}

extern "C" int qw_gpu_qkv_bf16(h3_gpu *g, h3_gpu_tensor *qo, h3_gpu_tensor *ko,
                               h3_gpu_tensor *vo, const h3_gpu_tensor *in,
                               const h3_gpu_tensor *wq, const h3_gpu_tensor *wk,
                               const h3_gpu_tensor *wv, uint32_t rows, uint32_t dim) {
    return h3_gpu_linear_bf16(g, qo, in, wq, NULL, rows, dim, dim) &&
           h3_gpu_linear_bf16(g, ko, in, wk, NULL, rows, dim, dim) &&
           h3_gpu_linear_bf16(g, vo, in, wv, NULL, rows, dim, dim);
}

static void *scratch(h3_gpu *g, size_t bytes) {
    if (g->scratch_bytes >= bytes) return g->scratch;
    hipStreamSynchronize(g->stream);
    if (g->scratch) hipFree(g->scratch);
    g->scratch = NULL;
    g->scratch_bytes = 0;
    if (hipMalloc(&g->scratch, bytes) != hipSuccess) return NULL;
    g->scratch_bytes = bytes;
    g->stats.allocated_bytes += bytes;
    return g->scratch;
}

extern "C" int h3_gpu_mlp_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in,
                               const h3_gpu_tensor *fc1, const h3_gpu_tensor *fc2,
                               uint32_t rows, uint32_t in_dim, uint32_t hidden,
                               uint32_t out_dim) {
    size_t wide = (size_t)rows * hidden * 2, act_n = (size_t)rows * hidden;
    if (rows > 8 && hidden % 8 == 0) { /* one launch for fc1 and the activation */
        unsigned char *s = (unsigned char *)scratch(g, act_n * 2);
        if (!s) return fail(g, "mlp: scratch allocation failed");
        if (!fc1 || fc1->dtype != H3_GPU_BF16) return fail(g, "linear_bf16: weight must be bf16");
        h3_gpu_tensor ta = {g, s, act_n, H3_GPU_BF16, 0};
        qw_linear_desc d = plain_linear(&ta, in, fc1, NULL, rows, in_dim, 2 * hidden);
        d.ldc = hidden;
        return qw_gpu_linear_swiglu(g, &d) &&
               h3_gpu_linear_bf16(g, out, &ta, fc2, NULL, rows, hidden, out_dim);
    }
    unsigned char *s = (unsigned char *)scratch(g, (wide + act_n) * 2 + 512);
    if (!s) return fail(g, "mlp: scratch allocation failed");
    h3_gpu_tensor tw = {g, s, wide, H3_GPU_BF16, 0};
    h3_gpu_tensor ta = {g, s + ((wide * 2 + 255) & ~(size_t)255), act_n, H3_GPU_BF16, 0};
    return h3_gpu_linear_bf16(g, &tw, in, fc1, NULL, rows, in_dim, 2 * hidden) &&
           qw_gpu_swiglu_bf16(g, &ta, &tw, rows, hidden) &&
           h3_gpu_linear_bf16(g, out, &ta, fc2, NULL, rows, hidden, out_dim);
}

/* ---- attention ----------------------------------------------------------- */

/* How an attention launch fills the CUs. A block of 256 queries takes its
 * CU 1.9 us a tile of 64 keys in full rounds (two waves per SIMD; 1.75 where
 * part of the chip idles), a block of 128 queries 1.32 us alone on a CU and
 * 2 us beside another; blocks that see few keys (text rows) fill in between.
 * Rounds of blocks that leave a last one partly filled (or do not fill the
 * first) are cut along the keys instead: the blocks past the full rounds
 * (`dp`) in `split` pieces, each a share of the key tiles, that meet in
 * memory (7 us, 1 to 1.5 more a piece, and the partials at 5 TB/s). 1 x 32
 * heads x 4119 rows (544 blocks, 2.1 rounds) 344 -> 278 us; 24 heads, 4096
 * queries of 8512 keys (1.5 rounds) 421 -> 369; 465 of 3323 71 -> 39. */
#define QW_ATTN_PART(waves) ((size_t)(waves) * (16 * 1024 + 512)) /* bytes of a piece's partial */
struct attn_plan {
    int small; /* 128-query blocks */
    uint32_t dp, split;
};
static attn_plan plan_attention(const h3_gpu *g, const qw_attention_desc *d) {
    const uint32_t C = g->cus, pairs = d->heads * d->batch, T = (d->kv_rows + 63) / 64;
    /* blocks of qb queries, and those of a (batch, head) pair that see few
     * keys: the leading ones, all text */
    auto blocks = [&](uint32_t qb) { return (d->q_rows + qb - 1) / qb; };
    auto light = [&](uint32_t qb) {
        return d->kv_limit || 2 * d->text_rows > d->kv_rows ? 0u : d->text_rows / qb;
    };
    const uint64_t nb8 = (uint64_t)blocks(256) * pairs;
    if (nb8 >= C) {
        const uint32_t per = blocks(256) - light(256);
        const uint64_t heavy = (uint64_t)per * pairs, full = heavy / C, R = heavy % C;
        attn_plan p = {0, 0, 1};
        if (!R) return p;
        /* whole blocks: the rounds and the partly filled one */
        double best = 0.97 * 1.75 * T * (full + 1);
        for (uint32_t s = 2; s <= 8 && T >= 4 * s; s++) {
            const double t = 1.9 * (T * full + (R * s + C - 1) / C * ((T + s - 1) / s)) + 7.0 +
                             1.5 * s + R * s * QW_ATTN_PART(8) * 2 / 5e6;
            if (t < best) {
                best = t;
                p.split = s;
            }
        }
        /* the first block past `full` rounds of heavy ones; pairs are walked
         * in order, light blocks first */
        const uint64_t h = full * C;
        p.dp = (uint32_t)(h / per * blocks(256) + (h % per ? light(256) + h % per : 0));
        return p;
    }
    const uint32_t heavy = (blocks(128) - light(128)) * pairs;
    auto us = [&](uint32_t s) { /* time of the launch in s pieces a block */
        const uint64_t n = (uint64_t)heavy * s;
        return (double)((n + 2 * C - 1) / (2 * C)) * ((T + s - 1) / s) * (n <= C ? 1.32 : 2.0) +
               (s > 1 ? 7.0 + s + n * QW_ATTN_PART(4) / 5e6 : 3.0);
    };
    attn_plan p = {1, 0, 1};
    double best = 0.95 * us(1);
    for (uint32_t s = 2; s <= 8 && T >= 2 * s; s++)
        if (us(s) < best) {
            best = us(s);
            p.split = s;
        }
    return p;
}

extern "C" int qw_gpu_attention_bf16(h3_gpu *g, const qw_attention_desc *d) {
    if (!g || !d) return 0;
    REQ_DT(d->out, H3_GPU_BF16, "attention out");
    REQ_DT(d->q, H3_GPU_BF16, "attention q");
    REQ_DT(d->k, H3_GPU_BF16, "attention k");
    REQ_DT(d->v, H3_GPU_BF16, "attention v");
    if (!d->batch || !d->q_rows || !d->heads) return 1;
    if (!d->kv_rows) return fail(g, "attention: no keys");
    const uint32_t hd = d->heads * 128;
    if (d->ldq < hd || d->ldk < hd || d->ldv < hd || d->ldo < hd)
        return fail(g, "attention: row strides smaller than heads * 128");
    if (d->ldq % 8 || d->ldk % 8 || d->ldv % 8 || d->ldo % 4 || d->q_offset % 8 ||
        d->k_offset % 8 || d->v_offset % 8 || d->out_offset % 4)
        return fail(g, "attention: rows must be 16-byte aligned");
    size_t qr = (size_t)d->batch * d->q_rows, kr = (size_t)d->batch * d->kv_rows;
    if (!fits(d->q, d->q_offset, (qr - 1) * d->ldq + hd) ||
        !fits(d->k, d->k_offset, (kr - 1) * d->ldk + hd) ||
        !fits(d->v, d->v_offset, (kr - 1) * d->ldv + hd) ||
        !fits(d->out, d->out_offset, (qr - 1) * d->ldo + hd))
        return fail(g, "attention: tensor too small");
    if (d->kv_limit) {
        REQ_DT(d->kv_limit, H3_GPU_U32, "attention kv_limit");
        if (!fits(d->kv_limit, 0, d->q_rows)) return fail(g, "attention: kv_limit too small");
    }
    if (!d->kv_limit && d->text_rows > d->q_rows)
        return fail(g, "attention: text_rows > q_rows");
    qw_attn_args a;
    a.out = (uint16_t *)d->out->ptr + d->out_offset;
    a.q = (const uint16_t *)d->q->ptr + d->q_offset;
    a.k = (const uint16_t *)d->k->ptr + d->k_offset;
    a.v = (const uint16_t *)d->v->ptr + d->v_offset;
    a.kv_limit = d->kv_limit ? (const uint32_t *)d->kv_limit->ptr : NULL;
    a.q_rows = d->q_rows;
    a.kv_rows = d->kv_rows;
    a.heads = d->heads;
    a.batch = d->batch;
    a.ldq = d->ldq;
    a.ldk = d->ldk;
    a.ldv = d->ldv;
    a.ldo = d->ldo;
    a.text_rows = d->text_rows;
    a.text_causal = d->text_causal;
    a.scale = d->scale;
    a.scale_log2 = d->scale * 1.4426950408889634f;
    g->stats.mps_sdpa_dispatches += 0;
    if (((uint64_t)(d->kv_rows - 1) * std::max(d->ldk, d->ldv) + hd) * 2 >= (1ull << 31))
        return fail(g, "attention: one batch entry's K/V exceed 2 GiB");
    a.dp_blocks = 0;
    a.split = 1;
    a.part = NULL;
    a.flag = NULL;
    const uint32_t aqb = g->attn_threads / 2; /* 32 query rows per 64-lane wave */
    const uint64_t nwg = (uint64_t)((d->q_rows + aqb - 1) / aqb) * d->heads * d->batch;
    if (nwg >= (1ull << 31)) return fail(g, "attention: grid too large");
    const attn_plan p = plan_attention(g, d);
    g->route_n = 0;
    /* the launch's own kernel: a small plan keeps its pieces on either */
    const int w4 = p.small && g->attn_small;
    const uint32_t threads = w4 ? g->attn4_threads : g->attn_threads, qb = threads / 2;
    const uint32_t nb = (d->q_rows + qb - 1) / qb * d->heads * d->batch;
    const uint64_t R = nb - p.dp, np = R * p.split;
    /* whole blocks where the pieces would not fit the workspace (a counter
     * a block, a partial a piece) or there is none to be had */
    if (p.split == 1 || R > (uint64_t)QW_FLAGS * g->cus ||
        np * QW_ATTN_PART(threads / 64) > (size_t)QW_SPLIT_MAX_PIECES * g->cus * 256 * 256 * 4 ||
        !split_workspace(g))
        return launch_step(g, w4 ? K_ATTN_W4 : K_ATTN, dim3(nb), dim3(threads), a, 1);
    a.dp_blocks = p.dp;
    a.split = p.split;
    a.part = g->sk_part;
    a.flag = g->sk_flag;
    return launch_step(g, w4 ? K_ATTN_W4_SPLIT : K_ATTN_SPLIT, dim3((uint32_t)(p.dp + np)),
                       dim3(threads), a, p.split, 0, p.dp);
}

static int sdpa_contig(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                       const h3_gpu_tensor *k, const h3_gpu_tensor *v,
                       const h3_gpu_tensor *limit, uint32_t q_rows, uint32_t kv_rows,
                       uint32_t heads, uint32_t head_dim, float scale, uint32_t text_rows,
                       int causal) {
    if (head_dim != 128) return fail(g, "sdpa: head_dim must be 128");
    qw_attention_desc d;
    memset(&d, 0, sizeof(d));
    d.out = out;
    d.q = q;
    d.k = k;
    d.v = v;
    d.ldo = d.ldq = d.ldk = d.ldv = heads * 128;
    d.kv_limit = limit;
    d.batch = 1;
    d.q_rows = q_rows;
    d.kv_rows = kv_rows;
    d.heads = heads;
    d.text_rows = text_rows;
    d.text_causal = causal;
    d.scale = scale;
    return qw_gpu_attention_bf16(g, &d);
}

extern "C" int qw_gpu_flash_sdpa_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                                      const h3_gpu_tensor *k, const h3_gpu_tensor *v,
                                      uint32_t q_rows, uint32_t kv_rows, uint32_t heads,
                                      uint32_t head_dim, float scale) {
    return sdpa_contig(g, out, q, k, v, NULL, q_rows, kv_rows, heads, head_dim, scale, 0, 0);
}

extern "C" int qw_gpu_sdpa_rect_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                                     const h3_gpu_tensor *k, const h3_gpu_tensor *v,
                                     uint32_t q_rows, uint32_t kv_rows, uint32_t heads,
                                     uint32_t head_dim, float scale) {
    return sdpa_contig(g, out, q, k, v, NULL, q_rows, kv_rows, heads, head_dim, scale, 0, 0);
}

extern "C" int qw_gpu_flash_sdpa_prefix_bf16(h3_gpu *g, h3_gpu_tensor *out,
                                             const h3_gpu_tensor *q, const h3_gpu_tensor *k,
                                             const h3_gpu_tensor *v,
                                             const h3_gpu_tensor *kv_limit, uint32_t q_rows,
                                             uint32_t kv_rows, uint32_t heads, uint32_t kv_heads,
                                             uint32_t head_dim, float scale) {
    if (kv_heads != heads) return fail(g, "sdpa_prefix: grouped K/V heads not supported");
    if (!kv_limit) return fail(g, "sdpa_prefix: kv_limit required");
    return sdpa_contig(g, out, q, k, v, kv_limit, q_rows, kv_rows, heads, head_dim, scale, 0, 0);
}

extern "C" int h3_gpu_gqa_causal_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *q,
                                      const h3_gpu_tensor *k, const h3_gpu_tensor *v,
                                      uint32_t seq, uint32_t qh, uint32_t kvh, uint32_t head_dim,
                                      float scale) {
    if (kvh != qh) return fail(g, "gqa_causal: grouped K/V heads not supported");
    return sdpa_contig(g, out, q, k, v, NULL, seq, seq, qh, head_dim, scale, seq, 1);
}
