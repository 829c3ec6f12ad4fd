/* What the library asks of the HIP runtime, written down: this program stands in for the runtime's calls (memory is the
 * host's, nothing runs) and makes calls of the C ABI.  One line a launch, event or pinned allocation; "+ event" where the
 * event rides on the launch.  Compiled and run by test_library_cpu.py. */
#include <hip/hip_runtime_api.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../include/deep_ep_hip.h"

static int capturing;

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { (void)e; return "error"; }
hipError_t hipMalloc(void** p, size_t n) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    printf("pinned%s%s\n", flags & hipHostMallocMapped ? " mapped" : "", flags & hipHostMallocCoherent ? " coherent" : "");
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned flags) { (void)flags; *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = calloc(1, 4 << 20); return hipSuccess; }
hipError_t hipModuleLoad(hipModule_t* m, const char* path) { (void)path; *m = (hipModule_t)1; return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t m, const char* name) {
    (void)m;
    *f = (hipFunction_t)strcpy(malloc(strlen(name) + 1), name);
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz,
                                 unsigned smem, hipStream_t stream, void** params, void** extra) {
    (void)gx, (void)gy, (void)gz, (void)bx, (void)by, (void)bz, (void)smem, (void)params, (void)extra;
    printf("%s on %d\n", (const char*)f, (int)(size_t)stream);
    return hipSuccess;
}
hipError_t hipExtModuleLaunchKernel(hipFunction_t f, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, uint32_t by, uint32_t bz,
                                    size_t smem, hipStream_t stream, void** params, void** extra, hipEvent_t start, hipEvent_t stop,
                                    uint32_t flags) {
    (void)gx, (void)gy, (void)gz, (void)bx, (void)by, (void)bz, (void)smem, (void)params, (void)extra, (void)start, (void)flags;
    printf("%s on %d%s\n", (const char*)f, (int)(size_t)stream, stop != NULL ? " + event" : "");
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t stream) {
    (void)e;
    printf("event on %d\n", (int)(size_t)stream);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status) {
    (void)s;
    *status = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}

static ep_tensor_t tensor(int dtype, int ndim, int64_t n0, int64_t n1) {
    static char storage[64];                       /* (looked at by nobody) */
    const ep_tensor_t t = {storage, dtype, ndim, {n0, ndim == 2 ? n1 : 0}, {ndim == 2 ? n1 : 1, ndim == 2 ? 1 : 0}};
    return t;
}

static void said(const char* what, int rc) {
    if (rc != 0) printf("%s refused: %s\n", what, ep_last_error());
}

enum { K = 4, E = 32, A = 8 };
static int64_t H = 256;

static ep_dispatch_args_t dispatch_args(int T, int R) {
    ep_dispatch_args_t a;
    memset(&a, 0, sizeof a);
    a.x = tensor(EP_DTYPE_BF16, 2, T, H);
    a.topk_idx = tensor(EP_DTYPE_I64, 2, T, K);
    a.psum_num_recv_tokens_per_rank = tensor(EP_DTYPE_I32, 1, R, 0);
    a.psum_num_recv_tokens_per_expert = a.num_unaligned_recv_tokens_per_expert = tensor(EP_DTYPE_I32, 1, E / R, 0);
    a.dst_buffer_slot_idx = a.dst_gsge_idx = tensor(EP_DTYPE_I32, 2, T, K);
    a.num_max_tokens_per_rank = T;
    a.num_experts = E;
    a.expert_alignment = A;
    a.stream = (void*)1;
    return a;
}

static ep_dispatch_epilogue_args_t epilogue_args(int T, int R, ep_buffer_t* b) {
    ep_dispatch_epilogue_args_t e;
    memset(&e, 0, sizeof e);
    e.x = tensor(EP_DTYPE_BF16, 2, T, H);
    e.psum_num_recv_tokens_per_rank = tensor(EP_DTYPE_I32, 1, R, 0);
    e.psum_num_recv_tokens_per_expert = tensor(EP_DTYPE_I32, 1, E / R, 0);
    e.recv_x = tensor(EP_DTYPE_BF16, 2, (int64_t)R * T * K, H);
    e.recv_src_metadata = tensor(EP_DTYPE_I32, 2, (int64_t)R * T, K + 2);
    e.num_topk = K;
    e.num_max_tokens_per_rank = T;
    e.num_experts = E;
    e.expert_alignment = A;
    e.do_zero_padding = 1;
    e.stream = (void*)2;
    e.dispatch_stamp = ep_dispatch_stamp(b);
    return e;
}

/* event T R alone|node|mapped [capture]: a dispatch and an owner-side reduce of partition 0, each with an event behind it */
static void event_behind_calls(int T, int R, const char* form) {
    ep_buffer_t* b[4];
    const int64_t bytes = ep_calculate_buffer_size(R, T, H, K, 0);
    const int n = strcmp(form, "node") == 0 ? R : 1;
    for (int i = 0; i < n; ++i) said("create", ep_buffer_create(i, R, bytes, 0, 1, 1, &b[i]));
    if (strcmp(form, "node") == 0) said("connect", ep_buffer_connect(b, R));
    if (strcmp(form, "mapped") == 0) {
        void* arenas[4];
        for (int i = 0; i < R; ++i) arenas[i] = ep_buffer_region(b[0], 0, NULL);
        said("set_peers", ep_buffer_set_peers(b[0], arenas, R));
    }
    ep_dispatch_args_t a = dispatch_args(T, R);
    ep_combine_args_t c;
    memset(&c, 0, sizeof c);
    c.x = tensor(EP_DTYPE_BF16, 2, (int64_t)R * T * K, H);
    c.src_metadata = tensor(EP_DTYPE_I32, 2, (int64_t)R * T, K + 2);
    c.combined_topk_idx = a.topk_idx;
    c.psum_num_recv_tokens_per_rank = a.psum_num_recv_tokens_per_rank;
    c.num_experts = E;
    c.num_max_tokens_per_rank = T;
    c.stream = (void*)1;
    for (int i = 0; i < n; ++i) said("dispatch", ep_dispatch_launch_event(b[i], &a, (void*)7));
    for (int i = 0; i < n; ++i) {
        ep_dispatch_recv_args_t r;
        memset(&r, 0, sizeof r);
        r.psum_num_recv_tokens_per_rank = a.psum_num_recv_tokens_per_rank;
        r.psum_num_recv_tokens_per_expert = r.num_unaligned_recv_tokens_per_expert = a.psum_num_recv_tokens_per_expert;
        r.recv_src_metadata = c.src_metadata;
        r.hidden_bytes = 2 * H;
        r.num_topk = K;
        r.num_max_tokens_per_rank = T;
        r.num_experts = E;
        r.expert_alignment = A;
        r.stream = (void*)2;
        r.dispatch_stamp = ep_dispatch_stamp(b[i]);
        said("receive", ep_dispatch_recv_launch(b[i], &r));
        ep_dispatch_epilogue_args_t e = epilogue_args(T, R, b[i]);
        said("epilogue", ep_dispatch_epilogue_launch(b[i], &e));
    }
    printf("combine\n");
    for (int i = 0; i < n; ++i) said("combine", ep_combine_begin_event(b[i], &c, (void*)7));
}

/* begin T next|only [H]: a dispatch of one partition on stream 1 and its copy epilogue on stream 2 */
static void begin_and_epilogue(int T, const char* form) {
    ep_buffer_t* b;
    said("create", ep_buffer_create(0, 1, ep_calculate_buffer_size(1, T, H, K, 0), 0, 1, 1, &b));
    ep_dispatch_args_t a = dispatch_args(T, 1);
    said("begin", strcmp(form, "only") == 0 ? ep_dispatch_begin_only(b, &a) : ep_dispatch_begin(b, &a));
    ep_dispatch_epilogue_args_t e = epilogue_args(T, 1, b);
    said("epilogue", ep_dispatch_epilogue_launch(b, &e));
}

int main(int argc, char** argv) {
    const int T = argc > 2 ? atoi(argv[2]) : 0, R = argc > 3 ? atoi(argv[3]) : 1;
    if (ep_init(NULL) != 0) {
        said("init", 1);
        return 1;
    }
    if (argc > 4 && strcmp(argv[1], "event") == 0) capturing = argc > 5, event_behind_calls(T, R, argv[4]);
    if (argc > 4 && strcmp(argv[1], "begin") == 0) H = atoi(argv[4]);
    if (argc > 3 && strcmp(argv[1], "begin") == 0) begin_and_epilogue(T, argv[3]);
    fflush(stdout);
    return 0;
}
