// Host runtime behind the C ABI of include/deep_ep_hip.h: argument contracts, the pooled arena,
// the mapped count page and the launches of the ahead-of-time built gfx950 kernels through
// hipModuleLaunchKernel.  It stands where the reference has csrc/buffers/ep.hpp (host class),
// csrc/kernels/ep/*.hpp (launchers) and csrc/runtime/jit.hpp (run-time compiler).
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <dlfcn.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/deep_ep_hip.h"
#include "ep_args.h"
#include "ep_fp8.h"

void ep_static_scratch_init();      // looks up this device's copy of the static scratch (end of this file)

namespace {

constexpr int64_t kAllocAlign = 2097152;       // reference: common/compiled.hpp:48
constexpr int kUbAlign = 32;                   // reference: common/compiled.hpp:39
constexpr int64_t kWorkspaceBytes = 16 * 1024 * 1024;

thread_local std::string g_err;

struct EpError {
    std::string msg;
};

std::string format(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    return buf;
}

#define EP_HOST_ASSERT(cond)                                                                        \
    do {                                                                                            \
        if (!(cond)) throw EpError{format("Assertion exception (%s:%d): %s", __FILE_NAME__, __LINE__, #cond)}; \
    } while (0)

#define EP_HOST_UNREACHABLE(reason) \
    throw EpError { format("Assertion exception (%s:%d): %s", __FILE_NAME__, __LINE__, reason) }

#define HIP_CHECK(cmd)                                                                              \
    do {                                                                                            \
        const hipError_t e_ = (cmd);                                                                \
        if (e_ != hipSuccess)                                                                       \
            throw EpError{format("HIP runtime exception (%s:%d): Error code: %d, detail: %s", __FILE_NAME__, \
                                 __LINE__, (int)e_, hipGetErrorString(e_))};                        \
    } while (0)

template <class F>
int guarded(F&& f) {
    try {
        f();
        return 0;
    } catch (const EpError& e) {
        g_err = e.msg;
        return 1;
    } catch (const std::exception& e) {
        g_err = e.what();
        return 1;
    }
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t align_up(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

// ---- token layout (reference: layout/ep/token.hpp:9-83) -------------------------------------
int64_t token_bytes(int hidden_bytes, int sf_bytes, int topk, bool with_metadata) {
    int64_t meta = (int64_t)topk * 4 + (with_metadata ? align_up((int64_t)topk * 8, kUbAlign) + 4 : 0);
    int64_t n = hidden_bytes;
    if (sf_bytes > 0) n += align_up(sf_bytes, kUbAlign);
    return n + align_up(meta, kUbAlign);
}

// Byte offsets inside a packed token (reference: layout/ep/token.hpp:59-82).
struct PackedToken {
    int64_t bytes;
    int sf_off, idx_off, w_off, src_off;
};

PackedToken packed_token(int hidden_bytes, int sf_bytes, int topk, bool with_metadata) {
    PackedToken p{};
    p.bytes = token_bytes(hidden_bytes, sf_bytes, topk, with_metadata);
    p.sf_off = (int)align_up(hidden_bytes, kUbAlign);
    p.idx_off = sf_bytes > 0 ? p.sf_off + (int)align_up(sf_bytes, kUbAlign) : hidden_bytes;
    p.w_off = p.idx_off + (with_metadata ? (int)align_up((int64_t)topk * 8, kUbAlign) : 0);
    p.src_off = p.w_off + topk * 4;
    return p;
}

int64_t dispatch_buffer_size(int max_tokens, int hidden, int sf_packs, int topk, int elem, int ranks) {
    return (int64_t)ranks * max_tokens * token_bytes(hidden * elem, sf_packs * 2, topk, true);
}

int64_t combine_buffer_size(int ranks, int max_tokens, int hidden, int topk) {
    return (int64_t)std::min(topk, ranks) * max_tokens * token_bytes(hidden * 2, 0, topk, false);
}

// ---- code object ------------------------------------------------------------------------------
struct Kernels {
    hipModule_t module = nullptr;
    hipFunction_t layout_count, layout_scan, layout_place, layout_assign[2][3];      // [sums the counts itself][EP_LAYOUT_SIDE_*]
    hipFunction_t scatter_copy, scatter_quant, scatter_quant_sw, sf_transpose;
    hipFunction_t scatter_copy_pack, scatter_quant_pack, scatter_quant_sw_pack;
    hipFunction_t small[2][3];       // [packs][copy, quant, quant_sw]
    hipFunction_t chunk[2][3];
    hipFunction_t layout_count_bits, layout_assign_bits;        // one partition, up to top-8: instead of layout_count and layout_assign
    hipFunction_t recv_copy;
    hipFunction_t combine[3][8];     // [mode][generic, k2 .. k8]
    hipFunction_t fp8_selftest, quant_rows;
    int device = -1;
};

std::mutex g_mutex;
Kernels g_k;
std::atomic<bool> g_fp8_hw{true};
// Workgroups of the single-partition combine kernel a CU holds at once, enforced through an unused dynamic LDS
// allocation (0: no cap, the registers decide: 5 to 8; negative: chosen by top-k, below).  The gather is fastest
// with about 150 KiB of row fetches in flight a CU (a wave fetches top-k x 2 KiB): more waves queue more fetches
// than the memory keeps open.  Measured at 16384 tokens x 7168 (microseconds at 2/3/4/5 workgroups and uncapped):
//   top-2  175 140 126 120 120      top-4  233 201 194 199 200
//   top-6  297 272 286 289 291      top-8  385 354 377 378 376
// and for the kernel that takes any top-k, which launches of this size take for top-1 and from top-9 on: top-1 best uncapped, with two
// biases (three rows) at 6, from top-9 to top-16 at 4.
// A bias row is one more row a wave fetches: top-6 with one / two biases 326 311 329 336 / 358 350 373 377 at 2/3/4/5.
// The two-phase kernels of the partitioned path do not react to it.
std::atomic<int> g_combine_blocks_per_cu{-1};
constexpr unsigned kLdsBytesPerCu = 160 * 1024;
// The unrolled kernels of odd top-k at 3/4/5/6 and uncapped: top-3 - 158 153 153 153, top-5 233 234 241 244 -, at 8192 tokens 123 119 120 122 -;
// top-7 314 329 335 - -, of 2560 channels at 8192 tokens 62.1 60.6 60.8 - -.  With one / two biases at 2/3/4/5/6 and uncapped, 16384 tokens: top-3 235 198
// 188 191 195 196 / 260 228 229 235 239 240; top-5 287 268 277 284 288 288 / 316 309 323 331 331 334; top-7 357 354 372 377 377 379 / 388 399 415 421 420
// 419 (the kernel for any top-k, at 4: 190 / 226, 272 / 308, 350 / 394); of 2560 channels top-7 137 127 128 130 131 130 / 149 140 142 145 145 145 (137 / 146).
unsigned combine_lds_cap(int num_topk, bool specialised, bool odd, int num_row_blocks, int hidden) {     // num_topk: rows a wave fetches, biases included
    int n = g_combine_blocks_per_cu;
    if (n < 0) {
        // a launch that fills the machine less than about twice over wants every wave it can get
        // (1024 tokens, top-6: 23.8 us uncapped, 25.4 at four workgroups; from 4096 tokens on the cap costs nothing),
        // and so do short rows (hidden 512 / 1536, top-8: 113 / 160 us uncapped, 124 / 170 at three; from 2048 on the
        // cap wins)
        if (num_row_blocks < 4096 or hidden < 2048) n = 0;
        else if (specialised and odd) n = num_topk <= 3 ? 6 : num_topk <= 5 or hidden < 4096 ? 4 : 3;
        else if (specialised) n = num_topk <= 2 ? 0 : num_topk <= 4 ? 4 : 3;
        else n = num_topk <= 2 ? 0 : num_topk == 3 ? 6 : 4;
    }
    // a workgroup can ask for 64 KiB at most, which lets two of them into a CU: a cap of one cannot be enforced this
    // way (it is served as two), and from 160 workgroups on a share of the LDS is too small to mean anything (no cap)
    if (n <= 0) return 0;
    const unsigned share = kLdsBytesPerCu / (unsigned)n;
    if (share <= 1024u) return 0;
    return std::min(64u * 1024u, share - 1024u);       // n of them fit a CU, n + 1 do not
}
// From here on the top-8 kernels send their first row's fetches ahead of the others.  Replayed combines of 7168 channels, us
// first row ahead / all at once: 32 tokens (56 row blocks) 5.3 / 5.1, 64 6.2 / 5.9, 128 7.0 / 6.7, 256 9.3 / 9.2, 1024 25.4 / 25.2,
// 2048 (3584 row blocks) 47.6 / 47.5, 4096 91.0 / 90.8, 6144 (10752) 136.5 / 137.1, 8192 181.7 / 183.3, 16384 354 / 362.
constexpr int kPacedRowBlocks = 8192;
std::atomic<int> g_recount_limit{-1};     // blocks x top-k up to which one partition's slot assignment counts all ids itself; negative: recount_pays
std::atomic<int> g_fold_max_blocks{256};    // up to this many layout workgroups the slot assignment sums the block counts itself

std::string library_dir() {
    Dl_info info;
    if (dladdr((void*)&library_dir, &info) == 0 || info.dli_fname == nullptr) return ".";
    std::string p = info.dli_fname;
    const auto pos = p.find_last_of('/');
    return pos == std::string::npos ? "." : p.substr(0, pos);
}

void load_kernels(const char* dir) {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_k.module != nullptr) return;
    const std::string path = (dir != nullptr ? std::string(dir) : library_dir()) + "/ep_kernels.hsaco";
    FILE* f = fopen(path.c_str(), "rb");
    if (f == nullptr) throw EpError{"cannot open the gfx950 code object " + path + " (build it first)"};
    fclose(f);
    int ndev = 0;
    HIP_CHECK(hipGetDeviceCount(&ndev));
    if (ndev <= 0) throw EpError{"no HIP device visible: the EP kernels only run on a gfx950 GPU"};
    HIP_CHECK(hipGetDevice(&g_k.device));
    hipModule_t m;
    HIP_CHECK(hipModuleLoad(&m, path.c_str()));
    auto get = [&](hipFunction_t& fn, const char* name) { HIP_CHECK(hipModuleGetFunction(&fn, m, name)); };
    get(g_k.layout_count, "ep_layout_count");
    get(g_k.layout_scan, "ep_layout_scan");
    get(g_k.layout_count_bits, "ep_layout_count_bits");
    get(g_k.layout_assign_bits, "ep_layout_assign_bits");
    get(g_k.layout_place, "ep_layout_place");
    const char* sides[3] = {"", "_send", "_recv"};      // EP_LAYOUT_SIDE_*
    for (int side = 0; side < 3; ++side) {
        get(g_k.layout_assign[0][side], (std::string("ep_layout_assign") + sides[side]).c_str());
        get(g_k.layout_assign[1][side], (std::string("ep_layout_assign_fold") + sides[side]).c_str());
    }
    get(g_k.scatter_copy, "ep_scatter_copy");
    get(g_k.scatter_quant, "ep_scatter_quant");
    get(g_k.scatter_quant_sw, "ep_scatter_quant_sw");
    get(g_k.scatter_copy_pack, "ep_scatter_copy_pack");
    get(g_k.scatter_quant_pack, "ep_scatter_quant_pack");
    get(g_k.scatter_quant_sw_pack, "ep_scatter_quant_sw_pack");
    const char* small_names[3] = {"copy", "quant", "quant_sw"};
    for (int i = 0; i < 3; ++i) {
        get(g_k.small[0][i], (std::string("ep_dispatch_small_") + small_names[i]).c_str());
        get(g_k.small[1][i], (std::string("ep_dispatch_small_") + small_names[i] + "_pack").c_str());
        get(g_k.chunk[0][i], (std::string("ep_dispatch_chunk_") + small_names[i]).c_str());
        get(g_k.chunk[1][i], (std::string("ep_dispatch_chunk_") + small_names[i] + "_pack").c_str());
    }
    get(g_k.recv_copy, "ep_recv_copy");
    get(g_k.sf_transpose, "ep_sf_transpose");
    const char* modes[3] = {"", "_partial", "_final"};
    const char* ks[8] = {"_generic", "_k2", "_k3", "_k4", "_k5", "_k6", "_k7", "_k8"};
    for (int mode = 0; mode < 3; ++mode)
        for (int k = 0; k < 8; ++k)
            get(g_k.combine[mode][k], (std::string("ep_combine") + modes[mode] + ks[k]).c_str());
    get(g_k.fp8_selftest, "ep_fp8_selftest");
    get(g_k.quant_rows, "ep_quant_rows");
    g_k.module = m;
}

// The event that a call leaves behind its launches.  Recorded by itself it is a packet of its own in the queue, with fences
// (2.7 us of the GPU behind a kernel that writes 16 MiB); as the stop event of the call's last kernel it is that kernel's
// completion signal and costs nothing there.  It rides where what the call stored is read by this process on this GPU: one
// partition, or all of a node's in this process.  What a partition alone or with arenas given by address has stored is read from outside
// (by a transport, by another GPU) behind the event: there, under capture, and where the call launches nothing, it is recorded.
// A pass of eight partitions, two deferred calls each: of 2048 tokens 1290 -> 1249 us; of 64 (bound by the host) a tenth less.
class DoneEvent {
public:
    DoneEvent(void* event, void* stream, const ep_buffer* b);
    // for the last launch of the call: the event to ride on it, or none
    hipEvent_t take(uint64_t threads) {
        if (event_ == nullptr or not rides_ or threads > UINT32_MAX) return nullptr;      // (that launch takes threads, not workgroups)
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream_, &status) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (status != hipStreamCaptureStatusNone) return nullptr;
        hipEvent_t taken = event_;
        event_ = nullptr;
        return taken;
    }
    void record() {
        if (event_ != nullptr) HIP_CHECK(hipEventRecord(event_, stream_));
        event_ = nullptr;
    }

private:
    hipEvent_t event_;
    hipStream_t stream_;
    bool rides_;
};

template <class A>
void launch(hipFunction_t fn, unsigned grid, unsigned block, unsigned smem, void* stream, A& args, DoneEvent* done = nullptr) {
    void* params[] = {&args};
    if (hipEvent_t stop = done != nullptr ? done->take((uint64_t)grid * block) : nullptr) {
        HIP_CHECK(hipExtModuleLaunchKernel(fn, grid * block, 1, 1, block, 1, 1, smem, (hipStream_t)stream, params, nullptr, nullptr, stop, 0));
        return;
    }
    HIP_CHECK(hipModuleLaunchKernel(fn, grid, 1, 1, block, 1, 1, smem, (hipStream_t)stream, params, nullptr));
}

// ---- tensor contracts -------------------------------------------------------------------------
bool present(const ep_tensor_t& t) { return t.data != nullptr; }

int elem_size(int dtype) {
    switch (dtype) {
        case EP_DTYPE_BF16: case EP_DTYPE_I16: return 2;
        case EP_DTYPE_FP8_E4M3: case EP_DTYPE_U8: return 1;
        case EP_DTYPE_I32: case EP_DTYPE_F32: return 4;
        case EP_DTYPE_I64: return 8;
        default: return 0;
    }
}

bool contiguous(const ep_tensor_t& t) {
    int64_t expect = 1;
    for (int d = t.ndim - 1; d >= 0; --d) {
        if (t.size[d] != 1 && t.stride[d] != expect) return false;
        expect *= t.size[d];
    }
    return true;
}

}  // namespace

struct ep_buffer {
    int rank_idx = 0, num_ranks = 1;
    int64_t num_buffer_bytes = 0, num_lb_bytes = 0;
    int cpu_timeout_secs = 300, gpu_timeout_secs = 100;
    char* arena = nullptr;       // workspace || buffer || lb storage
    int* host_page = nullptr;    // pinned + mapped
    int* host_page_dev = nullptr;
    int seq = 0;                 // sequence number of the last non-cached dispatch
    int64_t launch_stamp = 0;    // counts the non-cached ep_dispatch_launch calls; the latest one owns the workspace
    int64_t workspace_bytes = kWorkspaceBytes;
    bool is_static = false;      // a view over the library's static scratch: no arena, no count page, one partition
    bool destroyed = false;
    int device = 0;
    // node of partitions living in this process (ep_buffer_connect): every partition's arena is a peer
    bool connected = false;
    std::vector<ep_buffer*> peers;
    // how often each phase has been enqueued: the partitions of a node move in lockstep, which lets the
    // host catch a phase enqueued before the peers' previous phase (nothing on the device waits for it)
    int64_t num_sends = 0, num_expands = 0, num_partials = 0;
    // state handed from ep_dispatch_launch to ep_dispatch_epilogue_launch
    struct {
        bool valid = false;
        int64_t stamp = 0;
        int num_tokens = 0, num_topk = 0, num_experts = 0, alignment = 0, max_tokens = 0;
        int* slot_map = nullptr;
        int* tok_row = nullptr;
        bool notified = false;
        bool ships_ranks = false;   // more than one partition: the send sides leave counts and ranks in the receivers' boxes
        bool notifies_peers = false;// ... and their counts in the receivers' host boxes
        bool host_boxes = false;    // this partition's host counts come from its host boxes, filled by the send sides
        int send_seq = 0;           // the sequence number the sources left there
        int64_t counted_rows = -1;  // rows of the receive stream, once the host has read its host boxes
        bool layout_pending = false;// the layout is left to the copy launch, whatever stream that comes on
        bool place_pending = false; // receive side: the placing is left to the copy launch
        EpLayoutArgs pending{};     // (of either)
        bool copied = false;        // the copy launch has used it up: the workspace holds no layout to copy by again
        bool recv_done = false;     // more than one partition: the receive-side layout has been enqueued
    } last;

    char* const* peer_table() const { return (char* const*)(arena + EP_WS_PEERS_OFF); }
    const int* inbox() const { return (const int*)(arena + EP_WS_INBOX_OFF); }
    // rows the receive stream of this partition can hold
    int64_t recv_rows_bound(int num_tokens, int max_tokens) const {
        return connected ? (int64_t)num_ranks * max_tokens : num_tokens;
    }

    char* workspace() const { return arena; }
    char* buffer() const { return arena + workspace_bytes; }
    char* lb() const { return arena + workspace_bytes + num_buffer_bytes; }
};

DoneEvent::DoneEvent(void* event, void* stream, const ep_buffer* b)
    : event_((hipEvent_t)event), stream_((hipStream_t)stream), rides_(b->num_ranks == 1 or not b->peers.empty()) {}

namespace {
// LDS of the layout kernels: histograms / per-wave counters, the staged keys, the per-source row counts
unsigned layout_key_bytes(int K) { return 2u * EP_TOKENS_PER_BLOCK * K * sizeof(short); }
unsigned layout_count_lds(int E, int R, int K) {
    return (unsigned)(E + R + R + EP_LAYOUT_THREADS / 64) * sizeof(int) + layout_key_bytes(K);
}
// (cnt_stride > 0: the assignment sums the count rows itself and needs two rows of ints where the partial sums meet)
unsigned layout_assign_lds(int E, int R, int K, int count_experts, int cnt_stride) {
    const unsigned nw = EP_LAYOUT_THREADS / 64;
    return (unsigned)(count_experts + R + nw * (E + R) + nw + 1 + R + nw + 2 * cnt_stride) * sizeof(int) + layout_key_bytes(K);
}

unsigned layout_count_bits_lds(int cnt_stride) { return 4u * (unsigned)cnt_stride + 8u * (EP_TOKENS_PER_BLOCK * EP_BITS_TOPK / 64 + 1); }
unsigned layout_assign_bits_lds(int E, int cnt_stride) {
    constexpr unsigned entries = EP_TOKENS_PER_BLOCK * EP_BITS_TOPK;
    return 16u * (unsigned)E + 12u * (unsigned)cnt_stride + 8u * (entries / 64 + 1) + 8u + 2u * entries;
}

// Up to here one partition ranks in bit masks, behind histograms of its own (figures at the kernel; beyond top-8 a thread would hold more
// than four ids, and the masks of more experts leave a CU too few workgroups).  It is the faster form or level but for top-1 and top-2 of few
// experts at some multiples of 256 blocks, between which it gains.  us of a layout, ids ranked by match-any / in masks: top-1, 64 experts,
// 24576 tokens 10.3 / 9.7, 32768 10.6 / 10.6, 49152 12.6 / 12.0, 65536 12.9 / 13.1, 98304 18.9 / 18.8; 32 experts, 49152 12.3 / 11.8, 98304 16.3 / 16.8;
// top-2 17.0 / 17.4; top-3 18.4 / 17.5.
bool bits_layout(int K, int E) { return K <= EP_BITS_TOPK and E <= EP_SMALL_MASK_EXPERTS; }

// Where one launch that counts the ids of all blocks in every workgroup beats a histogram launch in front of the slot
// assignment.  It saves a launch; each further block is more ids to every workgroup, and one more of these.
// Against ep_layout_count + ep_layout_assign_fold (beyond top-8 or EP_SMALL_MASK_EXPERTS now), us of a replayed dispatch of 16 channels, 256 experts,
// two launches / one: top-1, 16 blocks 12.8 / 11.6, 24 12.9 / 13.9, 64 14.4 / 21.9; top-2, 12 13.0 / 12.5, 16 13.0 / 13.1, 32 13.6 / 17.8; top-3, 10 14.4 /
// 13.4, 16 14.6 / 15.6; top-4, 8 14.5 / 13.3, 16 14.8 / 17.0; top-6, 8 16.1 / 15.7, 10 16.3 / 17.3; top-8, 6 17.5 / 16.7, 8 17.6 / 18.3; top-12, 4 21.1 /
// 18.9; top-32, 2 37.3 / 31.5.  To a host that waits for the counts the saved launch was worth more (wall clock, 8 blocks, top-7 24.3 / 23.7,
// top-8 25.3 / 25.0).
// Against the two launches that rank in bit masks the line lies lower where no host waits, and lower still with more than a few experts, whose
// histograms every workgroup clears and scans.  us, two launches / one, 256 experts: top-1,
// 16 blocks 9.4 / 8.9; top-2, 8 9.3 / 8.2, 16 9.4 / 10.3; top-4, 4 9.7 / 8.8, 6 9.8 / 10.1; top-8, 2 10.3 / 10.5, 3 10.1 / 11.8; 1024 experts top-4
// 10.7 / 10.3, 10.8 / 11.6.  What one launch takes more, at 12 to 16, 18 to 24, 25 to 32 and 35 to 40 blocks x top-k, top-2 to 4 / top-5 to 8: 8 experts -3.2 / -2.7,
// -1.7 / -1.4, -1.3 / -1.2, 0 / 0.2; 32 -2.0 / -1.4, -0.6 / -0.2, -0.3 / 0 (top-7 and 8 0.2, 0.2), 1.1 / 1.3; 64 -1.6 / -0.9, -0.2 / 0.3, 0.1 / 0.5, 1.5 / 1.8; 128 -1.3 / -0.6, 0.1 / 0.7, 0.4 / 0.8.
// Where a host waits it is 48 blocks x top-k for every top-k: higher than against the other two for top-3 to top-5 (32 to 40 there), lower for top-7
// and top-8 (56, 64).  The ids come 16 a thread and trip: wall clock of a dispatch of exact sizes is level up to 48 and falls off beyond.  us, two
// launches / one: 256 experts, top-3, 10 blocks 26.2 / 25.0, 12 26.8 / 27.2, 16 26.7 / 26.8; top-4, 8 26.6 / 25.0, 10 26.3 / 26.1, 12 26.7 / 27.0, 14 26.6 / 28.4; top-5, 9
// 26.2 / 26.4, 10 26.2 / 27.2; top-6, 8 26.1 / 26.0, 9 26.3 / 27.3; top-7, 4 26.2 / 25.3, 6 26.5 / 26.7, 7 26.4 / 27.7, 8 26.3 / 27.3; top-8, 4 26.2 / 25.5, 6
// 26.3 / 26.5, 7 26.5 / 27.8, 8 26.3 / 27.5; 32 experts, top-8, 6 26.5 / 25.9, 7 26.4 / 27.0; 1024, 4 30.3 / 30.0, 6 30.1 / 30.7.
bool recount_pays(int num_blocks, int K, int E, bool host_waits) {
    const int most = 2 * EP_RECOUNT_DEPTH;
    const int limit = bits_layout(K, E) ? (host_waits ? 48 : E <= 32 and E * K <= 192 ? 32 : 16)
                                        : std::max(K > 8 ? most : std::min(8 * K, host_waits ? most : 48), 32);
    return num_blocks <= 16 and num_blocks * K <= limit;
}

// The layout pass: per-block histograms, then the slot assignment.  One block needs no histogram pass; up
// to g_fold_max_blocks blocks the assignment kernel sums the histograms of the blocks before it itself;
// beyond that a scan kernel turns them into prefixes first.
void launch_layout(EpLayoutArgs& la, int num_blocks, void* stream) {
    const int E = la.num_experts, R = la.num_ranks, K = la.num_topk, C = la.count_experts;
    // (the few shapes with more count columns than the summing instance has threads for, or whose LDS would not hold
    //  the rows where its sums meet, take the scan kernel at any size)
    // (what the summing costs is rows a thread: blocks x column groups of 8 / threads.  The limit is quoted in blocks at
    //  the headline's 264 columns, 33 groups; narrower rows, as the 40 columns of an EP32 partition, sum that many more)
    const bool fold = (int64_t)num_blocks * (la.cnt_stride / 8) <= (int64_t)g_fold_max_blocks * 33 and
                      la.cnt_stride <= 8 * EP_LAYOUT_THREADS and layout_assign_lds(E, R, K, C, la.cnt_stride) <= 64 * 1024;
    // a few blocks of one partition (send side): the slot assignment counts the ids of all blocks itself, a launch less
    // (two histograms of El + R ints and a byte a token on top of its LDS; at 64 blocks x top-k a thread holds 32 ids)
    const unsigned recount_extra = (unsigned)(2 * (E / R + R)) * sizeof(int) + (unsigned)num_blocks * EP_TOKENS_PER_BLOCK;
    const int side = la.recv_mode ? EP_LAYOUT_SIDE_RECV : R > 1 ? EP_LAYOUT_SIDE_SEND : EP_LAYOUT_SIDE_SINGLE;
    const int limit = g_recount_limit.load();
    const bool recount = side == EP_LAYOUT_SIDE_SINGLE and num_blocks >= 2 and
                         (limit < 0 ? recount_pays(num_blocks, K, E, la.notify_host != 0) : num_blocks <= std::min(limit, 2 * EP_RECOUNT_DEPTH) / K) and
                         layout_assign_lds(E, R, K, C, 0) + recount_extra <= 64 * 1024;
    la.scan_mode = num_blocks == 1 ? EP_LAYOUT_SINGLE
                   : recount       ? EP_LAYOUT_RECOUNTED
                   : fold          ? EP_LAYOUT_FOLDED
                                   : EP_LAYOUT_SCANNED;
    const unsigned smem_assign = layout_assign_lds(E, R, K, C, la.scan_mode == EP_LAYOUT_FOLDED ? la.cnt_stride : 0) +
                                 (la.scan_mode == EP_LAYOUT_RECOUNTED ? recount_extra : 0u);
    EP_HOST_ASSERT(smem_assign <= 64 * 1024);
    if (la.scan_mode == EP_LAYOUT_FOLDED and side == EP_LAYOUT_SIDE_SINGLE and bits_layout(K, E)) {
        launch(g_k.layout_count_bits, num_blocks, EP_LAYOUT_THREADS, layout_count_bits_lds(la.cnt_stride), stream, la);
        launch(g_k.layout_assign_bits, (unsigned)num_blocks + 1u, EP_LAYOUT_THREADS, layout_assign_bits_lds(E, la.cnt_stride), stream, la);
        return;
    }
    if (la.scan_mode == EP_LAYOUT_FOLDED or la.scan_mode == EP_LAYOUT_SCANNED)
        launch(g_k.layout_count, num_blocks, EP_LAYOUT_THREADS, layout_count_lds(E, R, K), stream, la);
    if (la.scan_mode == EP_LAYOUT_SCANNED)
        launch(g_k.layout_scan, (unsigned)ceil_div(la.cnt_stride, 16), EP_SCAN_THREADS, 0, stream, la);
    // (one workgroup more than blocks: it publishes the totals and ranks nothing)
    launch(g_k.layout_assign[la.scan_mode == EP_LAYOUT_FOLDED][side], (unsigned)num_blocks + 1u, EP_LAYOUT_THREADS,
           smem_assign, stream, la);
}

// Decode sizes: layout and copy in one launch.
unsigned small_lds(int E, int R) {
    const unsigned tokens = EP_TOKENS_PER_BLOCK / 8, masks = E <= EP_SMALL_MASK_EXPERTS ? (unsigned)E : 0u;
    return ((unsigned)R + masks) * tokens + (2u * (unsigned)align_up(E, 8) + 4u) * sizeof(int) +
           (EP_SMALL_ENTRIES + (masks > 0 ? EP_SMALL_REPEATS : 0)) * sizeof(short);
}
// Workgroups that zero the padding of such a dispatch: each counts all ids first, in LDS that grows with the experts, so they
// are no more than fit the chip at once with the row workgroups (1024), unless the padding may be more than 48 MiB.
// us of a replayed dispatch, two launches / one with 1024 / with 2048 workgroups: 128 tokens top-1, 2048 experts, 7168 FP8
// channels, alignment 16 14.9 / 13.2 / 17.3, 128 29.9 / 31.6 / 29.5; 4 tokens top-8, 1024 experts, 2048 BF16 channels, alignment 64
// 15.2 / 9.6 / 11.6; 128 tokens top-8, 1024 experts, alignment 128 (0.9 GB at most) 126 / 124 / 111, 256 experts 53 / 45 / 47;
// 32 tokens top-8, 512 experts, 2048 BF16 channels, alignment 64 (66 MB at most) 19.1 / 14.3 / 13.7.
unsigned small_pad_blocks(unsigned pieces, int num_tokens, int K, int num_experts, int alignment, int64_t row_bytes) {
    const int64_t most_padding = (int64_t)std::min(num_experts, num_tokens * K) * (alignment - 1) * row_bytes;
    return std::min(pieces, most_padding > (48 << 20) ? 2048u : 1024u);
}
// Up to here one launch is the faster form (us of a replayed dispatch without padding, 7168 BF16 channels, two launches / one):
// top-8 of 256, 1 token 10.4 / 6.0, 32 11.8 / 6.8, 96 12.9 / 9.9, 128 13.4 / 11.1; 128 tokens top-1 8.0 / 4.9, top-8 of 2048
// 16.9 / 12.8, 16384 channels 15.6 / 14.9; top-16, 64 tokens 17.6 / 12.8; top-32, 32 tokens 27.9 / 20.1.  One of eight partitions
// (FP8, top-8), 64 tokens 29.2 / 22.6, 128 30.6 / 25.4.  The line is one block of ids: a token's bit and its rank are kept for
// that many.  The form beyond (ep_dispatch_chunk_*) at these sizes is slower nearly everywhere (us, that form / this one): whole passes of a
// synchronised dispatch and a combine, 8 experts, 8 / 128 tokens 27.5 / 26.3, 27.6 / 26.7, 256 experts 28.9 / 27.8, 29.1 / 28.7; replayed passes of
// eight partitions top-2, 8 / 64 / 128 tokens 84.3 / 72.3, 92.5 / 78.5, 94.4 / 80.7, top-8 100.9 / 95.2, 114.2 / 106.4, 119.9 / 120.9; of two, 128
// tokens top-8 33.1 / 35.1.
bool small_dispatch(int num_tokens, int K) {
    return num_tokens > 0 and num_tokens <= EP_TOKENS_PER_BLOCK and num_tokens * K <= EP_SMALL_ENTRIES;
}
void launch_small(const EpLayoutArgs& la, const EpScatterArgs& sa, bool pack, bool quantise, int num_pad_blocks, void* stream,
                  DoneEvent* done = nullptr) {
    EpSmallArgs args{};
    args.l = la;
    args.s = sa;
    args.num_pad_blocks = num_pad_blocks;
    EP_HOST_ASSERT(sa.vecs_per_lane == 1);
    launch(g_k.small[pack][quantise ? (g_fp8_hw ? 1 : 2) : 0], 1u + (unsigned)sa.num_row_blocks + (unsigned)num_pad_blocks, EP_ROW_THREADS,
           small_lds(la.num_experts, la.num_ranks), stream, args, done);
}


// Chunk sizes: layout and copy in one launch as well, by workgroups that all count every id (ep_dispatch_chunk_*).
unsigned chunk_lds(int num_tokens, int K, int E, int R) {
    const unsigned marks = R > 1 ? (unsigned)num_tokens : (unsigned)ceil_div((int64_t)num_tokens * K, 64) * 2u + 2u;
    return (unsigned)(2 * E + 2 * R + EP_CHUNK_THREADS / 64 + 2 * EP_CHUNK_OWN) * sizeof(int) + EP_CHUNK_OWN * sizeof(short) + marks * sizeof(int);
}
// Up to here one launch is the faster form: what it costs is ids to every workgroup, what it saves is the launches and trips
// of the layout in front.  us of a replayed dispatch, two launches / one: 129 tokens x 256, top-2 9.1 / 6.7; 512 x 4096 top-32
// 60.4 / 34.6; 2048 x 7168 BF16 top-8 (16384 entries) 66.9 / 53.0, 108.6 / 105.2 with alignment 128; 2700 FP8 top-6 65.8 / 62.3;
// 4096 x 512 top-4 16.8 / 14.5; beyond: 3000 tokens FP8 top-6 67.0 / 65.7, 4096 top-6 58.7 / 60.1, top-8 BF16 152 / 157, 8192 x 512 top-2 16.3 / 22.1.
// Several partitions, all of a partition's dispatch: two of 2048 tokens x 2048 top-8 44.0 / 41.3, four of 1500 x 7168 top-8 94.3 / 86.4, 32 of 1024 top-6
// 54.8 / 48.0; beyond, four of 4096 top-4 89.3 / 90.2, two of 4096 x 2048 top-2 38.7 / 38.7 (a word a token is kept in LDS).
// (a partition is a bit of that word)
// Wide rows of many tokens are a copy long enough for its fixed shares a workgroup to cost more than the launch saved, most with hot
// experts.  Mean of BF16 and FP8, alignment 1, 16 and 128, uniform and Zipf (1.2) routing, two launches / one: 7168 channels, 2700 top-6
// 73.5 / 72.7, 2900 top-5 70.8 / 70.5, 3200 top-5 73.8 / 74.8, 3800 top-4 73.0 / 74.5, 4096 top-3 68.9 / 70.0, top-4 75.4 / 77.6 (Zipf, alignment
// 16, FP8 51.2 / 55.3), but 4096 top-2 56.7 / 53.1; 10240, 2400 top-6 91.5 / 92.0, 2700 96.5 / 99.6; 16384, 2048 top-6 112.5 / 108.4, 2700 134.0 /
// 136.1.  5120 channels are level at 4096 top-4 (59.1 / 59.5), 4096 gain (51.1 / 50.5).
bool chunk_dispatch(int num_tokens, int K, int E, int R, int num_parts) {
    if (num_tokens <= 0 or num_tokens > (R > 1 ? EP_CHUNK_TOKENS / 2 : EP_CHUNK_TOKENS) or num_tokens * K > EP_CHUNK_ENTRIES or R > 32) return false;
    const bool long_copy = num_parts >= 12 and num_tokens > (num_parts <= 16 ? 3072 : 2560) and num_tokens * K > 12000;
    return not long_copy and chunk_lds(num_tokens, K, E, R) <= 64 * 1024;
}
// (token, part) tasks a row of a dispatch falls into: 512 channels of a row being quantised, 1 KiB of any other
int row_parts(int64_t hidden, int64_t row_bytes, bool quantise) {
    return (int)std::max<int64_t>(1, quantise ? ceil_div(hidden, 512) : ceil_div(row_bytes, 1024));
}
// Workgroups: no more than one task a wave needs.  Two a CU keep twice the rows on the way, one a CU counts the ids half as
// often (us at 256 / 512 workgroups): 14 parts a row, 1021 tokens top-8 35.6 / 34.5, 2048 top-4 39.9 / 38.1, but 2048 top-8 53.0 / 60.3 and eight
// partitions of 2048 FP8 top-6 65.6 / 67.6; 10 parts, 1021 top-8 27.8 / 27.0; 8 parts, 2048 top-4 27.2 / 26.3, 1021 top-8 23.6 / 23.7, one of two
// partitions, all of a pass, 1021 top-8 59.7 / 62.4; 9 parts, 2048 top-4 28.6 / 28.8, eight partitions of 500 top-8 198.0 / 208.6; 5 parts, 1021 top-6
// 17.6 / 18.4; 2 parts, 4096 top-2 12.9 / 15.3.  (The publishing workgroup beside 512 costs nothing: with 511, 1021 x 7168 top-8 34.4 / 34.4.)
// Padding is shared by all workgroups: as many as there is padding for.  (Two a CU for it alone: 2048 experts at alignment 128 2 % faster, 64
// to 256 experts 0 to 15 % slower.  That much padding beside few tokens is the one case left where two launches were faster: 2048 experts, 2560
// channels, 500 tokens top-4 124.8 / 138.2, 200 top-8 112.5 / 115.4, 1000 top-8 205.6 / 199.7; whether padding is zeroed is not known at the begin.)
void launch_chunk(const EpLayoutArgs& la, const EpScatterArgs& sa, bool pack, bool quantise, unsigned pad_pieces, void* stream,
                  DoneEvent* done = nullptr) {
    EpSmallArgs args{};
    args.l = la;
    args.s = sa;
    args.zero_padding = pad_pieces > 0;
    EP_HOST_ASSERT(sa.vecs_per_lane == 1 and sa.num_rows_bound == la.num_tokens);
    const int64_t tasks = (int64_t)la.num_tokens * sa.num_parts;
    const bool two_a_cu = sa.num_parts >= 10 and la.num_tokens * la.num_topk <= EP_CHUNK_ENTRIES / 2;
    const int64_t most = two_a_cu ? EP_CHUNK_BLOCKS : EP_CHUNK_BLOCKS / 2;
    const int64_t blocks = std::min<int64_t>(most, ceil_div(tasks, EP_CHUNK_THREADS / 64));
    args.tasks_per_block = (int)ceil_div(tasks, blocks);
    const int64_t own = (args.tasks_per_block + sa.num_parts - 2) / sa.num_parts + 1;      // tokens that so many tasks can touch
    EP_HOST_ASSERT(own * la.num_topk <= EP_CHUNK_OWN);
    const int64_t pads = std::min<int64_t>(most, ceil_div((int64_t)pad_pieces, EP_CHUNK_THREADS / EP_ROW_THREADS));
    launch(g_k.chunk[pack][quantise ? (g_fp8_hw ? 1 : 2) : 0], 1u + (unsigned)std::max(blocks, pads), EP_CHUNK_THREADS,
           chunk_lds(la.num_tokens, la.num_topk, la.num_experts, la.num_ranks), stream, args, done);
}

// Scale packs (2 bytes) can move two at a time: packs side by side, rows that start on 4 bytes where they are read and written.
int sf_pairs(const EpScatterArgs& sa, const void* out) {
    return sa.sf != nullptr and out != nullptr and sa.num_sf_packs % 2 == 0 and sa.sf_pack_stride_bytes == 2 and
           sa.sf_token_stride_bytes % 4 == 0 and sa.out_sf_row_bytes % 4 == 0 and (((uintptr_t)sa.sf | (uintptr_t)out) & 3) == 0;
}

unsigned layout_place_lds(int E, int R, int K) {
    const unsigned nw = EP_LAYOUT_THREADS / 64;
    return (unsigned)(E + E / R + nw + R + nw + 2 * EP_TOKENS_PER_BLOCK) * sizeof(int) + EP_TOKENS_PER_BLOCK * K;
}

// The receive side of a node whose send sides ship ranks: placed and copied in one launch (ep_recv_copy), for as many sources as a
// wave has lanes.  It saves a launch and its trips; each workgroup adds up the counts of all experts instead.  us of all phases of a
// node (host included), two launches / one: 8 partitions of 64 tokens 409 / 401, of 2048 1378 / 1332; 32 of 16384 1243 / 1198
// a partition; 16 of 2048 with 2048 experts 1438 / 1385; 2 partitions, 2048 experts, 512 channels: 2048 tokens top-8 155 / 153, 4096 top-2
// 148 / 147, 8192 top-2 (3300 row blocks) 154 / 165, with 1024 experts 148 / 145.  Means over 512 to 7168 channels, top-2 and 8, replayed: two
// partitions, 64 experts, 64 / 4096 / 16384 tokens 34.4 / 26.6, 146 / 136, 401 / 408; eight, 64 experts 124 / 89, 487 / 459, 742 / 720, 512 experts
// 133 / 96, 497 / 478, 767 / 761, 1024 experts 144 / 106, 530 / 516, 807 / 828 (with a host sync, whose row blocks are those of rows that came, there too
// 786 / 763).
constexpr int kRecvCopyMaxRanks = 64;
unsigned recv_copy_lds(int E, int R) { return (unsigned)(E + 2 * (E / R) + EP_ROW_THREADS / 64) * sizeof(int); }
bool recv_copy_pays(int num_experts, int row_blocks) { return num_experts <= 1024 or row_blocks <= 2048; }

// Boxes of a connected partition's workspace, behind its header, at the same place in every arena of the node: counts
// per source and local expert [R][El], then per packed row the ranks of its entries inside their source [R * max_tokens][K].
struct RankBoxes {
    int64_t count_off = 0, rank_off = 0, end = EP_WS_HEADER_BYTES;
    bool used = false;
};
// Every partition of a node comes to the same answer: only what all of them agree on goes in.  Without room for the boxes
// beside the send side's scratch of max_tokens tokens (32 partitions of 16384 tokens at top-6 fit), or for the counters
// of all experts in LDS, the receive side counts and ranks itself.
RankBoxes rank_boxes(const ep_buffer* b, int max_tokens, int K, int E) {
    RankBoxes x;
    const int R = b->num_ranks;
    if (R == 1 or not b->connected) return x;
    auto a256 = [](int64_t n) { return align_up(std::max<int64_t>(n, 1), 256); };
    const int64_t W = align_up(E + R, 8), blocks = std::max<int64_t>(1, ceil_div(max_tokens, EP_TOKENS_PER_BLOCK));
    const int64_t counts = a256(4 * (int64_t)E), ranks = a256(4 * (int64_t)R * max_tokens * K);
    const int64_t scratch = a256(4 * W) + a256(4 * blocks * W) + a256(4 * (int64_t)max_tokens * K);
    if (EP_WS_HEADER_BYTES + counts + ranks + scratch > b->workspace_bytes) return x;
    if (layout_assign_lds(E, R, K, E, 0) > 64 * 1024 or layout_place_lds(E, R, K) > 64 * 1024) return x;
    x.count_off = EP_WS_HEADER_BYTES;
    x.rank_off = x.count_off + counts;
    x.end = x.rank_off + ranks;
    x.used = true;
    return x;
}

void write_peer_table(ep_buffer* b, const std::vector<char*>& arenas) {
    std::vector<char*> table(EP_MAX_RANKS, nullptr);
    for (size_t i = 0; i < arenas.size(); ++i) table[i] = arenas[i];
    HIP_CHECK(hipMemcpy(b->arena + EP_WS_PEERS_OFF, table.data(), sizeof(char*) * EP_MAX_RANKS, hipMemcpyHostToDevice));
}

void disconnect(ep_buffer* b) {
    write_peer_table(b, std::vector<char*>(b->num_ranks, b->arena));
    // the row counts the other partitions left while connected describe rows nobody will refresh
    HIP_CHECK(hipMemset(b->arena + EP_WS_INBOX_OFF, 0, sizeof(int) * EP_MAX_RANKS));
    b->connected = false;
    b->peers.clear();
}

// Phase order inside a node (ep_buffer_connect): `ready(peer)` must hold for every partition.
template <class F>
void check_peers(const ep_buffer* b, F&& ready, const char* what) {
    for (const ep_buffer* p : b->peers)
        if (not ready(*p)) throw EpError{format("Assertion exception (%s): partition %d of the node: %s", __FILE_NAME__, p->rank_idx, what)};
}

// The code object is loaded on one device and the arena lives there: calls must come with that
// device current.
void check_buffer(const ep_buffer* b) {
    EP_HOST_ASSERT(b != nullptr);
    EP_HOST_ASSERT(not b->destroyed);
    int dev = -1;
    HIP_CHECK(hipGetDevice(&dev));
    EP_HOST_ASSERT(dev == b->device and "the buffer belongs to another device");
}
}  // namespace

extern "C" {

const char* ep_last_error(void) { return g_err.c_str(); }

int ep_init(const char* dir) {
    return guarded([&] {
        load_kernels(dir);
        ep_static_scratch_init();      // the address of the static scratch on this device
    });
}

int64_t ep_get_num_allocation_alignment(void) { return kAllocAlign; }
int64_t ep_get_num_tma_alignment(void) { return 32; }
int64_t ep_get_num_rdma_alignment(void) { return 32; }

int ep_get_num_compute_units(void) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return n;
}

int64_t ep_get_dispatch_buffer_size(int max_tokens, int hidden, int sf_packs, int topk, int elem, int ranks) {
    return dispatch_buffer_size(max_tokens, hidden, sf_packs, topk, elem, ranks);
}

int64_t ep_get_combine_buffer_size(int ranks, int max_tokens, int hidden, int topk) {
    return combine_buffer_size(ranks, max_tokens, hidden, topk);
}

int64_t ep_calculate_buffer_size(int num_ranks, int max_tokens, int hidden, int num_topk, int use_fp8) {
    int64_t out = -1;
    const int rc = guarded([&] {
        EP_HOST_ASSERT(num_ranks > 0);
        EP_HOST_ASSERT(max_tokens > 0);
        EP_HOST_ASSERT(hidden > 0);
        EP_HOST_ASSERT(num_topk >= 0);
        const int topk = num_topk == 0 ? 32 : num_topk;            // room for the largest top-k
        const int sf_packs = use_fp8 ? (int)ceil_div(hidden, 32) : 0;   // the hint never sees the SF tensor
        const int64_t d = dispatch_buffer_size(max_tokens, hidden, sf_packs, topk, use_fp8 ? 1 : 2, num_ranks);
        const int64_t c = combine_buffer_size(num_ranks, max_tokens, hidden, topk);
        out = align_up(std::max(d, c), kAllocAlign);
    });
    return rc == 0 ? out : -1;
}

void ep_host_f32_to_e4m3fn(const float* src, uint8_t* dst, int64_t n) {
    for (int64_t i = 0; i < n; ++i) {
        uint32_t b;
        memcpy(&b, src + i, 4);
        dst[i] = (uint8_t)ep_f32_bits_to_e4m3fn(b);
    }
}

void ep_set_fp8_hw_convert(int enable) { g_fp8_hw = enable != 0; }

int ep_fp8_selftest(uint64_t first, uint64_t count, float limit, uint64_t out[2]) {
    return guarded([&] {
        load_kernels(nullptr);
        unsigned long long* dev = nullptr;
        HIP_CHECK(hipMalloc((void**)&dev, 16));
        const unsigned long long init[2] = {0ull, ~0ull};
        HIP_CHECK(hipMemcpy(dev, init, 16, hipMemcpyHostToDevice));
        EpFp8TestArgs args = {first, count, dev, limit, 0};
        launch(g_k.fp8_selftest, 4096, 256, 0, nullptr, args);
        HIP_CHECK(hipDeviceSynchronize());
        unsigned long long res[2];
        HIP_CHECK(hipMemcpy(res, dev, 16, hipMemcpyDeviceToHost));
        HIP_CHECK(hipFree(dev));
        out[0] = res[0];
        out[1] = res[1];
    });
}

int ep_per_token_cast_to_fp8(const ep_tensor_t* px, const ep_tensor_t* pq, const ep_tensor_t* psf, void* stream) {
    return guarded([&] {
        load_kernels(nullptr);
        EP_HOST_ASSERT(px != nullptr and pq != nullptr and psf != nullptr);
        const ep_tensor_t &x = *px, &q = *pq, &sf = *psf;
        EP_HOST_ASSERT(present(x) and x.ndim == 2 and x.dtype == EP_DTYPE_BF16 and contiguous(x));
        const int64_t rows = x.size[0], hidden = x.size[1];
        EP_HOST_ASSERT(hidden > 0 and hidden % 8 == 0 and hidden <= 16384);
        EP_HOST_ASSERT(present(q) and q.ndim == 2 and q.size[0] == rows and q.size[1] == hidden and contiguous(q));
        EP_HOST_ASSERT(q.dtype == EP_DTYPE_FP8_E4M3 or q.dtype == EP_DTYPE_U8);
        EP_HOST_ASSERT(present(sf) and sf.ndim == 2 and sf.size[0] == rows and sf.size[1] == ceil_div(hidden, 128));
        EP_HOST_ASSERT(sf.dtype == EP_DTYPE_F32 and contiguous(sf));
        EP_HOST_ASSERT(((uintptr_t)x.data & 15) == 0 and ((uintptr_t)q.data & 7) == 0);
        EpQuantArgs qa{};
        qa.x = x.data;
        qa.q = q.data;
        qa.sf = (float*)sf.data;
        qa.num_rows = (int)rows;
        qa.hidden = (int)hidden;
        qa.num_parts = (int)ceil_div(hidden, 512);
        qa.hw_convert = g_fp8_hw ? 1 : 0;
        const int64_t blocks = ceil_div(rows * qa.num_parts, EP_ROWS_PER_BLOCK);
        EP_HOST_ASSERT(rows <= INT32_MAX and blocks <= INT32_MAX);
        if (blocks > 0) launch(g_k.quant_rows, (unsigned)blocks, EP_ROW_THREADS, 0, stream, qa);
    });
}

// ---- buffer -----------------------------------------------------------------------------------
int ep_buffer_create(int rank_idx, int num_ranks, int64_t num_bytes, int64_t num_lb_bytes, int cpu_timeout_secs,
                     int gpu_timeout_secs, ep_buffer_t** out) {
    return guarded([&] {
        EP_HOST_ASSERT(out != nullptr);
        EP_HOST_ASSERT(num_bytes >= 0 and num_bytes % kAllocAlign == 0);
        EP_HOST_ASSERT(num_lb_bytes >= 0 and num_lb_bytes % kAllocAlign == 0);
        EP_HOST_ASSERT(num_ranks > 0 and num_ranks <= EP_MAX_RANKS and rank_idx >= 0 and rank_idx < num_ranks);
        EP_HOST_ASSERT(cpu_timeout_secs > 0 and gpu_timeout_secs > 0);
        load_kernels(nullptr);
        int cur = -1;
        HIP_CHECK(hipGetDevice(&cur));
        EP_HOST_ASSERT(cur == g_k.device and "the kernels were loaded on another device");
        auto* b = new ep_buffer();
        b->rank_idx = rank_idx;
        b->num_ranks = num_ranks;
        b->num_buffer_bytes = num_bytes;
        b->num_lb_bytes = num_lb_bytes;
        b->cpu_timeout_secs = cpu_timeout_secs;
        b->gpu_timeout_secs = gpu_timeout_secs;
        try {
            HIP_CHECK(hipGetDevice(&b->device));
            const int64_t total = kWorkspaceBytes + num_bytes + num_lb_bytes;
            HIP_CHECK(hipMalloc((void**)&b->arena, (size_t)total));
            HIP_CHECK(hipMemset(b->arena, 0, (size_t)total));
            const size_t page_bytes = (EP_HOST_PAGE_INTS + (num_ranks > 1 ? 2 * EP_HOST_BOX_INTS : 0)) * sizeof(int);
            // (coherent: the kernels' stores to it are announced by one more store behind them, with no release of a cache in front.
            //  That is the runtime's default too, unless its environment says otherwise)
            HIP_CHECK(hipHostMalloc((void**)&b->host_page, page_bytes, hipHostMallocMapped | hipHostMallocCoherent));
            memset(b->host_page, 0, page_bytes);
            HIP_CHECK(hipHostGetDevicePointer((void**)&b->host_page_dev, b->host_page, 0));
            write_peer_table(b, std::vector<char*>(num_ranks, b->arena));    // not connected: every peer is this arena
            HIP_CHECK(hipDeviceSynchronize());
        } catch (...) {
            if (b->arena != nullptr) (void)hipFree(b->arena);
            if (b->host_page != nullptr) (void)hipHostFree(b->host_page);
            delete b;
            throw;
        }
        *out = b;
    });
}

int ep_buffer_connect(ep_buffer_t** bufs, int n) {
    return guarded([&] {
        EP_HOST_ASSERT(bufs != nullptr and n > 1);
        std::vector<char*> arenas(n);
        for (int i = 0; i < n; ++i) {
            check_buffer(bufs[i]);
            EP_HOST_ASSERT(bufs[i]->num_ranks == n and bufs[i]->rank_idx == i);
            EP_HOST_ASSERT(bufs[i]->num_buffer_bytes == bufs[0]->num_buffer_bytes);
            EP_HOST_ASSERT(not bufs[i]->connected);
            arenas[i] = bufs[i]->arena;
        }
        HIP_CHECK(hipDeviceSynchronize());
        std::vector<int*> boxes(EP_HOST_BOXES_MAX_RANKS, nullptr);
        for (int i = 0; i < std::min(n, EP_HOST_BOXES_MAX_RANKS); ++i) boxes[i] = bufs[i]->host_page_dev + EP_HOST_PAGE_INTS;
        for (int i = 0; i < n; ++i) {
            write_peer_table(bufs[i], arenas);
            HIP_CHECK(hipMemcpy(bufs[i]->arena + EP_WS_HOST_BOXES_OFF, boxes.data(), sizeof(int*) * boxes.size(), hipMemcpyHostToDevice));
            memset(bufs[i]->host_page + EP_HOST_PAGE_INTS, 0, 2 * EP_HOST_BOX_INTS * sizeof(int));     // (a former node's counts)
            bufs[i]->connected = true;
            bufs[i]->peers.assign(bufs, bufs + n);
        }
    });
}

int ep_buffer_set_peers(ep_buffer_t* b, void* const* arena_bases, int n) {
    return guarded([&] {
        check_buffer(b);
        HIP_CHECK(hipDeviceSynchronize());
        if (arena_bases == nullptr) {
            disconnect(b);
            return;
        }
        EP_HOST_ASSERT(n == b->num_ranks and n > 1);
        std::vector<char*> arenas(n);
        for (int i = 0; i < n; ++i) {
            EP_HOST_ASSERT(arena_bases[i] != nullptr);
            arenas[i] = (char*)arena_bases[i];
        }
        EP_HOST_ASSERT(arenas[b->rank_idx] == b->arena and "a partition's own entry is its own arena");
        write_peer_table(b, arenas);
        b->connected = true;
        b->peers.clear();           // arenas the caller mapped: theirs to keep alive and to disconnect
    });
}

int ep_buffer_destroy(ep_buffer_t* b) {
    return guarded([&] {
        EP_HOST_ASSERT(b != nullptr);
        EP_HOST_ASSERT(not b->destroyed);
        HIP_CHECK(hipDeviceSynchronize());
        // the other partitions of a node must not keep pointers into this arena
        const std::vector<ep_buffer*> peers = b->peers;
        for (ep_buffer* p : peers)
            if (p != b) disconnect(p);
        b->peers.clear();
        HIP_CHECK(hipFree(b->arena));
        HIP_CHECK(hipHostFree(b->host_page));
        b->arena = nullptr;
        b->host_page = nullptr;
        b->destroyed = true;
        delete b;
    });
}

void* ep_buffer_region(ep_buffer_t* b, int which, int64_t* num_bytes) {
    if (b == nullptr || b->destroyed) return nullptr;
    switch (which) {
        case 0: if (num_bytes) *num_bytes = kWorkspaceBytes; return b->workspace();
        case 1: if (num_bytes) *num_bytes = b->num_buffer_bytes; return b->buffer();
        case 2: if (num_bytes) *num_bytes = b->num_lb_bytes; return b->lb();
        default: return nullptr;
    }
}

int ep_buffer_print_memory_usage(ep_buffer_t* b) {
    return guarded([&] {
        EP_HOST_ASSERT(b != nullptr and not b->destroyed);
        const double gib = 1 << 30;
        printf("[DeepEP memory usage] rank_idx=%d, num_ranks=%d, GPU total %.3f GiB "
               "(workspace %.3f GiB, buffer %.3f GiB, RDMA storage %.3f GiB), CPU total %.3f GiB\n",
               b->rank_idx, b->num_ranks, (kWorkspaceBytes + b->num_buffer_bytes + b->num_lb_bytes) / gib,
               kWorkspaceBytes / gib, b->num_buffer_bytes / gib, b->num_lb_bytes / gib, 0.0);
        fflush(stdout);
    });
}

// ---- dispatch ---------------------------------------------------------------------------------
// What the caller says of the copy epilogue: nothing (the layout is enqueued at once), that it is the next call (a decode-size layout
// is left to it), or that it is the only one, of the same experts and alignment, with no wait for counts in front (every
// layout that a copy launch can make is).
enum class Epilogue { any, next, only };

static int dispatch_launch(ep_buffer_t* b, const ep_dispatch_args_t* pa, Epilogue epilogue, void* event = nullptr) {
    return guarded([&] {
        EP_HOST_ASSERT(pa != nullptr);
        check_buffer(b);
        const ep_dispatch_args_t& a = *pa;
        DoneEvent done(event, a.stream, b);
        const bool cached_mode = a.cached_mode != 0;
        const bool do_cpu_sync = a.do_cpu_sync != 0;
        EP_HOST_ASSERT(not b->is_static or (not cached_mode and not do_cpu_sync and b->num_ranks == 1));
        if (cached_mode) {
            EP_HOST_ASSERT(not do_cpu_sync and "Cannot do CPU sync with cached mode");
            EP_HOST_ASSERT(not present(a.cumulative_local_expert_recv_stats));
        }

        // data tensor
        EP_HOST_ASSERT(present(a.x));
        EP_HOST_ASSERT(a.x.ndim == 2);
        const int num_tokens = (int)a.x.size[0];
        const int hidden = (int)a.x.size[1];
        const int num_ranks = b->num_ranks;
        EP_HOST_ASSERT(a.num_experts > 0 and a.num_experts <= EP_MAX_EXPERTS);
        EP_HOST_ASSERT(a.num_experts % num_ranks == 0);
        const int num_experts_per_rank = a.num_experts / num_ranks;
        EP_HOST_ASSERT(contiguous(a.x));
        EP_HOST_ASSERT(num_tokens <= a.num_max_tokens_per_rank);
        EP_HOST_ASSERT(a.num_max_tokens_per_rank > 0);
        EP_HOST_ASSERT(a.expert_alignment > 0);

        int num_sf_packs = 0;
        if (present(a.sf)) {
            EP_HOST_ASSERT(not a.fused_fp8_quant);
            EP_HOST_ASSERT(a.x.dtype == EP_DTYPE_FP8_E4M3);
            EP_HOST_ASSERT(a.sf.ndim == 2 and a.sf.size[0] == num_tokens);
            EP_HOST_ASSERT(elem_size(a.sf.dtype) == 2);
            EP_HOST_ASSERT(a.sf.stride[0] == 1 or a.sf.stride[1] == 1);
            EP_HOST_ASSERT(a.sf.stride[0] <= INT32_MAX and a.sf.stride[1] <= INT32_MAX);
            num_sf_packs = (int)a.sf.size[1];
        } else {
            EP_HOST_ASSERT(a.x.dtype == EP_DTYPE_BF16);
        }
        const int x_elem = elem_size(a.x.dtype);
        EP_HOST_ASSERT((int64_t)hidden * x_elem % 16 == 0);
        if (a.fused_fp8_quant) {
            EP_HOST_ASSERT(hidden % 8 == 0 and hidden <= 16384);
        }

        // top-k
        EP_HOST_ASSERT(present(a.topk_idx) and a.topk_idx.ndim == 2);
        const int num_topk = (int)a.topk_idx.size[1];
        EP_HOST_ASSERT(a.topk_idx.size[0] == num_tokens);
        EP_HOST_ASSERT(a.topk_idx.dtype == EP_DTYPE_I64);
        EP_HOST_ASSERT(contiguous(a.topk_idx));
        EP_HOST_ASSERT(num_topk > 0 and num_topk <= EP_MAX_TOPK);
        if (present(a.topk_weights)) {
            EP_HOST_ASSERT(a.topk_weights.ndim == 2);
            EP_HOST_ASSERT(a.topk_weights.size[0] == num_tokens and a.topk_weights.size[1] == num_topk);
            EP_HOST_ASSERT(contiguous(a.topk_weights));
            EP_HOST_ASSERT(a.topk_weights.dtype == EP_DTYPE_F32);
        }
        if (present(a.cumulative_local_expert_recv_stats)) {
            const auto& s = a.cumulative_local_expert_recv_stats;
            EP_HOST_ASSERT(s.ndim == 1 and s.size[0] == num_experts_per_rank);
            EP_HOST_ASSERT(contiguous(s));
            EP_HOST_ASSERT(s.dtype == EP_DTYPE_I32);
        }

        // buffer size (the packed regions of csrc/buffers/ep.hpp:196-198)
        const int packed_elem = a.fused_fp8_quant ? 1 : x_elem;
        const int packed_sf = a.fused_fp8_quant ? 2 * (int)ceil_div(hidden, 128) : num_sf_packs;
        // (the static view has no buffer: with one partition the packed regions are never materialised)
        EP_HOST_ASSERT(b->is_static or dispatch_buffer_size(a.num_max_tokens_per_rank, hidden, packed_sf, num_topk, packed_elem,
                                                            num_ranks) <= b->num_buffer_bytes);
        // packed rows put the scales at the next multiple of 32 bytes behind the payload while the row size adds the
        // payload unaligned (layout/ep/token.hpp:36-43,59-61, whose own check of this is commented out :29): rows
        // would overlap their neighbours
        EP_HOST_ASSERT(num_ranks == 1 or packed_sf == 0 or (int64_t)hidden * packed_elem % kUbAlign == 0);

        // handle tensors
        const auto& psum_rank = a.psum_num_recv_tokens_per_rank;
        const auto& psum_expert = a.psum_num_recv_tokens_per_expert;
        const auto& unaligned = a.num_unaligned_recv_tokens_per_expert;
        EP_HOST_ASSERT(present(psum_rank) and present(psum_expert) and present(unaligned));
        EP_HOST_ASSERT(present(a.dst_buffer_slot_idx) and present(a.dst_gsge_idx));
        EP_HOST_ASSERT(psum_rank.ndim == 1 and psum_rank.size[0] == num_ranks);
        EP_HOST_ASSERT(psum_expert.ndim == 1 and psum_expert.size[0] == num_experts_per_rank);
        EP_HOST_ASSERT(unaligned.ndim == 1 and unaligned.size[0] == num_experts_per_rank);
        EP_HOST_ASSERT(a.dst_buffer_slot_idx.ndim == 2 and a.dst_buffer_slot_idx.size[0] == num_tokens and
                       a.dst_buffer_slot_idx.size[1] == num_topk);
        EP_HOST_ASSERT(a.dst_gsge_idx.ndim == 2 and a.dst_gsge_idx.size[0] == num_tokens and
                       a.dst_gsge_idx.size[1] == num_topk);
        EP_HOST_ASSERT(contiguous(psum_rank) and contiguous(psum_expert) and contiguous(unaligned));
        EP_HOST_ASSERT(contiguous(a.dst_buffer_slot_idx) and contiguous(a.dst_gsge_idx));
        EP_HOST_ASSERT(psum_rank.dtype == EP_DTYPE_I32 and psum_expert.dtype == EP_DTYPE_I32);
        EP_HOST_ASSERT(unaligned.dtype == EP_DTYPE_I32);
        EP_HOST_ASSERT(a.dst_buffer_slot_idx.dtype == EP_DTYPE_I32 and a.dst_gsge_idx.dtype == EP_DTYPE_I32);

        const RankBoxes boxes = cached_mode ? RankBoxes{} : rank_boxes(b, a.num_max_tokens_per_rank, num_topk, a.num_experts);
        int* rank_map = nullptr;
        const EpLayoutArgs* own_layout = nullptr;       // the pack launch works out the layout as well
        // geometry of the packed rows of the partition-major regions (only materialised when R > 1)
        const PackedToken pk = packed_token(hidden * packed_elem, packed_sf * 2, num_topk, not cached_mode);
        auto launch_pack = [&]() {
            EpScatterArgs sa{};
            sa.mode = EP_SCATTER_PACK;
            sa.x = a.x.data;
            sa.sf = a.sf.data;
            sa.topk_weights = (const float*)a.topk_weights.data;
            sa.topk_idx = (const int64_t*)a.topk_idx.data;
            sa.dst_slot_idx = (const int*)a.dst_buffer_slot_idx.data;
            sa.recv_x = b->buffer();
            sa.recv_sf = packed_sf > 0 ? b->buffer() + pk.sf_off : nullptr;
            sa.x_row_bytes = (int64_t)hidden * x_elem;
            sa.copy_bytes = sa.x_row_bytes;
            sa.out_row_bytes = pk.bytes;
            sa.out_sf_row_bytes = pk.bytes;
            if (present(a.sf)) {
                sa.sf_token_stride_bytes = a.sf.stride[0] * 2;
                sa.sf_pack_stride_bytes = a.sf.stride[1] * 2;
            }
            sa.hidden = hidden;
            sa.num_topk = num_topk;
            sa.num_rows_bound = num_tokens;
            sa.num_tokens = num_tokens;
            sa.rank_idx = b->rank_idx;
            sa.max_tokens = a.num_max_tokens_per_rank;
            sa.num_sf_packs = num_sf_packs;
            sa.num_experts = a.num_experts;
            sa.experts_per_rank = num_experts_per_rank;
            sa.with_metadata = cached_mode ? 0 : 1;
            sa.idx_off = pk.idx_off;
            sa.w_off = pk.w_off;
            sa.src_off = pk.src_off;
            sa.num_out_rows = num_ranks * a.num_max_tokens_per_rank;
            // unconnected: the regions of this arena, one per destination; in a node: region `rank_idx` of
            // the destination's own arena, where its receive side will look for them
            sa.peer_arenas = b->peer_table();
            sa.buffer_off = b->workspace_bytes;
            sa.region_by_source = b->connected ? 1 : 0;
            sa.num_ranks = num_ranks;
            sa.pack_sf_off = pk.sf_off;
            sa.sf_pairs = sf_pairs(sa, sa.recv_sf);
            sa.slot_map = rank_map;
            sa.rank_box_off = boxes.used ? boxes.rank_off : 0;
            sa.vecs_per_lane = 1;
            sa.num_parts = row_parts(hidden, sa.copy_bytes, a.fused_fp8_quant != 0);
            sa.num_row_blocks = (int)ceil_div((int64_t)num_tokens * sa.num_parts, EP_ROWS_PER_BLOCK);
            if (sa.num_row_blocks == 0) return;
            if (own_layout != nullptr) {
                if (small_dispatch(num_tokens, num_topk)) launch_small(*own_layout, sa, true, a.fused_fp8_quant != 0, 0, a.stream, &done);
                else launch_chunk(*own_layout, sa, true, a.fused_fp8_quant != 0, 0, a.stream, &done);
                return;
            }
            hipFunction_t fn = a.fused_fp8_quant ? (g_fp8_hw ? g_k.scatter_quant_pack : g_k.scatter_quant_sw_pack)
                                                 : g_k.scatter_copy_pack;
            launch(fn, (unsigned)sa.num_row_blocks, EP_ROW_THREADS, 0, a.stream, sa, &done);
        };

        // the rows about to be packed overwrite what the peers received last time
        if (num_ranks > 1)
            check_peers(b, [&](const ep_buffer& p) { return p.num_expands >= b->num_sends; },
                        "has not run the copy epilogue of the previous dispatch yet");
        // (counted once everything is enqueued: a dispatch that is refused on the way is none to the peers, whose receive
        //  sides would otherwise take the counts of the one before for its)
        const int64_t send = b->num_sends + 1;
        if (cached_mode) {
            // the cached handle already holds the whole layout: only the packed regions are refreshed
            b->last.valid = b->last.layout_pending = b->last.place_pending = false;
            if (num_ranks > 1) {
                launch_pack();
                b->num_sends = send;
            }
            done.record();
            return;
        }

        // scratch carved from the workspace
        const int E = a.num_experts, R = num_ranks, K = num_topk;
        const int num_blocks = std::max<int>(1, (int)ceil_div(num_tokens, EP_TOKENS_PER_BLOCK));
        int* ws = (int*)b->workspace();
        int64_t off = boxes.end / sizeof(int);
        auto carve = [&](int64_t n) {
            int* p = ws + off;
            off += align_up(std::max<int64_t>(n, 1), 64);
            return p;
        };
        EpLayoutArgs la{};
        la.count_experts = boxes.used ? E : E / R;
        la.count_lo = boxes.used ? 0 : b->rank_idx * (E / R);
        la.count_box_off = boxes.used ? boxes.count_off : 0;
        la.cnt_stride = (int)align_up(la.count_experts + R, 8);
        la.col_total = carve(la.cnt_stride);
        la.blk_cnt = carve((int64_t)num_blocks * la.cnt_stride);
        if (R == 1 or boxes.used) la.slot_map = carve((int64_t)num_tokens * K);
        if (R == 1) la.tok_row = carve(num_tokens);
        rank_map = la.slot_map;
        if (b->is_static and off * (int64_t)sizeof(int) > b->workspace_bytes)
            throw EpError{format("Assertion exception (%s:%d): the layout scratch of %d tokens x top-%d over %d experts (%lld bytes) "
                                 "exceeds the library's static scratch of %lld bytes", __FILE_NAME__, __LINE__, num_tokens, K, E,
                                 (long long)(off * (int64_t)sizeof(int)), (long long)b->workspace_bytes)};
        EP_HOST_ASSERT(off * (int64_t)sizeof(int) <= b->workspace_bytes);
        // more than one partition: this launch is the send side only (slots in the destinations' regions, row
        // counts into their inboxes); the receive side is ep_dispatch_recv_launch
        la.peer_arenas = b->peer_table();
        la.connected = b->connected ? 1 : 0;

        la.topk_idx = (const int64_t*)a.topk_idx.data;
        la.num_tokens = num_tokens;
        la.num_topk = K;
        la.num_experts = E;
        la.num_ranks = R;
        la.rank_idx = b->rank_idx;
        la.expert_alignment = a.expert_alignment;
        la.max_tokens = a.num_max_tokens_per_rank;
        la.experts_per_rank = num_experts_per_rank;
        la.num_blocks = num_blocks;
        la.seq = R == 1 ? ++b->seq : (int)send;
        la.notify_host = do_cpu_sync and R == 1 ? 1 : 0;
        // a node in this process: the counts go to every receiver's host as well (arenas that were only mapped here
        // have no host pages this process knows: their counts come from the receive side)
        const bool notify_peers = boxes.used and do_cpu_sync and not b->peers.empty() and R <= EP_HOST_BOXES_MAX_RANKS;
        if (notify_peers) {
            la.host_boxes = (int* const*)(b->workspace() + EP_WS_HOST_BOXES_OFF);
            la.host_box_slot = (send & 1) * EP_HOST_BOX_INTS;
        }
        la.dst_buffer_slot_idx = (int*)a.dst_buffer_slot_idx.data;
        la.dst_gsge_idx = (int*)a.dst_gsge_idx.data;
        la.psum_rank = (int*)psum_rank.data;
        la.psum_expert = (int*)psum_expert.data;
        la.unaligned_expert = (int*)unaligned.data;
        la.cumulative_stats = (int*)a.cumulative_local_expert_recv_stats.data;
        la.host_page = b->host_page_dev;

        const bool small = small_dispatch(num_tokens, K);
        const bool one_launch = small or chunk_dispatch(num_tokens, K, E, R, row_parts(hidden, (int64_t)hidden * x_elem, a.fused_fp8_quant != 0));
        b->last.layout_pending = b->last.place_pending = b->last.copied = false;
        if (one_launch and num_ranks > 1) {
            own_layout = &la;
        } else if ((small and epilogue == Epilogue::next) or (one_launch and epilogue == Epilogue::only)) {
            b->last.layout_pending = true;
            b->last.pending = la;
        } else {
            launch_layout(la, num_blocks, a.stream);
        }

        if (num_ranks > 1) {
            launch_pack();
            b->num_sends = send;
        }

        b->last.valid = true;
        b->last.stamp = ++b->launch_stamp;
        b->last.num_tokens = num_tokens;
        b->last.num_topk = K;
        b->last.num_experts = E;
        b->last.alignment = a.expert_alignment;
        b->last.max_tokens = a.num_max_tokens_per_rank;
        b->last.slot_map = la.slot_map;
        b->last.tok_row = la.tok_row;
        b->last.ships_ranks = boxes.used;
        b->last.notifies_peers = notify_peers;
        b->last.host_boxes = false;
        b->last.notified = do_cpu_sync and R == 1;
        b->last.recv_done = false;
        done.record();
    });
}

int ep_dispatch_launch(ep_buffer_t* b, const ep_dispatch_args_t* pa) { return dispatch_launch(b, pa, Epilogue::any); }
int ep_dispatch_launch_event(ep_buffer_t* b, const ep_dispatch_args_t* pa, void* event) { return dispatch_launch(b, pa, Epilogue::any, event); }
int ep_dispatch_begin(ep_buffer_t* b, const ep_dispatch_args_t* pa) { return dispatch_launch(b, pa, Epilogue::next); }
int ep_dispatch_begin_only(ep_buffer_t* b, const ep_dispatch_args_t* pa) { return dispatch_launch(b, pa, Epilogue::only); }

int64_t ep_dispatch_stamp(ep_buffer_t* b) {
    return (b == nullptr || b->destroyed || !b->last.valid) ? 0 : b->last.stamp;
}

void ep_set_layout_fold_max_blocks(int num_blocks) { g_fold_max_blocks = num_blocks; }

void ep_set_layout_recount_limit(int blocks_times_topk) { g_recount_limit = blocks_times_topk; }

void ep_set_combine_blocks_per_cu(int num_blocks) { g_combine_blocks_per_cu = num_blocks; }

static void launch_place(const ep_buffer_t* b, EpLayoutArgs& la, void* stream) {
    launch(g_k.layout_place, (unsigned)la.num_blocks + 1u, EP_LAYOUT_THREADS,
           layout_place_lds(la.num_experts, la.num_ranks, la.num_topk), stream, la);
}

static int dispatch_recv(ep_buffer_t* b, const ep_dispatch_recv_args_t* pa, bool epilogue_follows) {
    return guarded([&] {
        EP_HOST_ASSERT(pa != nullptr);
        check_buffer(b);
        const ep_dispatch_recv_args_t& a = *pa;
        const int R = b->num_ranks;
        if (R == 1) return;             // one partition: ep_dispatch_launch has produced the whole layout
        EP_HOST_ASSERT(b->last.valid and not b->last.recv_done and "follows this buffer's own ep_dispatch_launch");
        EP_HOST_ASSERT(a.dispatch_stamp == b->last.stamp and "the receive side belongs to the latest dispatch launch of this buffer");
        check_peers(b, [&](const ep_buffer& p) { return p.num_sends >= b->num_sends; },
                    "its ep_dispatch_launch comes before any receive side");
        const int K = a.num_topk, E = a.num_experts;
        EP_HOST_ASSERT(K == b->last.num_topk and E == b->last.num_experts);
        EP_HOST_ASSERT(a.expert_alignment == b->last.alignment and a.num_max_tokens_per_rank == b->last.max_tokens);
        const int El = E / R;
        const auto& psum_rank = a.psum_num_recv_tokens_per_rank;
        const auto& psum_expert = a.psum_num_recv_tokens_per_expert;
        const auto& unaligned = a.num_unaligned_recv_tokens_per_expert;
        EP_HOST_ASSERT(present(psum_rank) and psum_rank.ndim == 1 and psum_rank.size[0] == R);
        EP_HOST_ASSERT(present(psum_expert) and psum_expert.ndim == 1 and psum_expert.size[0] == El);
        EP_HOST_ASSERT(present(unaligned) and unaligned.ndim == 1 and unaligned.size[0] == El);
        EP_HOST_ASSERT(psum_rank.dtype == EP_DTYPE_I32 and psum_expert.dtype == EP_DTYPE_I32);
        EP_HOST_ASSERT(unaligned.dtype == EP_DTYPE_I32);
        EP_HOST_ASSERT(contiguous(psum_rank) and contiguous(psum_expert) and contiguous(unaligned));
        if (present(a.cumulative_local_expert_recv_stats)) {
            const auto& st = a.cumulative_local_expert_recv_stats;
            EP_HOST_ASSERT(st.ndim == 1 and st.size[0] == El and contiguous(st) and st.dtype == EP_DTYPE_I32);
        }
        const auto& meta = a.recv_src_metadata;
        EP_HOST_ASSERT(present(meta) and meta.ndim == 2 and meta.size[1] == K + 2);
        EP_HOST_ASSERT(contiguous(meta) and meta.dtype == EP_DTYPE_I32);
        const int64_t rows_bound = b->recv_rows_bound(b->last.num_tokens, a.num_max_tokens_per_rank);
        EP_HOST_ASSERT(meta.size[0] >= rows_bound and "room for every row that can arrive");
        EP_HOST_ASSERT(rows_bound <= INT32_MAX);
        EP_HOST_ASSERT(a.hidden_bytes > 0 and a.num_sf_packs >= 0);
        const PackedToken pk = packed_token(a.hidden_bytes, a.num_sf_packs * 2, K, true);
        EP_HOST_ASSERT((int64_t)R * a.num_max_tokens_per_rank * pk.bytes <= b->num_buffer_bytes);
        EP_HOST_ASSERT(a.num_sf_packs == 0 or a.hidden_bytes % kUbAlign == 0);      // see ep_dispatch_launch

        const int num_blocks = std::max<int>(1, (int)ceil_div(rows_bound, EP_TOKENS_PER_BLOCK));
        int* ws = (int*)b->workspace();
        const RankBoxes boxes = rank_boxes(b, a.num_max_tokens_per_rank, K, E);
        int64_t off = boxes.end / sizeof(int);
        auto carve = [&](int64_t n) {
            int* p = ws + off;
            off += align_up(std::max<int64_t>(n, 1), 64);
            return p;
        };
        EP_HOST_ASSERT(boxes.used == b->last.ships_ranks and "the node is connected as it was at the dispatch launch");
        EpLayoutArgs la{};
        la.count_experts = El;
        la.count_lo = b->rank_idx * El;
        la.cnt_stride = (int)align_up(E / R + R, 8);
        if (boxes.used) {
            la.count_box = (const int*)(b->workspace() + boxes.count_off);
            la.rank_box = (const int*)(b->workspace() + boxes.rank_off);
        } else {
            la.col_total = carve(la.cnt_stride);
            la.blk_cnt = carve((int64_t)num_blocks * la.cnt_stride);
        }
        EP_HOST_ASSERT(off * (int64_t)sizeof(int) <= b->workspace_bytes and "layout scratch of the receive stream fits the workspace");
        la.recv_mode = 1;
        la.num_tokens = (int)rows_bound;
        la.num_topk = K;
        la.num_experts = E;
        la.num_ranks = R;
        la.rank_idx = b->rank_idx;
        la.expert_alignment = a.expert_alignment;
        la.max_tokens = a.num_max_tokens_per_rank;
        la.experts_per_rank = El;
        la.num_blocks = num_blocks;
        // every source has left its counts with this partition's host (or will, before this launch runs)
        bool told = boxes.used and not b->peers.empty();
        for (const ep_buffer* p : b->peers) told = told and p->last.valid and p->last.notifies_peers and p->num_sends == b->num_sends;
        la.seq = ++b->seq;
        la.notify_host = a.do_cpu_sync and not told ? 1 : 0;
        la.psum_rank = (int*)psum_rank.data;
        la.psum_expert = (int*)psum_expert.data;
        la.unaligned_expert = (int*)unaligned.data;
        la.cumulative_stats = (int*)a.cumulative_local_expert_recv_stats.data;
        la.host_page = b->host_page_dev;
        la.peer_arenas = b->peer_table();
        la.connected = b->connected ? 1 : 0;
        la.inbox = b->inbox();
        la.packed_base = b->buffer();
        la.packed_row_bytes = pk.bytes;
        la.idx_off = pk.idx_off;
        la.src_off = pk.src_off;
        la.recv_src_metadata = (int*)meta.data;
        la.rows_cap = (int)std::min<int64_t>(meta.size[0], INT32_MAX);
        // (a host that waits for counts of this launch waits before the epilogue: then it cannot be left to it)
        b->last.place_pending = epilogue_follows and boxes.used and R <= kRecvCopyMaxRanks and la.notify_host == 0;
        if (b->last.place_pending)
            b->last.pending = la;
        else if (boxes.used)
            launch_place(b, la, a.stream);
        else
            launch_layout(la, num_blocks, a.stream);
        b->last.recv_done = true;
        b->last.notified = a.do_cpu_sync != 0;
        b->last.host_boxes = a.do_cpu_sync != 0 and told;
        b->last.counted_rows = -1;
        b->last.send_seq = (int)b->num_sends;
    });
}

int ep_dispatch_recv_launch(ep_buffer_t* b, const ep_dispatch_recv_args_t* pa) { return dispatch_recv(b, pa, false); }
int ep_dispatch_recv_begin(ep_buffer_t* b, const ep_dispatch_recv_args_t* pa) { return dispatch_recv(b, pa, true); }

int ep_dispatch_wait_counts(ep_buffer_t* b, int* num_recv_tokens, int* num_expanded_tokens, int* per_expert) {
    return guarded([&] {
        EP_HOST_ASSERT(b != nullptr and not b->destroyed);
        EP_HOST_ASSERT(b->last.valid);
        EP_HOST_ASSERT(not b->last.layout_pending and "the copy epilogue of an ep_dispatch_begin comes before the counts");
        EP_HOST_ASSERT(b->last.notified and "the last dispatch was launched with do_cpu_sync (nothing else publishes the counts)");
        const auto deadline = std::chrono::steady_clock::now() + std::chrono::seconds(b->cpu_timeout_secs);
        volatile int* page = b->host_page;
        if (b->last.host_boxes) {
            // sum what the sources left here; the host does not wait for this partition's own receive side
            const int R = b->num_ranks, El = b->last.num_experts / R;
            volatile int* box = page + EP_HOST_PAGE_INTS + (b->last.send_seq & 1) * EP_HOST_BOX_INTS;
            int rows = 0, expanded = 0;
            for (int s = 0; s < R; ++s) {
                while (__atomic_load_n(&box[EP_HOST_BOX_SEQ_OFF + s], __ATOMIC_ACQUIRE) != b->last.send_seq) {
                    if (std::chrono::steady_clock::now() >= deadline) EP_HOST_UNREACHABLE("reduction timeout");
                }
                rows += box[EP_HOST_BOX_ROWS_OFF + s];
            }
            for (int e = 0; e < El; ++e) {
                int count = 0;
                for (int s = 0; s < R; ++s) count += box[s * El + e];
                const int aligned = (int)align_up(count, b->last.alignment);
                if (per_expert != nullptr) per_expert[e] = aligned;
                expanded += aligned;
            }
            if (num_recv_tokens != nullptr) *num_recv_tokens = rows;
            if (num_expanded_tokens != nullptr) *num_expanded_tokens = expanded;
            b->last.counted_rows = rows;
            return;
        }
        while (__atomic_load_n(&page[0], __ATOMIC_ACQUIRE) != b->seq) {
            if (std::chrono::steady_clock::now() >= deadline) EP_HOST_UNREACHABLE("reduction timeout");
        }
        if (num_recv_tokens != nullptr) *num_recv_tokens = page[1];
        if (num_expanded_tokens != nullptr) *num_expanded_tokens = page[2];
        if (per_expert != nullptr) {
            const int El = b->last.num_experts / b->num_ranks;
            for (int e = 0; e < El; ++e) per_expert[e] = page[EP_HOST_EXPERT_OFF + e];
        }
    });
}

int ep_dispatch_worst_case_sizes(ep_buffer_t* b, int max_tokens, int num_topk, int num_experts, int alignment,
                                 int* num_recv_tokens, int* num_expanded_tokens) {
    return guarded([&] {
        EP_HOST_ASSERT(b == nullptr or not b->destroyed);
        const int num_ranks = b == nullptr ? 1 : b->num_ranks;      // no buffer: one partition
        EP_HOST_ASSERT(num_experts % num_ranks == 0 and alignment > 0);
        const int El = num_experts / num_ranks;
        int64_t n = (int64_t)num_ranks * max_tokens * std::min(num_topk, El);
        n += (int64_t)(alignment - 1) * El;
        n = align_up(n, alignment);
        EP_HOST_ASSERT(n <= INT32_MAX);
        *num_recv_tokens = num_ranks * max_tokens;
        *num_expanded_tokens = (int)n;
    });
}

int ep_dispatch_epilogue_launch(ep_buffer_t* b, const ep_dispatch_epilogue_args_t* pa) {
    return guarded([&] {
        EP_HOST_ASSERT(pa != nullptr);
        check_buffer(b);
        const ep_dispatch_epilogue_args_t& a = *pa;
        const bool cached_mode = a.cached_mode != 0;
        EP_HOST_ASSERT(present(a.x) and a.x.ndim == 2 and contiguous(a.x));
        const int num_tokens = (int)a.x.size[0];
        const int hidden = (int)a.x.size[1];
        const int K = a.num_topk;
        const int R = b->num_ranks;
        EP_HOST_ASSERT(K > 0 and K <= EP_MAX_TOPK);
        EP_HOST_ASSERT(a.num_experts % R == 0);
        const int El = a.num_experts / R;
        const bool fused = a.fused_fp8_quant != 0;
        // the same input contract as ep_dispatch_launch: this entry point may be called on its own
        if (present(a.sf)) {
            EP_HOST_ASSERT(not fused and a.x.dtype == EP_DTYPE_FP8_E4M3);
            EP_HOST_ASSERT(a.sf.ndim == 2 and a.sf.size[0] == num_tokens and elem_size(a.sf.dtype) == 2);
            EP_HOST_ASSERT(a.sf.stride[0] == 1 or a.sf.stride[1] == 1);
            EP_HOST_ASSERT(a.sf.stride[0] <= INT32_MAX and a.sf.stride[1] <= INT32_MAX);
        } else {
            EP_HOST_ASSERT(a.x.dtype == EP_DTYPE_BF16);
        }
        EP_HOST_ASSERT(not fused or (hidden % 8 == 0 and hidden <= 16384));
        EP_HOST_ASSERT(a.num_max_tokens_per_rank > 0 and num_tokens <= a.num_max_tokens_per_rank);
        EP_HOST_ASSERT(a.expert_alignment > 0);
        EP_HOST_ASSERT(present(a.recv_x) and a.recv_x.ndim == 2 and a.recv_x.size[1] == hidden);
        EP_HOST_ASSERT(contiguous(a.recv_x));
        EP_HOST_ASSERT(a.recv_x.dtype == (fused ? (int)EP_DTYPE_FP8_E4M3 : a.x.dtype));
        const int64_t num_expanded = a.recv_x.size[0];
        const bool has_sf = present(a.sf) or fused;
        int num_sf_packs = 0;
        if (has_sf) {
            EP_HOST_ASSERT(present(a.recv_sf) and a.recv_sf.ndim == 2 and a.recv_sf.size[0] == num_expanded);
            if (fused) {
                EP_HOST_ASSERT(a.recv_sf.dtype == EP_DTYPE_F32 and a.recv_sf.size[1] == ceil_div(hidden, 128));
            } else {
                EP_HOST_ASSERT(elem_size(a.recv_sf.dtype) == 2 and a.recv_sf.size[1] == a.sf.size[1]);
                num_sf_packs = (int)a.sf.size[1];
            }
            // row-major scale rows (csrc/kernels/ep/dispatch.hpp:112-113), or the column-major result of
            // the reference's transposing pass (csrc/buffers/ep.hpp:379-381) written in place
            EP_HOST_ASSERT(a.recv_sf_layout >= EP_SF_ROW_MAJOR and a.recv_sf_layout <= EP_SF_COL_MAJOR_COUNTED);
            if (a.recv_sf_layout == EP_SF_ROW_MAJOR) {
                EP_HOST_ASSERT(a.recv_sf.stride[1] == 1 and a.recv_sf.stride[0] == a.recv_sf.size[1]);
            } else {
                EP_HOST_ASSERT(a.recv_sf.stride[0] == 1 and a.recv_sf.stride[1] == a.recv_sf.size[0]);
                // the copy kernel writes scale rows into the staging tensor, a second kernel turns them
                const ep_tensor_t& st = a.recv_sf_staging;
                EP_HOST_ASSERT(present(st) and st.ndim == 2 and st.dtype == a.recv_sf.dtype);
                EP_HOST_ASSERT(st.size[0] == a.recv_sf.size[0] and st.size[1] == a.recv_sf.size[1]);
                EP_HOST_ASSERT(st.stride[1] == 1 and st.stride[0] == st.size[1] and st.data != a.recv_sf.data);
            }
        }
        if (present(a.topk_weights)) {
            EP_HOST_ASSERT(present(a.recv_topk_weights) and a.recv_topk_weights.ndim == 1);
            EP_HOST_ASSERT(a.recv_topk_weights.size[0] == num_expanded and a.recv_topk_weights.dtype == EP_DTYPE_F32);
            EP_HOST_ASSERT(a.topk_weights.ndim == 2 and a.topk_weights.size[0] == num_tokens and a.topk_weights.size[1] == K);
            EP_HOST_ASSERT(contiguous(a.topk_weights) and a.topk_weights.dtype == EP_DTYPE_F32);
            EP_HOST_ASSERT(contiguous(a.recv_topk_weights));
        }
        EP_HOST_ASSERT(present(a.recv_src_metadata) and a.recv_src_metadata.ndim == 2);
        EP_HOST_ASSERT(a.recv_src_metadata.size[1] == K + 2);
        EP_HOST_ASSERT(contiguous(a.recv_src_metadata));
        EP_HOST_ASSERT(a.recv_src_metadata.dtype == EP_DTYPE_I32);
        for (const ep_tensor_t* ps : {&a.psum_num_recv_tokens_per_rank, &a.psum_num_recv_tokens_per_expert})
            EP_HOST_ASSERT(present(*ps) and ps->ndim == 1 and contiguous(*ps) and ps->dtype == EP_DTYPE_I32);
        EP_HOST_ASSERT(a.psum_num_recv_tokens_per_rank.size[0] == R and a.psum_num_recv_tokens_per_expert.size[0] == El);
        if (not cached_mode) {
            EP_HOST_ASSERT(b->last.valid and "the copy epilogue follows its own dispatch launch");
            // the slot map and the receive order live in the workspace, which every dispatch launch overwrites
            EP_HOST_ASSERT(a.dispatch_stamp == b->last.stamp and "the copy epilogue belongs to the latest dispatch launch of this buffer");
            EP_HOST_ASSERT(b->last.num_tokens == num_tokens and b->last.num_topk == K);
            EP_HOST_ASSERT((R == 1 or b->last.recv_done) and "the receive-side layout comes before the copy");
        }
        if (R > 1) {
            check_peers(b, [&](const ep_buffer& p) { return p.num_sends >= b->num_sends; },
                        "its ep_dispatch_launch comes before any copy epilogue");
            b->num_expands = b->num_sends;
        }

        EpScatterArgs sa{};
        sa.topk_weights = (const float*)a.topk_weights.data;
        sa.slot_map = b->last.slot_map;
        sa.tok_row = b->last.tok_row;
        sa.num_recv_ptr = (const int*)a.psum_num_recv_tokens_per_rank.data + (R - 1);
        sa.recv_src_metadata = (int*)a.recv_src_metadata.data;
        sa.recv_x = a.recv_x.data;
        const bool sf_columns = has_sf and a.recv_sf_layout != EP_SF_ROW_MAJOR;
        sa.recv_sf = has_sf ? (sf_columns ? a.recv_sf_staging.data : a.recv_sf.data) : nullptr;
        sa.recv_topk_weights = present(a.topk_weights) ? (float*)a.recv_topk_weights.data : nullptr;
        sa.psum_expert = (const int*)a.psum_num_recv_tokens_per_expert.data;
        sa.out_row_bytes = (int64_t)hidden * elem_size(a.recv_x.dtype);
        sa.out_sf_row_bytes = has_sf ? a.recv_sf.size[1] * elem_size(a.recv_sf.dtype) : 0;
        sa.hidden = hidden;
        sa.num_topk = K;
        // never walk past the rows the metadata tensor holds
        sa.num_rows_bound = (int)std::min<int64_t>(b->recv_rows_bound(num_tokens, a.num_max_tokens_per_rank),
                                                   a.recv_src_metadata.size[0]);
        sa.num_meta_rows = (int)std::min<int64_t>(a.recv_src_metadata.size[0], INT32_MAX);
        sa.num_tokens = num_tokens;
        sa.rank_idx = b->rank_idx;
        sa.max_tokens = a.num_max_tokens_per_rank;
        sa.cached = cached_mode ? 1 : 0;
        sa.num_local_experts = El;
        sa.expert_alignment = a.expert_alignment;
        sa.num_out_rows = (int)std::min<int64_t>(num_expanded, INT32_MAX);
        bool quantise_here = fused;
        if (R == 1) {
            // one partition: the packed intermediate is skipped, rows come straight from x
            sa.mode = EP_SCATTER_EXPAND;
            if (not cached_mode) {
                // the tasks walk the tokens, not the receive stream: no device count bounds them
                sa.num_recv_ptr = nullptr;
                sa.num_rows_bound = num_tokens;
            }
            // a cached handle that holds one metadata row per token: row i is token i (the rows ascend with the token)
            sa.rows_are_tokens = cached_mode and a.recv_src_metadata.size[0] == num_tokens ? 1 : 0;
            sa.x = a.x.data;
            sa.sf = a.sf.data;
            sa.x_row_bytes = (int64_t)hidden * elem_size(a.x.dtype);
            sa.copy_bytes = sa.x_row_bytes;
            if (present(a.sf)) {
                sa.sf_token_stride_bytes = a.sf.stride[0] * 2;
                sa.sf_pack_stride_bytes = a.sf.stride[1] * 2;
            }
            sa.num_sf_packs = num_sf_packs;
        } else {
            // expand this partition's own region of the packed rows written by ep_dispatch_launch
            const int payload_elem = fused ? 1 : elem_size(a.x.dtype);
            const int sf_packs = fused ? 2 * (int)ceil_div(hidden, 128) : num_sf_packs;
            const PackedToken pk = packed_token(hidden * payload_elem, sf_packs * 2, K, not cached_mode);
            EP_HOST_ASSERT((int64_t)R * a.num_max_tokens_per_rank * pk.bytes <= b->num_buffer_bytes);
            EP_HOST_ASSERT(sf_packs == 0 or (int64_t)hidden * payload_elem % kUbAlign == 0);   // see ep_dispatch_launch
            sa.mode = EP_SCATTER_REGION;
            sa.psum_rank = (const int*)a.psum_num_recv_tokens_per_rank.data;
            sa.num_ranks = R;
            sa.x = b->buffer();
            sa.x_row_bytes = pk.bytes;
            sa.copy_bytes = (int64_t)hidden * payload_elem;
            sa.sf = sf_packs > 0 ? b->buffer() + pk.sf_off : nullptr;
            sa.sf_token_stride_bytes = pk.bytes;
            sa.sf_pack_stride_bytes = 2;
            sa.num_sf_packs = sf_packs;
            sa.w_off = pk.w_off;
            quantise_here = false;
        }
        sa.sf_pairs = quantise_here ? 0 : sf_pairs(sa, sa.recv_sf);
        // a wave task covers 1 KiB of a verbatim row (4 KiB of a packed row, which mostly has one destination
        // among this partition's few experts), or 512 channels of a row being quantised
        sa.vecs_per_lane = sa.mode == EP_SCATTER_REGION ? 4 : 1;
        sa.num_parts = row_parts(hidden, ceil_div(sa.copy_bytes, sa.vecs_per_lane), quantise_here);
        const int64_t row_blocks = ceil_div((int64_t)sa.num_rows_bound * sa.num_parts, EP_ROWS_PER_BLOCK);
        EP_HOST_ASSERT(row_blocks <= INT32_MAX / 2);
        sa.num_row_blocks = (int)row_blocks;
        // rows are read in 16-byte vectors; the verbatim kernel writes them so, the quantising one 8 bytes a lane
        EP_HOST_ASSERT(sa.x_row_bytes % 16 == 0 and sa.out_row_bytes % (quantise_here ? 8 : 16) == 0);
        // an expert has at most alignment - 1 padding rows: about one workgroup per 8 of them (measured: 16 a
        // expert at alignment 128 and 32 or 64 give the same time; one per 4 KiB chunk, 223 a expert, is 10-20 %
        // slower: every workgroup first waits for the expert's row count)
        sa.pad_blocks_per_expert = std::max(1, std::min(EP_MAX_PAD_BLOCKS_PER_EXPERT, a.expert_alignment / 8));
        const unsigned pad_blocks = a.do_zero_padding and a.expert_alignment > 1 ? (unsigned)(El * sa.pad_blocks_per_expert) : 0u;
        const unsigned grid = (unsigned)sa.num_row_blocks + pad_blocks;
        const bool pending = not cached_mode and b->last.layout_pending;      // (a cached epilogue in between leaves it waiting)
        // the receive side of an ep_dispatch_recv_begin: placed by the copy launch where that writes what the begin was given
        // (every row that can have arrived, into the same tensors, padded alike), else by a launch in front of it
        bool place_here = not cached_mode and b->last.place_pending;
        if (place_here) {
            EpLayoutArgs& la = b->last.pending;
            EP_HOST_ASSERT(b->connected and "the node is connected as it was at the receive side");
            const int64_t rows = b->last.counted_rows >= 0 ? b->last.counted_rows : std::min<int64_t>(la.num_tokens, la.rows_cap);
            place_here = sa.num_rows_bound >= rows and la.recv_src_metadata == sa.recv_src_metadata and la.psum_rank == sa.psum_rank and
                         la.psum_expert == sa.psum_expert and la.num_topk == K and la.num_experts == a.num_experts and
                         la.expert_alignment == a.expert_alignment and la.max_tokens == sa.max_tokens and
                         la.packed_row_bytes == sa.x_row_bytes and recv_copy_pays(a.num_experts, sa.num_row_blocks);
            if (not place_here) {
                launch_place(b, la, a.stream);
                b->last.place_pending = false;
            }
        }
        EP_HOST_ASSERT((cached_mode or not b->last.copied) and "an ep_dispatch_begin has one copy epilogue");
        if (pending) {
            // (one partition, tokens and metadata rows at hand: there are row workgroups.  The layout runs on this call's
            // stream, whichever the begin came on: a caller who changes streams has ordered this one behind the begin)
            EP_HOST_ASSERT(sa.num_row_blocks > 0);
            // the one launch sizes its LDS by the begin's experts and pads by the epilogue's
            EP_HOST_ASSERT(a.num_experts == b->last.num_experts and a.expert_alignment == b->last.alignment and
                           "the copy epilogue has the experts and the alignment of its ep_dispatch_begin");
            if (small_dispatch(num_tokens, K))
                launch_small(b->last.pending, sa, false, quantise_here,
                             (int)small_pad_blocks(pad_blocks, num_tokens, K, El, a.expert_alignment, sa.out_row_bytes), a.stream);
            else
                launch_chunk(b->last.pending, sa, false, quantise_here, pad_blocks, a.stream);
            b->last.layout_pending = false;
            b->last.copied = true;
        } else if (place_here) {
            EpSmallArgs args{};
            args.l = b->last.pending;
            args.s = sa;
            args.num_pad_blocks = (int)pad_blocks;
            EP_HOST_ASSERT(args.l.notify_host == 0);       // (that kernel announces nothing)
            launch(g_k.recv_copy, 1u + grid, EP_ROW_THREADS, recv_copy_lds(a.num_experts, R), a.stream, args);
            b->last.place_pending = false;
        } else if (grid > 0) {
            hipFunction_t fn = quantise_here ? (g_fp8_hw ? g_k.scatter_quant : g_k.scatter_quant_sw) : g_k.scatter_copy;
            launch(fn, grid, EP_ROW_THREADS, 0, a.stream, sa);
        }
        if (sf_columns and num_expanded > 0) {
            EpSfTransposeArgs ta{};
            ta.src = a.recv_sf_staging.data;
            ta.dst = a.recv_sf.data;
            ta.psum_expert = sa.psum_expert;
            ta.num_rows = sa.num_out_rows;
            ta.num_cols = (int)a.recv_sf.size[1];
            ta.elem_bytes = elem_size(a.recv_sf.dtype);
            ta.counted = a.recv_sf_layout == EP_SF_COL_MAJOR_COUNTED ? 1 : 0;
            ta.num_local_experts = El;
            ta.expert_alignment = a.expert_alignment;
            launch(g_k.sf_transpose, (unsigned)ceil_div(ta.num_rows, EP_SF_TILE), EP_LAYOUT_THREADS, 0, a.stream, ta);
        }
    });
}

// ---- combine ----------------------------------------------------------------------------------
static int combine_launch(ep_buffer_t* b, const ep_combine_args_t* pa, int phase, void* event) {
    return guarded([&] {
        EP_HOST_ASSERT(pa != nullptr);
        check_buffer(b);
        const ep_combine_args_t& a = *pa;
        DoneEvent done(event, a.stream, b);
        const int R = b->num_ranks;
        EP_HOST_ASSERT(a.num_experts > 0 and a.num_experts % R == 0);

        EP_HOST_ASSERT(present(a.x) and a.x.ndim == 2);
        const int num_tokens = (int)a.x.size[0];
        const int hidden = (int)a.x.size[1];
        EP_HOST_ASSERT(contiguous(a.x));
        EP_HOST_ASSERT(a.x.dtype == EP_DTYPE_BF16);
        EP_HOST_ASSERT(hidden % 8 == 0);

        EP_HOST_ASSERT(present(a.combined_topk_idx) and a.combined_topk_idx.ndim == 2);
        const int num_combined_tokens = (int)a.combined_topk_idx.size[0];
        const int K = (int)a.combined_topk_idx.size[1];
        EP_HOST_ASSERT(K > 0 and K <= EP_MAX_TOPK);
        EP_HOST_ASSERT(num_combined_tokens <= a.num_max_tokens_per_rank);
        EP_HOST_ASSERT(contiguous(a.combined_topk_idx));
        EP_HOST_ASSERT(a.combined_topk_idx.dtype == EP_DTYPE_I64);
        EP_HOST_ASSERT(present(a.src_metadata) and a.src_metadata.ndim == 2 and a.src_metadata.size[1] == K + 2);
        EP_HOST_ASSERT(a.src_metadata.size[0] <= (int64_t)R * a.num_max_tokens_per_rank);
        EP_HOST_ASSERT(contiguous(a.src_metadata));
        EP_HOST_ASSERT(a.src_metadata.dtype == EP_DTYPE_I32);
        const auto& psum_rank = a.psum_num_recv_tokens_per_rank;
        EP_HOST_ASSERT(present(psum_rank) and psum_rank.ndim == 1);
        EP_HOST_ASSERT(psum_rank.size[0] == R);
        EP_HOST_ASSERT(contiguous(psum_rank));
        EP_HOST_ASSERT(psum_rank.dtype == EP_DTYPE_I32);

        if (present(a.topk_weights)) {
            EP_HOST_ASSERT(a.topk_weights.ndim == 1 and a.topk_weights.size[0] == num_tokens);
            EP_HOST_ASSERT(contiguous(a.topk_weights));
            EP_HOST_ASSERT(a.topk_weights.dtype == EP_DTYPE_F32);
        }
        EP_HOST_ASSERT(not a.apply_weights or present(a.topk_weights));
        const ep_tensor_t* biases[2] = {&a.bias_0, &a.bias_1};
        for (const ep_tensor_t* bias : biases) {
            if (present(*bias)) {
                EP_HOST_ASSERT(bias->ndim == 2);
                EP_HOST_ASSERT(bias->size[0] == num_combined_tokens and bias->size[1] == hidden);
                EP_HOST_ASSERT(contiguous(*bias));
                EP_HOST_ASSERT(bias->dtype == a.x.dtype);
            }
        }
        EP_HOST_ASSERT(combine_buffer_size(R, a.num_max_tokens_per_rank, hidden, K) <= b->num_buffer_bytes);
        EP_HOST_ASSERT(phase == 0 or phase == 1);
        EP_HOST_ASSERT(not a.apply_weights or R == 1);
        const int unrolled = K >= 2 and K <= 8 ? K - 1 : 0;      // (0: the kernel for any top-k)
        const int64_t combine_token = token_bytes(hidden * 2, 0, K, false);

        EpCombineArgs ca{};
        ca.expanded_weights = (const float*)a.topk_weights.data;
        ca.recv_src_metadata = (const int*)a.src_metadata.data;
        ca.topk_idx = (const int64_t*)a.combined_topk_idx.data;
        ca.hidden = hidden;
        ca.num_topk = K;
        ca.num_tokens = num_combined_tokens;
        ca.rank_idx = b->rank_idx;
        ca.max_tokens = a.num_max_tokens_per_rank;
        ca.num_parts = (int)std::max<int64_t>(1, ceil_div(hidden, 1024));
        ca.num_experts = a.num_experts;
        ca.num_ranks = R;
        ca.experts_per_rank = a.num_experts / R;
        ca.num_groups = std::min(K, R);

        if (phase == 0) {
            if (R == 1) return done.record();       // single partition: the whole reduction is one token-side launch
            // the partials land where the peers' packed rows are
            check_peers(b, [&](const ep_buffer& p) { return p.num_expands >= p.num_sends and p.num_sends >= b->num_sends; },
                        "runs its copy epilogue before any combine");
            ++b->num_partials;
            // owner side: one partial per received row into this GPU's combine buffer
            ca.y = a.x.data;
            ca.y_row_bytes = (int64_t)hidden * 2;
            ca.num_in_rows = num_tokens;
            ca.num_recv_ptr = (const int*)psum_rank.data + (R - 1);
            ca.num_rows_bound = (int)a.src_metadata.size[0];
            ca.combined_x = b->buffer();
            ca.peer_arenas = b->peer_table();
            ca.buffer_off = b->workspace_bytes;
            ca.out_row_bytes = combine_token;
            // With few slots a row (less than two selections a partition) the rows are short of loads in flight, and from
            // about 16384 of them on there are enough tasks to give each 2048 channels.  us a launch with 1024 / 2048 / whole
            // rows, top-6 unless noted: 16 partitions, 21k rows 140 / 135 / 151; 8 partitions, 22k (top-8) 166 / 163 / 174;
            // 4 partitions, 27k 200 / 201 / 228; against them 2 partitions, 33k (top-8) 399 / 418 / 466.  At 9k rows of 8
            // partitions the forms are level (68.6 / 68.6 us).
            if (ca.num_rows_bound >= 16384 and K < 2 * R) {
                ca.long_parts = 1;
                ca.num_parts = (int)std::max<int64_t>(1, ceil_div(hidden, EP_COMBINE_LONG_PART));
            }
            ca.num_row_blocks = (int)ceil_div((int64_t)ca.num_rows_bound * ca.num_parts, EP_ROWS_PER_BLOCK);
            // Odd top-k: the unrolled kernels ask for all slots of a row at once and save trips to memory (top-3 with as many registers: 63
            // against 62).  Launches of many wide rows wait for bandwidth, and where most positions are none the shorter bursts of the kernel for any
            // top-k win, as they do for one partition.  us of both reduces of all partitions, that one / unrolled, top-3 / 5 / 7: eight of 64 tokens x
            // 7168 (top-3, top-7) 81.8 / 76.4, 125 / 121; 1024 x 2560 137 / 131, 176 / 171, 214 / 210; 4096 x 1024 186 / 183, 242 / 240, 306 / 301; but 2048 x
            // 7168 460 / 471, 666 / 681, 849 / 852; 4096 x 4096 526 / 548, 752 / 768, in long parts (top-7) 1029 / 1010; 4096 x 7168 851 / 888, 1254 / 1286,
            // in long parts 1682 / 1657.  Four of 1024 x 7168 125 / 125, 160 / 160, 188 / 187; of 4096 394 / 409, 521 / 528, 627 / 633.  16 of 2048 x 2560
            // 433 / 434, 600 / 610, 782 / 813; three and four of 4096 x 2560 top-3 123 / 122, 168 / 168.  Two of 2048 x 7168 93 / 94, 117 / 116, 140 / 137; 8192 x
            // 4096 192 / 200, 245 / 250, 301 / 300; 16384 x 4096 379 / 388, 469 / 491, 578 / 593; x 7168 632 / 640, 789 / 798, 980 / 963.
            const bool few = K < 2 * R, wide = hidden >= 4096;
            const bool one_by_one = K % 2 != 0 and not ca.long_parts and
                                    (few ? ca.num_row_blocks >= 4000 and (wide or (K > 3 and K <= R)) : ca.num_row_blocks >= 12000 and wide and K <= 2 * R + 1);
            if (ca.num_row_blocks > 0)
                launch(g_k.combine[EP_COMBINE_PARTIAL][one_by_one ? 0 : unrolled], (unsigned)ca.num_row_blocks, EP_ROW_THREADS, 0, a.stream, ca, &done);
            return done.record();
        }

        EP_HOST_ASSERT(present(a.combined_x) and a.combined_x.ndim == 2);
        EP_HOST_ASSERT(a.combined_x.size[0] == num_combined_tokens and a.combined_x.size[1] == hidden);
        EP_HOST_ASSERT(contiguous(a.combined_x) and a.combined_x.dtype == EP_DTYPE_BF16);
        if (present(a.topk_weights)) {
            const auto& w = a.combined_topk_weights;
            EP_HOST_ASSERT(present(w) and w.ndim == 2 and w.size[0] == num_combined_tokens and w.size[1] == K);
            EP_HOST_ASSERT(contiguous(w) and w.dtype == EP_DTYPE_F32);
        }
        ca.bias_0 = a.bias_0.data;
        ca.bias_1 = a.bias_1.data;
        ca.combined_x = a.combined_x.data;
        ca.combined_topk_weights = present(a.topk_weights) ? (float*)a.combined_topk_weights.data : nullptr;
        ca.out_row_bytes = (int64_t)hidden * 2;
        if (R == 1) {
            ca.y = a.x.data;
            ca.y_row_bytes = (int64_t)hidden * 2;
            ca.num_in_rows = num_tokens;
            ca.num_recv_ptr = (const int*)psum_rank.data + (R - 1);
            ca.num_rows_bound = (int)a.src_metadata.size[0];
            ca.weighted = a.apply_weights ? 1 : 0;
            ca.num_row_blocks = (int)ceil_div((int64_t)ca.num_rows_bound * ca.num_parts, EP_ROWS_PER_BLOCK);
            const unsigned grid = (unsigned)ca.num_row_blocks + (unsigned)ceil_div(num_combined_tokens, EP_ROW_THREADS);
            if (grid == 0) return;
            // odd top-k: a launch of up to three row blocks a CU, all on their way at once, waits for its trips to memory and takes the unrolled
            // kernel, and so does one that fills the chip several times over; between the two the general one's shorter bursts win.
            // us, general / unrolled, four outputs in turn, top-3 / 5 / 7, 2560 channels unless noted: 384 blocks 6.5 / 6.1, 8.2 / 7.1, 9.9 / 8.4; 766 7.6 /
            // 7.3, 9.5 / 9.0, 11.6 / 11.1; 7168 channels 764 8.2 / 7.8, 10.0 / 9.9, 11.9 / 12.2; 776 8.0 / 7.8, 10.1 / 10.6, 11.8 / 12.8; 800 8.4 / 8.5, 10.3 / 11.0,
            // 12.3 / 13.4 (the same of 1024 to 5120 channels; the third, half part of 2560 puts the line at 860, 790 and 770; top-7 loses from 720 full
            // blocks on: 720 11.7 / 11.7, 750 11.8 / 12.0); 896 8.7 / 9.0, 10.5 / 10.9,
            // 13.0 / 13.7; 1787 13.2 / 14.0, 18.4 / 18.8, 22.8 / 23.5; 3584 24.1 / 24.3, 33.4 / 33.7, 43.2 / 43.7; 5376 33.3 / 32.9, 50.6 / 47.9, 68.2 / 66.0;
            // 28672 155 / 153, 233 / 234, 319 / 314; 6144 (2560 channels) 34.3 / 32.3, 49.6 / 45.6, 67.6 / 60.6
            ca.paced = ca.num_row_blocks >= kPacedRowBlocks ? 1 : 0;
            const bool odd = unrolled != 0 and K % 2 != 0;
            const bool once = ca.num_row_blocks <= 3 * 256 and (K < 7 or (int64_t)ca.num_rows_bound * hidden <= 720 * 4096);
            const int kidx = odd and not once and ca.num_row_blocks < 4096 ? 0 : unrolled;
            const unsigned cap = combine_lds_cap(K + (ca.bias_0 != nullptr) + (ca.bias_1 != nullptr), kidx != 0, odd, ca.num_row_blocks, hidden);
            launch(g_k.combine[EP_COMBINE_FUSED][kidx], grid, EP_ROW_THREADS, cap, a.stream, ca);
        } else {
            check_peers(b, [&](const ep_buffer& p) { return p.num_partials >= b->num_partials; },
                        "its owner-side reduce (phase 0) comes before any token-side reduce");
            // token side: biases + the partial of every master, read from the combine buffer
            ca.y = b->buffer();
            ca.y_row_bytes = combine_token;
            ca.num_in_rows = ca.num_groups * a.num_max_tokens_per_rank;
            ca.num_recv_ptr = nullptr;
            ca.num_rows_bound = num_combined_tokens;
            ca.num_row_blocks = (int)ceil_div((int64_t)ca.num_rows_bound * ca.num_parts, EP_ROW_THREADS / 64);
            if (ca.num_row_blocks == 0) return;
            ca.paced = ca.num_row_blocks >= kPacedRowBlocks ? 1 : 0;
            // The unrolled kernels fetch a row for every position, a master's again where a position is none: most of them with few
            // partitions.  Launches that have more than a trip to wait for take the kernel that goes master by master there, and for
            // top-2 and 3, where it has the more waves.  us of both reduces of all partitions (7168 channels, captured), unrolled / that: two of 64 /
            // 256 / 1024 / 2048 tokens top-8 21.3 / 21.2, 32.6 / 31.3, 90.5 / 79.3, 164 / 143, of 256 top-4 24.5 / 24.0, top-2 21.1 / 21.4; four of 256
            // / 512 / 2048 top-8 77.1 / 79.6, 122 / 117, 379 / 358; eight of 256 / 800 / 2048 top-3 101.5 / 105.9, 228 / 210, 476 / 463, top-6 146 / 163,
            // 346 / 348, a pass of them with a host sync 1234 / 1243; two, three and four of 640 to 2048 tokens top-3 0 to 6 % less; top-2 of five to eight
            // partitions, 960 row blocks of 2560 channels 1 to 2 % more, 1120 of 7168 1 % less.  That against unrolled in % over 1024 to 7168 channels, at 900 / 1000 / 1100 / 1400 / 2000 row blocks: three partitions
            // top-4 0 / 0 / -2 / -2 / -2, top-5 -2 / -1 / -3 / -4 / -4, top-8 -6 / -5 / -9 / -9 / -8; four top-6 -1 / -1 / -2 / -4 / -3, top-8 -3 / -3 / -6 / -6 / -5, but top-5
            // +2 / +2 / 0 / -1 / -1, top-4 +3 / +3 / +1 / 0 / 0 (2560 channels +5 / +4 / +3 / +1 / -3).  Two, at 448 / 520 / 760: top-4 -1 / -2 / -2, top-8 -4 / -7 / -6.
            const int from = R == 2 ? 448 : R == 4 and K == 4 ? 1500 : R == 4 and K == 5 ? 1100 : K == 2 ? 1024 : 896;
            const bool master_by_master = ca.num_row_blocks >= from and (R <= 4 ? K > 2 : K <= 3);
            launch(g_k.combine[EP_COMBINE_FINAL][master_by_master ? 0 : unrolled], (unsigned)ca.num_row_blocks, EP_ROW_THREADS, 0, a.stream, ca);
        }
    });
}

int ep_combine_launch(ep_buffer_t* b, const ep_combine_args_t* pa, int phase) { return combine_launch(b, pa, phase, nullptr); }
int ep_combine_begin_event(ep_buffer_t* b, const ep_combine_args_t* pa, void* event) { return combine_launch(b, pa, 0, event); }

}  // extern "C"

// ---- dispatch without any allocation ------------------------------------------------------------
// For callers that cannot call hipMalloc (code under HIP graph capture, serving loops, harnesses that
// forbid it): the layout scratch that ep_dispatch_launch carves from a buffer's arena lives in a
// file-scope device array instead, so no ep_buffer (whose creation allocates) is needed at all.  Every
// GPU holds its own copy of the array until the process ends; its device address is looked up once per
// device and kept.  The kernels take that address as an argument, exactly as they take the arena's
// workspace.  Every call on a GPU shares the array: calls that overlap on one GPU race.  Nothing in it
// has to start at zero (every word the kernels read was written earlier in the same call).
#define EP_STATIC_SCRATCH_BYTES (4 * 1024 * 1024)
static __device__ __align__(256) unsigned char scratch[EP_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
ep_buffer g_static_view[kMaxDevices];       // host-side views: arena = the device's copy of `scratch`
std::mutex g_static_mutex;

ep_buffer* static_view_of_current_device() {
    int dev = -1;
    HIP_CHECK(hipGetDevice(&dev));
    EP_HOST_ASSERT(dev >= 0 and dev < kMaxDevices);
    EP_HOST_ASSERT(dev == g_k.device and "the kernels were loaded on another device");
    std::lock_guard<std::mutex> lock(g_static_mutex);
    ep_buffer* v = &g_static_view[dev];
    if (v->arena == nullptr) {
        void* ptr = nullptr;
        HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));     // this device's copy; never the array's name
        EP_HOST_ASSERT(ptr != nullptr);
        v->arena = (char*)ptr;
        v->device = dev;
        v->rank_idx = 0;
        v->num_ranks = 1;
        v->num_buffer_bytes = 0;
        v->workspace_bytes = EP_STATIC_SCRATCH_BYTES;
        v->is_static = true;
    }
    return v;
}
}  // namespace

void ep_static_scratch_init() { (void)static_view_of_current_device(); }

// Bytes of the static scratch a single-partition dispatch of this shape carves: the header, then the column
// totals, the count matrix, the slot map and the token -> row map, each rounded up to 64 ints (what
// ep_dispatch_launch carves from a workspace, restated).
extern "C" int64_t ep_dispatch_static_scratch_bytes(int num_tokens, int num_topk, int num_experts) {
    if (num_tokens < 0 or num_topk <= 0 or num_experts <= 0) return -1;
    auto a64 = [](int64_t n) { return align_up(std::max<int64_t>(n, 1), 64); };
    const int64_t W = align_up((int64_t)num_experts + 1, 8);
    const int64_t B = std::max<int64_t>(1, ceil_div(num_tokens, EP_TOKENS_PER_BLOCK));
    return EP_WS_HEADER_BYTES + 4 * (a64(W) + a64(B * W) + a64((int64_t)num_tokens * num_topk) + a64(num_tokens));
}
extern "C" int64_t ep_dispatch_static_scratch_capacity(void) { return EP_STATIC_SCRATCH_BYTES; }

extern "C" int ep_dispatch_static_launch(const ep_dispatch_args_t* d, const ep_dispatch_epilogue_args_t* e) {
    int rc = guarded([&] {
        EP_HOST_ASSERT(d != nullptr and e != nullptr);
        load_kernels(nullptr);
        EP_HOST_ASSERT(not d->cached_mode and not d->do_cpu_sync and not e->cached_mode);
        EP_HOST_ASSERT(d->stream == e->stream);
    });
    if (rc != 0) return rc;
    ep_buffer* v = nullptr;
    rc = guarded([&] { v = static_view_of_current_device(); });
    if (rc != 0) return rc;
    // (an epilogue that pads for other experts or another alignment than the layout's comes behind a layout of its own)
    rc = dispatch_launch(v, d, d->num_experts == e->num_experts and d->expert_alignment == e->expert_alignment ? Epilogue::only : Epilogue::any);
    if (rc != 0) return rc;
    ep_dispatch_epilogue_args_t ee = *e;
    ee.dispatch_stamp = v->last.stamp;
    return ep_dispatch_epilogue_launch(v, &ee);
}
