// Device code object for the EP dispatch/combine path on gfx950 (wave64).  Built ahead of time with
// `hipcc --genco` and launched by the host runtime through hipModuleLaunchKernel.
//
// Kernels (all HBM-bound, no MFMA):
//   ep_layout_count / ep_layout_assign (/ ep_layout_scan)  stable counting sort of the (token, slot)
//       entries by destination partition and by local expert -> every handle tensor; with several
//       partitions once on the send side (slots in the destinations' regions) and, where the send sides
//       ship no ranks, once on the receive side (slots of the rows that arrived).  Two launches up to a few hundred workgroups (the
//       assignment sums the histograms of the workgroups before it itself), three beyond.
//   ep_layout_count_bits / ep_layout_assign_bits           the same two launches for one partition, up to top-8
//   ep_layout_place                                        receive side of a node out of the shipped counts and ranks
//   ep_scatter_copy / ep_scatter_quant                     token (or receive-stream row) -> its expanded slots
//   ep_scatter_copy_pack / ep_scatter_quant_pack           token -> one packed row per destination partition
//   ep_recv_copy                                           ep_layout_place and the copy of the received rows in one launch
//   ep_dispatch_small_*                                    layout and copy (or pack) of a decode-size dispatch in one launch
//   ep_dispatch_chunk_*                                    the same of a dispatch of up to a few thousand tokens
//   ep_sf_transpose                                        scale rows -> scale columns
//   ep_quant_rows                                          the quantiser alone (rows in place)
//   ep_combine_k<K> / ep_combine_generic                   K-way gather + fp32 reduce back to token order
//   ep_combine_partial_* / ep_combine_final_*              the same reduce in its owner-side and token-side halves
//   ep_fp8_selftest                                        hardware vs integer e4m3fn conversion
// (The calibration code object of the benchmarks, ep_calib.hip, includes this file and instantiates some of
// its bodies once more; nothing of it is built into this code object.)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ep_args.h"
#include "ep_fp8.h"

#define WAVE 64

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Streaming stores of the row kernels.  The policy bits of the store instruction (sc0, sc1 = scope,
// nt = non-temporal) decide how the L2 treats the lines; which combination moves rows fastest is a
// measured choice per kernel (EP_*_ST_POL below; bit 0 = nt, bit 1 = sc0, bit 2 = sc1).
template <int POL>
__device__ __forceinline__ void stream_store(u32x4* p, u32x4 v) {
    if (POL == 0) *p = v;
    else if (POL == 1) __builtin_nontemporal_store(v, p);
    else if (POL == 2) asm volatile("global_store_dwordx4 %0, %1, off sc0" ::"v"(p), "v"(v) : "memory");
    else if (POL == 3) asm volatile("global_store_dwordx4 %0, %1, off sc0 nt" ::"v"(p), "v"(v) : "memory");
    else if (POL == 4) asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
    else if (POL == 5) asm volatile("global_store_dwordx4 %0, %1, off sc1 nt" ::"v"(p), "v"(v) : "memory");
    else if (POL == 6) asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt" ::"v"(p), "v"(v) : "memory");
}
template <int POL>
__device__ __forceinline__ void stream_store(u32x2* p, u32x2 v) {
    if (POL == 0) *p = v;
    else if (POL == 1) __builtin_nontemporal_store(v, p);
    else if (POL == 2) asm volatile("global_store_dwordx2 %0, %1, off sc0" ::"v"(p), "v"(v) : "memory");
    else if (POL == 3) asm volatile("global_store_dwordx2 %0, %1, off sc0 nt" ::"v"(p), "v"(v) : "memory");
    else if (POL == 4) asm volatile("global_store_dwordx2 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
    else if (POL == 5) asm volatile("global_store_dwordx2 %0, %1, off sc1 nt" ::"v"(p), "v"(v) : "memory");
    else if (POL == 6) asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1 nt" ::"v"(p), "v"(v) : "memory");
}
#ifndef EP_SCATTER_ST_POL
#define EP_SCATTER_ST_POL 1
#endif
#ifndef EP_PAD_ST_POL
#define EP_PAD_ST_POL 1
#endif
#ifndef EP_COMBINE_ST_POL
#define EP_COMBINE_ST_POL 1
#endif

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }
__device__ __forceinline__ int wave_id() { return threadIdx.x >> 6; }
__device__ __forceinline__ int align_up(int x, int a) { return (x + a - 1) / a * a; }

__device__ __forceinline__ int readlane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Lanes of the wave holding the same key.  Every lane must call it; `key` < 2^nbits.
__device__ __forceinline__ uint64_t match_any(int key, int nbits) {
    uint64_t peers = ~0ull;
    for (int b = 0; b < nbits; ++b) {
        const bool bit = (key >> b) & 1;
        const uint64_t ones = __ballot(bit);
        peers &= bit ? ones : ~ones;
    }
    return peers;
}

// Every lane must be active.  (DPP shifts inside a row of 16 lanes, then the rows' last lanes broadcast to the rows behind: six
// dependent VALU operations, where shuffles are six trips through the LDS: a replayed decode of 32 tokens 17.7 -> 17.5 us, larger calls
// level.)
__device__ __forceinline__ int wave_inclusive_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);      // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);      // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);      // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // row_bcast:15 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);      // row_bcast:31 to rows 2 and 3
    return v;
}

// Counts for the host go to its pinned page (fine-grained memory) with stores that pass the L2, one by one; when a workgroup's have
// arrived, one more says so; it orders them and nothing else.  A release at system scope would write the whole L2 back in front of
// it: 1 us where nothing is dirty, and far longer beside the stores of a copy in the same launch.  Whole host-synchronised cases, three pairs of
// processes, release / this (us): 128 tokens of a toy layer 25.0 / 24.9, a chunk of 1021 tokens 35.4 / 28.2, eight partitions of 2048 1293 / 1252.
__device__ __forceinline__ void host_store(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
__device__ __forceinline__ void host_stores_arrived() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// Reads one word of every 64 bytes of the kernel's arguments, all in one trip.  The compiler fetches arguments where they are
// first used, in some kernels four or five times in a row along the way to the first store, and each first touch of a
// cache line is a trip to memory.  Whole cases, three pairs of processes, without / with (us): prefill of 4096 tokens top-8 246.4 / 244.6, a
// training step of 8192 269.1 / 267.2, prefill of 32768 1202.4 / 1201.5, a replayed decode of 32 17.5 / 17.5; in the combine kernels
// of eight partitions of 2048 tokens 1242.7 / 1239.0, replayed, 600 tokens 473.0 / 468.8.
template <typename Args>
__device__ __forceinline__ void fetch_arguments() {
    typedef const unsigned __attribute__((address_space(4)))* words_t;
    const words_t words = (words_t)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int LINES = (int)(sizeof(Args) + 63) / 64, LAST = (int)sizeof(Args) / 4 - 1;
    unsigned v[10];
    static_assert(LINES <= 10, "one word a line");
#pragma unroll
    for (int i = 0; i < 10; ++i) v[i] = words[16 * i <= LAST ? 16 * i : LAST];
    asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]), "s"(v[6]), "s"(v[7]), "s"(v[8]), "s"(v[9]));
}

// A word that every lane reads alike and nothing of the launch writes, by way of the scalar cache.  The compiler takes the asm of
// fetch_arguments for a store and reads such words behind it with a vector load: two trips in a row in the owner-side reduce (eight
// partitions of 2048 tokens, three pairs of processes, 1252.0 -> 1241.7 us).  Not in the copy kernels, where the one word comes back no later than
// the metadata row beside it (a training step 264.6 -> 266.2).
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p) {
    return *(const T __attribute__((address_space(4)))*)p;
}

// ------------------------------------------------------------------------------------------------
// Entries of the layout passes: (token, j) of topk_idx on the send side, (row, j) of the receive
// stream on the receive side.
// ------------------------------------------------------------------------------------------------
// Receive side: inclusive row counts per source partition from the inbox, in LDS.  Every thread of
// the workgroup calls it (blockDim >= R); returns the length of the receive stream.  s_psum holds
// R + blockDim/64 ints.
__device__ __forceinline__ int recv_scan_sources(const EpLayoutArgs& a, int* s_psum) {
    const int R = a.num_ranks, tid = threadIdx.x, lane = lane_id(), w = wave_id();
    int* s_w = s_psum + R;
    int v = 0;
    if (tid < R) v = max(0, min(a.inbox[tid], a.max_tokens));
    const int incl = wave_inclusive_sum(v);
    if (lane == WAVE - 1) s_w[w] = incl;
    __syncthreads();
    int off = 0;
    for (int i = 0; i < w; ++i) off += s_w[i];
    if (tid < R) s_psum[tid] = off + incl;
    __syncthreads();
    return s_psum[R - 1];
}

// Row g of the receive stream (the regions of the source partitions one after the other, each up to
// its row count: the PSumIterator of dispatch_copy_epilogue.hpp:130-174) -> packed row index.
__device__ __forceinline__ int64_t recv_packed_row(const int* psum, int R, int max_tokens, int g) {
    int lo = 0, hi = R - 1;                       // first source whose inclusive count exceeds g
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (psum[mid] > g) hi = mid; else lo = mid + 1;
    }
    return (int64_t)lo * max_tokens + (g - (lo ? psum[lo - 1] : 0));
}

// Stages the expert ids of this workgroup's entries.  Send side: entry (t, j) of topk_idx.  Receive
// side: entry (row, j) of the receive stream, read from the packed row; partitions play no role there.
// num_rows: rows (tokens) the entries range over (layout_num_rows).
// (recv: a.recv_mode, or the constant an instance of the slot assignment was built for)
__device__ __forceinline__ int layout_num_rows(const EpLayoutArgs& a, int* s_psum, bool recv) {
    return recv ? recv_scan_sources(a, s_psum) : a.num_tokens;
}
__device__ __forceinline__ void layout_load_keys(const EpLayoutArgs& a, short* s_key, short* s_rk, const int* s_psum,
                                                 int num_rows, bool recv, int block) {
    const int K = a.num_topk;
    const int n = EP_TOKENS_PER_BLOCK * K;
    if (recv) {
        const int N = num_rows;
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const int row = i / K, j = i - row * K;
            const int g = block * EP_TOKENS_PER_BLOCK + row;
            int e = -1;
            if (g < N) {
                const int64_t pr = recv_packed_row(s_psum, a.num_ranks, a.max_tokens, g);
                const int64_t v = ((const int64_t*)(a.packed_base + pr * a.packed_row_bytes + a.idx_off))[j];
                e = (v >= 0 && v < a.num_experts) ? (int)v : -1;
            }
            s_key[i] = (short)e;
            s_rk[i] = -1;
        }
        return;
    }
    const int64_t base = (int64_t)block * n;
    const int64_t total = (int64_t)a.num_tokens * K;
    if (total <= 0) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) s_key[i] = s_rk[i] = -1;
        return;
    }
    // four loads a thread in flight, none under a per-lane condition (an entry past the end re-reads the last one
    // and is masked): the ids come from memory, and one trip for a workgroup's entries is all this pass waits for
    for (int i0 = threadIdx.x; i0 < n; i0 += 4 * blockDim.x) {
        int64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = a.topk_idx[min(base + i0 + u * (int)blockDim.x, total - 1)];
        __builtin_amdgcn_sched_barrier(0);      // (the scheduler otherwise uses the first value before it issues the other loads)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * (int)blockDim.x;
            if (i >= n) break;
            const int e = (base + i < total && v[u] >= 0 && v[u] < a.num_experts) ? (int)v[u] : -1;
            s_key[i] = (short)e;
            s_rk[i] = (short)(e < 0 ? -1 : e / a.experts_per_rank);
        }
    }
}

// Destination partition of entry idx if it is the last slot of its token going there, else -1
// (the "master" of common/simt.hpp:24-34).
__device__ __forceinline__ int master_rank(const short* s_rk, int idx, int j, int K) {      // j = idx % K
    const int r = s_rk[idx];
    if (r < 0) return -1;
    for (int jj = j + 1; jj < K; ++jj)
        if (s_rk[idx - j + jj] == r) return -1;
    return r;
}

// ------------------------------------------------------------------------------------------------
// Layout pass A: per-block histograms of expert ids and of destination-partition masters.
// Reference semantics: impls/ep/dispatch.hpp:166-194 (expert histogram, dedup by partition).
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_count(EpLayoutArgs a) {
    fetch_arguments<EpLayoutArgs>();
    extern __shared__ int smem[];
    const int E = a.num_experts, R = a.num_ranks, K = a.num_topk;
    int* s_ecnt = smem;                 // [E]
    int* s_rcnt = s_ecnt + E;           // [R]
    short* s_key = (short*)(s_rcnt + R);
    short* s_rk = s_key + EP_TOKENS_PER_BLOCK * K;
    int* s_psum = (int*)(s_rk + EP_TOKENS_PER_BLOCK * K);      // [R + waves]  (receive side)
    for (int i = threadIdx.x; i < E + R; i += blockDim.x) smem[i] = 0;
    const int num_rows = layout_num_rows(a, s_psum, a.recv_mode != 0);
    // the scan stops at the last workgroup that has rows: the ones behind it leave nothing
    if ((int)blockIdx.x > 0 && (int)blockIdx.x * EP_TOKENS_PER_BLOCK >= num_rows) return;
    layout_load_keys(a, s_key, s_rk, s_psum, num_rows, a.recv_mode != 0, blockIdx.x);
    __syncthreads();
    const int n = EP_TOKENS_PER_BLOCK * K;
    // (the position of an entry inside its token is carried along: a division by a run-time top-k is forty instructions)
    int j = (int)threadIdx.x % K;
    const int jstep = (int)blockDim.x % K;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int e = s_key[i];
        if (e >= 0) atomicAdd(&s_ecnt[e], 1);
        const int mr = master_rank(s_rk, i, j, K);
        if (mr >= 0) atomicAdd(&s_rcnt[mr], 1);
        j += jstep;
        if (j >= K) j -= K;
    }
    __syncthreads();
    // one row of the count matrix: the counted experts, then the partitions, then zero fill.  For the scan kernel
    // the counts are ints; the slot assignment that sums the rows itself takes them as 16-bit halves (a count is at
    // most EP_TOKENS_PER_BLOCK * EP_MAX_TOPK = 4096), eight columns a 16-byte load and two columns an add.
    const int El = a.count_experts, lo = a.count_lo;
    if (a.scan_mode == EP_LAYOUT_FOLDED) {
        unsigned* row = (unsigned*)a.blk_cnt + (int64_t)blockIdx.x * (a.cnt_stride >> 1);
        auto count_of = [&](int i) -> unsigned { return i < El ? s_ecnt[lo + i] : (i < El + R ? s_rcnt[i - El] : 0); };
        for (int i = threadIdx.x; i < (a.cnt_stride >> 1); i += blockDim.x) row[i] = count_of(2 * i) | count_of(2 * i + 1) << 16;
        return;
    }
    int* row = a.blk_cnt + (int64_t)blockIdx.x * a.cnt_stride;
    for (int i = threadIdx.x; i < a.cnt_stride; i += blockDim.x)
        row[i] = i < El ? s_ecnt[lo + i] : (i < El + R ? s_rcnt[i - El] : 0);
}

// ------------------------------------------------------------------------------------------------
// Layout pass B: exclusive prefix over the workgroups of pass A for every histogram column, plus
// column totals.  One workgroup owns 16 columns; its 1024 threads are 64 row groups x 16 columns, a
// thread walks the rows of its group (consecutive threads read consecutive columns of one row).
// ------------------------------------------------------------------------------------------------
#define EP_SCAN_COLS 16
#define EP_SCAN_GROUPS (EP_SCAN_THREADS / EP_SCAN_COLS)

extern "C" __global__ __launch_bounds__(EP_SCAN_THREADS) void ep_layout_scan(EpLayoutArgs a) {
    fetch_arguments<EpLayoutArgs>();
    __shared__ int s_part[EP_SCAN_GROUPS][EP_SCAN_COLS + 1];
    __shared__ int s_rows;
    const int R = a.num_ranks, W = a.cnt_stride;
    int B = a.num_blocks;
    if (a.recv_mode) {
        // rows exist only up to the length of the receive stream
        if (threadIdx.x == 0) s_rows = 0;
        __syncthreads();
        if ((int)threadIdx.x < R) atomicAdd(&s_rows, max(0, min(a.inbox[threadIdx.x], a.max_tokens)));
        __syncthreads();
        B = min(B, max(1, (s_rows + EP_TOKENS_PER_BLOCK - 1) / EP_TOKENS_PER_BLOCK));
    }
    const int c = threadIdx.x % EP_SCAN_COLS, g = threadIdx.x / EP_SCAN_COLS;
    const int col = blockIdx.x * EP_SCAN_COLS + c;
    const bool live = col < W;
    int* base = a.blk_cnt + col;
    const int rpg = (B + EP_SCAN_GROUPS - 1) / EP_SCAN_GROUPS;
    const int r0 = min(B, g * rpg), r1 = min(B, r0 + rpg);
    int sum = 0;
    if (live)
        for (int r = r0; r < r1; ++r) sum += base[(int64_t)r * W];
    s_part[g][c] = sum;
    __syncthreads();
    int off = 0, total = 0;
    for (int i = 0; i < EP_SCAN_GROUPS; ++i) {
        const int v = s_part[i][c];
        if (i < g) off += v;
        total += v;
    }
    if (live) {
        int run = off;
        for (int r = r0; r < r1; ++r) {
            const int v = base[(int64_t)r * W];
            base[(int64_t)r * W] = run;
            run += v;
        }
        if (g == 0) a.col_total[col] = total;
    }
}

// ------------------------------------------------------------------------------------------------
// Layout pass C: slot of every entry.
//   dst_buffer_slot_idx[t,j] = number of earlier tokens with a master for the same partition
//                               (masters only)                       -- impls/ep/dispatch.hpp:258-281
//   slot_map[t,j]            = expert_start[e] + number of earlier (t',j') entries with the same
//                               local expert (lexicographic order)    -- dispatch_copy_epilogue.hpp:471-488
//                               with the canonical order of deep_ep/buffers/ep.py:100-160
// One workgroup (the only one, or one launched beside the ranking ones) publishes the per-partition / per-expert
// counts and prefix sums (impls/ep/dispatch.hpp:469-545) and, when asked, the host count page.
//
// Where the counts of the other blocks come from (a.scan_mode):
//   EP_LAYOUT_SCANNED  ep_layout_scan left exclusive prefixes in blk_cnt and totals in col_total
//   EP_LAYOUT_FOLDED   ep_layout_count left plain counts in blk_cnt (16-bit halves): every block sums the rows
//                      before it itself (cheaper than a launch of its own up to a few hundred blocks)
//   EP_LAYOUT_SINGLE   one block owns every token: nothing ran before, its own LDS counts are the totals
//   EP_LAYOUT_RECOUNTED  a few blocks of one partition: nothing ran before, every workgroup counts the ids of all
//                      blocks itself (a launch less; the ids of 1024 tokens are 48 KB)
// Only the local experts and the partitions need prefixes: slots of other experts are never used.
// ------------------------------------------------------------------------------------------------
#define EP_FOLD_DEPTH 22
#define EP_KEY_MASTER 0x4000          // flag in a staged key: the entry is the master of its partition (ids < 2048)
#define EP_LAYOUT_MAX_COLS_PER_THREAD ((EP_MAX_EXPERTS + EP_MAX_RANKS + EP_LAYOUT_THREADS - 1) / EP_LAYOUT_THREADS)

// Six instances.  FOLD: for EP_LAYOUT_FOLDED (the other modes run one without the summing code).  SIDE: one partition, or
// the send or the receive side of several.  (With the send side's shipping of counts in the instance of one partition, which
// never runs it, that instance took 11.0 instead of 10.2 us at 129 tokens and 12.1 instead of 11.6 at 1024, top-8 of 256.)
enum LayoutSide { SIDE_SINGLE = EP_LAYOUT_SIDE_SINGLE, SIDE_SEND = EP_LAYOUT_SIDE_SEND, SIDE_RECV = EP_LAYOUT_SIDE_RECV };
template <bool FOLD, LayoutSide SIDE>
__device__ __forceinline__ void layout_assign_body(const EpLayoutArgs& a) {
    constexpr bool RECV = SIDE == SIDE_RECV, SEND = SIDE == SIDE_SEND;
    extern __shared__ int smem[];
    const int E = a.num_experts, R = a.num_ranks, K = a.num_topk, A = a.expert_alignment;
    const int El = RECV ? a.experts_per_rank : a.count_experts;
    const int NW = EP_LAYOUT_THREADS / WAVE;
    const int b = blockIdx.x;
    int* s_tot = smem;                     // [El + R] totals of the counted experts, then of the partitions
    int* s_we = s_tot + El + R;            // [NW][E] per-wave counts, then running slot counters
    int* s_wr = s_we + NW * E;             // [NW][R]
    int* s_tmp = s_wr + NW * R;            // [NW + 1]
    short* s_key = (short*)(s_tmp + NW + 1);
    short* s_rk = s_key + EP_TOKENS_PER_BLOCK * K;
    int* s_psum = (int*)(s_rk + EP_TOKENS_PER_BLOCK * K);      // [R + NW]  (receive side)
    const int tid = threadIdx.x, lane = lane_id(), w = wave_id();
    const int lo = RECV ? a.rank_idx * El : a.count_lo;
    const int ncols = El + R;              // column c < El: expert lo + c; else partition c - El

    // The launch has one workgroup more than blocks of tokens.  It ranks nothing: it gets the totals like the others
    // (a single block: it counts that block's ids once more) and publishes them (handle tensors, inboxes, the host count
    // page and the wait for its stores), so that no ranking workgroup has that on its way.
    const bool single = !FOLD && a.scan_mode == EP_LAYOUT_SINGLE;     // (the summing instance never runs alone)
    const bool publisher = b == a.num_blocks, worker = !publisher;
    const int kb = single ? 0 : b;         // the block whose ids this workgroup stages
    const int num_rows = layout_num_rows(a, s_psum, RECV);
    if (!publisher && b > 0 && b * EP_TOKENS_PER_BLOCK >= num_rows) return;      // nothing to rank here

    // ---- counts of the workgroups before this one (kept in registers) and totals over all of them ----
    int pre[EP_LAYOUT_MAX_COLS_PER_THREAD], tot[EP_LAYOUT_MAX_COLS_PER_THREAD];
#pragma unroll
    for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) pre[k] = tot[k] = 0;
    if (!FOLD && a.scan_mode == EP_LAYOUT_SCANNED) {
#pragma unroll
        for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) {
            const int c = tid + k * EP_LAYOUT_THREADS;
            if (c >= ncols) continue;
            if (worker) pre[k] = a.blk_cnt[(int64_t)b * a.cnt_stride + c];
            tot[k] = a.col_total[c];
        }
    }
    const int nkeys = EP_TOKENS_PER_BLOCK * K;
    const int64_t key_base = (int64_t)kb * nkeys, key_total = (int64_t)a.num_tokens * K;
    // EP_LAYOUT_RECOUNTED (one partition, a few blocks, send side): every workgroup reads the ids of all blocks in one
    // go: a histogram of all of them (the totals), one of the blocks before its own, its own block's ids staged on the
    // way.  With one partition the master of a token is its last valid position: the partition's column counts the
    // tokens that have a valid id at all (flags in LDS, counted by ballot).
    const bool recount = !FOLD && SIDE == SIDE_SINGLE && a.scan_mode == EP_LAYOUT_RECOUNTED;
    if (recount) {
        int* s_rpre = s_psum + R + NW;                         // [ncols]
        int* s_rtot = s_rpre + ncols;                          // [ncols]
        int* s_any = s_rtot + ncols;                           // [num_blocks * EP_TOKENS_PER_BLOCK / 4] one byte a token
        unsigned char* s_anyb = (unsigned char*)s_any;
        const int ntok_all = a.num_blocks * EP_TOKENS_PER_BLOCK, n_all = a.num_blocks * nkeys;
        for (int i = tid; i < 2 * ncols + ntok_all / 4; i += blockDim.x) s_rpre[i] = 0;
        for (int i = tid; i < NW * (E + R); i += blockDim.x) s_we[i] = 0;
        for (int i = tid; i < nkeys; i += blockDim.x) s_key[i] = s_rk[i] = -1;
        __syncthreads();
        if (key_total > 0) {
            // (token and position of an id are carried along from load to load instead of divided out)
            const int tok_step = EP_LAYOUT_THREADS / K, pos_step = EP_LAYOUT_THREADS - tok_step * K;
            int tok = tid / K, pos = tid - tok * K;
            // all ids at once, in up to four goes of eight a thread (as many as there are blocks to read: the same in
            // every thread, so that a short launch neither asks for nor looks at the rest)
            constexpr int GOES = 4, GO = EP_RECOUNT_DEPTH / GOES;
            const int goes = (n_all + GO * EP_LAYOUT_THREADS - 1) / (GO * EP_LAYOUT_THREADS);      // 1..4 (the host's limit)
            int64_t v[GOES][GO];
#pragma unroll
            for (int c = 0; c < GOES; ++c) {
                if (c >= goes) break;
#pragma unroll
                for (int u = 0; u < GO; ++u) v[c][u] = a.topk_idx[min((int64_t)tid + (c * GO + u) * EP_LAYOUT_THREADS, key_total - 1)];
            }
            __builtin_amdgcn_sched_barrier(0);      // (every id is asked for before the first is looked at)
#pragma unroll
            for (int c = 0; c < GOES; ++c) {
                if (c >= goes) break;
#pragma unroll
                for (int u = 0; u < GO; ++u) {
                    const int i = tid + (c * GO + u) * EP_LAYOUT_THREADS;
                    const bool valid = i < n_all && i < key_total && v[c][u] >= 0 && v[c][u] < a.num_experts;
                    const int e = valid ? (int)v[c][u] : -1;
                    if (valid) {
                        atomicAdd(&s_rtot[e], 1);
                        if (i < b * nkeys) atomicAdd(&s_rpre[e], 1);
                        s_anyb[tok] = 1;
                    }
                    const int own = i - b * nkeys;
                    if (own >= 0 && own < nkeys) {
                        s_key[own] = (short)e;
                        s_rk[own] = (short)(valid ? 0 : -1);
                    }
                    tok += tok_step;
                    pos += pos_step;
                    if (pos >= K) { pos -= K; ++tok; }
                }
            }
        }
        __syncthreads();
        for (int t0 = 0; t0 < ntok_all; t0 += blockDim.x) {
            const int t = t0 + tid;
            const bool any = t < ntok_all && s_anyb[t] != 0;
            const int all = __popcll(__ballot(any)), before = __popcll(__ballot(any && t < b * EP_TOKENS_PER_BLOCK));
            if (lane == 0 && all > 0) {
                atomicAdd(&s_rtot[El], all);
                if (before > 0) atomicAdd(&s_rpre[El], before);
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) {
            const int c = tid + k * EP_LAYOUT_THREADS;
            if (c >= ncols) continue;
            pre[k] = s_rpre[c];
            tot[k] = s_rtot[c];
        }
    }
    // This workgroup's expert ids are asked for first (send side, up to four ids a thread).
    const bool folded = FOLD;
    const bool keys_early = folded && !RECV && nkeys <= 4 * EP_LAYOUT_THREADS && key_total > 0;
    // EP_LAYOUT_FOLDED: ep_layout_count has finished and left plain counts as 16-bit halves; the rows before this
    // workgroup's (and all rows) are summed here.  A thread takes 8 adjacent columns (one 16-byte load a row) of every
    // S-th row, EP_FOLD_DEPTH loads in flight, and adds them two columns an instruction: each half of the rows in flight
    // has 16-bit sums of its own (EP_FOLD_DEPTH / 2 rows of at most 4096 stay below 2^16), widened at its end; the S
    // partial sums of a column meet in LDS.  The rows come from memory (other XCDs wrote
    // them) and that trip is the longest wait of the kernel: the first turn's rows are asked for here and summed only
    // after the keys have been staged and counted per wave, which needs none of them.
    const int W = a.cnt_stride, FG = W >> 3;
    int* s_fpre = s_psum + R + NW;         // [W]  (EP_LAYOUT_FOLDED only)
    int* s_ftot = s_fpre + W;              // [W]
    const int nb = min(a.num_blocks, max(1, (num_rows + EP_TOKENS_PER_BLOCK - 1) / EP_TOKENS_PER_BLOCK));
    const int S = FG >= EP_LAYOUT_THREADS ? 1 : EP_LAYOUT_THREADS / FG;
    const int s0 = FG >= EP_LAYOUT_THREADS ? 0 : tid / FG;
    const int g0 = FG >= EP_LAYOUT_THREADS ? tid : tid - s0 * FG;
    // (rows are addressed by a 32-bit offset from the uniform base: two instructions a load)
    const unsigned row_bytes = (unsigned)W * 2u, step = (unsigned)S * row_bytes;
    auto fold_loads = [&](u32x4 (&v)[EP_FOLD_DEPTH], int r, int g) {
        const unsigned off = (unsigned)r * row_bytes + 16u * g, last = (unsigned)(nb - 1) * row_bytes + 16u * g;
        // unconditional loads (a row past the end re-reads the last one and is masked in the sums), so that all of
        // them are in flight before the first is waited for
#pragma unroll
        for (int u = 0; u < EP_FOLD_DEPTH; ++u) v[u] = *(const u32x4*)((const char*)a.blk_cnt + min(off + u * step, last));
        __builtin_amdgcn_sched_barrier(0);          // (the scheduler otherwise sums the first rows before it asks for the last)
    };
    auto fold_sums = [&](const u32x4 (&v)[EP_FOLD_DEPTH], int r, int (&p)[8], int (&t)[8]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // (a short launch has no rows in the second half of a turn: its adds are skipped)
            if (h == 1 && r + (EP_FOLD_DEPTH / 2) * S >= nb) break;
            u16x2 ts[4], ps[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) ts[q] = ps[q] = u16x2{0, 0};
#pragma unroll
            for (int u = h * (EP_FOLD_DEPTH / 2); u < (h + 1) * (EP_FOLD_DEPTH / 2); ++u) {
                const int rr = r + u * S;
                const unsigned mt = rr < nb ? ~0u : 0u, mp = rr < b ? ~0u : 0u;      // b <= nb - 1
                ts[0] += __builtin_bit_cast(u16x2, v[u].x & mt); ps[0] += __builtin_bit_cast(u16x2, v[u].x & mp);
                ts[1] += __builtin_bit_cast(u16x2, v[u].y & mt); ps[1] += __builtin_bit_cast(u16x2, v[u].y & mp);
                ts[2] += __builtin_bit_cast(u16x2, v[u].z & mt); ps[2] += __builtin_bit_cast(u16x2, v[u].z & mp);
                ts[3] += __builtin_bit_cast(u16x2, v[u].w & mt); ps[3] += __builtin_bit_cast(u16x2, v[u].w & mp);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                t[2 * q] += (int)ts[q].x;
                t[2 * q + 1] += (int)ts[q].y;
                p[2 * q] += (int)ps[q].x;
                p[2 * q + 1] += (int)ps[q].y;
            }
        }
    };
    // (Lanes are 8 columns apart: column 8 g + q lives at 8 g + ((q + g / 4) & 7), which spreads the 32 lanes of one
    //  add over the 32 banks instead of four.)
    auto fold_meet = [&](int g, const int (&p)[8], const int (&t)[8]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int at = 8 * g + ((q + (g >> 2)) & 7);
            atomicAdd(&s_fpre[at], p[q]);
            atomicAdd(&s_ftot[at], t[q]);
        }
    };
    // (the host sends shapes with more than 8 * EP_LAYOUT_THREADS count columns to the scan kernel: one column group a thread)
    const bool fold_mine = folded && s0 < S && g0 < FG;        // this thread sums rows

    // ---- A: stage this block's keys, clear the per-wave counters (and where the sums of the rows meet) ----
    // Every thread asks for rows and only the ones that sum look at what arrives; both ways through this phase leave
    // the same EP_FOLD_DEPTH loads in flight.  (The compiler counts the loads in flight along every path: with the
    // rows asked for on one path only, or under a per-thread condition, it waits for all of them at the next loop.)
    u32x4 v_first[EP_FOLD_DEPTH];
    auto clear_counters = [&]() {
        for (int i = tid; i < NW * (E + R); i += blockDim.x) s_we[i] = 0;
        if (folded)
            for (int i = tid; i < 2 * W; i += blockDim.x) s_fpre[i] = 0;
    };
    if (keys_early) {
        // ids first, rows behind them; the ids are staged while the rows are on their way
        int64_t pk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) pk[u] = a.topk_idx[min(key_base + tid + u * EP_LAYOUT_THREADS, key_total - 1)];
        __builtin_amdgcn_sched_barrier(0);
        if (FOLD) fold_loads(v_first, s0, min(g0, FG - 1));
        clear_counters();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = tid + u * EP_LAYOUT_THREADS;
            if (i >= nkeys) break;
            const int e = (key_base + i < key_total && pk[u] >= 0 && pk[u] < a.num_experts) ? (int)pk[u] : -1;
            s_key[i] = (short)e;
            s_rk[i] = (short)(e < 0 ? -1 : e / a.experts_per_rank);
        }
    } else if (!recount) {            // (recounted: the ids are staged and the counters clear already)
        clear_counters();
        layout_load_keys(a, s_key, s_rk, s_psum, num_rows, RECV, kb);
        if (FOLD) fold_loads(v_first, s0, min(g0, FG - 1));
    }
    __syncthreads();

    // ---- B: per-wave counts: wave w owns entries [w*epw, (w+1)*epw) of this block's chunk ----
    const int n = EP_TOKENS_PER_BLOCK * K;
    const int rounds = (n + EP_LAYOUT_THREADS - 1) / EP_LAYOUT_THREADS;
    const int epw = rounds * WAVE;
    // (token and position of this lane's entry of a round are carried along instead of divided out every round)
    const int tok0 = (w * epw + lane) / K, pos0 = (w * epw + lane) - tok0 * K;
    const int tok_step = WAVE / K, pos_step = WAVE - tok_step * K;
    for (int rd = 0, pos = pos0; rd < rounds; ++rd) {
        const int idx = w * epw + rd * WAVE + lane;
        if (idx < n) {
            const int e = s_key[idx];
            if (e >= 0) atomicAdd(&s_we[w * E + e], 1);
            const int mr = master_rank(s_rk, idx, pos, K);
            if (mr >= 0) {
                atomicAdd(&s_wr[w * R + mr], 1);
                s_key[idx] = (short)(e | EP_KEY_MASTER);        // remembered for the ranking (only this thread reads it)
            }
        }
        pos += pos_step;
        if (pos >= K) pos -= K;
    }

    // ---- the rows asked for at the top: counts of the workgroups before this one, totals over all ----
    if (fold_mine) {
        int p[8], t[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] = t[q] = 0;
        fold_sums(v_first, s0, p, t);
        for (int r = s0 + EP_FOLD_DEPTH * S; r < nb; r += EP_FOLD_DEPTH * S) {
            u32x4 v[EP_FOLD_DEPTH];
            fold_loads(v, r, g0);
            fold_sums(v, r, p, t);
        }
        fold_meet(g0, p, t);
    }
    __syncthreads();
    if (folded) {
#pragma unroll
        for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) {
            const int c = tid + k * EP_LAYOUT_THREADS;
            if (c >= ncols) continue;
            const int at = (c & ~7) | ((c + (c >> 5)) & 7);
            pre[k] = s_fpre[at];
            tot[k] = s_ftot[at];
        }
    }

    // ---- C: totals over all workgroups into LDS (one workgroup: its own per-wave counts are the totals) ----
#pragma unroll
    for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) {
        const int c = tid + k * EP_LAYOUT_THREADS;
        if (c >= ncols) continue;
        if (a.scan_mode == EP_LAYOUT_SINGLE) {
            const bool is_expert = c < El;
            const int* wc = is_expert ? s_we + lo + c : s_wr + (c - El);
            const int stride = is_expert ? E : R;
            int t = 0;
            for (int i = 0; i < NW; ++i) t += wc[i * stride];
            tot[k] = t;
        }
        s_tot[c] = tot[k];
    }
    __syncthreads();

    // ---- D + E: aligned exclusive scan over the local experts (totals are replaced in place by the
    //      first slot of each expert); the publishing workgroup writes the handle tensors and the host count page ----
    int* s_start = s_tot;
    const int per = (El + EP_LAYOUT_THREADS - 1) / EP_LAYOUT_THREADS;
    const int e0 = min(El, tid * per), e1 = min(El, e0 + per);
    int mine = 0;
    for (int e = e0; e < e1; ++e) mine += align_up(s_tot[e], A);
    if (publisher && !RECV && (SEND ? a.host_boxes != nullptr : a.notify_host != 0))
        // (the host's copy, in adjacent words: every other word of a line is a transfer of its own, 384 experts 27 us later)
        for (int e = tid; e < El; e += EP_LAYOUT_THREADS) {
            const int r = SEND ? e / a.experts_per_rank : 0, at = a.rank_idx * a.experts_per_rank + (e - r * a.experts_per_rank);
            if (SEND) host_store(&a.host_boxes[r][a.host_box_slot + at], s_tot[e]);
            else host_store(&a.host_page[EP_HOST_EXPERT_OFF + e], align_up(s_tot[e], A));
        }
    const int incl = wave_inclusive_sum(mine);
    if (lane == WAVE - 1) s_tmp[w] = incl;
    __syncthreads();
    int wave_off = 0, grand = 0;
    for (int i = 0; i < NW; ++i) {
        if (i < w) wave_off += s_tmp[i];
        grand += s_tmp[i];
    }
    {
        int run = wave_off + incl - mine;
        for (int e = e0; e < e1; ++e) {
            const int c = s_tot[e];
            if (publisher && !SEND) {
                a.unaligned_expert[e] = c;
                a.psum_expert[e] = run + c;
                if (a.cumulative_stats != nullptr) atomicAdd(&a.cumulative_stats[e], c);
            }
            if (SEND) {
                // slots are the receivers' business: ranks count from 0, and the receivers get the counts they need
                // to place them (a partition that is not connected to a node ships nothing)
                if (publisher && a.count_box_off != 0) {
                    const int r = e / a.experts_per_rank, at = a.rank_idx * a.experts_per_rank + (e - r * a.experts_per_rank);
                    ((int*)(a.peer_arenas[r] + a.count_box_off))[at] = c;
                }
                s_start[e] = 0;
                continue;
            }
            s_start[e] = run;
            run += align_up(c, A);
        }
    }
    if (publisher && SEND) {
        // rows this partition sends to every partition, left in the receivers' inboxes: the count half of
        // the reference's cross-rank reduction (impls/ep/dispatch.hpp:469-545)
        // (a partition that is not connected to a node only has its own inbox)
        for (int r = tid; r < R; r += blockDim.x)
            if (a.connected || r == a.rank_idx)
                ((int*)(a.peer_arenas[r] + EP_WS_INBOX_OFF))[a.rank_idx] = min(s_tot[El + r], a.max_tokens);
        if (a.host_boxes != nullptr) {
            // the hosts' copies: a receiver's host then sizes its outputs without waiting for its receive side, which
            // in a stream of phases comes behind the copies of the partitions before it (eight partitions of 2048 tokens:
            // 18-21 us of idle GPU a partition, all phases 1436 -> 1384 us)
            for (int r = tid; r < R; r += blockDim.x)
                host_store(&a.host_boxes[r][a.host_box_slot + EP_HOST_BOX_ROWS_OFF + a.rank_idx], min(s_tot[El + r], a.max_tokens));
            host_stores_arrived();
            for (int r = tid; r < R; r += blockDim.x)
                host_store(&a.host_boxes[r][a.host_box_slot + EP_HOST_BOX_SEQ_OFF + a.rank_idx], a.seq);
        }
    }
    if (publisher && !SEND) {
        // one partition: the receive stream is this partition's own routed tokens; several: the rows counted
        // in the inbox (csrc/buffers/ep.hpp:205-246 names the tensors)
        const int n_recv = RECV ? num_rows : s_tot[El + a.rank_idx];
        for (int r = tid; r < R; r += blockDim.x) {
            const int upto = RECV ? s_psum[r] : n_recv;
            const int from = RECV && r ? s_psum[r - 1] : 0;
            a.psum_rank[r] = upto;
            if (a.notify_host) host_store(&a.host_page[EP_HOST_RANK_OFF + r], upto - from);
        }
        if (a.notify_host) {
            if (RECV) {                 // (from the first slots: ahead of the scan its registers spill)
                __syncthreads();
                for (int e = tid; e < El; e += EP_LAYOUT_THREADS)
                    host_store(&a.host_page[EP_HOST_EXPERT_OFF + e], (e + 1 < El ? s_start[e + 1] : grand) - s_start[e]);
            }
            if (tid == 0) {
                host_store(&a.host_page[1], n_recv);
                host_store(&a.host_page[2], grand);
            }
            host_stores_arrived();
            if (tid == 0) host_store(&a.host_page[0], a.seq);
        }
    }
    if (!worker) return;
    __syncthreads();

    // ---- F: counts -> starting slots (global base + blocks before + waves before) ----
#pragma unroll
    for (int k = 0; k < EP_LAYOUT_MAX_COLS_PER_THREAD; ++k) {
        const int c = tid + k * EP_LAYOUT_THREADS;
        if (c >= ncols) continue;
        const bool is_expert = c < El;
        int* wc = is_expert ? s_we + lo + c : s_wr + (c - El);
        const int stride = is_expert ? E : R;
        int run = pre[k] + (is_expert ? s_start[c] : 0);
        for (int i = 0; i < NW; ++i) {
            const int cnt = wc[i * stride];
            wc[i * stride] = run;
            run += cnt;
        }
    }
    __syncthreads();

    // ---- G: stable ranking, 64 consecutive entries per wave per round ----
    const int ebits = 32 - __builtin_clz(E);       // keys+1 in [0, E]
    const int rbits = 32 - __builtin_clz(R);
    const uint64_t lt = (1ull << lane) - 1ull;
    const int64_t total = (int64_t)num_rows * K;
    for (int rd = 0, tok = tok0, pos = pos0; rd < rounds; ++rd) {
        const int idx = w * epw + rd * WAVE + lane;
        const bool in = idx < n;
        const int key = in ? s_key[idx] : -1;
        const int e = key < 0 ? -1 : key & (EP_KEY_MASTER - 1);
        const int le = e - lo;
        const bool local = e >= 0 && le >= 0 && le < El;
        const int mr = (key >= 0 && (key & EP_KEY_MASTER)) ? s_rk[idx] : -1;
        const uint64_t pe = match_any(local ? e + 1 : 0, ebits);
        const uint64_t pr = match_any(mr + 1, rbits);
        int eslot = -1, rslot = -1;
        if (local) {
            eslot = s_we[w * E + e] + __popcll(pe & lt);
            if ((pe >> lane) == 1ull) s_we[w * E + e] = eslot + 1;      // highest peer advances the counter
        }
        if (mr >= 0) {
            rslot = s_wr[w * R + mr] + __popcll(pr & lt);
            if ((pr >> lane) == 1ull) s_wr[w * R + mr] = rslot + 1;
        }
        const int64_t g = (int64_t)b * n + idx;
        if (in && g < total) {
            if (RECV) {
                const int64_t row = g / K;
                if (row < a.rows_cap) a.recv_src_metadata[row * (K + 2) + (g - row * K)] = eslot;
            } else {
                a.dst_buffer_slot_idx[g] = rslot;
                a.dst_gsge_idx[g] = -1;             // every copy is local: no transport descriptors
                if (!SEND || a.slot_map != nullptr) a.slot_map[g] = eslot;
                if (!SEND && mr == a.rank_idx) a.tok_row[b * EP_TOKENS_PER_BLOCK + tok] = rslot;
            }
        }
        // the running counters of a wave are touched by that wave only and the LDS operations of a wave
        // complete in order: no block barrier (which would also wait for the stores above) is needed
        __builtin_amdgcn_wave_barrier();
        tok += tok_step;
        pos += pos_step;
        if (pos >= K) { pos -= K; ++tok; }
    }
    if (RECV) {
        // the two trailing columns of the metadata rows: source token and last local selection
        // (dispatch_copy_epilogue.hpp:514-522)
        for (int row = tid; row < EP_TOKENS_PER_BLOCK; row += blockDim.x) {
            const int g = b * EP_TOKENS_PER_BLOCK + row;
            if (g >= num_rows || g >= a.rows_cap) continue;
            int master = -1;
            for (int j = 0; j < K; ++j) {
                const int key = s_key[row * K + j];
                const int le = (key < 0 ? -1 : key & (EP_KEY_MASTER - 1)) - lo;
                if (key >= 0 && le >= 0 && le < El) master = j;
            }
            const int64_t pr = recv_packed_row(s_psum, R, a.max_tokens, g);
            int* m = a.recv_src_metadata + (int64_t)g * (K + 2);
            m[K] = *(const int*)(a.packed_base + pr * a.packed_row_bytes + a.src_off);
            m[K + 1] = master;
        }
    }
}

extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<false, SIDE_SINGLE>(a); }
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_send(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<false, SIDE_SEND>(a); }
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_recv(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<false, SIDE_RECV>(a); }
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_fold(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<true, SIDE_SINGLE>(a); }
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_fold_send(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<true, SIDE_SEND>(a); }
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_fold_recv(EpLayoutArgs a) { fetch_arguments<EpLayoutArgs>(); layout_assign_body<true, SIDE_RECV>(a); }

// ------------------------------------------------------------------------------------------------
// Receive side of a node whose send sides ship ranks: nothing is counted or ranked here.  An entry's slot is
//   first slot of its expert + entries of the same expert from the sources before its own + its rank inside its source,
// the first two out of the count box [R][El] that the sources filled, the last out of the rank box beside the packed
// rows: the order of the receive stream (sources in turn, a source's tokens ascending) makes that the lexicographic
// (row, j) rank of the general receive side above.  Same outputs; two dependent trips to memory (counts, then ids and
// ranks) where the general form has a histogram launch, a trip for its rows and a ranking.
// Bound by those trips and the launch.  Workgroup 0 publishes (handle tensors, host count page), the others place 128 rows each.
// Eight partitions of 64 / 2048 tokens, a partition: count 7.4 + assign 14.0 -> 5.7 us / 6.1 + 11.3 -> 5.5 us (the send side,
// which now counts all experts, 11.2 -> 10.7 / 17.0 -> 16.9 us); all phases of the node 543 -> 397 / 1522 -> 1436 us.
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_place(EpLayoutArgs a) {
    fetch_arguments<EpLayoutArgs>();
    extern __shared__ int smem[];
    constexpr int NW = EP_LAYOUT_THREADS / WAVE;
    const int E = a.num_experts, R = a.num_ranks, K = a.num_topk, El = a.experts_per_rank, A = a.expert_alignment;
    int* s_box = smem;                     // [E]  counts per source and local expert, then the first slot of each pair
    int* s_tot = s_box + E;                // [El]
    int* s_tmp = s_tot + El;               // [NW]
    int* s_psum = s_tmp + NW;              // [R + NW]
    int* s_pr = s_psum + R + NW;           // [EP_TOKENS_PER_BLOCK]  packed row of this workgroup's rows
    int* s_at = s_pr + EP_TOKENS_PER_BLOCK;                    // [EP_TOKENS_PER_BLOCK]  their source's place in s_box
    signed char* s_local = (signed char*)(s_at + EP_TOKENS_PER_BLOCK);     // [EP_TOKENS_PER_BLOCK * K]  entry is local
    const int tid = threadIdx.x, lane = lane_id(), w = wave_id();
    const bool publisher = blockIdx.x == 0;
    const int b = (int)blockIdx.x - 1, lo = a.rank_idx * El;
    for (int i = tid; i < E; i += EP_LAYOUT_THREADS) s_box[i] = a.count_box[i];
    const int num_rows = recv_scan_sources(a, s_psum);          // (its barriers cover s_box)
    if (!publisher && b * EP_TOKENS_PER_BLOCK >= num_rows) return;

    // counts -> entries of the sources before, totals; then the aligned scan over the experts
    for (int e = tid; e < El; e += EP_LAYOUT_THREADS) {
        int run = 0;
        for (int s = 0; s < R; ++s) {
            const int c = s_box[s * El + e];
            s_box[s * El + e] = run;
            run += c;
        }
        s_tot[e] = run;
    }
    __syncthreads();
    const int per = (El + EP_LAYOUT_THREADS - 1) / EP_LAYOUT_THREADS;
    const int e0 = min(El, tid * per), e1 = min(El, e0 + per);
    int mine = 0;
    for (int e = e0; e < e1; ++e) mine += align_up(s_tot[e], A);
    if (publisher && a.notify_host)                 // (in adjacent words, as in the slot assignment)
        for (int e = tid; e < El; e += EP_LAYOUT_THREADS) host_store(&a.host_page[EP_HOST_EXPERT_OFF + e], align_up(s_tot[e], A));
    const int incl = wave_inclusive_sum(mine);
    if (lane == WAVE - 1) s_tmp[w] = incl;
    __syncthreads();
    int run = incl - mine, grand = 0;
    for (int i = 0; i < NW; ++i) {
        if (i < w) run += s_tmp[i];
        grand += s_tmp[i];
    }
    for (int e = e0; e < e1; ++e) {
        const int c = s_tot[e];
        if (publisher) {
            a.unaligned_expert[e] = c;
            a.psum_expert[e] = run + c;
            if (a.cumulative_stats != nullptr) atomicAdd(&a.cumulative_stats[e], c);
        }
        s_tot[e] = run;
        run += align_up(c, A);
    }
    if (publisher) {
        for (int r = tid; r < R; r += EP_LAYOUT_THREADS) {
            const int upto = s_psum[r], from = r ? s_psum[r - 1] : 0;
            a.psum_rank[r] = upto;
            if (a.notify_host) host_store(&a.host_page[EP_HOST_RANK_OFF + r], upto - from);
        }
        if (a.notify_host) {
            if (tid == 0) {
                host_store(&a.host_page[1], num_rows);
                host_store(&a.host_page[2], grand);
            }
            host_stores_arrived();
            if (tid == 0) host_store(&a.host_page[0], a.seq);
        }
        return;
    }
    const int first = b * EP_TOKENS_PER_BLOCK;
    const int nrow = min(EP_TOKENS_PER_BLOCK, num_rows - first), n = nrow * K;
    int src = 0;
    if (tid < nrow) {
        const int64_t pr = recv_packed_row(s_psum, R, a.max_tokens, first + tid);
        s_pr[tid] = (int)pr;
        s_at[tid] = (int)pr / a.max_tokens * El;
        src = *(const int*)(a.packed_base + pr * a.packed_row_bytes + a.src_off);
    }
    __syncthreads();

    // the entries of this workgroup's rows, four a thread in flight (an entry past the end re-reads the last one);
    // row and position of an entry are carried along instead of divided out
    const int row_step = EP_LAYOUT_THREADS / K, pos_step = EP_LAYOUT_THREADS - row_step * K;
    int row = tid / K, pos = tid - row * K;
    for (int i0 = tid; i0 < n; i0 += 4 * EP_LAYOUT_THREADS) {
        int64_t id[4];
        int rank[4], rows[4], js[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool in = row < nrow;
            rows[u] = in ? row : nrow - 1;
            js[u] = in ? pos : K - 1;
            const int64_t pr = s_pr[rows[u]];
            id[u] = ((const int64_t*)(a.packed_base + pr * a.packed_row_bytes + a.idx_off))[js[u]];
            rank[u] = a.rank_box[pr * K + js[u]];
            row += row_step;
            pos += pos_step;
            if (pos >= K) { pos -= K; ++row; }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i0 + u * EP_LAYOUT_THREADS >= n) break;
            const bool local = id[u] >= lo && id[u] < lo + El;
            const int le = local ? (int)id[u] - lo : 0;
            const int slot = local ? s_tot[le] + s_box[s_at[rows[u]] + le] + rank[u] : -1;
            s_local[rows[u] * K + js[u]] = local;
            if (first + rows[u] < a.rows_cap) a.recv_src_metadata[(int64_t)(first + rows[u]) * (K + 2) + js[u]] = slot;
        }
    }
    __syncthreads();
    // the two trailing columns: source token and last local selection (dispatch_copy_epilogue.hpp:514-522)
    if (tid < nrow && first + tid < a.rows_cap) {
        int master = -1;
        for (int j = 0; j < K; ++j)
            if (s_local[tid * K + j]) master = j;
        int* m = a.recv_src_metadata + (int64_t)(first + tid) * (K + 2);
        m[K] = src;
        m[K + 1] = master;
    }
}

// ------------------------------------------------------------------------------------------------
// Scatter (dispatch copy epilogue): a wave task is one column part of one row (a token, or a row of the receive stream).
// Reference semantics: impls/ep/dispatch_copy_epilogue.hpp:450-545 (expand), :547-620 (zero padding).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float bf16_lo(unsigned int u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(unsigned int u) { return __uint_as_float(u & 0xffff0000u); }

// Largest magnitude over the 16 lanes of a DPP row, result in every lane of the row.  The operands
// are the bit patterns of |x|: as unsigned integers they order like the floats, +inf above every
// finite value and NaN above +inf, so a NaN anywhere in the group comes out as the group's maximum,
// as it does from torch's amax (deep_ep/utils/math.py:36).
__device__ __forceinline__ unsigned row16_umax(unsigned x) {
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x128, 0xf, 0xf, false));  // row_ror:8
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x124, 0xf, 0xf, false));  // row_ror:4
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x122, 0xf, 0xf, false));  // row_ror:2
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x121, 0xf, 0xf, false));  // row_ror:1
    return x;
}

template <bool HW>
__device__ __forceinline__ u32x2 quant8(const float* f, float inv) {
    u32x2 o;
    if (HW) {
        int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0] * inv, f[1] * inv, 0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2] * inv, f[3] * inv, w0, true);
        int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4] * inv, f[5] * inv, 0, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6] * inv, f[7] * inv, w1, true);
        o.x = (unsigned)w0;
        o.y = (unsigned)w1;
    } else {
        unsigned b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = ep_f32_bits_to_e4m3fn(__float_as_uint(f[i] * inv));
        o.x = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
        o.y = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
    }
    return o;
}

struct RowCtx {
    int t;            // local token index of the row (expand and pack)
    int myslot;       // lane j < K: destination row of (row, j) or -1
    uint64_t mybase;  // lane j < K: first byte of the regions that row belongs to (pack)
    int64_t src_row;  // row of the source matrix holding the payload
};

// Stream row i of the receive side -> packed row of this partition's regions, with the inclusive row
// counts per source in global memory.  Every lane of the wave calls it.
__device__ __forceinline__ int64_t region_row_of_stream(const int* psum, int R, int max_tokens, int i) {
    const int lane = lane_id();
    int q = 0;                                         // sources whose rows all come before row i
    for (int r0 = 0; r0 < R; r0 += WAVE) {
        const bool before = r0 + lane < R && psum[r0 + lane] <= i;
        q += __popcll(__ballot(before));
    }
    q = min(q, R - 1);
    const int slot = min(i - (q ? psum[q - 1] : 0), max_tokens - 1);      // counts of a stale handle cannot lead outside
    return (int64_t)q * max_tokens + max(slot, 0);
}

// First byte of the rows that destination j of the task writes, and of their scales.
template <bool PACK>
__device__ __forceinline__ char* out_rows_of(const EpScatterArgs& a, const RowCtx& c, int j) {
    if (!PACK) return (char*)a.recv_x;
    const unsigned lo = (unsigned)readlane((int)(unsigned)c.mybase, j);
    const unsigned hi = (unsigned)readlane((int)(unsigned)(c.mybase >> 32), j);
    return (char*)(((uint64_t)hi << 32) | lo);
}
template <bool PACK>
__device__ __forceinline__ char* out_sf_of(const EpScatterArgs& a, char* rows) {
    return PACK ? rows + a.pack_sf_off : (char*)a.recv_sf;
}

// Part 0 of a packed row's task: the metadata of the row and its ranks, in every destination.  Lane j < K holds the
// expert id, the gate weight and the rank of entry (t, j).  Lane l of a round stores item l % K of destination l / K: as many
// destinations a round as fit a wave.  (A destination after the other is K times the address arithmetic and the store queue's turns, which
// the other parts of the row do not have: 64 tokens x 7168 top-8, each of eight partitions, dispatches of all
// 93.4 -> 88.3 us.  us of a dispatch and its receive side, all of eight partitions in a captured graph, one after the other / so: 256 tokens top-8,
// 2048 BF16 channels 126.0 / 113.3, 7168 FP8 143.5 / 136.8; top-1 94.1 / 95.5 (97 with integer division for the quotients: it cost more than the
// rounds save up to top-2; 98 with the loop kept beside this form for up to two destinations, for the registers and the code).  Two
// partitions of 2048 tokens, 7168 FP8 channels, stay 2 % behind the loop.)
__device__ __forceinline__ void pack_row_metadata(const EpScatterArgs& a, const RowCtx& c, int64_t e, float w, int rank) {
    const int lane = lane_id(), K = a.num_topk;
    // (quotients of small integers: (x + 1/2) / K is at least 1 / 2K away from the next integer, far more than the reciprocal is off)
    const float per_row = __builtin_amdgcn_rcpf((float)K);
    const int at_once = (int)((float)(2 * WAVE + 1) * 0.5f * per_row), jj = (int)(((float)lane + 0.5f) * per_row), k = lane - jj * K;
    const unsigned e_lo = (unsigned)__shfl((int)(unsigned)e, k), e_hi = (unsigned)__shfl((int)(e >> 32), k);
    const int rank_k = __shfl(rank, k);
    const float w_k = __shfl(w, k);
    for (int j0 = 0; j0 < K; j0 += at_once) {
        const int j = j0 + jj;
        const int g = __shfl(c.myslot, j);
        const unsigned lo = (unsigned)__shfl((int)(unsigned)c.mybase, j), hi = (unsigned)__shfl((int)(unsigned)(c.mybase >> 32), j);
        if (jj >= at_once || j >= K || g < 0) continue;
        char* rows = (char*)((uint64_t)hi << 32 | lo);
        char* row = rows + (int64_t)g * a.out_row_bytes;
        if (a.rank_box_off != 0) ((int*)(rows - a.buffer_off + a.rank_box_off))[(int64_t)g * K + k] = rank_k;
        if (a.with_metadata) ((int64_t*)(row + a.idx_off))[k] = (int64_t)((uint64_t)e_hi << 32 | e_lo);
        ((float*)(row + a.w_off))[k] = w_k;
        if (a.with_metadata && k == 0) *(int*)(row + a.src_off) = a.rank_idx * a.max_tokens + c.t;
    }
}

// A wave task is (row, column part).  Resolves the row's token, its source row and its destination
// rows; the task of part 0 also writes the row's small items.  Three modes:
//   EP_SCATTER_EXPAND  rows are tokens (non-cached: slots from the slot map) or rows of the receive stream
//                      (cached: slots and token from the metadata row), payload read from x[token]; destinations
//                      are the expanded slots; part 0 writes the metadata row (non-cached) and the gate weights
//   EP_SCATTER_PACK    rows are tokens; destinations are rows of the partition-major regions
//                      (partition * max_tokens + slot of dst_buffer_slot_idx); part 0 writes the packed
//                      metadata [all K topk_idx | all K weights | src_token_global_idx] into each of them
//                      (impls/ep/dispatch.hpp:768-794, layout/ep/token.hpp:59-82)
//   EP_SCATTER_REGION  rows of the receive stream (the regions of every source partition in turn), payload,
//                      scales and weights read from the packed rows; destinations come from the metadata
//                      rows the receive-side layout wrote (dispatch_copy_epilogue.hpp:459-522)
template <bool PACK>
__device__ __forceinline__ bool scatter_row_prologue(const EpScatterArgs& a, int i, int part, RowCtx& c) {
    const int lane = lane_id();
    const int K = a.num_topk;
    int myslot = -1, t;
    float early_w = 0.0f;          // gate weight fetched ahead of its use (token-walking expand)
    if (PACK) {
        uint64_t mybase = 0;
        t = i;
        int64_t e = -1;
        if (lane < K) {
            e = a.topk_idx[(int64_t)t * K + lane];
            const int s = a.dst_slot_idx[(int64_t)t * K + lane];
            if (s >= 0 && s < a.max_tokens && e >= 0 && e < a.num_experts) {
                const int peer = (int)(e / a.experts_per_rank);
                myslot = (a.region_by_source ? a.rank_idx : peer) * a.max_tokens + s;
                mybase = (uint64_t)(a.peer_arenas[peer] + a.buffer_off);
            }
        }
        c.t = t;
        c.myslot = myslot;
        c.mybase = mybase;
        c.src_row = t;
        if (part == 0) {
            const float w = (a.topk_weights != nullptr && lane < K) ? a.topk_weights[(int64_t)t * K + lane] : 0.0f;
            const int rank = (a.rank_box_off != 0 && lane < K) ? a.slot_map[(int64_t)t * K + lane] : 0;
            pack_row_metadata(a, c, e, w, rank);
        }
        return true;
    }
    c.mybase = 0;
    if (a.mode == EP_SCATTER_REGION) {
        // the metadata rows are complete before this kernel runs: written by the receive-side layout, or cached
        const int v = lane < K + 2 ? a.recv_src_metadata[(int64_t)i * (K + 2) + lane] : -1;
        if (i >= *a.num_recv_ptr) return false;          // (checked after the row's own load has been issued)
        if (lane < K && v >= 0 && v < a.num_out_rows) myslot = v;
        c.src_row = region_row_of_stream(a.psum_rank, a.num_ranks, a.max_tokens, i);
        if (part == 0 && a.recv_topk_weights != nullptr && myslot >= 0)
            a.recv_topk_weights[myslot] = ((const float*)((const char*)a.x + c.src_row * a.x_row_bytes + a.w_off))[lane];
        c.t = i;
        c.myslot = myslot;
        return true;
    }
    if (!a.cached) {
        // the tasks walk the tokens (nothing has to be looked up before the row of x can be fetched); the row of
        // the receive stream a token became is only needed for its metadata row
        t = i;
        if (lane < K) myslot = a.slot_map[(int64_t)t * K + lane];
        // the task that writes the token's metadata row and weights fetches what it needs for that in the same trip
        // (both are indexed by the token alone; tok_row holds nothing meaningful for a token nobody receives)
        int row = -1;
        if (part == 0) {
            row = a.tok_row[t];
            if (a.recv_topk_weights != nullptr && lane < K) early_w = a.topk_weights[(int64_t)t * K + lane];
        }
        const uint64_t vm = __ballot(myslot >= 0);
        if (vm == 0) return false;                       // a token nobody receives
        if (part == 0) {
            const int master = 63 - __builtin_clzll(vm);
            // [slot_0 .. slot_{K-1}, src_token_global_idx, last local j]  (dispatch_copy_epilogue.hpp:514-522)
            const int v = lane < K ? myslot : (lane == K ? a.rank_idx * a.max_tokens + t : master);
            if (lane < K + 2 && row >= 0 && row < a.num_meta_rows) a.recv_src_metadata[(int64_t)row * (K + 2) + lane] = v;
        }
    } else {
        const int v = lane < K + 2 ? a.recv_src_metadata[(int64_t)i * (K + 2) + lane] : -1;
        if (i >= *a.num_recv_ptr) return false;          // (checked after the row's own load has been issued)
        if (lane < K) myslot = v;
        t = readlane(v, K) - a.rank_idx * a.max_tokens;
        if (t < 0 || t >= a.num_tokens) return false;
    }
    if (lane < K && (myslot < 0 || myslot >= a.num_out_rows)) myslot = -1;
    c.src_row = (int64_t)t;
    if (part == 0 && a.recv_topk_weights != nullptr && lane < K && myslot >= 0)
        a.recv_topk_weights[myslot] = a.cached ? a.topk_weights[(int64_t)t * K + lane] : early_w;
    c.t = t;
    c.myslot = myslot;
    return true;
}

// Source row of task row i if it is known before the prologue has run, else -1.
template <bool PACK>
__device__ __forceinline__ int64_t scatter_guess_source_row(const EpScatterArgs& a, int i) {
    if (PACK) return i;                                            // rows are tokens
    if (a.mode == EP_SCATTER_EXPAND && (!a.cached || a.rows_are_tokens)) return i;
    return -1;
}

// The padding rows of an expert, [psum[e], align(psum[e], A)), are one contiguous span of each output:
// the workgroups that share it walk the span 4 KiB at a time, 16 bytes per lane
// (dispatch_copy_epilogue.hpp:547-620).
__device__ __forceinline__ void zero_span(char* base, int64_t nbytes, int part, int nparts) {
    const u32x4 z = {0u, 0u, 0u, 0u};
    const int64_t tid = (int64_t)part * EP_ROW_THREADS + (threadIdx.x & (EP_ROW_THREADS - 1));    // among the threads sharing the span
    const int64_t nthreads = (int64_t)nparts * EP_ROW_THREADS;
    // 16-byte stores over the aligned body; the ends in 2-byte units (every element here is 2 or 4 bytes wide)
    const int64_t head = min((int64_t)((16 - ((uintptr_t)base & 15)) & 15), nbytes);
    const int64_t body = (nbytes - head) & ~(int64_t)15;
    for (int64_t o = tid * 16; o < body; o += nthreads * 16) stream_store<EP_PAD_ST_POL>((u32x4*)(base + head + o), z);
    for (int64_t o = tid * 2; o < head; o += nthreads * 2) *(unsigned short*)(base + o) = 0;
    for (int64_t o = head + body + tid * 2; o < nbytes; o += nthreads * 2) *(unsigned short*)(base + o) = 0;
}

// (end: one past the expert's last row)
__device__ __forceinline__ void zero_padding_piece(const EpScatterArgs& a, int end, int part) {
    const int rows = min(align_up(end, a.expert_alignment), a.num_out_rows) - end;     // never past the outputs
    if (end < 0 || rows <= 0) return;
    zero_span((char*)a.recv_x + (int64_t)end * a.out_row_bytes, (int64_t)rows * a.out_row_bytes, part,
              a.pad_blocks_per_expert);
    if (a.recv_sf != nullptr && part == 0)
        zero_span((char*)a.recv_sf + (int64_t)end * a.out_sf_row_bytes, (int64_t)rows * a.out_sf_row_bytes, 0, 1);
    if (a.recv_topk_weights != nullptr && part == a.pad_blocks_per_expert - 1)
        zero_span((char*)(a.recv_topk_weights + end), (int64_t)rows * 4, 0, 1);
}
__device__ __forceinline__ void zero_padding_rows(const EpScatterArgs& a) {
    const int pb = blockIdx.x - a.num_row_blocks;
    const int e = pb / a.pad_blocks_per_expert, part = pb % a.pad_blocks_per_expert;
    if (e < a.num_local_experts) zero_padding_piece(a, a.psum_expert[e], part);
}

// The stores of a verbatim task: d[u] = vector (part * vecs_per_lane + u) * 64 + lane of the row; part 0 also carries the
// scale packs of pre-quantised rows.
// Scale packs two at a time where rows and strides allow it: fetched behind the payload (early_scales), one store a
// destination for up to 128 packs (6007 tokens, top-6, 112 packs: 93.2 -> 92.2 us; receive side of eight partitions of 2048
// tokens 32.8 -> 32.1 us a partition).
__device__ __forceinline__ unsigned early_scales(const EpScatterArgs& a, int64_t src_row, int part) {
    const int lane = lane_id();
    if (!a.sf_pairs || part != 0 || lane >= (a.num_sf_packs >> 1)) return 0u;
    return *(const unsigned*)((const char*)a.sf + src_row * a.sf_token_stride_bytes + 4 * lane);
}
// (VECS: the most vectors a lane moves per task)
template <bool PACK, int VECS>
__device__ __forceinline__ void copy_row_out(const EpScatterArgs& a, const RowCtx& c, int part, const u32x4 (&d)[VECS], unsigned scales) {
    const int lane = lane_id(), K = a.num_topk, U = VECS == 1 ? 1 : a.vecs_per_lane;
    const int nvec = (int)(a.copy_bytes >> 4);
    for (int j = 0; j < K; ++j) {
        const int s = readlane(c.myslot, j);
        if (s < 0) continue;
        u32x4* row = (u32x4*)(out_rows_of<PACK>(a, c, j) + (int64_t)s * a.out_row_bytes);
#pragma unroll
        for (int u = 0; u < VECS; ++u) {
            const int v = (part * U + u) * WAVE + lane;
            if (u < U && v < nvec) stream_store<EP_SCATTER_ST_POL>(row + v, d[u]);
        }
    }
    if (part == 0 && a.sf_pairs) {
        const int P2 = a.num_sf_packs >> 1;
        const char* sfrow = (const char*)a.sf + c.src_row * a.sf_token_stride_bytes;
        for (int p = lane; p < P2; p += WAVE) {
            if (p >= WAVE) scales = ((const unsigned*)sfrow)[p];
            for (int j = 0; j < K; ++j) {
                const int s = readlane(c.myslot, j);
                if (s < 0) continue;
                ((unsigned*)(out_sf_of<PACK>(a, out_rows_of<PACK>(a, c, j)) + (int64_t)s * a.out_sf_row_bytes))[p] = scales;
            }
        }
    } else if (part == 0 && a.recv_sf != nullptr) {
        const int P = a.num_sf_packs;
        const char* sfrow = (const char*)a.sf + c.src_row * a.sf_token_stride_bytes;
        for (int p = lane; p < P; p += WAVE) {
            const unsigned short val = *(const unsigned short*)(sfrow + (int64_t)p * a.sf_pack_stride_bytes);
            for (int j = 0; j < K; ++j) {
                const int s = readlane(c.myslot, j);
                if (s < 0) continue;
                ((unsigned short*)(out_sf_of<PACK>(a, out_rows_of<PACK>(a, c, j)) + (int64_t)s * a.out_sf_row_bytes))[p] = val;
            }
        }
    }
}

// Verbatim rows: BF16 payload, or FP8 payload with its 2-byte scale packs.  A task moves 1 KiB of
// the row (16 bytes per lane) to every slot; many short tasks keep far more loads in flight than
// one wave walking a whole row.
template <bool PACK>
__device__ __forceinline__ void scatter_copy_body(const EpScatterArgs& a) {
    if ((int)blockIdx.x >= a.num_row_blocks) {
        zero_padding_rows(a);
        return;
    }
    const int lane = lane_id();
    const int task = blockIdx.x * EP_ROWS_PER_BLOCK + wave_id();
    const int i = task / a.num_parts, part = task - i * a.num_parts;
    if (i >= a.num_rows_bound) return;
    const int nvec = (int)(a.copy_bytes >> 4);
    // a task moves vecs_per_lane KiB of the row: 1 where a row fans out to several slots, more where
    // nearly every row has a single destination and the set-up above would outweigh the copy
    const int U = a.vecs_per_lane;
    u32x4 d[4];
    // Where the source row of a task is known up front (tokens are walked, or every token was received so that
    // row i of the receive stream is token i), its payload is fetched while the prologue looks up the slots;
    // a prologue that names another row after all fetches again.
    const int64_t guess = scatter_guess_source_row<PACK>(a, i);
    if (guess >= 0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int v = (part * U + u) * WAVE + lane;
            if (u < U && v < nvec)
                d[u] = __builtin_nontemporal_load((const u32x4*)((const char*)a.x + guess * a.x_row_bytes) + v);
        }
    }
    unsigned scales = guess >= 0 ? early_scales(a, guess, part) : 0u;
    RowCtx c;
    if (!scatter_row_prologue<PACK>(a, i, part, c)) return;
    if (c.src_row != guess) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int v = (part * U + u) * WAVE + lane;
            if (u < U && v < nvec)
                d[u] = __builtin_nontemporal_load((const u32x4*)((const char*)a.x + c.src_row * a.x_row_bytes) + v);
        }
        scales = early_scales(a, c.src_row, part);
    }
    copy_row_out<PACK>(a, c, part, d, scales);
}

// Fused BF16 -> e4m3fn quantisation (deep_ep/utils/math.py:30-38) + scatter.  A task owns 512
// channels of a row: a lane holds 8 of them, a 128-channel group is one DPP row of 16 lanes, so the
// task produces 512 payload bytes and 4 fp32 scales per slot.
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_copy(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_copy_body<false>(a);
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_copy_pack(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_copy_body<true>(a);
}

// Quantises the 8 channels a lane holds (vector v of the row; a 128-channel group is one DPP row of 16 lanes) and stores
// them, and the group's scale, into every destination of the row.
template <bool HW, bool PACK>
__device__ __forceinline__ void quant_row_out(const EpScatterArgs& a, const RowCtx& c, int v, bool live, const u32x4& d) {
    const int lane = lane_id(), K = a.num_topk;
    float f[8] = {bf16_lo(d.x), bf16_hi(d.x), bf16_lo(d.y), bf16_hi(d.y),
                  bf16_lo(d.z), bf16_hi(d.z), bf16_lo(d.w), bf16_hi(d.w)};
    unsigned mbits = 0u;
#pragma unroll
    for (int q = 0; q < 8; ++q) mbits = max(mbits, __float_as_uint(f[q]) & 0x7fffffffu);
    const float m = __uint_as_float(row16_umax(mbits));
    const float amax = m < 1e-4f ? 1e-4f : m;       // clamp(min=1e-4): a NaN stays a NaN
    const float inv = (1.0f / amax) * 448.0f;       // torch evaluates `448.0 / t` as t.reciprocal() * 448.0
    const float scale = amax / 448.0f;
    u32x2 q8 = quant8<HW>(f, inv);
    if (amax != amax) q8 = u32x2{0x7f7f7f7fu, 0x7f7f7f7fu};   // every product is NaN: e4m3fn has one NaN, sign clear
    if (!live) return;
    const bool writes_scale = (lane & 15) == 0;
    for (int j = 0; j < K; ++j) {
        const int s = readlane(c.myslot, j);
        if (s < 0) continue;
        char* rows = out_rows_of<PACK>(a, c, j);
        stream_store<EP_SCATTER_ST_POL>((u32x2*)(rows + (int64_t)s * a.out_row_bytes) + v, q8);
        if (writes_scale) ((float*)(out_sf_of<PACK>(a, rows) + (int64_t)s * a.out_sf_row_bytes))[v >> 4] = scale;
    }
}

// (LOADS = false exists for the benchmarks' calibration code object only: the same tasks and stores with a
// made-up payload in place of the row of x.)
template <bool HW, bool PACK, bool LOADS = true>
__device__ __forceinline__ void scatter_quant_body(const EpScatterArgs& a) {
    if ((int)blockIdx.x >= a.num_row_blocks) {
        zero_padding_rows(a);
        return;
    }
    const int lane = lane_id();
    const int task = blockIdx.x * EP_ROWS_PER_BLOCK + wave_id();
    const int i = task / a.num_parts, part = task - i * a.num_parts;
    if (i >= a.num_rows_bound) return;
    const int nvec = a.hidden >> 3;                      // 16-byte vectors of 8 BF16
    const int v = part * WAVE + lane;
    const bool live = v < nvec;
    u32x4 d = {0u, 0u, 0u, 0u};
    // the payload is fetched while the prologue looks up the slots wherever the source row is known up front
    const int64_t guess = scatter_guess_source_row<PACK>(a, i);
    if (live && LOADS && guess >= 0) d = __builtin_nontemporal_load((const u32x4*)((const char*)a.x + guess * a.x_row_bytes) + v);
    RowCtx c;
    if (!scatter_row_prologue<PACK>(a, i, part, c)) return;
    if (live && LOADS && c.src_row != guess)
        d = __builtin_nontemporal_load((const u32x4*)((const char*)a.x + c.src_row * a.x_row_bytes) + v);
    if (!LOADS) d = u32x4{0x3f803f80u + (unsigned)v, 0x40004000u, 0xbf80bf80u, 0x3f003f00u};
    quant_row_out<HW, PACK>(a, c, v, live, d);
}

extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_quant(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_quant_body<true, false>(a);
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_quant_sw(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_quant_body<false, false>(a);
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_quant_pack(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_quant_body<true, true>(a);
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_scatter_quant_sw_pack(EpScatterArgs a) {
    fetch_arguments<EpScatterArgs>();
    scatter_quant_body<false, true>(a);
}

// What the publishing workgroup of a one-launch dispatch (below) leaves: the handle tensors and the host count page, or
// (several partitions) the counts in the receivers' inboxes and boxes.
template <bool PACK, typename CountOf, typename TokensTo>
__device__ __forceinline__ void publish_dispatch(const EpLayoutArgs& l, int grand, CountOf count_of, const int* s_start, TokensTo tokens_to) {
    const int E = l.num_experts, R = l.num_ranks, A = l.expert_alignment, El = l.experts_per_rank, tid = threadIdx.x;
    for (int e = tid; e < E; e += (int)blockDim.x) {
        const int c = count_of(e);
        if (PACK) {
            const int r = e / El, at = l.rank_idx * El + (e - r * El);
            if (l.count_box_off != 0) ((int*)(l.peer_arenas[r] + l.count_box_off))[at] = c;
            if (l.host_boxes != nullptr) host_store(&l.host_boxes[r][l.host_box_slot + at], c);
        } else {
            l.unaligned_expert[e] = c;
            l.psum_expert[e] = s_start[e] + c;
            if (l.cumulative_stats != nullptr) atomicAdd(&l.cumulative_stats[e], c);
            if (l.notify_host) host_store(&l.host_page[EP_HOST_EXPERT_OFF + e], align_up(c, A));
        }
    }
    for (int r = tid; r < R; r += (int)blockDim.x) {
        const int rows = min(tokens_to(r), l.max_tokens);
        if (PACK) {
            if (l.connected || r == l.rank_idx) ((int*)(l.peer_arenas[r] + EP_WS_INBOX_OFF))[l.rank_idx] = rows;
            if (l.host_boxes != nullptr) host_store(&l.host_boxes[r][l.host_box_slot + EP_HOST_BOX_ROWS_OFF + l.rank_idx], rows);
        } else {
            l.psum_rank[r] = rows;
            if (l.notify_host) host_store(&l.host_page[EP_HOST_RANK_OFF + r], rows);
        }
    }
    if (PACK ? l.host_boxes != nullptr : l.notify_host != 0) {
        if (!PACK && tid == 0) {
            host_store(&l.host_page[1], tokens_to(0));
            host_store(&l.host_page[2], grand);
        }
        host_stores_arrived();
        if (PACK) {
            for (int r = tid; r < R; r += (int)blockDim.x)
                host_store(&l.host_boxes[r][l.host_box_slot + EP_HOST_BOX_SEQ_OFF + l.rank_idx], l.seq);
        } else if (tid == 0) {
            host_store(&l.host_page[0], l.seq);
        }
    }
}

// A block's entries that have an expert, a bit each: those of the token whose first entry is `at`.
__device__ __forceinline__ unsigned entry_marks(const uint64_t* s_mark, int at, int K) {
    const uint64_t lo = s_mark[at >> 6] >> (at & 63), hi = (at & 63) ? s_mark[(at >> 6) + 1] << (64 - (at & 63)) : 0ull;
    return (unsigned)(lo | hi) & ((1u << K) - 1u);
}

// ------------------------------------------------------------------------------------------------
// The histograms in front of ep_layout_assign_bits: what ep_layout_count leaves for EP_LAYOUT_FOLDED, of one partition and up to top-8: a
// token is received where one of its entries has an expert, which a bit an entry tells without a look at its neighbours.
// Bound by the launch and the trip for the ids.  us of a layout (both launches, several in a captured graph) of 256 experts behind ep_layout_count
// and this one: 4096 tokens top-8 11.7 / 10.7, top-4 10.4 / 9.9, 16384 top-4 11.2 / 10.6, 32768 top-2 14.0 / 13.7.  A thread asks for four ids
// whatever the top-k, no further than its block's own: beyond those, the next blocks' ids came along, two to eight times the bytes at top-4
// to top-1 (both kernels, 32768 tokens of 64 experts top-1 10.70 -> 10.59, 40960 of 32 experts top-2 11.64 -> 11.47, level at top-4).
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_count_bits(EpLayoutArgs a) {
    fetch_arguments<EpLayoutArgs>();
    extern __shared__ int smem[];
    constexpr int NT = EP_LAYOUT_THREADS, PER = EP_TOKENS_PER_BLOCK * EP_BITS_TOPK / NT;
    const int E = a.num_experts, K = a.num_topk, n = EP_TOKENS_PER_BLOCK * K, W = a.cnt_stride, tid = threadIdx.x, lane = lane_id();
    int* s_cnt = smem;                                  // [W]
    uint64_t* s_mark = (uint64_t*)(s_cnt + W);          // [n / 64 + 1] entries with an expert, a bit each
    const int64_t base = (int64_t)blockIdx.x * n, total = (int64_t)a.num_tokens * K;
    int64_t id[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) id[u] = a.topk_idx[min(base + min(tid + u * NT, n - 1), total - 1)];
    __builtin_amdgcn_sched_barrier(0);
    for (int i = tid; i < W; i += NT) s_cnt[i] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = tid + u * NT;
        const bool valid = i < n && base + i < total && id[u] >= 0 && id[u] < E;
        const uint64_t bits = __ballot(valid);
        if (lane == 0 && i < n) s_mark[i >> 6] = bits;
        if (valid) atomicAdd(&s_cnt[(int)id[u]], 1);
    }
    __syncthreads();
    const int rows = __popcll(__ballot(entry_marks(s_mark, lane * K, K) != 0u)) + __popcll(__ballot(entry_marks(s_mark, (lane + WAVE) * K, K) != 0u));
    auto count_of = [&](int c) -> unsigned { return c < E ? (unsigned)s_cnt[c] : c == E ? (unsigned)rows : 0u; };
    unsigned* row = (unsigned*)a.blk_cnt + (int64_t)blockIdx.x * (W >> 1);
    for (int i = tid; i < (W >> 1); i += NT) row[i] = count_of(2 * i) | count_of(2 * i + 1) << 16;
}

// ------------------------------------------------------------------------------------------------
// The slot assignment of one partition behind ep_layout_count_bits, up to top-8 and EP_SMALL_MASK_EXPERTS experts: what
// ep_layout_assign_fold does, with ranks from bit masks.  A block's ids leave a bit a token and expert in LDS, and an entry's rank is
// the number of bits below its token (where tokens select an expert more than once, the second, third, .. selections leave their bits
// one after the other in passes of their own); the last valid position of a token and the tokens with one come from a bit an entry.  Neither counts per
// wave nor rounds of match-any, and two barriers: one behind the clearing of the LDS, one behind bits and sums of the count rows.
// Each wave makes the scan over the experts alone.
// Bound by the launch and its trips to memory (ids and count rows, asked for together).  us of a layout (both launches, several in a
// captured graph), ep_layout_count + ep_layout_assign_fold / ep_layout_count_bits + this one: 256 experts, 2048 tokens top-8 14.6 / 10.6, 4096
// top-8 14.6 / 10.7, top-6 13.4 / 10.2, 8192 top-4 12.1 / 10.0, 16384 top-2 11.4 / 10.3; 64 experts 4096 top-8 14.2 / 10.7, 32768 top-2
// 11.0 / 10.9.  With repeated selections, 4096 tokens top-8 of 256 experts, ids of one repeated once 14.6 / 12.7, of all 14.6 / 12.8, drawn with
// repetitions 14.6 / 13.1, every token on one expert 14.8 / 15.8 (up to 64 experts 14.3 / 15.9), every entry on one 15.9 / 16.4; top-4 12.1 /
// 11.0, 11.0, 11.0, 12.0, 12.4.  (The repetitions in a list that every entry looks through: 12.6, 22.4, 15.1, 80, 81; passes that take bits
// away instead of setting them, a barrier less each but all of a token's ids to compare in front: 13.2, 13.2, 13.6, 17.0, 17.5.)  (Every workgroup counting all ids in one launch, as ep_dispatch_chunk_* does: 1024 top-8 7.8, 2048 9.6, 4096 13.1, 8192 top-4
// 13.7: better only where that launch copies as well.)
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_layout_assign_bits(EpLayoutArgs a) {
    fetch_arguments<EpLayoutArgs>();
    extern __shared__ int smem[];
    constexpr int NT = EP_LAYOUT_THREADS, PER = EP_TOKENS_PER_BLOCK * EP_BITS_TOPK / NT, TW = EP_TOKENS_PER_BLOCK / 32;
    const int E = a.num_experts, K = a.num_topk, A = a.expert_alignment, b = blockIdx.x, nb = a.num_blocks;
    const bool publisher = b == nb;
    const int n = EP_TOKENS_PER_BLOCK * K, W = a.cnt_stride, FG = W >> 3;      // W: the experts, the partition, up to 8 columns
    u32x4* s_mask = (u32x4*)smem;                       // [E] tokens of the block that selected an expert, a bit each
    int* s_pre = (int*)(s_mask + E);                    // [W] entries in the blocks before, columns rotated as below
    int* s_tot = s_pre + W;                             // [W] entries in all blocks
    int* s_start = s_tot + W;                           // [W] first slot of an expert
    uint64_t* s_mark = (uint64_t*)(s_start + W);        // [n / 64 + 1] entries with an expert, a bit each
    int* s_last = (int*)(s_mark + EP_TOKENS_PER_BLOCK * EP_BITS_TOPK / WAVE + 1);      // [2] last pass over repeated selections, 0: there are none
    short* s_key = (short*)(s_last + 2);                // [n] expert of an entry, -1: none
    const int tid = threadIdx.x, lane = lane_id();

    // ---- ids first, count rows behind them: a thread takes 8 adjacent columns of every S-th row (see ep_layout_assign_fold) ----
    const int64_t base = (int64_t)min(b, nb - 1) * n, total = (int64_t)a.num_tokens * K;
    int64_t id[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) id[u] = a.topk_idx[min(base + min(tid + u * NT, n - 1), total - 1)];
    __builtin_amdgcn_sched_barrier(0);
    const int S = FG >= NT ? 1 : NT / FG, s0 = FG >= NT ? 0 : tid / FG, g0 = FG >= NT ? tid : tid - s0 * FG;
    const unsigned row_bytes = (unsigned)W * 2u, step = (unsigned)S * row_bytes;
    u32x4 v[EP_FOLD_DEPTH];
    auto fold_loads = [&](int r) {
        const unsigned off = (unsigned)r * row_bytes + 16u * min(g0, FG - 1), last = (unsigned)(nb - 1) * row_bytes + 16u * min(g0, FG - 1);
#pragma unroll
        for (int u = 0; u < EP_FOLD_DEPTH; ++u) v[u] = *(const u32x4*)((const char*)a.blk_cnt + min(off + u * step, last));
        __builtin_amdgcn_sched_barrier(0);
    };
    fold_loads(s0);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int i = tid; i < E + (W >> 1); i += NT) s_mask[i] = zero;      // masks and both rows of sums
    if (tid == 0) *s_last = 0;
    __syncthreads();

    // ---- a bit a token and expert, a bit an entry ----
    const float per_token = 1.0f / (float)K;            // (as in the one-launch kernels: exact for these quotients)
    int tok[PER], key[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = tid + u * NT;
        const bool valid = i < n && base + i < total && id[u] >= 0 && id[u] < E;
        tok[u] = (int)(((float)i + 0.5f) * per_token);
        key[u] = valid ? (int)id[u] : -1;
        const uint64_t bits = __ballot(valid);
        if (lane == 0 && i < n) s_mark[i >> 6] = bits;
        if (i < n) s_key[i] = (short)key[u];
        if (valid && !publisher) {
            const unsigned bit = 1u << (tok[u] & 31);
            if (atomicOr((unsigned*)&s_mask[key[u]] + (tok[u] >> 5), bit) & bit) *s_last = 1;
        }
    }
    // ---- sums of the count rows: blocks before this one, and all ----
    if (s0 < S && g0 < FG) {
        int p[8], t[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] = t[q] = 0;
        for (int r = s0;;) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {               // (11 rows of at most 128 top-k entries stay below 2^16)
                if (h == 1 && r + (EP_FOLD_DEPTH / 2) * S >= nb) break;
                u16x2 ts[4], ps[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) ts[q] = ps[q] = u16x2{0, 0};
#pragma unroll
                for (int u = h * (EP_FOLD_DEPTH / 2); u < (h + 1) * (EP_FOLD_DEPTH / 2); ++u) {
                    const int rr = r + u * S;
                    const unsigned mt = rr < nb ? ~0u : 0u, mp = rr < min(b, nb) ? ~0u : 0u;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        ts[q] += __builtin_bit_cast(u16x2, v[u][q] & mt);
                        ps[q] += __builtin_bit_cast(u16x2, v[u][q] & mp);
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    t[2 * q] += (int)ts[q].x;
                    t[2 * q + 1] += (int)ts[q].y;
                    p[2 * q] += (int)ps[q].x;
                    p[2 * q + 1] += (int)ps[q].y;
                }
            }
            r += EP_FOLD_DEPTH * S;
            if (r >= nb) break;
            fold_loads(r);
        }
        // (the lanes of an add are 8 columns apart: column 8 g + q lives at 8 g + ((q + g / 4) & 7), which spreads them over the banks)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int at = 8 * g0 + ((q + (g0 >> 2)) & 7);
            atomicAdd(&s_pre[at], p[q]);
            atomicAdd(&s_tot[at], t[q]);
        }
    }
    __syncthreads();
    auto at_of = [](int c) { return (c & ~7) | ((c + (c >> 5)) & 7); };

    // ---- aligned exclusive scan over the experts, eight a lane ----
    const bool pow2 = (A & (A - 1)) == 0;
    int grand = 0;
    for (int e0 = 0; e0 < E; e0 += 8 * WAVE) {
        const int e = e0 + 8 * lane;
        int before[8], sum = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int x = e + q < E ? s_tot[at_of(e + q)] : 0;
            before[q] = sum;
            sum += pow2 ? (x + A - 1) & -A : align_up(x, A);
        }
        const int incl = wave_inclusive_sum(sum), run = grand + incl - sum;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (e + q < E) s_start[e + q] = run + before[q];
        grand += readlane(incl, WAVE - 1);
    }
    __builtin_amdgcn_wave_barrier();                    // (the LDS operations of a wave complete in order)
    if (publisher) {
        publish_dispatch<false>(a, grand, [&](int e) { return s_tot[at_of(e)]; }, s_start, [&](int) { return s_tot[at_of(E)]; });
        return;
    }
    // ---- tokens with an expert, a bit each (a wave has 128 tokens in two ballots) ----
    auto marks_of = [&](int t) { return entry_marks(s_mark, t * K, K); };
    const uint64_t any_lo = __ballot(marks_of(lane) != 0u), any_hi = __ballot(marks_of(lane + WAVE) != 0u);
    const int rows_before = s_pre[at_of(E)];
    // ---- rank: the bits of the expert below the token ----
    auto below = [&](int e, int t) -> int {
        const u32x4 m = s_mask[e];
        int c = 0;
#pragma unroll
        for (int q = 0; q < TW; ++q) {
            const int bits = min(max(t - 32 * q, 0), 32);
            c += __popc(m[q] & (bits == 32 ? ~0u : (1u << bits) - 1u));
        }
        return c;
    };
    int rank[PER];                                      // (where a token selects an expert more than once)
    const bool repeats = __builtin_amdgcn_readfirstlane(*s_last) != 0;
    if (repeats) {
        // entries with as many equal ones in front of them in their token leave their bits together, a pass each
        int met[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            rank[u] = below(max(key[u], 0), tok[u]);
            met[u] = 0;
            if (key[u] < 0) continue;
            for (int at = tok[u] * K; at < tid + u * NT; ++at) met[u] += s_key[at] == key[u] ? 1 : 0;
            rank[u] += met[u];
        }
        for (int pass = 1, last = pass; pass <= last; ++pass) {
            __syncthreads();                            // (masks and last pass have been read)
            for (int i = tid; i < E; i += NT) s_mask[i] = zero;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                if (met[u] == pass) atomicOr((unsigned*)&s_mask[key[u]] + (tok[u] >> 5), 1u << (tok[u] & 31));
                if (met[u] > pass) *s_last = pass + 1;
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < PER; ++u) rank[u] += below(max(key[u], 0), tok[u]);
            last = __builtin_amdgcn_readfirstlane(*s_last);
        }
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = tid + u * NT, t = tok[u], e = key[u];
        if (i >= n || base + i >= total) continue;
        const int pos = i - t * K;
        int slot = -1, rslot = -1;
        if (e >= 0) {
            slot = s_start[e] + s_pre[at_of(e)] + (repeats ? rank[u] : below(e, t));
            if ((marks_of(t) >> pos) == 1u)             // the last one of its token
                rslot = rows_before + (t < WAVE ? __popcll(any_lo & ((1ull << t) - 1ull))
                                                : __popcll(any_lo) + __popcll(any_hi & ((1ull << (t - WAVE)) - 1ull)));
        }
        a.dst_buffer_slot_idx[base + i] = rslot;
        a.dst_gsge_idx[base + i] = -1;                  // every copy is local: no transport descriptors
        a.slot_map[base + i] = slot;
        if (rslot >= 0) a.tok_row[b * EP_TOKENS_PER_BLOCK + t] = rslot;
    }
}

// ------------------------------------------------------------------------------------------------
// A dispatch of at most EP_TOKENS_PER_BLOCK tokens and EP_SMALL_ENTRIES entries in one launch.  Instead of a slot
// assignment in front of the copy (a launch that one or two workgroups of the chip work at, bound by its own dependent
// phases), every workgroup counts all ids in LDS and leaves a bit a token and expert there; its waves rank the one token each of
// them copies by the bits below it, a position a lane.  (A token that selects an expert twice has one bit for both and an entry in a
// list, which is looked through 64 entries at a time.  With more than EP_SMALL_REPEATS of them, and beyond EP_SMALL_MASK_EXPERTS, whose masks
// would leave a CU too few workgroups, the ids in front of the token are compared expert by expert.)
// The payload is fetched before the ids are looked at.  Workgroup 0 publishes what the assignment's publishing workgroup
// does, the next ones copy (or, with several partitions, pack) as the kernels above, the last zero the padding.
// Bound by the launch, two trips to memory and the phases in LDS between them.  Assignment + copy -> this kernel with ids compared (us): 32 tokens,
// top-8 of 256, FP8 8.8 + 6.2 -> 9.0; 61 tokens x 5120, top-6 of 160, BF16 7.5 + 4.2 -> 8.2; 128 tokens, top-8, 230 MB of
// padding 10.0 + 31.2 -> 35.3; one of eight partitions of 64 tokens 11.2 + 5.6 -> 10.1.
// Ids compared -> masks, and a scan that each wave makes alone (us a dispatch, several in a captured graph; stamps had the ranking at 2.4 of
// 6.3): 256 experts, BF16, top-8, 7168 channels 1 / 32 / 61 tokens 5.7 / 6.4 / 7.5 -> 4.3 / 4.9 / 5.7, 256 channels 128 tokens 8.2 -> 5.8; top-6, FP8,
// alignment 16, 96 tokens 8.0 -> 6.5; 1024 experts, 61 tokens top-8 7.4 -> 5.8; top-1 level; all of a dispatch of eight partitions of 64 tokens
// top-8, metadata above included, 110.0 -> 88.3.  Masks at 2048 experts: 1 token top-1 with padding 8.3 -> 10.8, compared so 8.2.
// Repeated selections, ids compared without masks / compared behind masks / listed: 128 tokens x 7168 top-8 of 256, one repeated once
// 10.9 / 11.1 / 9.2, ids drawn with repetitions 11.0 / 11.2 / 9.7; one repeated by every token, 61 tokens x 5120 top-6 7.1 / 7.2 / 6.7, 100 x 2048 7.9 /
// 7.8 / 7.4; beyond the list (that form compares) 128 tokens x 7168, one repeated by every token 11.2 / 11.4 / 11.9, every token on one expert 11.4 / 11.9 /
// 12.4, every entry on one 12.5 / 14.1 / 14.5, of 256 channels 9.6 / 10.2 / 10.6: the masks' and the list's words are contended.
// ------------------------------------------------------------------------------------------------
template <bool QUANT, bool HW, bool PACK>
__device__ __forceinline__ void dispatch_small_body(const EpSmallArgs& a) {
    extern __shared__ int smem[];
    constexpr int CH = EP_SMALL_ENTRIES / WAVE, PER = EP_SMALL_ENTRIES / EP_ROW_THREADS, TW = EP_TOKENS_PER_BLOCK / 32;
    const EpLayoutArgs& l = a.l;
    const EpScatterArgs& s = a.s;
    const int E = l.num_experts, R = l.num_ranks, K = l.num_topk, A = l.expert_alignment, El = l.experts_per_rank;
    const int Ep = (E + 7) & ~7;
    const bool publisher = blockIdx.x == 0;
    const int rb = (int)blockIdx.x - 1;
    const bool copies = !publisher && rb < s.num_row_blocks;
    const bool masks = copies && E <= EP_SMALL_MASK_EXPERTS;            // (who ranks nothing needs none)
    u32x4* s_tok = (u32x4*)smem;                        // [R] tokens that go to a partition, a bit each
    u32x4* s_mask = s_tok + R;                          // [E] tokens that selected an expert, a bit each (E <= EP_SMALL_MASK_EXPERTS)
    int* s_cnt = (int*)(s_mask + (masks ? E : 0));      // [Ep] entries per expert
    int* s_more = s_cnt + Ep;                           // [4] entries that s_list has, or would have
    int* s_start = s_more + 4;                          // [Ep] first slot of each expert (one partition)
    short* s_key = (short*)(s_start + Ep);              // [EP_SMALL_ENTRIES] expert of every entry, -1: none
    short* s_list = s_key + EP_SMALL_ENTRIES;           // [EP_SMALL_REPEATS] entries beyond the first of a token for an expert (masks)
    const int tid = threadIdx.x, lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    const int n = l.num_tokens * K;

    // all ids, the ids of this wave's own token, then the payload of its task, all in flight together
    int64_t id[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) id[u] = l.topk_idx[min(tid + u * EP_ROW_THREADS, n - 1)];
    const int task = copies ? rb * EP_ROWS_PER_BLOCK + w : 0;
    const int t = task / s.num_parts, part = task - t * s.num_parts;
    const bool works = copies && t < s.num_rows_bound;
    const int64_t own = l.topk_idx[works ? t * K + min(lane, K - 1) : 0];
    const int nvec = QUANT ? s.hidden >> 3 : (int)(s.copy_bytes >> 4);
    const int v = part * WAVE + lane;
    const bool live = works && v < nvec;
    u32x4 d[1] = {{0u, 0u, 0u, 0u}};
    if (live) d[0] = __builtin_nontemporal_load((const u32x4*)((const char*)s.x + (int64_t)t * s.x_row_bytes) + v);
    const unsigned scales = !QUANT && works ? early_scales(s, t, part) : 0u;
    float gate = 0.0f;
    if (works && part == 0 && lane < K && s.topk_weights != nullptr) gate = s.topk_weights[(int64_t)t * K + lane];

    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int i = tid; i < R + (masks ? E : 0) + (Ep >> 2) + 1; i += EP_ROW_THREADS) s_tok[i] = zero;
    __syncthreads();
    // (quotients of small integers: (x + 1/2) / y is at least 1 / 2y away from the next integer, far more than the products round)
    const float per_token = 1.0f / (float)K, per_partition = 1.0f / (float)El;
    auto partition_of = [&](int e) { return (int)(((float)e + 0.5f) * per_partition); };
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (u * EP_ROW_THREADS >= n) break;
        const int i = tid + u * EP_ROW_THREADS;
        const bool valid = i < n && id[u] >= 0 && id[u] < E;
        const int e = valid ? (int)id[u] : -1;
        s_key[i] = (short)e;
        if (valid) {
            const int tok = (int)(((float)i + 0.5f) * per_token);
            const unsigned bit = 1u << (tok & 31);
            atomicAdd(&s_cnt[e], 1);
            atomicOr((unsigned*)&s_tok[PACK ? partition_of(e) : 0] + (tok >> 5), bit);
            if (masks && (atomicOr((unsigned*)&s_mask[e] + (tok >> 5), bit) & bit)) {
                const int x = atomicAdd(s_more, 1);
                if (x < EP_SMALL_REPEATS) s_list[x] = (short)i;
            }
        }
    }
    // (own ids are here by now, and with them the arenas of the token's partitions, which are a trip of their own)
    const int e = (works && lane < K && own >= 0 && own < E) ? (int)own : -1;
    const int r = e < 0 ? -1 : PACK ? partition_of(e) : 0;
    char* peer = nullptr;
    if (PACK && works) peer = s.peer_arenas[max(r, 0)];
    __syncthreads();
    int grand = 0;
    if (!PACK) {
        // aligned exclusive scan over the experts, eight a lane: every wave makes all of it (and writes the same words), which
        // costs less than meeting twice
        const bool pow2 = (A & (A - 1)) == 0;
        for (int e0 = 8 * lane; e0 - 8 * lane < E; e0 += 8 * WAVE) {
            u32x4 c[2] = {zero, zero};
            if (e0 < E) {
                c[0] = *(const u32x4*)(s_cnt + e0);
                c[1] = *(const u32x4*)(s_cnt + e0 + 4);
            }
            int before[8], sum = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int x = (int)c[q >> 2][q & 3];
                before[q] = sum;
                sum += pow2 ? (x + A - 1) & -A : align_up(x, A);
            }
            const int incl = wave_inclusive_sum(sum), run = grand + incl - sum;
            if (e0 < E) {
                *(u32x4*)(s_start + e0) = u32x4{(unsigned)run, (unsigned)(run + before[1]), (unsigned)(run + before[2]), (unsigned)(run + before[3])};
                *(u32x4*)(s_start + e0 + 4) = u32x4{(unsigned)(run + before[4]), (unsigned)(run + before[5]), (unsigned)(run + before[6]), (unsigned)(run + before[7])};
            }
            grand += readlane(incl, WAVE - 1);
        }
        __builtin_amdgcn_wave_barrier();                // (a wave's lanes read each other's words: its LDS operations complete in order)
    }
    auto below = [&](const u32x4& m, int before) -> int {      // bits of m below `before`
        int c = 0;
#pragma unroll
        for (int q = 0; q < TW; ++q) {
            const int bits = min(max(before - 32 * q, 0), 32);
            c += __popc(m[q] & (bits == 32 ? ~0u : (1u << bits) - 1u));
        }
        return c;
    };

    if (publisher) {
        publish_dispatch<PACK>(l, grand, [&](int e) { return s_cnt[e]; }, s_start,
                               [&](int r) { return below(s_tok[r], EP_TOKENS_PER_BLOCK); });
        return;
    }
    if (!copies) {
        const int pieces = s.num_local_experts * s.pad_blocks_per_expert;
        for (int p = rb - s.num_row_blocks; p < pieces; p += a.num_pad_blocks) {
            const int e = p / s.pad_blocks_per_expert;
            zero_padding_piece(s, s_start[e] + s_cnt[e], p - e * s.pad_blocks_per_expert);
        }
        return;
    }
    if (!works) return;

    // ---- rank of the token's entries: earlier entries with the same expert ----
    int rank = 0;
    const int more = __builtin_amdgcn_readfirstlane(*s_more);
    if (masks && more <= EP_SMALL_REPEATS) {
        rank = below(s_mask[max(e, 0)], t);             // earlier tokens that selected it, and beyond that their repetitions
        for (int x0 = 0; x0 < more; x0 += WAVE) {
            const int at = s_list[min(x0 + lane, more - 1)];
            const int earlier = x0 + lane < more && at < t * K ? s_key[at] : -2;
            for (int j = 0; j < K; ++j) {
                const int c0 = __popcll(__ballot(earlier == readlane(e, j)));
                if (lane == j) rank += c0;
            }
        }
        if (more > 0)                                   // (and the same expert earlier in the own token)
            for (int j = 1; j < K; ++j) {
                const int c0 = __popcll(__ballot(e == readlane(e, j)) & ((1ull << j) - 1ull));
                if (lane == j) rank += c0;
            }
    } else {
        const int before = t * K, chunks = (before + WAVE - 1) / WAVE;
        int key[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int i = c * WAVE + lane;
            key[c] = i < before ? s_key[i] : -2;        // (-2 equals no expert and no missing selection)
        }
        for (int j = 0; j < K; ++j) {
            const int ej = readlane(e, j);
            if (ej < 0) continue;
            // (the same expert twice in one token: the earlier one counts too)
            int c0 = __popcll(__ballot(e == ej) & ((1ull << j) - 1ull));
#pragma unroll
            for (int c = 0; c < CH; c += 4)             // (four chunks a branch; a break would keep the loop from being unrolled)
                if (c < chunks) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) c0 += __popcll(__ballot(key[c + q] == ej));
                }
            if (lane == j) rank = c0;
        }
    }
    // ---- masters: the last entry of the token for a partition; its slot there ----
    const uint64_t peers = PACK ? match_any(r + 1, 32 - __builtin_clz(R)) : __ballot(r == 0);
    const int rslot = r >= 0 && (peers >> lane) == 1ull ? below(s_tok[r], t) : -1;
    if (part == 0 && lane < K) {
        l.dst_buffer_slot_idx[(int64_t)t * K + lane] = rslot;
        l.dst_gsge_idx[(int64_t)t * K + lane] = -1;     // every copy is local: no transport descriptors
    }
    RowCtx c;
    c.t = t;
    c.src_row = t;
    c.mybase = 0;
    c.myslot = -1;
    if (PACK) {
        if (rslot >= 0 && rslot < s.max_tokens) {
            c.myslot = (s.region_by_source ? s.rank_idx : r) * s.max_tokens + rslot;
            c.mybase = (uint64_t)(peer + s.buffer_off);
        }
        if (part == 0) pack_row_metadata(s, c, lane < K ? own : 0, gate, e >= 0 ? rank : -1);
    } else {
        const uint64_t vm = __ballot(e >= 0);
        if (vm == 0) return;                            // a token nobody receives
        const int slot = e >= 0 ? s_start[e] + rank : -1;
        if (part == 0) {
            const int last = 63 - __builtin_clzll(vm);
            const int row = readlane(rslot, last);
            // [slot_0 .. slot_{K-1}, src_token_global_idx, last local j]  (dispatch_copy_epilogue.hpp:514-522)
            const int mv = lane < K ? slot : (lane == K ? s.rank_idx * s.max_tokens + t : last);
            if (lane < K + 2 && row >= 0 && row < s.num_meta_rows) s.recv_src_metadata[(int64_t)row * (K + 2) + lane] = mv;
        }
        c.myslot = slot < s.num_out_rows ? slot : -1;
        if (part == 0 && s.recv_topk_weights != nullptr && c.myslot >= 0) s.recv_topk_weights[c.myslot] = gate;
    }
    if (QUANT) quant_row_out<HW, PACK>(s, c, v, live, d[0]);
    else copy_row_out<PACK>(s, c, part, d, scales);
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_copy(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<false, true, false>(a); }
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_quant(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<true, true, false>(a); }
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_quant_sw(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<true, false, false>(a); }
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_copy_pack(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<false, true, true>(a); }
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_quant_pack(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<true, true, true>(a); }
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_dispatch_small_quant_sw_pack(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_small_body<true, false, true>(a); }

// ------------------------------------------------------------------------------------------------
// A dispatch of up to EP_CHUNK_ENTRIES entries in one launch.  Workgroups that fill the chip once, each with an equal share of the
// (token, part) tasks of the copy: every one of them counts the ids of all tokens (all, and those of the tokens before its own
// first, in the two halves of one counter an expert), ranks the entries of the few tokens it copies in one wave, and copies (or
// packs) them.  The payload of a wave's first task is on its way meanwhile; the next one's is fetched ahead of each task's stores.
// Bound by the copy's traffic behind the phases in front of it; those by the launch, a trip to memory for the ids and the
// instructions a thread spends on each (1024 threads of a workgroup, eight waves a SIMD with two workgroups a CU).  At 2048 tokens top-8,
// us from the kernel's start (stamps, 256 workgroups): ids on the way and LDS cleared 1.4, counted 3.0, scanned and ranked 1.8; with a
// mark byte a token, quotients carried along and a token a wave ranked position by position 6.4 + 2.7 + 1.6 at 512 workgroups,
// now 5.0 + 2.2.  A replayed dispatch, two launches / this one (us): 200 tokens x 7168 FP8, top-8, alignment 128 56.7 / 49.2; 512 tokens
// without padding 19.6 / 13.0; 1021 x 2560 BF16, top-7 23.3 / 14.6; 1024 x 7168 BF16, top-8 41.1 / 30.4; 2048 x 7168 66.9 / 53.0; 4096 x
// 1024 top-2 16.4 / 12.9; one of eight partitions, FP8, all of its dispatch: 256 tokens top-8 32.4 / 18.5, 2048 top-6 71.4 / 65.6.
// With several partitions a workgroup counts the ids up to its own tokens' and no further (ranks and places in a partition
// count what is before), so that half of the chip's share of that work falls away and the first workgroups copy meanwhile.  us a
// dispatch and its receive side, all partitions in a captured graph, before / after: eight of 2048 tokens FP8 top-6 532 / 518 (a whole pass with
// both reduces, 1235, is level), of 512 185.7 / 182.7, of 256 125.9 / 125.2; four of 1024 x 4096 top-8 148.1 / 147.3, top-4 106.5 / 106.7.
// (Padding as equal shares of all padding rows in place of pieces of experts: 256 tokens 50.8 -> 56.9; the ids of two goes in flight:
// spills, or one workgroup a CU and level; each id of the next go asked for as one of this go is used: 2048 x 2560 19.8 -> 18.7, but one go
// 1 to 2 % slower.)
// ------------------------------------------------------------------------------------------------
template <bool QUANT, bool HW, bool PACK>
__device__ __forceinline__ void dispatch_chunk_body(const EpSmallArgs& a) {
    extern __shared__ int smem[];
    constexpr int NT = EP_CHUNK_THREADS, NW = NT / WAVE, GO = 8;
    const EpLayoutArgs& l = a.l;
    const EpScatterArgs& s = a.s;
    const int E = l.num_experts, R = l.num_ranks, K = l.num_topk, A = l.expert_alignment, El = l.experts_per_rank;
    const int T = l.num_tokens, n = T * K;
    unsigned* s_cnt = (unsigned*)smem;                  // [E] entries per expert; high half: those before the ones being ranked
    int* s_start = (int*)(s_cnt + E);                   // [E] first slot of each expert (one partition)
    unsigned* s_rcnt = (unsigned*)(s_start + E);        // [R] tokens per partition; high half: those before this workgroup's
    int* s_rown = (int*)(s_rcnt + R);                   // [R] of this workgroup's, those ranked so far
    int* s_tmp = s_rown + R;                            // [NW]
    int* s_rank = s_tmp + NW;                           // [EP_CHUNK_OWN] of an own entry: entries of the same expert before it
    int* s_rslot = s_rank + EP_CHUNK_OWN;               // [EP_CHUNK_OWN] own tokens before its own in its partition (masters), or -1
    short* s_key = (short*)(s_rslot + EP_CHUNK_OWN);    // [EP_CHUNK_OWN] its expert, -1: none
    unsigned* s_mask = (unsigned*)(s_key + EP_CHUNK_OWN);              // [T] partitions a token goes to, a bit each (several), or
                                                        // [entries / 32 + 2] entries with an expert, a bit each (one partition)
    const int tid = threadIdx.x, lane = lane_id(), w = wave_id();
    const bool publisher = blockIdx.x == 0;
    const int wg = (int)blockIdx.x - 1;
    const int tasks = T * s.num_parts;
    const int task0 = publisher ? 0 : min(tasks, wg * a.tasks_per_block), task1 = publisher ? 0 : min(tasks, task0 + a.tasks_per_block);
    const int first = task0 / s.num_parts, own = task1 > task0 ? (task1 - 1) / s.num_parts - first + 1 : 0;
    // who packs needs the ids up to its own and no further (the slots are the receivers' business)
    const int upto = PACK && !publisher ? (first + own) * K : n;
    const int nvec = QUANT ? s.hidden >> 3 : (int)(s.copy_bytes >> 4);

    u32x2 id[GO];
    auto fetch_ids = [&](int i0) {
#pragma unroll
        for (int u = 0; u < GO; ++u) id[u] = *(const u32x2*)((const char*)l.topk_idx + 8u * (unsigned)min(i0 + tid + u * NT, n - 1));
    };
    fetch_ids(0);
    u32x4 next = {0u, 0u, 0u, 0u};
    unsigned next_scales = 0u;
    float next_gate = 0.0f;
    auto fetch_task = [&](int task) {
        if (task >= task1) return;
        const int t = task / s.num_parts, part = task - t * s.num_parts, v = part * WAVE + lane;
        next = u32x4{0u, 0u, 0u, 0u};                   // (channels past the end of the row count as zeros in their group)
        if (v < nvec) next = __builtin_nontemporal_load((const u32x4*)((const char*)s.x + (int64_t)t * s.x_row_bytes) + v);
        if (!QUANT) next_scales = early_scales(s, t, part);
        if (part == 0 && lane < K && s.topk_weights != nullptr) next_gate = s.topk_weights[(int64_t)t * K + lane];
    };
    fetch_task(task0 + w);

    for (int i = tid; i < E; i += NT) s_cnt[i] = 0u;
    if (PACK)
        for (int i = tid; i < T; i += NT) s_mask[i] = 0u;
    if (tid < R) {
        s_rcnt[tid] = 0u;
        s_rown[tid] = 0;
    }
    __syncthreads();
    // (quotients of small integers: (x + 1/2) / y is at least 1 / 2y away from the next integer, far more than the products round)
    const float per_token = 1.0f / (float)K, per_partition = 1.0f / (float)El;
    auto partition_of = [&](int e) { return (int)(((float)e + 0.5f) * per_partition); };
    {
        const int own0 = first * K, nown = own * K, wave0 = __builtin_amdgcn_readfirstlane(w) * WAVE;
        for (int i0 = 0; i0 < upto; i0 += GO * NT) {
            if (i0 > 0) fetch_ids(i0);
#pragma unroll
            for (int u = 0; u < GO; ++u) {
                const int i = i0 + tid + u * NT;
                if (i0 + u * NT + wave0 >= upto) break;
                const bool valid = id[u].y == 0u && id[u].x < (unsigned)E && i < upto;
                if (!PACK) {
                    const uint64_t bits = __ballot(valid);
                    if (lane == 0) ((uint64_t*)s_mask)[i >> 6] = bits;
                }
                if (valid) {
                    atomicAdd(&s_cnt[id[u].x], i < own0 ? 0x10001u : 1u);
                    if (PACK) atomicOr(&s_mask[(int)(((float)i + 0.5f) * per_token)], 1u << partition_of((int)id[u].x));
                }
                if ((unsigned)(i - own0) < (unsigned)nown) s_key[i - own0] = valid ? (short)id[u].x : (short)-1;
            }
        }
    }
    __syncthreads();
    // ---- tokens per partition; aligned exclusive scan over the experts (one partition) ----
    {
        unsigned sum = 0u;                              // lane r < R: of partition r
        for (int t0 = w * WAVE; t0 < (PACK && !publisher ? first : T); t0 += NT) {
            const int t = t0 + lane, at = t * K;
            const uint64_t earlier = __ballot(t < first);
            if (PACK) {
                const unsigned m = t < T ? s_mask[t] : 0u;
                for (int r = 0; r < R; ++r) {
                    const uint64_t to = __ballot((m >> r) & 1u);
                    if (lane == r) sum += (unsigned)__popcll(to) | (unsigned)__popcll(to & earlier) << 16;
                }
            } else {
                const uint64_t bits = t < T ? ((uint64_t)s_mask[(at >> 5) + 1] << 32 | s_mask[at >> 5]) >> (at & 31) : 0ull;
                const uint64_t to = __ballot((bits & ((1ull << K) - 1ull)) != 0ull);
                if (lane == 0) sum += (unsigned)__popcll(to) | (unsigned)__popcll(to & earlier) << 16;
            }
        }
        if (lane < R && sum != 0u) atomicAdd(&s_rcnt[lane], sum);
    }
    int grand = 0, mine = 0, incl = 0;
    const int per = (E + NT - 1) / NT, e0 = min(E, tid * per), e1 = min(E, e0 + per);
    if (!PACK) {
        for (int e = e0; e < e1; ++e) mine += align_up((int)(s_cnt[e] & 0xffffu), A);
        incl = wave_inclusive_sum(mine);
        if (lane == WAVE - 1) s_tmp[w] = incl;
    }
    // ---- meanwhile one wave ranks the own entries, whole tokens at a time: earlier entries with the same expert, masters (the
    //      last entry of a token for a partition), earlier masters of the same partition ----
    if (w == NW - 1) {
        const int ebits = 32 - __builtin_clz(E), rbits = 32 - __builtin_clz(R);
        const int toks = WAVE / K, pos = lane - lane / K * K;
        const uint64_t lt = (1ull << lane) - 1ull, later = (1ull << (K - 1 - pos)) - 1ull;
        for (int c = 0; c < own; c += toks) {
            const int at = c * K + lane;
            const bool in = lane < toks * K && at < own * K;
            const int e = in ? s_key[at] : -1, r = e < 0 ? -1 : PACK ? partition_of(e) : 0;
            const uint64_t pe = match_any(e + 1, ebits), pr = PACK ? match_any(r + 1, rbits) : __ballot(r == 0);
            const bool master = r >= 0 && (pr >> lane >> 1 & later) == 0ull;
            const uint64_t pm = PACK ? match_any(master ? r + 1 : 0, rbits) : __ballot(master);
            int rank = -1, rslot = -1;
            if (e >= 0) {
                const unsigned cnt = s_cnt[e];
                rank = (int)(cnt >> 16) + __popcll(pe & lt);
                if ((pe >> lane) == 1ull) s_cnt[e] = cnt + ((unsigned)__popcll(pe) << 16);      // highest peer
            }
            if (master) {
                const int before = s_rown[r];
                rslot = before + __popcll(pm & lt);
                if ((pm >> lane) == 1ull) s_rown[r] = rslot + 1;
            }
            if (in) {
                s_rank[at] = rank;
                s_rslot[at] = rslot;
            }
            __builtin_amdgcn_wave_barrier();            // (the LDS operations of a wave complete in order)
        }
    }
    if (!PACK) {
        __syncthreads();
        int run = incl - mine;
        for (int i = 0; i < NW; ++i) {
            if (i < w) run += s_tmp[i];
            grand += s_tmp[i];
        }
        for (int e = e0; e < e1; ++e) {
            s_start[e] = run;
            run += align_up((int)(s_cnt[e] & 0xffffu), A);
        }
    }
    __syncthreads();
    if (publisher) {
        publish_dispatch<PACK>(l, grand, [&](int e) { return (int)(s_cnt[e] & 0xffffu); }, s_start,
                               [&](int r) { return (int)(s_rcnt[r] & 0xffffu); });
        return;
    }
    // ---- the tasks ----
    for (int task = task0 + w; task < task1; task += NW) {
        const u32x4 d[1] = {next};
        const unsigned scales = next_scales;
        const float gate = next_gate;
        fetch_task(task + NW);
        const int t = task / s.num_parts, part = task - t * s.num_parts, at = (t - first) * K + lane;
        const int e = lane < K ? s_key[at] : -1, r = PACK ? partition_of(e) : 0;
        int rank = -1, rslot = -1, slot = -1;
        if (e >= 0) {
            rank = s_rank[at];
            if (PACK || part == 0) {
                rslot = s_rslot[at];
                if (rslot >= 0) rslot += (int)(s_rcnt[r] >> 16);
            }
            if (!PACK) slot = s_start[e] + rank;
            else if (rslot >= 0 && rslot < s.max_tokens) slot = (s.region_by_source ? s.rank_idx : r) * s.max_tokens + rslot;
        }
        RowCtx c;
        c.t = t;
        c.src_row = t;
        c.mybase = PACK && slot >= 0 ? (uint64_t)(s.peer_arenas[r] + s.buffer_off) : 0;
        c.myslot = slot;
        if (part == 0) {
            if (lane < K) {
                l.dst_buffer_slot_idx[(int64_t)t * K + lane] = rslot;
                l.dst_gsge_idx[(int64_t)t * K + lane] = -1;             // every copy is local: no transport descriptors
            }
            if (PACK) {
                pack_row_metadata(s, c, lane < K && e < 0 ? l.topk_idx[(int64_t)t * K + lane] : e, gate, rank);
            } else {
                const uint64_t vm = __ballot(slot >= 0);
                const int last = vm != 0 ? 63 - __builtin_clzll(vm) : 0;
                const int row = readlane(rslot, last);
                // [slot_0 .. slot_{K-1}, src_token_global_idx, last local j]  (dispatch_copy_epilogue.hpp:514-522)
                const int mv = lane < K ? slot : (lane == K ? s.rank_idx * s.max_tokens + t : last);
                if (vm != 0 && lane < K + 2 && row >= 0 && row < s.num_meta_rows) s.recv_src_metadata[(int64_t)row * (K + 2) + lane] = mv;
            }
        }
        if (!PACK) {
            c.myslot = slot < s.num_out_rows ? slot : -1;
            if (part == 0 && s.recv_topk_weights != nullptr && c.myslot >= 0) s.recv_topk_weights[c.myslot] = gate;
        }
        const int v = part * WAVE + lane;
        if (QUANT) quant_row_out<HW, PACK>(s, c, v, v < nvec, d[0]);
        else copy_row_out<PACK>(s, c, part, d, scales);
    }
    // ---- padding, in pieces of a 256-thread workgroup ----
    if (!PACK && a.zero_padding) {
        constexpr int GROUPS = NT / EP_ROW_THREADS;
        const int pieces = s.num_local_experts * s.pad_blocks_per_expert;
        for (int p = wg * GROUPS + __builtin_amdgcn_readfirstlane(tid / EP_ROW_THREADS); p < pieces; p += ((int)gridDim.x - 1) * GROUPS) {
            const int e = p / s.pad_blocks_per_expert;
            const int end = __builtin_amdgcn_readfirstlane(s_start[e] + (int)(s_cnt[e] & 0xffffu));
            zero_padding_piece(s, end, p - e * s.pad_blocks_per_expert);
        }
    }
}
#define EP_CHUNK_KERNEL(NAME, QUANT, HW, PACK) \
    extern "C" __global__ __launch_bounds__(EP_CHUNK_THREADS, 8) void ep_dispatch_chunk_##NAME(EpSmallArgs a) { fetch_arguments<EpSmallArgs>(); dispatch_chunk_body<QUANT, HW, PACK>(a); }
EP_CHUNK_KERNEL(copy, false, true, false)
EP_CHUNK_KERNEL(quant, true, true, false)
EP_CHUNK_KERNEL(quant_sw, true, false, false)
EP_CHUNK_KERNEL(copy_pack, false, true, true)
EP_CHUNK_KERNEL(quant_pack, true, true, true)
EP_CHUNK_KERNEL(quant_sw_pack, true, false, true)

// ------------------------------------------------------------------------------------------------
// Receive side of a node whose send sides ship ranks, placing and copying in one launch: what ep_layout_place and the
// copy kernel of received rows do, for at most 64 partitions.  Every workgroup adds the counts up itself: the row counts of
// the sources in registers (a lane a source), the counts per source and expert in LDS; a wave then knows the slots of its
// row's entries from their ids and shipped ranks.  The row's payload is fetched with its ids.  Workgroup 0 writes the handle tensors (no
// host waits for counts of this launch), the next ones copy, the last zero the padding.
// Bound by two trips to memory (counts; ids, ranks and payload) and the launch at decode sizes, by the copy's traffic beyond.
// Eight partitions of 2048 tokens, all phases 1372 -> 1325 us; of 64 tokens (bound by the host's calls) 409 -> 383 us.
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_recv_copy(EpSmallArgs a) {
    fetch_arguments<EpSmallArgs>();
    extern __shared__ int smem[];
    constexpr int NW = EP_ROW_THREADS / WAVE;
    const EpLayoutArgs& l = a.l;
    const EpScatterArgs& s = a.s;
    const int E = l.num_experts, R = l.num_ranks, K = l.num_topk, El = l.experts_per_rank, A = l.expert_alignment;
    int* s_box = smem;                     // [R][El] counts per source and local expert
    int* s_start = s_box + E;              // [El] first slot of each expert
    int* s_cnt = s_start + El;             // [El]
    int* s_tmp = s_cnt + El;               // [NW]
    const int tid = threadIdx.x, lane = lane_id(), w = wave_id();
    const bool publisher = blockIdx.x == 0;
    const int rb = (int)blockIdx.x - 1, lo = l.rank_idx * El;
    const bool copies = !publisher && rb < s.num_row_blocks;

    // ---- counts of all sources; the row of the receive stream that a wave works on ----
    const int mine = lane < R ? max(0, min(l.inbox[lane], l.max_tokens)) : 0;
    for (int i = tid; i < E; i += EP_ROW_THREADS) s_box[i] = l.count_box[i];
    const int upto = wave_inclusive_sum(mine);           // lane r < R: rows of the sources up to r
    const int num_rows = readlane(upto, WAVE - 1);
    const int task = copies ? rb * EP_ROWS_PER_BLOCK + w : 0;
    const int i = task / s.num_parts, part = task - i * s.num_parts;
    if (copies && rb * EP_ROWS_PER_BLOCK / s.num_parts >= num_rows) return;
    const bool works = copies && i < min(num_rows, s.num_rows_bound);
    const int q = works ? __popcll(__ballot(lane < R && upto <= i)) : 0;       // sources whose rows all come before row i
    const int slot_in = works ? i - (q ? readlane(upto, q - 1) : 0) : 0;
    const int64_t pr = (int64_t)q * l.max_tokens + slot_in;
    const char* packed = l.packed_base + pr * l.packed_row_bytes;
    const int nvec = (int)(s.copy_bytes >> 4), U = s.vecs_per_lane;
    u32x4 d[4];
    int64_t id = -1;
    int rank = 0, src = 0;
    float gate = 0.0f;
    unsigned scales = 0u;
    if (works) {
        if (lane < K) {
            id = ((const int64_t*)(packed + l.idx_off))[lane];
            rank = l.rank_box[pr * K + lane];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int v = (part * U + u) * WAVE + lane;
            if (u < U && v < nvec) d[u] = __builtin_nontemporal_load((const u32x4*)packed + v);
        }
        scales = early_scales(s, pr, part);
        if (part == 0) {
            src = *(const int*)(packed + l.src_off);
            if (lane < K && s.recv_topk_weights != nullptr) gate = ((const float*)(packed + s.w_off))[lane];
        }
    }
    __syncthreads();

    // ---- totals, aligned scan over the experts ----
    const int per = (El + EP_ROW_THREADS - 1) / EP_ROW_THREADS;
    const int e0 = min(El, tid * per), e1 = min(El, e0 + per);
    int aligned = 0;
    for (int e = e0; e < e1; ++e) {
        int c = 0;
        for (int r = 0; r < R; ++r) c += s_box[r * El + e];
        s_cnt[e] = c;
        aligned += align_up(c, A);
    }
    const int incl = wave_inclusive_sum(aligned);
    if (lane == WAVE - 1) s_tmp[w] = incl;
    __syncthreads();
    int run = incl - aligned;
    for (int k = 0; k < NW; ++k)
        if (k < w) run += s_tmp[k];
    for (int e = e0; e < e1; ++e) {
        s_start[e] = run;
        run += align_up(s_cnt[e], A);
    }
    __syncthreads();

    if (publisher) {
        for (int e = tid; e < El; e += EP_ROW_THREADS) {
            const int c = s_cnt[e];
            l.unaligned_expert[e] = c;
            l.psum_expert[e] = s_start[e] + c;
            if (l.cumulative_stats != nullptr) atomicAdd(&l.cumulative_stats[e], c);
        }
        if (tid < R) l.psum_rank[tid] = upto;            // (the first wave: R <= 64)
        return;
    }
    if (!copies) {
        const int pieces = El * s.pad_blocks_per_expert;
        for (int p = rb - s.num_row_blocks; p < pieces; p += a.num_pad_blocks) {
            const int e = p / s.pad_blocks_per_expert;
            zero_padding_piece(s, s_start[e] + s_cnt[e], p - e * s.pad_blocks_per_expert);
        }
        return;
    }
    if (!works) return;

    // ---- slots: first slot of the expert, entries of the sources before, rank inside the source ----
    const bool local = id >= lo && id < lo + El;
    const int le = local ? (int)id - lo : 0;
    int slot = s_start[le] + rank;
    for (int r = 0; r < q; ++r) slot += s_box[r * El + le];
    if (!local) slot = -1;
    if (part == 0) {
        const uint64_t vm = __ballot(local);
        // [slot_0 .. slot_{K-1}, src_token_global_idx, last local j]  (dispatch_copy_epilogue.hpp:514-522)
        const int v = lane < K ? slot : (lane == K ? src : (vm != 0 ? 63 - __builtin_clzll(vm) : -1));
        if (lane < K + 2 && i < l.rows_cap) l.recv_src_metadata[(int64_t)i * (K + 2) + lane] = v;
    }
    RowCtx c;
    c.t = i;
    c.mybase = 0;
    c.src_row = pr;
    c.myslot = slot >= 0 && slot < s.num_out_rows ? slot : -1;
    if (part == 0 && s.recv_topk_weights != nullptr && c.myslot >= 0) s.recv_topk_weights[c.myslot] = gate;
    copy_row_out<false>(s, c, part, d, scales);
}

// The quantiser alone (deep_ep/utils/math.py:30-38, what a caller runs before a dispatch of pre-quantised rows):
// the arithmetic of the fused kernel above, rows written in place of being scattered.
template <bool HW>
__device__ __forceinline__ void quant_rows_body(const EpQuantArgs& a) {
    const int lane = lane_id();
    const int task = blockIdx.x * EP_ROWS_PER_BLOCK + wave_id();
    const int t = task / a.num_parts, part = task - t * a.num_parts;
    if (t >= a.num_rows) return;
    const int nvec = a.hidden >> 3;
    const int v = part * WAVE + lane;
    const bool live = v < nvec;
    u32x4 d = {0u, 0u, 0u, 0u};
    if (live) d = __builtin_nontemporal_load((const u32x4*)((const char*)a.x + (int64_t)t * a.hidden * 2) + v);
    float f[8] = {bf16_lo(d.x), bf16_hi(d.x), bf16_lo(d.y), bf16_hi(d.y),
                  bf16_lo(d.z), bf16_hi(d.z), bf16_lo(d.w), bf16_hi(d.w)};
    unsigned mbits = 0u;
#pragma unroll
    for (int q = 0; q < 8; ++q) mbits = max(mbits, __float_as_uint(f[q]) & 0x7fffffffu);
    const float m = __uint_as_float(row16_umax(mbits));
    const float amax = m < 1e-4f ? 1e-4f : m;
    const float inv = (1.0f / amax) * 448.0f;
    u32x2 q8 = quant8<HW>(f, inv);
    if (amax != amax) q8 = u32x2{0x7f7f7f7fu, 0x7f7f7f7fu};
    if (!live) return;
    ((u32x2*)((char*)a.q + (int64_t)t * a.hidden))[v] = q8;
    if ((lane & 15) == 0) a.sf[(int64_t)t * ((a.hidden + 127) >> 7) + (v >> 4)] = amax / 448.0f;
}
extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_quant_rows(EpQuantArgs a) {
    if (a.hw_convert) quant_rows_body<true>(a);
    else quant_rows_body<false>(a);
}

// Column-major scales (use_tma_aligned_col_major_sf): the copy kernels write scale rows, this
// kernel turns them into columns.  The reference does the same with a generic transposing copy
// (csrc/buffers/ep.hpp:379-381); writing columns straight from the copy kernel was measured and is
// slower, since every 4-byte scale then lands in a cache line of its own.
template <typename E>
__device__ __forceinline__ void sf_transpose_body(const EpSfTransposeArgs& a, int n, unsigned (*tile)[EP_SF_TILE + 1]) {
    const int r0 = blockIdx.x * EP_SF_TILE;
    const int tx = threadIdx.x % EP_SF_TILE, ty = threadIdx.x / EP_SF_TILE;
    constexpr int STEP = EP_LAYOUT_THREADS / EP_SF_TILE;
    const E* src = (const E*)a.src;
    E* dst = (E*)a.dst;
    for (int c0 = 0; c0 < a.num_cols; c0 += EP_SF_TILE) {
        for (int rr = ty; rr < EP_SF_TILE; rr += STEP)
            if (r0 + rr < n && c0 + tx < a.num_cols) tile[rr][tx] = src[(int64_t)(r0 + rr) * a.num_cols + c0 + tx];
        __syncthreads();
        for (int cc = ty; cc < EP_SF_TILE; cc += STEP)
            if (c0 + cc < a.num_cols && r0 + tx < n) dst[(int64_t)(c0 + cc) * n + r0 + tx] = (E)tile[tx][cc];
        __syncthreads();
    }
}

// Whole rows through LDS, from a 16-byte aligned source: 64 rows of at most EP_SF_WIDE_ROW_BYTES, half as many at a time per
// doubling of the row (8 at the widest).  They are one contiguous piece of the source: the piece goes to LDS in 16-byte loads,
// all of a thread's in flight, and leaves as V adjacent rows of a column a
// store: 16 bytes where columns start on 16 bytes (16 to 256 bytes a column and piece), else 4, else one element.
// 52 thousand rows of 112 2-byte packs: 11.2 us with pairs of packs and two barriers per 64 columns, 7.7 us so (fetching the
// rows before the row count is known, to save its trip, measured 8.4: the workgroups beyond the rows then fetch as well).
// Wider rows, whole calls (pairs of packs / element by element / so): 3000 tokens top-2, 192 packs 171 / 184 / 161 us; 2501 tokens
// top-4, 256 packs 157 / 170 / 150; 2000 tokens top-8, 320 packs 535 / 557 / 527.
template <typename E, int V>
__device__ __forceinline__ void sf_columns_out(const EpSfTransposeArgs& a, int n, int r0, int log_rows, int rows, int pitch,
                                               const unsigned char* lds) {
    typedef E vec_t __attribute__((ext_vector_type(V)));
    const int log_groups = log_rows - __builtin_ctz(V);                // 2^log_groups vectors of V rows a column
    const int rr = ((int)threadIdx.x & ((1 << log_groups) - 1)) * V;
    for (int c = (int)threadIdx.x >> log_groups; c < a.num_cols; c += EP_LAYOUT_THREADS >> log_groups) {
        E* out = (E*)a.dst + (int64_t)c * n + r0 + rr;
        vec_t x;
#pragma unroll
        for (int q = 0; q < V; ++q) x[q] = *(const E*)(lds + (rr + q) * pitch + c * (int)sizeof(E));
        if (rr + V <= rows) *(vec_t*)out = x;
        else
            for (int q = 0; q < V; ++q)
                if (rr + q < rows) out[q] = x[q];
    }
}
template <typename E>
__device__ __forceinline__ void sf_transpose_wide(const EpSfTransposeArgs& a, int n, int r0, int log_rows, unsigned char* lds) {
    constexpr int VEC = 16 / (int)sizeof(E), MAXV = EP_SF_TILE * EP_SF_WIDE_ROW_BYTES / 16 / EP_LAYOUT_THREADS;
    const int cols = a.num_cols, rows = min(1 << log_rows, n - r0);
    // rows of an odd number of words: the rows that neighbouring lanes read spread over the banks
    const int pitch = ((cols * (int)sizeof(E) + 3) / 4 | 1) * 4;
    const int count = rows * cols, nvec = count / VEC;
    const E* src = (const E*)a.src + (int64_t)r0 * cols;
    u32x4 v[MAXV];
#pragma unroll
    for (int u = 0; u < MAXV; ++u) {
        const int i = threadIdx.x + u * EP_LAYOUT_THREADS;
        if (i < nvec) v[u] = ((const u32x4*)src)[i];
    }
#pragma unroll
    for (int u = 0; u < MAXV; ++u) {
        const int i = threadIdx.x + u * EP_LAYOUT_THREADS;
        if (i >= nvec) break;
        int r = i * VEC / cols, c = i * VEC - r * cols;
        E x[VEC];
        __builtin_memcpy(x, &v[u], 16);
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
            *(E*)(lds + r * pitch + c * (int)sizeof(E)) = x[q];
            if (++c == cols) { c = 0; ++r; }
        }
    }
    if ((int)threadIdx.x < count - nvec * VEC) {            // the last, partial vector
        const int i = nvec * VEC + threadIdx.x, r = i / cols;
        *(E*)(lds + r * pitch + (i - r * cols) * (int)sizeof(E)) = src[i];
    }
    __syncthreads();
    const int step = n * (int)sizeof(E) | (int)((uintptr_t)a.dst & 15);
    if ((step & 15) == 0) sf_columns_out<E, VEC>(a, n, r0, log_rows, rows, pitch, lds);
    else if ((step & 3) == 0) sf_columns_out<E, 4 / (int)sizeof(E)>(a, n, r0, log_rows, rows, pitch, lds);
    else sf_columns_out<E, 1>(a, n, r0, log_rows, rows, pitch, lds);
}
// The 64 rows of a workgroup: at once (a case of its own: with the number of rows in a register narrow rows lose 3 % of a
// call, 160 thousand rows of 16 packs), or in pieces of fewer where the rows are wider.
template <typename E>
__device__ __forceinline__ void sf_transpose_pieces(const EpSfTransposeArgs& a, int n, unsigned char* lds) {
    constexpr int LOG_TILE = __builtin_ctz(EP_SF_TILE);
    const int r0 = blockIdx.x * EP_SF_TILE, row_bytes = a.num_cols * (int)sizeof(E);
    if (row_bytes <= EP_SF_WIDE_ROW_BYTES) {
        sf_transpose_wide<E>(a, n, r0, LOG_TILE, lds);
        return;
    }
    int log_rows = LOG_TILE - 1;
    while (row_bytes << log_rows > EP_SF_TILE * EP_SF_WIDE_ROW_BYTES) --log_rows;
    const int end = min(r0 + EP_SF_TILE, n);
    for (int r = r0; r < end; r += 1 << log_rows) {
        if (r != r0) __syncthreads();                       // (the piece before has left the LDS)
        sf_transpose_wide<E>(a, n, r, log_rows, lds);
    }
}

extern "C" __global__ __launch_bounds__(EP_LAYOUT_THREADS) void ep_sf_transpose(EpSfTransposeArgs a) {
    __shared__ __align__(16) unsigned char lds[EP_SF_TILE * (EP_SF_WIDE_ROW_BYTES + 4)];
    int n = a.num_rows;
    if (a.counted) n = min(n, align_up(a.psum_expert[a.num_local_experts - 1], a.expert_alignment));
    if ((int)blockIdx.x * EP_SF_TILE >= n) return;
    // (8 rows: the fewest that still make a 16-byte store of 2-byte packs; wider rows, and a source that does not start on 16
    // bytes, go element by element)
    const bool wide = a.num_cols * a.elem_bytes <= EP_SF_WIDE_ROW_BYTES * EP_SF_TILE / 8 && ((uintptr_t)a.src & 15) == 0;
    if (a.elem_bytes == 4) {
        if (wide) sf_transpose_pieces<unsigned>(a, n, lds);
        else sf_transpose_body<unsigned>(a, n, (unsigned (*)[EP_SF_TILE + 1])lds);
    } else {
        if (wide) sf_transpose_pieces<unsigned short>(a, n, lds);
        else sf_transpose_body<unsigned short>(a, n, (unsigned (*)[EP_SF_TILE + 1])lds);
    }
}

// ------------------------------------------------------------------------------------------------
// Combine, single partition: gather the row's expanded slots, sum in fp32 in ascending slot
// order, round once to BF16, then add the biases the same way.
// Reference semantics: impls/ep/combine.hpp:291-324 + combine_utils.hpp:14-93 (owner side),
// combine_reduce_epilogue.hpp:96-154 (token side); with one partition each token has one partial.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned f32_to_bf16_bits(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

__device__ __forceinline__ void unpack8(const u32x4& d, float* f) {
    f[0] = bf16_lo(d.x); f[1] = bf16_hi(d.x); f[2] = bf16_lo(d.y); f[3] = bf16_hi(d.y);
    f[4] = bf16_lo(d.z); f[5] = bf16_hi(d.z); f[6] = bf16_lo(d.w); f[7] = bf16_hi(d.w);
}

__device__ __forceinline__ u32x4 pack8(const float* f) {
    u32x4 o;
    o.x = f32_to_bf16_bits(f[0]) | (f32_to_bf16_bits(f[1]) << 16);
    o.y = f32_to_bf16_bits(f[2]) | (f32_to_bf16_bits(f[3]) << 16);
    o.z = f32_to_bf16_bits(f[4]) | (f32_to_bf16_bits(f[5]) << 16);
    o.w = f32_to_bf16_bits(f[6]) | (f32_to_bf16_bits(f[7]) << 16);
    return o;
}

// out = BF16(f32 b0 + f32 b1 + f32 partial), left to right; a single input is copied verbatim.
__device__ __forceinline__ u32x4 add_biases(const EpCombineArgs& a, int t, int v, bool have_partial, u32x4 partial) {
    const int64_t rowvec = a.hidden >> 3;
    float acc[8], g[8];
    int nin = 0;
    u32x4 last = {0u, 0u, 0u, 0u};
    const void* biases[2] = {a.bias_0, a.bias_1};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        if (biases[b] == nullptr) continue;
        last = ((const u32x4*)biases[b])[(int64_t)t * rowvec + v];
        unpack8(last, g);
        if (nin == 0) { for (int q = 0; q < 8; ++q) acc[q] = g[q]; }
        else { for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q]; }
        ++nin;
    }
    if (have_partial) {
        last = partial;
        unpack8(partial, g);
        if (nin == 0) { for (int q = 0; q < 8; ++q) acc[q] = g[q]; }
        else { for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q]; }
        ++nin;
    }
    if (nin <= 1) return last;          // zero inputs -> zeros, one input -> verbatim
    return pack8(acc);
}

// The same with the bias vectors already in registers (fetched together with the rows): the biases that exist, in
// order, then the partial.  (Registers of their own and uniform flags: a run-time index into an array of loaded
// vectors would make the compiler wait for the loads where they are issued.)
__device__ __forceinline__ u32x4 add_loaded_biases(bool has0, u32x4 x0, bool has1, u32x4 x1, u32x4 partial) {
    if (!has0 && !has1) return partial;
    float acc[8], g[8];
    if (has0) {
        unpack8(x0, acc);
        if (has1) {
            unpack8(x1, g);
            for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q];
        }
    } else {
        unpack8(x1, acc);
    }
    unpack8(partial, g);
    for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q];
    return pack8(acc);
}

// Tokens with no valid slot are never received: their output is the bias sum (or zero).
__device__ __forceinline__ void combine_unrouted(const EpCombineArgs& a) {
    const int lane = lane_id();
    const int K = a.num_topk;
    const int tb = ((int)blockIdx.x - a.num_row_blocks) * EP_ROW_THREADS + wave_id() * WAVE;
    const int t = tb + lane;
    bool unrouted = false;
    if (t < a.num_tokens) {
        unrouted = true;
        for (int j = 0; j < K; ++j) {
            const int64_t e = a.topk_idx[(int64_t)t * K + j];
            if (e >= 0 && e < a.num_experts) unrouted = false;
        }
    }
    uint64_t m = __ballot(unrouted);
    const int nvec = a.hidden >> 3;
    const u32x4 z = {0u, 0u, 0u, 0u};
    while (m != 0) {
        const int l = __builtin_ctzll(m);
        m &= m - 1;
        const int tt = tb + l;
        for (int v = lane; v < nvec; v += WAVE)
            ((u32x4*)a.combined_x)[(int64_t)tt * nvec + v] = add_biases(a, tt, v, false, z);
        if (a.combined_topk_weights != nullptr && lane < K) a.combined_topk_weights[(int64_t)tt * K + lane] = 0.0f;
    }
}

// A wave task is (row, 1024-channel part): two 16-byte vectors per lane and input row, all loads
// issued before the first add.  MODE selects which reduction of the reference the task performs:
//   EP_COMBINE_FUSED    one partition: rows are the receive stream; out = BF16(sum_j f32 y[slot_j]), then
//                       BF16(f32 b0 + f32 b1 + f32 that) when biases are given (the two levels of
//                       combine.hpp:291-324 and combine_reduce_epilogue.hpp:114-140 for a single master)
//   EP_COMBINE_PARTIAL  owner side: same sum, stored with its K-wide weight vector in the combine buffer
//                       at [group * max_tokens + source token]            (combine.hpp:94-106,301-324)
//   EP_COMBINE_FINAL    token side: rows are tokens; inputs = b0, b1, then the partial of every master
//                       (last top-k position per destination partition) in ascending position, summed
//                       left to right in fp32 and rounded once; weight vectors OR-merged
//                       (combine_reduce_epilogue.hpp:96-153)
// LOADS / STORES: the benchmarks' calibration code object builds the single-partition kernel once without its row
// fetches and once without its stores (what each stream costs alone); the library's kernels have both.
template <int KT, int MODE, bool LOADS = true, bool STORES = true>
__device__ __forceinline__ void combine_body(const EpCombineArgs& a) {
    static_assert((LOADS && STORES) || (KT > 0 && MODE == EP_COMBINE_FUSED), "only the unrolled single-partition kernel is taken apart");
    if (MODE == EP_COMBINE_FUSED && (int)blockIdx.x >= a.num_row_blocks) {
        combine_unrouted(a);
        return;
    }
    const int lane = lane_id();
    const int K = KT > 0 ? KT : a.num_topk;
    const int task = blockIdx.x * EP_ROWS_PER_BLOCK + wave_id();
    const int i = task / a.num_parts, part = task - i * a.num_parts;
    if (i >= a.num_rows_bound) return;

    int myslot = -1, t, group = 0, src_rank = 0;
    if (MODE == EP_COMBINE_FINAL) {
        t = i;
        int r = -1;
        if (lane < K) {
            const int64_t e = a.topk_idx[(int64_t)t * K + lane];
            if (e >= 0 && e < a.num_experts) r = (int)(e / a.experts_per_rank);
        }
        bool master = r >= 0;
        for (int jj = 1; jj < K; ++jj) {
            const int rj = readlane(r, jj);
            if (lane < jj && rj == r) master = false;          // a later position goes to the same partition
        }
        if (master) myslot = (a.num_ranks < K ? r : lane) * a.max_tokens + t;
    } else {
        const int mv = lane < K + 2 ? a.recv_src_metadata[(int64_t)i * (K + 2) + lane] : -1;
        const int num_recv = MODE == EP_COMBINE_PARTIAL ? uniform_load(a.num_recv_ptr) : *a.num_recv_ptr;
        if (i >= num_recv) return;                       // (checked after the row's own load has been issued)
        if (lane < K && mv >= 0 && mv < a.num_in_rows) myslot = mv;
        const int src = readlane(mv, K);                        // source partition * max_tokens + its token
        if (MODE == EP_COMBINE_PARTIAL) {
            src_rank = src / a.max_tokens;
            if (src < 0 || src_rank >= a.num_ranks) return;
            t = src - src_rank * a.max_tokens;
        } else {
            t = src - a.rank_idx * a.max_tokens;
            if (t < 0 || t >= a.max_tokens || t >= a.num_tokens) return;
        }
        group = a.num_ranks < K ? a.rank_idx : readlane(mv, K + 1);
        if (MODE == EP_COMBINE_PARTIAL && (group < 0 || group >= a.num_groups)) return;
    }
    const int nvalid = __popcll(__ballot(myslot >= 0));
    // Owner side with long parts (32 / 16 / 4 partitions of 4096 / 4096 / 8192 tokens, top-6: 157 / 152 / 227 us with a wave a
    // row, 136 / 136 / 199 so): a received row mostly has one or two slots among this partition's few experts, and one
    // slot's partial is that row verbatim: 4 vectors a lane and slot in flight, the second slot's behind the first's.
    const bool verbatim = MODE == EP_COMBINE_PARTIAL && a.long_parts && nvalid == 1;
    const int nvec = a.hidden >> 3;
    const int64_t yvec = a.y_row_bytes >> 4;
    const u32x4* y = (const u32x4*)a.y;
    // a partial goes to the combine buffer of the partition its token came from (impls/ep/combine.hpp:291-324)
    char* out_row = MODE == EP_COMBINE_PARTIAL
        ? uniform_load(&a.peer_arenas[src_rank]) + a.buffer_off + ((int64_t)group * a.max_tokens + t) * a.out_row_bytes
        : (char*)a.combined_x + (int64_t)t * a.out_row_bytes;

    // ---- gate weights ----
    float myw = 0.0f;
    if (MODE == EP_COMBINE_FINAL) {
        if (part == 0 && a.combined_topk_weights != nullptr) {
            unsigned acc = 0;
            if (KT > 0 && nvalid > 0) {
                // the weight vectors of all masters in one trip: no branch and no per-lane condition between the
                // loads (a position that is no master re-reads the first master's vector and is left out)
                const int s_any = readlane(myslot, (int)__builtin_ctzll(__ballot(myslot >= 0)));
                const int wl = min(lane, K - 1);
                unsigned wv[KT > 0 ? KT : 1];
#pragma unroll
                for (int j = 0; j < KT; ++j) {
                    const int s = readlane(myslot, j);
                    wv[j] = ((const unsigned*)((const char*)a.y + (int64_t)(s >= 0 ? s : s_any) * a.y_row_bytes + (a.hidden << 1)))[wl];
                }
#pragma unroll
                for (int j = 0; j < KT; ++j)
                    if (readlane(myslot, j) >= 0) acc |= wv[j];
            } else {
                for (int j = 0; j < K; ++j) {
                    const int s = readlane(myslot, j);
                    if (s < 0) continue;
                    if (lane < K) acc |= ((const unsigned*)((const char*)a.y + (int64_t)s * a.y_row_bytes + (a.hidden << 1)))[lane];
                }
            }
            if (lane < K) ((unsigned*)a.combined_topk_weights)[(int64_t)t * K + lane] = acc;
        }
    } else {
        const bool need_w = part == 0 || (MODE == EP_COMBINE_FUSED && a.weighted);
        if (LOADS && need_w && a.expanded_weights != nullptr && myslot >= 0) myw = a.expanded_weights[myslot];
        if (part == 0 && lane < K) {
            if (STORES && MODE == EP_COMBINE_FUSED && a.combined_topk_weights != nullptr)
                a.combined_topk_weights[(int64_t)t * K + lane] = myw;
            // (the verbatim path below stores them behind its row fetches, so that the two trips become one)
            if (MODE == EP_COMBINE_PARTIAL && a.expanded_weights != nullptr && !verbatim)
                ((float*)(out_row + (a.hidden << 1)))[lane] = myw;
        }
    }

    u32x4* out = (u32x4*)out_row;
    const bool has0 = a.bias_0 != nullptr, has1 = a.bias_1 != nullptr;
    const bool weighted = MODE == EP_COMBINE_FUSED && a.weighted;
    constexpr int LONG = EP_COMBINE_LONG_PART / (8 * WAVE);       // vectors a lane of a long part
    const bool long_parts = MODE == EP_COMBINE_PARTIAL && a.long_parts;
    if (long_parts && nvalid >= 1 && nvalid <= 2) {
        const uint64_t vm = __ballot(myslot >= 0);
        const u32x4* src0 = y + (int64_t)readlane(myslot, __builtin_ctzll(vm)) * yvec;
        const u32x4* src1 = y + (int64_t)readlane(myslot, 63 - __builtin_clzll(vm)) * yvec;
        // (a lane past the end of the row re-reads the last vector and stores nothing)
        const int vb = part * LONG * WAVE + lane;
        u32x4 d0[LONG], d1[LONG];
#pragma unroll
        for (int u = 0; u < LONG; ++u) d0[u] = __builtin_nontemporal_load(src0 + min(vb + u * WAVE, nvec - 1));
        if (verbatim) {
            if (part == 0 && lane < K && a.expanded_weights != nullptr) ((float*)(out_row + (a.hidden << 1)))[lane] = myw;
#pragma unroll
            for (int u = 0; u < LONG; ++u)
                if (vb + u * WAVE < nvec) stream_store<EP_COMBINE_ST_POL>(out + vb + u * WAVE, d0[u]);
            return;
        }
#pragma unroll
        for (int u = 0; u < LONG; ++u) d1[u] = __builtin_nontemporal_load(src1 + min(vb + u * WAVE, nvec - 1));
#pragma unroll
        for (int u = 0; u < LONG; ++u) {
            float f[8], g[8];
            unpack8(d0[u], f);
            unpack8(d1[u], g);
            for (int q = 0; q < 8; ++q) f[q] = f[q] + g[q];
            if (vb + u * WAVE < nvec) stream_store<EP_COMBINE_ST_POL>(out + vb + u * WAVE, pack8(f));
        }
        return;
    }
    // a task is one 1024-channel part of its row, or (owner side, long parts) several in turn
    const int part_end = long_parts ? min((part + 1) * (LONG / 2), (nvec + 2 * WAVE - 1) / (2 * WAVE)) : part + 1;
    for (int cp = long_parts ? part * (LONG / 2) : part; cp < part_end; ++cp) {
    const int v0 = cp * 2 * WAVE + lane, v1 = v0 + WAVE;
    const bool live0 = v0 < nvec, live1 = v1 < nvec;
    // the gate weights are scattered 4-byte loads: only the task that carries them back (part 0) or multiplies
    // by them has read them; the other tasks hold zeros
    const u32x4 zero = {0u, 0u, 0u, 0u};
    if (KT > 0) {
        // Every load of the task is issued before the first add: the biases of the token (not on the owner side), then
        // both 16-byte vectors of every input row.  The two vectors are then reduced one after the other, which
        // keeps the live registers at the loaded vectors plus one accumulator (72 VGPRs at K = 6: seven waves a SIMD).
        // No load depends on the lane being live: a lane past the end of the row fetches the row's last vector and
        // stores nothing.  (A load under a per-lane condition has to be merged with the register's old value when it
        // returns, and the compiler then waits for the first such load before it issues the next.)
        const int c0 = min(v0, nvec - 1), c1 = min(v1, nvec - 1);
        u32x4 d0[KT > 0 ? KT : 1], d1[KT > 0 ? KT : 1];
        // bias vectors: p0* of bias_0, p1* of bias_1, *a for the first vector of the task, *b for the second
        u32x4 p0a = zero, p0b = zero, p1a = zero, p1b = zero;
        if (MODE != EP_COMBINE_PARTIAL) {
            if (has0) {
                const u32x4* bp = (const u32x4*)a.bias_0 + (int64_t)t * nvec;
                p0a = __builtin_nontemporal_load(bp + c0);
                p0b = __builtin_nontemporal_load(bp + c1);
            }
            if (has1) {
                const u32x4* bp = (const u32x4*)a.bias_1 + (int64_t)t * nvec;
                p1a = __builtin_nontemporal_load(bp + c0);
                p1b = __builtin_nontemporal_load(bp + c1);
            }
        }
        // token side: the biases open the one accumulation; single partition: they are added to the rounded sum of
        // the rows in a second one (the two levels of the reference)
        const bool first0 = MODE == EP_COMBINE_FINAL && has0, first1 = MODE == EP_COMBINE_FINAL && has1;
        if (MODE == EP_COMBINE_PARTIAL) {
            // owner side: a received row has one or two of its K positions on this partition: fetch those only
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                const int s = readlane(myslot, j);
                if (s < 0) continue;
                d0[j] = __builtin_nontemporal_load(y + (int64_t)s * yvec + c0);
                d1[j] = __builtin_nontemporal_load(y + (int64_t)s * yvec + c1);
            }
        } else if (!LOADS) {
            const u32x4 filler = {(unsigned)lane, (unsigned)i, 0x3f803f80u, 0x3f803f80u};
#pragma unroll
            for (int j = 0; j < KT; ++j) d0[j] = d1[j] = filler;
        } else if (nvalid > 0) {
            // nearly every position is valid: one straight run of 2 K loads with no branch in it, a position without
            // a row re-reads the first valid one (the same cache lines again) and is left out of the sum below
            const int s_any = readlane(myslot, (int)__builtin_ctzll(__ballot(myslot >= 0)));
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                const int s = readlane(myslot, j);
                const int64_t row = (int64_t)(s >= 0 ? s : s_any) * yvec;
                d0[j] = __builtin_nontemporal_load(y + row + c0);
                d1[j] = __builtin_nontemporal_load(y + row + c1);
                // sixteen and more fetches a wave are better sent in two goes, the first row ahead of the others
                // (top-8 at 16384 / 32768 tokens: 354 / 707 us against 362 / 730 all at once; top-6 and below lose:
                // 277 against 272), unless the launch waits for its trips to memory and not for their bandwidth
                if (KT >= 8 && j == 0 && a.paced) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
        }
        // inputs in order: b0, b1, then the rows in ascending position; zero inputs -> zeros, one input -> verbatim
        // copy, more -> one rounding of the fp32 sum (a weighted single row is a product: rounded as well)
        auto reduce = [&](u32x4 x0, u32x4 x1, const u32x4* d) -> u32x4 {
            float acc[8], g[8];
            u32x4 first = zero;
            int nin = 0;
            if (first0) {
                unpack8(x0, acc);
                first = x0;
                ++nin;
            }
            if (first1) {
                unpack8(x1, g);
                if (nin == 0) { for (int q = 0; q < 8; ++q) acc[q] = g[q]; first = x1; }
                else { for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q]; }
                ++nin;
            }
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                const int s = readlane(myslot, j);
                if (s < 0) continue;
                unpack8(d[j], g);
                if (weighted) {
                    const float wj = __int_as_float(readlane(__float_as_int(myw), j));
                    for (int q = 0; q < 8; ++q) g[q] = g[q] * wj;
                }
                if (nin == 0) { for (int q = 0; q < 8; ++q) acc[q] = g[q]; first = d[j]; }
                else { for (int q = 0; q < 8; ++q) acc[q] = acc[q] + g[q]; }
                ++nin;
            }
            if (nin >= 2 || (weighted && nin == 1)) return pack8(acc);
            return first;
        };
        // (without stores the sums still have to be formed: they are stored under a condition that never holds)
        if (live0) {
            u32x4 res = reduce(p0a, p1a, d0);
            if (MODE == EP_COMBINE_FUSED) res = add_loaded_biases(has0, p0a, has1, p1a, res);
            if (STORES || ((res.x ^ res.y ^ res.z ^ res.w) == 0x9E3779B1u && a.num_in_rows < 0)) stream_store<EP_COMBINE_ST_POL>(out + v0, res);
        }
        if (live1) {
            u32x4 res = reduce(p0b, p1b, d1);
            if (MODE == EP_COMBINE_FUSED) res = add_loaded_biases(has0, p0b, has1, p1b, res);
            if (STORES || ((res.x ^ res.y ^ res.z ^ res.w) == 0x9E3779B1u && a.num_in_rows < 0)) stream_store<EP_COMBINE_ST_POL>(out + v1, res);
        }
        continue;
    }
    float acc0[8], acc1[8];
    u32x4 res0 = zero, res1 = zero;
    int nin = 0;                                              // inputs accumulated so far
    u32x4 p0a = zero, p0b = zero, p1a = zero, p1b = zero;     // single partition: biases fetched ahead of the rows
    if (MODE == EP_COMBINE_FUSED) {
        if (has0) {
            const u32x4* bp = (const u32x4*)a.bias_0 + (int64_t)t * nvec;
            if (live0) p0a = __builtin_nontemporal_load(bp + v0);
            if (live1) p0b = __builtin_nontemporal_load(bp + v1);
        }
        if (has1) {
            const u32x4* bp = (const u32x4*)a.bias_1 + (int64_t)t * nvec;
            if (live0) p1a = __builtin_nontemporal_load(bp + v0);
            if (live1) p1b = __builtin_nontemporal_load(bp + v1);
        }
    }
    if (MODE == EP_COMBINE_FINAL) {
        const void* biases[2] = {a.bias_0, a.bias_1};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if (biases[b] == nullptr) continue;
            const u32x4* bp = (const u32x4*)biases[b] + (int64_t)t * nvec;
            u32x4 e0 = zero, e1 = zero;
            if (live0) e0 = __builtin_nontemporal_load(bp + v0);
            if (live1) e1 = __builtin_nontemporal_load(bp + v1);
            float g0[8], g1[8];
            unpack8(e0, g0);
            unpack8(e1, g1);
            if (nin == 0) { for (int q = 0; q < 8; ++q) { acc0[q] = g0[q]; acc1[q] = g1[q]; } res0 = e0; res1 = e1; }
            else { for (int q = 0; q < 8; ++q) { acc0[q] = acc0[q] + g0[q]; acc1[q] = acc1[q] + g1[q]; } }
            ++nin;
        }
    }
    for (int j = 0; j < K; ++j) {
        const int s = readlane(myslot, j);
        if (s < 0) continue;
        u32x4 e0 = zero, e1 = zero;
        if (live0) e0 = __builtin_nontemporal_load(y + (int64_t)s * yvec + v0);
        if (live1) e1 = __builtin_nontemporal_load(y + (int64_t)s * yvec + v1);
        float g0[8], g1[8];
        unpack8(e0, g0);
        unpack8(e1, g1);
        if (weighted) {
            const float wj = __int_as_float(readlane(__float_as_int(myw), j));
            for (int q = 0; q < 8; ++q) { g0[q] = g0[q] * wj; g1[q] = g1[q] * wj; }
        }
        if (nin == 0) { for (int q = 0; q < 8; ++q) { acc0[q] = g0[q]; acc1[q] = g1[q]; } res0 = e0; res1 = e1; }
        else { for (int q = 0; q < 8; ++q) { acc0[q] = acc0[q] + g0[q]; acc1[q] = acc1[q] + g1[q]; } }
        ++nin;
    }
    // zero inputs -> zeros, one input -> verbatim copy, more -> one rounding of the fp32 sum
    if (nin >= 2 || (weighted && nvalid == 1)) {
        res0 = pack8(acc0);
        res1 = pack8(acc1);
    }
    if (live0) {
        if (MODE == EP_COMBINE_FUSED) res0 = add_loaded_biases(has0, p0a, has1, p1a, res0);
        stream_store<EP_COMBINE_ST_POL>(out + v0, res0);
    }
    if (live1) {
        if (MODE == EP_COMBINE_FUSED) res1 = add_loaded_biases(has0, p0b, has1, p1b, res1);
        stream_store<EP_COMBINE_ST_POL>(out + v1, res1);
    }
    }
}

// Unrolled for top-2 to top-8, and one for any top-k; which of the two a launch takes is the host's rule.  (Odd top-k, all rows in one trip
// instead of one trip a row: 61 tokens x 5120, flushed, top-3 / 5 / 7 8.0 / 9.2 / 10.7 -> 7.3 / 7.6 / 8.2 us; both reduces of eight partitions
// of 64 tokens x 7168, top-3 / 5 / 7 81.8 / 104 / 125 -> 70.7 / 75.8 / 85.8.)
#define EP_COMBINE_KERNEL(NAME, KT, MODE) \
    extern "C" __global__ __launch_bounds__(EP_ROW_THREADS) void ep_combine##NAME(EpCombineArgs a) { fetch_arguments<EpCombineArgs>(); combine_body<KT, MODE>(a); }
#define EP_COMBINE_KERNELS(SUFFIX, MODE)           \
    EP_COMBINE_KERNEL(SUFFIX##_generic, 0, MODE)   \
    EP_COMBINE_KERNEL(SUFFIX##_k2, 2, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k3, 3, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k4, 4, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k5, 5, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k6, 6, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k7, 7, MODE)        \
    EP_COMBINE_KERNEL(SUFFIX##_k8, 8, MODE)

EP_COMBINE_KERNELS(, EP_COMBINE_FUSED)
EP_COMBINE_KERNELS(_partial, EP_COMBINE_PARTIAL)
EP_COMBINE_KERNELS(_final, EP_COMBINE_FINAL)

// ------------------------------------------------------------------------------------------------
// Self-test: hardware e4m3fn conversion against the integer conversion over a range of fp32 bit
// patterns.  out[0] = number of mismatches, out[1] = first mismatching pattern (if any).
// ------------------------------------------------------------------------------------------------
extern "C" __global__ __launch_bounds__(256) void ep_fp8_selftest(EpFp8TestArgs a) {
    unsigned long long bad = 0, firstbad = ~0ull;
    for (unsigned long long k = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; k < a.count;
         k += (unsigned long long)gridDim.x * blockDim.x) {
        const unsigned bits = (unsigned)(a.first + k);
        const float f = __uint_as_float(bits);
        if (!(fabsf(f) <= a.limit)) continue;
        const unsigned hw = (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(f, 0.0f, 0, false) & 0xffu;
        const unsigned sw = ep_f32_bits_to_e4m3fn(bits);
        if (hw != sw) {
            ++bad;
            if (firstbad == ~0ull) firstbad = bits;
        }
    }
    if (bad != 0) {
        atomicAdd(&a.out[0], bad);
        atomicMin(&a.out[1], firstbad);
    }
}
