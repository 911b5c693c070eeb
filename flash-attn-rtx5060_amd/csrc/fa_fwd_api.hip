// C ABI of the gfx950 FlashAttention forward library (see include/fa_fwd.h).
//
// Role of the reference's launcher run_flash_attention / run_kernel<>
// (reference src/flash_forward.h:369-665): argument checking, derived
// parameters, kernel selection and launch.  Unlike the reference it never
// exits, aborts or throws, launches asynchronously on the caller's stream,
// keeps no global descriptor state, and does not time or print.
#include <hip/hip_runtime.h>
#include <dlfcn.h>
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "fa_fwd.h"
#include "fa_bwd.h"
#include "fa_bwd_args.h"
#include "fa_bwd_layout.h"
#include "fa_device_state.h"
#include "fa_kernel_args.h"
#include "fa_sched.h"

hipError_t fa_launch_forward_contiguous(const FaKernelArgs &a, int bf16, int D, int masked, int shape, unsigned grid,
                                        hipStream_t stream);
hipError_t fa_launch_forward_strided(const FaKernelArgs &a, int bf16, int D, int masked, int shape, unsigned grid,
                                     hipStream_t stream);
hipError_t fa_launch_forward_general(const FaKernelArgs &a, int bf16, int D, int masked, int shape, unsigned grid,
                                     hipStream_t stream);
hipError_t fa_launch_forward_dropout(const FaKernelArgs &a, int bf16, int D, int masked, int shape, unsigned grid,
                                     hipStream_t stream);
hipError_t fa_launch_forward_dropout_regular(const FaKernelArgs &a, int bf16, int D, int masked, int shape, unsigned grid,
                                             hipStream_t stream);
hipError_t fa_launch_forward_decode(const FaKernelArgs &a, int bf16, int D, int rows, int streaming, hipStream_t stream,
                                    bool configure_only = false);
hipError_t fa_configure_forward_decode();
hipError_t fa_launch_forward_small(const FaKernelArgs &a, int bf16, int D, int waves, hipStream_t stream, bool configure_only = false);
hipError_t fa_configure_forward_small();
hipError_t fa_launch_combine_splits(const FaKernelArgs &a, int bf16, int D, hipStream_t stream);
hipError_t fa_launch_backward(const FaBwdArgs &a, int bf16, int D, int masked, int general, int alibi, int compute_units,
                              hipStream_t stream, bool configure_only = false);
hipError_t fa_launch_backward_dropout(const FaBwdArgs &a, int bf16, int D, int alibi, int compute_units, hipStream_t stream,
                                      bool configure_only = false);
hipError_t fa_launch_backward_strided(const FaBwdArgs &a, int bf16, int D, int masked, int compute_units, hipStream_t stream,
                                      bool configure_only = false);
// the LDS opt-in (hipFuncSetAttribute) of every kernel instantiation of a translation unit, for the current device
hipError_t fa_configure_forward_contiguous();
hipError_t fa_configure_forward_strided();
hipError_t fa_configure_forward_general();
hipError_t fa_configure_forward_dropout();
hipError_t fa_configure_forward_dropout_regular();
hipError_t fa_configure_backward();
hipError_t fa_configure_backward_dropout();
hipError_t fa_launch_backward_dropout_regular(const FaBwdArgs &a, int bf16, int D, int masked, int strided, int compute_units,
                                              hipStream_t stream, bool configure_only = false);
hipError_t fa_configure_backward_dropout_regular();
hipError_t fa_launch_backward_alibi_regular(const FaBwdArgs &a, int bf16, int D, int masked, int strided, int compute_units,
                                            hipStream_t stream, bool configure_only = false);
hipError_t fa_configure_backward_alibi_regular();
hipError_t fa_configure_backward_strided();

namespace {
constexpr int kBlockKeysHost = 64;
// MI355X; the persistent grid, and which problems are small, go by the device at run time.  (Split counts are chosen without a device, for
// this many: on one with fewer, a chunk that is left whole for the kernel of 32-row blocks may be the tile kernels'.)
constexpr int kComputeUnits = 256;

// Workgroup shape for a problem.  The 8-wave kernel (256 query rows, one workgroup per CU) shares every K/V
// tile among more rows; the 4-wave kernel (128 rows, two workgroups per CU, each with its own barrier, so that the
// two waves of a SIMD are never lined up by one) has twice as many, smaller work items.  It wins when there are
// too few of the large items to fill and balance the chip, and when the items are short, i.e. when no query sees
// more than 1024 keys (at head dimension 64, where a tile carries half the matrix work per barrier, 4096 under a
// mask and 2048 without one): short sequences, and windows on long ones.  Measured, causal fp16, 4 waves against 8, TFLOP/s in one process: B8 H32
// S1024 D64 504 against 432, B8 H16 S1024 D64 443 against 391, B16 H16 S512 D64 275 against 252, B8 H32 S1024 D128 653
// against 590, B16 H16 S512 D128 369 against 340, c2 (B4 H16 S2048 D64) 568-580 against 541-563, B4 H32 S2048 D64 638
// against 626; windows: 512 keys at B1 H32 S16384 D128 604 against 546, 1024 keys at B2 H32 S8192 D64 618 against 578,
// 256 keys at B4 H32 S2048 D64 275 against 241; without a mask B8 H32 S1024 D64 734 against 718; and the other way
// round a window of 2048 keys at B1 H32 S16384 D128 867 against 899, B2 H32 S4096 D128 907 against 958, B1 H32 S8192
// D64 796 against 818, c3 973-1002 against 1029-1051; level: c4 (window 1024, D128, which stays with 8 waves) 780
// against 782.  Head dimension 64 at 4096 keys: causal B2 H32 751 against 744, B8 H32 774 against 748, B1 H16 455
// against 443, windows of 3000 and 4096 keys at B2 H32 S8192 728 against 688 and 736 against 683; without a mask B2 H32
// S4096 868 against 888.
// (`keys`: the largest number of keys a query can see, the key length without a mask)
int waves_for(int B, int N, int S, int d, long long keys, bool masked)
{
    if (S < 256) return 4;              // (few queries per head, e.g. decoding: a 256-row block would be mostly empty)
    if (keys <= (d == 64 ? (masked ? 4096 : 2048) : 1024)) return 4;
    const long long big_items = (long long)B * N * ((S + 255) / 256);
    return big_items >= 2LL * kComputeUnits ? 8 : 4;
}
// the same from the mask as the boundary states it
int waves_for_mask(int B, int N, int S, int S_kv, int d, int is_causal, int window_left, int window_right)
{
    const int sk = S_kv > 0 ? S_kv : S, s_max = sk > S ? sk : S;
    int L, R;
    fa_mask_bounds(s_max, is_causal, window_left, window_right, &L, &R);
    const long long keys = (long long)L + R + 1;
    return waves_for(B, N, S, d, keys < sk ? keys : sk, L < s_max || R < s_max);
}
int waves_of(const fa_fwd_params *p)
{
    return waves_for_mask(p->B, p->N, p->S, p->S_kv, p->d, p->is_causal, p->window_size_left, p->window_size_right);
}

thread_local char g_last_error[256] = "";

std::atomic<unsigned> g_capture_ticket[kFaMaxDevices], g_merge_ticket[kFaMaxDevices];     // captured launches with counters so far, per device
// Eager launches: which stream owns which counter set of a device.  A stream is named by its handle AND the id
// the runtime gave it at creation (hipStreamGetId): a handle value can come back for a new stream after the old
// one was destroyed, while the old stream's last launch may still be running on its counters; the id never does.
struct SlotOwner {
    uintptr_t handle;           // 0 = free
    unsigned long long id;
};
std::mutex g_slot_mutex;
// hipStreamGetId exists from HIP 7.1 on; a process may have loaded an older runtime (PyTorch wheels bring their
// own), so it is looked up at run time.  Without it a stream is named by its handle alone, and a caller that
// destroys streams has to release their sets first (fa_release_work_queue).
typedef hipError_t (*StreamIdFn)(hipStream_t, unsigned long long *);
bool stream_id(hipStream_t stream, unsigned long long *id)
{
    static const StreamIdFn fn = reinterpret_cast<StreamIdFn>(dlsym(RTLD_DEFAULT, "hipStreamGetId"));
    *id = 0;
    return fn == nullptr || fn(stream, id) == hipSuccess;
}
SlotOwner g_slot_owner[kFaMaxDevices][kFaEagerQueueSlots], g_merge_owner[kFaMaxDevices][kFaEagerMergeSlots];

// A counter set for one FA_SCHED_QUEUE launch, or null when none can be given safely (the caller then walks the
// list with the fixed snake: same results, no counters).  Eager launches: a set belongs to a stream -- launches on
// one stream run one after the other, so they may share it, and every launch leaves it rewound; a device hands out
// sixteen sets, to the first sixteen streams that ask, and a stream keeps its set until fa_release_work_queue or
// fa_reset_work_queues; further streams get none.  hipStreamPerThread gets none either: it is one handle value
// for a different stream in every host thread.  A launch that is being captured into a graph keeps its set for
// every replay of that graph, and a replay may run next to anything: every captured launch gets a set of its own
// from the remaining 240, for good, and when those are used up captured launches get none.  No two launches that
// can run at the same time ever share counters.
// (Likewise the sets of the decoding kernel's merges: 64 for streams, 192 for captured launches; what gets none has its key
// splits merged by a second launch.)  Returns the set's number, or -1.
int counter_set_for_launch(SlotOwner *owners, int eager, int all, std::atomic<unsigned> *captured, hipStream_t stream)
{
    if (stream == hipStreamPerThread) return -1;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const bool capturing = stream != nullptr && stream != hipStreamLegacy && hipStreamIsCapturing(stream, &status) == hipSuccess &&
                           status == hipStreamCaptureStatusActive;
    if (capturing) {
        const unsigned n = captured->load(std::memory_order_relaxed) < (unsigned)(all - eager) ? captured->fetch_add(1u, std::memory_order_relaxed) : ~0u;
        return n < (unsigned)(all - eager) ? eager + (int)n : -1;
    }
    // (the two names of the legacy default stream are one stream)
    const bool legacy = stream == nullptr || stream == hipStreamLegacy;
    const uintptr_t handle = legacy ? (uintptr_t)1 : reinterpret_cast<uintptr_t>(stream);
    unsigned long long id = 0;
    if (!legacy && !stream_id(stream, &id)) return -1;
    std::lock_guard<std::mutex> lock(g_slot_mutex);
    int free_slot = -1;
    for (int i = 0; i < eager; ++i) {
        if (owners[i].handle == handle && owners[i].id == id) return i;
        if (owners[i].handle == 0 && free_slot < 0) free_slot = i;
    }
    if (free_slot >= 0) owners[free_slot] = SlotOwner{handle, id};
    return free_slot;
}
unsigned *work_queue_for_launch(const FaDeviceState *ds, hipStream_t stream)
{
    const int dev = fa_launch_device(), set = counter_set_for_launch(g_slot_owner[dev], kFaEagerQueueSlots, kFaQueueSlots, &g_capture_ticket[dev], stream);
    return set < 0 ? nullptr : ds->queues + 16u * (unsigned)set;
}
unsigned *merge_counters_for_launch(const FaDeviceState *ds, hipStream_t stream)
{
    const int dev = fa_launch_device(), set = counter_set_for_launch(g_merge_owner[dev], kFaEagerMergeSlots, kFaMergeSlots, &g_merge_ticket[dev], stream);
    return set < 0 ? nullptr : ds->merges + (size_t)(kFaMergeHeads * kFaMergeStride) * (unsigned)set;
}
// Whether the decoding kernel merges a call's key splits itself: a counter per K/V head, at most the 32 KB of parts a head
// that one workgroup's threads load at once, eight of 16 bytes each, and one pass of its 256 threads, four elements of the head's rows
// each.  So the device is level or faster too, and the launch that goes is 1.5 to 2.5 us of a short call's host time; a second pass
// costs the device more than the second launch.  Graphs, second launch / inside, us (a library's place in memory alone moves
// them by 1.5 %): 8 K/V heads, 4 rows, D128, S_kv 1003 8.39 / 7.88; 64 heads, 1 row, S_kv 1000 10.08 / 9.38; 2 heads, 8 rows, D64,
// S_kv 3000 8.25 / 7.87; the least work, one row of one head, D64, S_kv 2000, 7.95 / 8.14 (called one by one 12.1 / 7.9).  Two passes: 1
// head, 16 rows, D128, S_kv 900 9.20 / 10.05, 32 rows, D64, S_kv 1000 9.60 / 10.39; four: 32 rows, D128, S_kv 500 11.25 / 14.22.  128 KB
// of parts: B4 H32/8 S8 S_kv 2000 13.4 / 16.3.  Calls that read more than 64 MB of K and V, 10 us, hide a launch's host time and
// keep the second one: B16 H32/8 S_kv 8192 (537 MB) 82.6, inside 83.1.
bool merge_inside(long long kv_heads, long long rows, long long keys, int d, int splits)
{
    return kv_heads <= kFaMergeHeads && rows * d <= 4 * 256 && (double)kv_heads * (double)keys * d * 4.0 <= 64e6 && rows * d * 4 * splits <= 32 << 10;
}

int device_fail(hipError_t e, const char *what)
{
    snprintf(g_last_error, sizeof(g_last_error), "%s: %s", what, hipGetErrorString(e));
    return FA_ERR_DEVICE;
}
}  // namespace

extern "C" {

const char *fa_strerror(int status)
{
    switch (status) {
    case FA_OK: return "ok";
    case FA_ERR_NULL_POINTER: return "Q, K, V or O is NULL";
    case FA_ERR_BAD_SHAPE: return "batch, heads and seqlen must be positive";
    case FA_ERR_HEAD_DIM: return "head_dim must be 64 or 128";
    case FA_ERR_SEQLEN_MULTIPLE: return "reserved (seqlen no longer has to be a multiple of 128)";
    case FA_ERR_WORKSPACE: return "needs a 16-byte aligned workspace of fa_fwd_workspace_bytes() (split_num > 1) or fa_bwd_workspace_bytes() bytes";
    case FA_ERR_LAYOUT: return "strides must be multiples of 8 elements (row strides at least head_dim), n_kv_heads must divide heads, pointers must be 16-byte aligned";
    case FA_ERR_UNSUPPORTED: return "dropout_prob must be at least 0 and below 1";
    case FA_ERR_DTYPE: return "dtype must be FA_DTYPE_F16 or FA_DTYPE_BF16";
    case FA_ERR_SCALE: return "softmax_scale must be finite and positive";
    case FA_ERR_DEVICE: return "HIP runtime error";
    case FA_ERR_NO_DEVICE: return "no gfx950 device visible";
    case FA_ERR_TOO_LARGE: return "problem too large for the kernel's index range";
    case FA_ERR_SCRATCH_LIMIT: return "the partial results of this call exceed the library's static scratch (fa_fwd_static_scratch_bytes): use fewer splits or fa_fwd with a workspace";
    default: return "unknown status";
    }
}

const char *fa_last_device_error(void) { return g_last_error; }

int fa_sched_block_rows(int B, int N, int S, int d, int is_causal, int window_left, int window_right)
{
    return 32 * waves_for_mask(B, N, S, S, d, is_causal, window_left, window_right);
}
int fa_sched_block_keys(int d) { (void)d; return kBlockKeysHost; }

long long fa_sched_num_items(int B, int N, int S, int d, int is_causal, int window_left, int window_right)
{
    const int br = fa_sched_block_rows(B, N, S, d, is_causal, window_left, window_right);
    return (long long)B * N * ((S + br - 1) / br);
}

int fa_sched_item(int B, int N, int S, int d, int is_causal, int window_left, int window_right,
                  long long item, int *bh, int *q_begin)
{
    if (B <= 0 || N <= 0 || S <= 0 || !bh || !q_begin) return FA_ERR_BAD_SHAPE;
    const int br = fa_sched_block_rows(B, N, S, d, is_causal, window_left, window_right);
    const int nqb = (S + br - 1) / br;
    if (item < 0 || item >= (long long)B * N * nqb) return FA_ERR_BAD_SHAPE;
    int L, R, qb;
    fa_mask_bounds(S, is_causal, window_left, window_right, &L, &R);
    fa_item_decode(item, B * N, nqb, (L < S || R < S) ? 1 : 0, bh, &qb);
    *q_begin = qb * br;
    return FA_OK;
}

int fa_sched_heads(int N, int n_kv_heads, int bh, int *batch, int *q_head, int *kv_head)
{
    const int hk = n_kv_heads > 0 ? n_kv_heads : N;
    if (N <= 0 || hk > N || N % hk != 0 || bh < 0 || !batch || !q_head || !kv_head) return FA_ERR_BAD_SHAPE;
    *batch = fa_strided_heads(bh, N, hk, q_head, kv_head);
    return FA_OK;
}

void fa_sched_tile_range(int S, int block_keys, int is_causal, int window_left, int window_right,
                         int q_begin, int rows, int *tile_lo, int *tile_hi)
{
    int L, R;
    fa_mask_bounds(S, is_causal, window_left, window_right, &L, &R);
    fa_tile_range(S, block_keys, L, R, q_begin, rows, tile_lo, tile_hi);
}

int fa_sched_classify(int block_keys, int is_causal, int window_left, int window_right,
                      int q_begin, int rows, int tile)
{
    // "unbounded" only has to exceed every reachable |i-j|
    const int big = 0x3fffffff;
    int L = window_left < 0 ? big : window_left;
    int R = window_right < 0 ? big : window_right;
    if (is_causal) R = 0;
    return fa_tile_class(block_keys, L, R, q_begin, rows, tile);
}

long long fa_count_pairs(int S, int is_causal, int window_left, int window_right)
{
    int L, R;
    fa_mask_bounds(S, is_causal, window_left, window_right, &L, &R);
    long long pairs = 0;
    for (int i = 0; i < S; ++i) {
        int lo = i - L < 0 ? 0 : i - L;
        int hi = i + R > S - 1 ? S - 1 : i + R;
        pairs += hi - lo + 1;
    }
    return pairs;
}

double fa_algorithmic_flops(int B, int N, int S, int d, int is_causal, int window_left, int window_right)
{
    return 4.0 * (double)B * (double)N * (double)d * (double)fa_count_pairs(S, is_causal, window_left, window_right);
}

int fa_dropout_threshold(float dropout_prob)
{
    if (!(dropout_prob > 0.0f)) return 0;
    const long t = lrintf(dropout_prob * 256.0f);
    return t > 255 ? 255 : (int)t;
}

int fa_dropout_keep(unsigned long long seed, long long bh, int i, int j, int threshold)
{
    // One Philox4x32-10 block per (query, 32-key block, (j / 4) % 2): sixteen bytes for sixteen keys.
    uint32_t c0 = (uint32_t)(2 * (j >> 5) + ((j >> 2) & 1)), c1 = (uint32_t)i, c2 = (uint32_t)bh, c3 = 0x44524F50u;
    uint32_t k0 = (uint32_t)(seed & 0xffffffffull), k1 = (uint32_t)(seed >> 32);
    for (int round = 0; round < 10; ++round) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1; c3 = (uint32_t)p0; c0 = n0; c2 = n2;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    const uint32_t w[4] = {c0, c1, c2, c3};
    const int r = 4 * ((j & 31) >> 3) + (j & 3);
    return (int)((w[r >> 2] >> (8 * (r & 3))) & 255u) >= threshold;
}

namespace {
int key_tiles(const fa_fwd_params *p) { return ((p->S_kv > 0 ? p->S_kv : p->S) + kBlockKeysHost - 1) / kBlockKeysHost; }
// splits actually used: at most one per key tile
// Query heads per K/V head packed into the rows of one work item (1 = not packed): when there are few
// queries behind long keys (decoding), all query heads of a K/V head fit one 128-row workgroup and K and V
// are then read once per group instead of once per query head.
int packed_group(const fa_fwd_params *p)
{
    const int hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N;
    if (hk <= 0 || hk >= p->N || p->N % hk != 0) return 1;
    const int group = p->N / hk, sk = p->S_kv > 0 ? p->S_kv : p->S;
    if (sk <= p->S) return 1;                                  // queries must sit behind earlier keys
    if ((long long)group * p->S > 32LL * waves_of(p)) return 1;
    return group;
}
// work items before key splits
long long base_items(const fa_fwd_params *p)
{
    const int pack = packed_group(p);
    if (pack > 1) return (long long)p->B * (p->N / pack);
    return fa_sched_num_items(p->B, p->N, p->S, p->d, p->is_causal, p->window_size_left, p->window_size_right);
}
// Key tiles that a work item visits at most: those of the keys from its first row's left bound to its last row's right one
int block_tiles(const fa_fwd_params *p)
{
    const long long sk = p->S_kv > 0 ? p->S_kv : p->S;
    const int s_max = sk > p->S ? (int)sk : p->S, block_rows = 32 * waves_of(p), rows = p->S < block_rows ? p->S : block_rows;
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    const long long keys = (long long)L + rows + R, tiles = (keys + kBlockKeysHost - 2) / kBlockKeysHost + 1;
    return tiles < key_tiles(p) ? (int)tiles : key_tiles(p);
}
int effective_splits(const fa_fwd_params *p)
{
    if (p->split_num <= 1) return 1;
    const int tiles = key_tiles(p);
    return p->split_num < tiles ? p->split_num : tiles;
}
// Whether the decoding kernel (fa_fwd_decode.hip) takes the problem: every query row of a K/V head fits its 32.
// (Rows that the default forward computes in the verifier's arithmetic, and dropout, belong to the tile kernels.  So do
// 2^24 and more K/V heads times `splits`: a workgroup each, of 256 threads, and a launch has fewer than 2^32 of them.)
constexpr long long kDecodeMostGroups = (1LL << 24) - 1;
bool decode_problem(const fa_fwd_params *p, bool causal_type, int splits)
{
    const int hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N, sk = p->S_kv > 0 ? p->S_kv : p->S;
    if ((long long)p->B * hk * splits > kDecodeMostGroups) return false;
    if ((long long)(p->N / hk) * p->S > 32 || sk < p->S || fa_dropout_threshold(p->dropout_prob) != 0) return false;
    if (causal_type && sk - p->S < 32 && packed_group(p) == 1 && !p->exact_first_rows) return false;
    // The decoding kernel's set-up and its merge of four waves' 32 rows at head dimension 128 cost as much as three key tiles:
    // up to there, with four workgroups and more per compute unit and no mask or a group's rows packed into one block, the
    // tile kernels are the faster ones.  bf16, decoding against tile kernel, us: B64 H16 S32 S_kv 64 17.9 / 12.8, S_kv 128
    // 22.3 / 17.3, S_kv 192 25.8 / 22.1; B256 H16 S17 S_kv 64 53.6 / 37.7, S24 S_kv 128 72.0 / 62.6, S32 S_kv 64 ALiBi 64 / 42; B512
    // H16 S32 S_kv 64 111 / 89, S_kv 96 123 / 130; B1024 H16/2 S4 S_kv 128 causal 42.8 / 35.2; and beyond: B48 H16 S32 S_kv 96
    // 16.9 / 17.7, B256 H16 S32 S_kv 200 101 / 104, S16 S_kv 100 42.4 / 63.7, S32 S_kv 100 D64 34.7 / 50.1, S_kv 128 causal 77 / 142.
    if (p->d == 128 && (long long)(p->N / hk) * p->S > 16 && sk <= 192 && (long long)p->B * hk >= 4 * kComputeUnits) {
        int L, R;
        fa_mask_bounds(sk, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
        if ((L >= sk && R >= sk) || packed_group(p) > 1) return false;
    }
    return true;
}
// Workgroups of the tile kernels that a device keeps resident
long long resident_groups(int compute_units, int waves) { return (long long)compute_units * (waves == 8 ? 1 : 2); }
// Rows in the verifier's arithmetic in workgroups of their own (FaKernelArgs.first_parts), in launches of one workgroup per item:
// whether the launch has such rows in items that could leave them, and into how many parts per head they go, 0 to leave them in
// the items.  Behind a tile loop the path is a chain of latencies, 4 us for eight rows and 8 to 15 for 32, which short items
// cannot hide; beside the items it costs slots.  As many parts as fit next to the items into the slots that a device has at a
// time, times two (head dimension 64, where the path is shorter: times 7/4), since the first blocks of a head are short
// themselves.  Causal, us, in the items / apart: B1 H4 S256 D64 14.1 / 8.7, B4 H32 S128 D128 bf16 30.3 / 16.4, B5 H16 S284 D128
// 23.2 / 14.4, B1 H32 S512 D128 20.3 / 15.2, B1 H384 S128 D64 19.4 / 17.7, B1 H256 S256 D128 31.4 / 29.2; further parts, H512 S100
// D64 21.6 / 21.9, H128 S500 D64 22.1 / 22.5, and at four times the slots H200 S256 D64 15.9 (two) / 21.6.
bool first_rows_few_keys(const fa_fwd_params *p, int R)
{
    const int pos_off = (p->S_kv > 0 ? p->S_kv : p->S) - p->S;
    return R == 0 && pos_off >= 0 && pos_off < 32 && packed_group(p) == 1 && !p->exact_first_rows;
}
int first_rows_parts(long long items, long long heads, int d, long long resident)
{
    int parts = 8;
    while (parts > 0 && items + parts * heads > (d == 128 ? 8 : 7) * resident / 4) parts /= 2;
    return parts;
}
// How a call reaches the device: by the decoding kernel, whose workgroups (one per K/V head and key split) the hardware
// hands out, with the streaming hint or without; by the kernel of 32-row blocks, which it hands out too, with small_waves waves each
// (0: not by it) and small_parts for FaKernelArgs.first_parts; else the schedule of the tile kernels' work items and theirs.
struct Launch {
    bool decode, streaming;
    int small_waves, small_parts;
    int sched, first_parts;
};
// The kernel of 32-row blocks whose waves share the keys (fa_fwd_small.hip).  The key tiles, in its own units, that a block visits
// at most; whether a problem is small enough for it, and with how many waves.
int small_tiles(const fa_fwd_params *p)
{
    const long long sk = p->S_kv > 0 ? p->S_kv : p->S, keys_per_tile = p->d == 64 ? 64 : 32;
    const int s_max = sk > p->S ? (int)sk : p->S;
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    const long long seen = ((long long)L + 32 + R + keys_per_tile - 2) / keys_per_tile + 1, all = (sk + keys_per_tile - 1) / keys_per_tile;
    return (int)(seen < all ? seen : all);
}
// At most the workgroups that a device holds at a time, two per compute unit; twice as many where a causal walk of at least
// 2048 queries makes the tile kernels wait for their longest blocks.  GPU time, tile kernels / this, us: no mask H16 S1024 D64 (512
// workgroups) 14.2 / 10.5, H8 S2048 D128 (512) 34.1 / 27.9, H64 S256 D128 (512) 9.5 / 9.4, H32 S1024 D64 (1024) 15.4 / 18.9; causal
// H8 S4096 D128 (1024) 68.6 / 56.1, H16 S2048 D64 (1024) 26.9 / 22.0, H32 S1024 D64 (1024) 16.9 / 17.3, H16 S4096 D128 (2048) 101 /
// 107.  With more than a workgroup per unit the tile kernels keep what they do in one or two tiles at full width: 128 queries on as many
// keys, no mask H72 to H128 D64 5.5 to 5.7 / 5.7 to 5.9, D128 7.2 to 7.5 / 7.7 to 8.1, causal H96 7.4 / 7.8 and 9.8 / 10.2; 64 keys that are a
// whole tile without a mask, D128 H130 S64 6.4 / 7.1, H256 6.7 / 7.7, H110 S96 6.6 / 7.4, H33 S320 6.8 / 7.4, D64 H165 S40 4.9 / 5.4, H256 S64
// 5.2 / 5.6, H170 S96 5.5 / 5.6, but H82 S100 5.4 / 5.35, H66 S160 5.6 / 5.4; with a mask 40 to the left D128 H165 S64 7.8 / 7.5, with 48 keys
// 7.8 / 7.5, with 100 9.2 / 8.0, with 128 7.8 / 7.7.
// First rows go in four parts of eight, a row to each half-wave: in eight parts half of their waves have none, and beside short blocks the
// workgroups that do not fit any more are what the call waits for (tile kernels / eight / four parts: bf16 H56 S64 D64 6.2 / 8.0 / 5.6, H52
// S97 D128 10.0 / 11.8 / 8.2, H40 S256 D64 9.1 / 9.5 / 6.7, fp16 H64 S169 D64 9.0 / 8.5 / 7.8, H16 S1024 D128 22.3 / 16.6 / 16.6).  Where a quarter
// of the slots more does not hold them (head dimension 128: eight of them per head, or all at once), the tile kernels are level: H64
// S256 D128 11.0 / 11.2.  Their bf16 products take longer: two 128-row blocks at head dimension 64 whose first rows do not fit
// beside them stay too, H60 S192 8.6 / 9.4, H64 S148 8.5 / 9.1.  (1900 random causal problems, us: none slower than the tile
// kernels by more than 1 %, 1.40 times as fast on average.)  Eight waves: no mask H4 S2048 D64 12.7 (four) / 11.1, D128 22.0 / 17.3, H8 S1024 D64 8.1 / 7.9,
// causal 8.4 / 9.4.
int small_waves_for(const fa_fwd_params *p, int compute_units, int *first_parts)
{
    const int sk = p->S_kv > 0 ? p->S_kv : p->S, s_max = sk > p->S ? sk : p->S;
    const long long heads = (long long)p->B * p->N, items = heads * ((p->S + 31) / 32), slots = 2LL * compute_units;
    *first_parts = 0;
    if (effective_splits(p) != 1 || fa_dropout_threshold(p->dropout_prob) != 0) return 0;
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    const bool uneven = R == 0 && L >= s_max && sk == p->S && p->S >= 2048;
    const bool one_whole_tile = sk == kBlockKeysHost && L >= s_max && R >= s_max && (p->d == 128 || p->S <= 96);
    if (items > (uneven ? 2 : 1) * slots || (items > compute_units && ((sk <= 128 && p->S % 128 == 0) || one_whole_tile))) return 0;
    if (first_rows_few_keys(p, R)) {              // (in workgroups of their own, or the problem stays with the tile kernels)
        const int rows = 32 - (sk - p->S) < p->S ? 32 - (sk - p->S) : p->S;
        const long long most = (uneven ? 2 : 1) * slots + slots / 4;
        if (p->d == 64 ? items + 4 * heads > most : items + 8 * heads > most && items + 4 * heads > slots) return 0;
        const bool beside = items + heads * ((rows + 7) / 8) <= slots;
        if (!beside && p->d == 64 && p->dtype == FA_DTYPE_BF16 && p->S > 128 && p->S <= 256) return 0;
        *first_parts = 4;
    }
    return items <= compute_units && small_tiles(p) >= 24 ? 8 : 4;
}
Launch launch_of(const fa_fwd_params *p, int compute_units)
{
    const int sk = p->S_kv > 0 ? p->S_kv : p->S, hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N;
    const int s_max = sk > p->S ? sk : p->S, waves = waves_of(p), pack = packed_group(p);
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    Launch l;
    l.decode = decode_problem(p, R == 0, effective_splits(p));
    l.small_parts = 0;
    l.small_waves = l.decode ? 0 : small_waves_for(p, compute_units, &l.small_parts);      // (whatever the schedule: the same bits)
    // (the streaming hint from where the K and V that are read -- under a left window the last S + L keys -- do not stay in
    // the 256 MB memory-side cache: measured beside the kernel)
    const long long visible = (long long)p->S + L < sk ? (long long)p->S + L : sk;
    l.streaming = l.decode && (double)p->B * hk * (double)visible * p->d * 4.0 > 128e6;
    // FA_SCHED_AUTO: with at most one item per resident workgroup there is nothing to schedule (and the
    // queue's counter round trips, 2.3 us each, would double the run time of a 7 us problem).  With fewer than
    // eight items per workgroup the fixed snake wins: it pairs every long item with a short one, knows its next
    // item without asking, and its items' loads can be requested before the current item's epilogue without a
    // counter in between -- causal fp16 problems, snake against queue: B8 H32 S1024 D64 (four items per workgroup)
    // 67 against 100 us, B4 H32 S2048 D64 (four) 111 against 138, B2 H32 S4096 D128 (four) 290 against 312, c2 (two)
    // 611 against 448 TFLOP/s.  At eight per workgroup the two are level (c3 1016 against 1018 TFLOP/s, B1 H32 S16384
    // 2097 us both); beyond, the queue's balancing is worth more than its counters cost (c5, 32 items per workgroup:
    // 16.2 against 17.0 ms; B8 H32 S8192 D64 2.75 against 2.80 ms).
    l.sched = p->sched;
    // Items that are all alike (no mask, or a window of at most half the length: all but the first few query blocks
    // of a head see the same number of tiles) need no balancing either, and the fixed order saves them the
    // counters' barriers: c4 766 against 748 TFLOP/s, c3's shape without a mask 1101 against 1096.
    const long long blocks = pack > 1 ? 1 : (p->S + 32 * waves - 1) / (32 * waves);
    const long long items = (long long)p->B * p->N / pack * blocks * effective_splits(p), resident = resident_groups(compute_units, waves);
    if (l.sched == FA_SCHED_AUTO) {
        const bool alike = !(L < s_max || R < s_max) || 2LL * L <= (long long)p->S;
        l.sched = items <= resident ? FA_SCHED_DISPATCH : (items < 8 * resident || alike) ? FA_SCHED_PERSISTENT : FA_SCHED_QUEUE;
    }
    const bool apart = l.sched == FA_SCHED_DISPATCH && effective_splits(p) == 1 && first_rows_few_keys(p, R);
    l.first_parts = apart ? first_rows_parts(items, (long long)p->B * p->N, p->d, resident) : 0;
    return l;
}
}  // namespace

int fa_sched_launch(const fa_fwd_params *p, int compute_units, int *decoding, int *streaming)
{
    const int st = fa_fwd_validate(p);
    if (st != FA_OK) return st;
    const Launch l = launch_of(p, compute_units);
    if (decoding) *decoding = l.decode;
    if (streaming) *streaming = l.streaming;
    return l.decode || l.small_waves > 0 ? FA_SCHED_DISPATCH : l.sched;
}

int fa_sched_small(const fa_fwd_params *p, int compute_units, int *first_parts)
{
    const int st = fa_fwd_validate(p);
    if (st != FA_OK) return st;
    const Launch l = launch_of(p, compute_units);
    if (first_parts) *first_parts = l.decode ? 0 : l.small_waves > 0 ? l.small_parts : l.first_parts;
    return l.small_waves;
}

unsigned long long fa_fwd_workspace_bytes(const fa_fwd_params *p)
{
    if (!p || p->B <= 0 || p->N <= 0 || p->S <= 0 || p->d <= 0) return 0;
    const int n = effective_splits(p);
    if (n <= 1) return 0;
    return (unsigned long long)n * p->B * p->N * p->S * (unsigned long long)(p->d + 1) * 4ull;
}

namespace {
// The tile kernels' estimated time of a call with n splits, us: 128-row blocks that visit `tiles` key tiles
double tile_kernels_us(const fa_fwd_params *p, int tiles, long long n, double second_launch_us)
{
    const double tile_us = p->d == 64 ? 0.55 : 0.85, partial = (double)p->B * p->N * p->S * p->d * 8.0 / 5.2e6;
    const long long per_cu = (base_items(p) * n + kComputeUnits - 1) / kComputeUnits;
    const double us = (double)per_cu * ((tiles + n - 1) / n * tile_us + 1.4) * (per_cu == 1 ? 1.4 : 1.0);
    return n > 1 ? us + second_launch_us + partial * (double)n : us;
}
// the count from 1 to `most` with the least of it
int least_time_splits(const fa_fwd_params *p, int tiles, int most, double second_launch_us)
{
    int best = 1;
    double best_us = 0.0;
    for (int n = 1; n == 1 || n <= most; ++n) {
        const double us = tile_kernels_us(p, tiles, n, second_launch_us);
        if (n == 1 || us < best_us) { best = n; best_us = us; }
    }
    return best;
}
// The 32-row kernel's estimated time of a call, us, or -1 where it does not take it: the tiles of its longest block in turns of
// its waves, and what lies beside them, for four waves with one and with two workgroups on a compute unit and for eight (within
// 10 % of 24 calls without a mask of 4 to 64 heads and 256 to 4096 keys).  Causal [B,S,H,D], split tile kernels / this, us: H32 S256
// S_kv 1231 D128 23.0 / 13.2, D64 17.7 / 9.3, H8 S512 S_kv 2000 D128 24.2 / 15.8, H64 S128 S_kv 400 D64 12.9 / 6.0; left where they
// were: H16 S64 S_kv 4000 D128 17.5 / 25.9, H32 S500 S_kv 4596 D128 56 / 58, H4 S100 S_kv 20000 D64 17.2 / 66.
double small_kernel_us(const fa_fwd_params *p)
{
    fa_fwd_params whole = *p;
    whole.split_num = 1;
    int first_parts;
    const int waves = small_waves_for(&whole, kComputeUnits, &first_parts);
    if (waves == 0) return -1.0;
    const double turns = (small_tiles(p) + waves - 1) / waves;
    const bool alone = (long long)p->B * p->N * ((p->S + 31) / 32) <= kComputeUnits;
    if (p->d == 64) return waves == 8 ? 4.7 + 1.6 * turns : alone ? 3.5 + 1.15 * turns : 4.1 + 1.65 * turns;
    return waves == 8 ? 6.0 + 1.4 * turns : alone ? 4.8 + 1.07 * turns : 7.0 + 1.3 * turns;
}
}  // namespace

int fa_fwd_suggest_splits(const fa_fwd_params *p)
{
    if (!p || p->B <= 0 || p->N <= 0 || p->S <= 0) return 1;
    // work items without splits against the workgroups the device keeps resident; split until the device is
    // filled once (the items of such a problem are all alike, so one full round has no tail; measured against
    // filling it twice: 98 against 106 us on B16 H32/8 S1 S_kv8192, 53 against 61 us on B8 H32/8 S4 S_kv8192,
    // 370 against 361 us on B4 H32 S1 S_kv32768), with at least four key tiles (256 keys) per split
    const long long items = base_items(p);
    const long long resident = (long long)kComputeUnits * (waves_of(p) == 8 ? 1 : 2);
    if (items >= resident) return 1;
    long long n = (resident + items - 1) / items;
    if (n > key_tiles(p) / 4) n = key_tiles(p) / 4;
    // A left window leaves a block a few of these tiles, and splits beyond them write empty partial results for the merge
    // to read: no more than one per tile, and the tile kernels of 128-row blocks take the count with the least estimated
    // time (fa_fwd_auto_splits; the second launch costs 3 us here, where the first one is short).
    const int sk = p->S_kv > 0 ? p->S_kv : p->S, s_max = sk > p->S ? sk : p->S, tiles = block_tiles(p);
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    if (n > tiles) n = tiles;
    if (L < s_max && waves_of(p) != 8 && !decode_problem(p, R == 0, 1)) n = least_time_splits(p, tiles, (int)n, 3.0);
    return n < 1 ? 1 : (int)n;
}

int fa_fwd_auto_splits(const fa_fwd_params *p)
{
    if (!p || p->B <= 0 || p->N <= 0 || p->S <= 0 || p->d <= 0) return 1;
    const int hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N, sk = p->S_kv > 0 ? p->S_kv : p->S;
    if (p->N % hk != 0) return 1;
    const int s_max = sk > p->S ? sk : p->S;
    int L, R;
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    if (!decode_problem(p, R == 0, 1)) {
        // The tile kernels, 128-row blocks, queries behind a cache (what else ran is left at the count that fills the device):
        // the least estimated time as well.  Workgroups per compute unit times (key tiles of a split, 0.85 us each at head
        // dimension 128 and 0.55 at 64, + 1.4), 1.4 of that per workgroup where a unit has only one; a second launch costs
        // 4.6 us and the partial results' traffic.  Filling the device once took just over one round to two: 512 slots for
        // 528 items are as slow as 1024.  Causal bf16 [B,S,H,D], items before splits, filled once against this, splits: us --
        // B1 H32/8 S700 S_kv 4700 192 3: 94.9, 4: 82.4; B1 H32 S300 S_kv 4000 D64 96 6: 38.9, 5: 29.1; B3 H8/2 S150 S_kv 10000 48 11:
        // 61.3, 10: 43.9; B4 H32/8 S256 S_kv 2000 256 2: 54.4, 1: 48.9; B4 H16 S600 S_kv 3000 320 2: 94.1, 1: 82.8; B1 H32/8 S500
        // S_kv 4596 128 4: 55.6 both.  Sixty random shapes where the two differ: 0.97 to 1.68 times as fast, 1.21 on average.
        const long long items = base_items(p);
        const int tiles = key_tiles(p);
        if (sk <= p->S || L < s_max || waves_of(p) == 8 || items >= 2 * kComputeUnits) return fa_fwd_suggest_splits(p);
        // (at least three tiles a split, B2 H16/4 S91 S_kv 636 5: 19.1, 2: 18.6; at most four workgroups on every slot)
        const long long slots = 8 * kComputeUnits / items;
        const int n = least_time_splits(p, tiles, (int)(slots < tiles / 3 ? slots : tiles / 3), 4.6);
        // (no split where the kernel of 32-row blocks, whose waves split the keys among them, is estimated to be as fast)
        const double whole = small_kernel_us(p);
        return whole >= 0.0 && whole <= tile_kernels_us(p, tiles, n, 4.6) ? 1 : n;
    }
    // The decoding kernel: the splits with the least estimated time.  The chip's bandwidth is shared by its CUs, so K and V
    // take as long as the CU with the most workgroups: (their bytes at 6.5 TB/s) * ceil(load) / load with load workgroups
    // per CU, 5 % more where a CU has only one (four waves do not keep enough bytes in flight); a second launch costs 4 us
    // and the partial results' traffic, one more trip to memory per 64 splits.  No wave without at least one piece of its own
    // (32 keys at head dimension 128, 64 at 64, four waves per workgroup) among the keys that some query sees.  Both
    // launches of a call, splits (workgroups per CU): us -- B17 H4 S_kv 27819 8 (2.1): 195, 15 (3.98): 149; B14 H32 S_kv
    // 8806 D64 2 (3.5): 169, 4 (7.0): 155; B33 H4 S_kv 10356 4 (2.06): 140, 5 (2.6): 117; B26 H32 S4 S_kv 1616 D64 1 (3.25): 86,
    // 4 (13): 63; B38 H32/4 S_kv 6599 4 (2.4): 94, 5 (2.97): 84.5; B4 H32 S_kv 32768 2 (1): 327, 4 (2): 308; B1 H32/8 S_kv 1003
    // 4: 9.9, 8: 8.3; B10 H16 S_kv 1000 D64 1 (0.6): 12.2, 3 (1.9): 13.8.
    const long long heads = (long long)p->B * hk, visible = (long long)p->S + L < sk ? (long long)p->S + L : sk;
    long long most = visible / (p->d == 64 ? 256 : 128);
    if (most > key_tiles(p)) most = key_tiles(p);
    const long long loaded = (4LL * kComputeUnits + heads - 1) / heads;         // beyond four workgroups per CU: up to eight splits
    if (most > (loaded > 8 ? loaded : 8)) most = loaded > 8 ? loaded : 8;
    if (most * heads > kDecodeMostGroups) most = kDecodeMostGroups / heads;
    const double base = heads * (double)visible * p->d * 4.0 / 6.5e6, partial = (double)p->B * p->N * p->S * p->d * 8.0 / 5e6;
    long long best = 1;
    double best_us = 0.0;
    for (long long n = 1; n <= most || n == 1; ++n) {
        const long long groups = heads * n, per_cu = (groups + kComputeUnits - 1) / kComputeUnits;
        double us = base * (double)(per_cu * kComputeUnits) / (double)groups * (per_cu == 1 ? 1.05 : 1.0);
        if (n > 1) us += 4.0 + partial * (double)n + (double)((n - 1) / 64);
        if (n == 1 || us < best_us) { best = n; best_us = us; }
    }
    return (int)best;
}

namespace {
int validate_layout(const fa_fwd_params *p);
// everything but the workspace of a call with key splits
int validate_no_workspace(const fa_fwd_params *p)
{
    if (!p || !p->Q || !p->K || !p->V || !p->O) return FA_ERR_NULL_POINTER;
    if (p->B <= 0 || p->N <= 0 || p->S <= 0) return FA_ERR_BAD_SHAPE;
    if (p->d != 64 && p->d != 128) return FA_ERR_HEAD_DIM;
    if (p->dtype != FA_DTYPE_F16 && p->dtype != FA_DTYPE_BF16) return FA_ERR_DTYPE;
    if (!(p->dropout_prob >= 0.0f) || !(p->dropout_prob < 1.0f)) return FA_ERR_UNSUPPORTED;
    if (!(p->softmax_scale > 0.0f) || !isfinite(p->softmax_scale)) return FA_ERR_SCALE;
    const long long bh = (long long)p->B * p->N;
    if (bh > 0x7fffffffLL || fa_sched_num_items(p->B, p->N, p->S, p->d, p->is_causal, p->window_size_left, p->window_size_right) > 0x7fffffffLL) return FA_ERR_TOO_LARGE;
    if (p->S_kv < 0) return FA_ERR_BAD_SHAPE;
    if ((long long)p->S + (p->S_kv > 0 ? p->S_kv : p->S) > 0x3fffffffLL) return FA_ERR_TOO_LARGE;   // tile and mask arithmetic is 32-bit
    if (base_items(p) * effective_splits(p) > 0x7fffffffLL) return FA_ERR_TOO_LARGE;
    return validate_layout(p);
}
}  // namespace

int fa_fwd_validate(const fa_fwd_params *p)
{
    const int st = validate_no_workspace(p);
    if (st != FA_OK) return st;
    if (effective_splits(p) > 1 && (p->workspace == nullptr || reinterpret_cast<uintptr_t>(p->workspace) % 16 != 0 ||
                                    p->workspace_bytes < fa_fwd_workspace_bytes(p))) return FA_ERR_WORKSPACE;
    return FA_OK;
}

namespace {
int validate_layout(const fa_fwd_params *p)
{
    if (p->n_kv_heads < 0 || (p->n_kv_heads > 0 && p->N % p->n_kv_heads != 0)) return FA_ERR_LAYOUT;
    const void *ptrs[4] = {p->Q, p->K, p->V, p->O};
    const long long *strides[4] = {p->q_strides, p->k_strides, p->v_strides, p->o_strides};
    for (int t = 0; t < 4; ++t) {
        if (reinterpret_cast<uintptr_t>(ptrs[t]) % 16 != 0) return FA_ERR_LAYOUT;
        const long long *st = strides[t];
        if (st[0] == 0 && st[1] == 0 && st[2] == 0) continue;       // contiguous
        for (int k = 0; k < 3; ++k)
            if (st[k] < 0 || st[k] % 8 != 0) return FA_ERR_LAYOUT;
        if (st[2] < p->d) return FA_ERR_LAYOUT;
        if (st[2] > (1LL << 24)) return FA_ERR_TOO_LARGE;           // per-lane byte offsets inside a tile are 32-bit
        // an output whose batch or head stride is zero would have several writers per element
        if (t == 3 && ((p->B > 1 && st[0] == 0) || (p->N > 1 && st[1] == 0))) return FA_ERR_LAYOUT;
    }
    return FA_OK;
}

// The forward pass with the partial results of key splits in `workspace` (ignored without splits).
int forward(const fa_fwd_params *p, void *workspace, const FaDeviceState *ds, void *stream)
{
    FaKernelArgs a;
    a.Q = static_cast<const uint16_t *>(p->Q);
    a.K = static_cast<const uint16_t *>(p->K);
    a.V = static_cast<const uint16_t *>(p->V);
    a.O = static_cast<uint16_t *>(p->O);
    a.lse = p->L;
    a.alibi = p->alibi_slopes_ptr;
    a.H = p->N;
    a.BH = p->B * p->N;
    a.S = p->S;
    // layout: contiguous [B,N,S,d] unless strides are given; K and V have n_kv_heads heads
    a.Hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N;
    a.Sk = p->S_kv > 0 ? p->S_kv : p->S;
    a.n_splits = effective_splits(p);
    a.o_part = static_cast<float *>(workspace);
    a.lse_part = a.o_part != nullptr ? a.o_part + (size_t)a.n_splits * p->B * p->N * p->S * p->d : nullptr;
    a.pack = packed_group(p);
    bool general = a.pack > 1 || p->S % 128 != 0 || a.Sk != p->S || a.n_splits > 1;
    // the regular problem, not stored contiguous [B,N,S,d], or with K/V heads shared by groups of query heads
    bool strided = a.Hk != p->N;
    {
        const long long *strides[4] = {p->q_strides, p->k_strides, p->v_strides, p->o_strides};
        long long eff[4][3];
        for (int t = 0; t < 4; ++t) {
            const long long heads = (t == 1 || t == 2) ? a.Hk : p->N;
            const long long len = (t == 1 || t == 2) ? a.Sk : p->S;
            const long long dense[3] = {heads * len * p->d, len * p->d, p->d};
            const long long *st = strides[t];
            const bool given = st[0] != 0 || st[1] != 0 || st[2] != 0;
            for (int k = 0; k < 3; ++k) {
                eff[t][k] = given ? st[k] : dense[k];
                if (eff[t][k] != dense[k]) strided = true;
            }
        }
        a.q_bs = eff[0][0]; a.q_hs = eff[0][1]; a.q_rs = (int)eff[0][2];
        a.k_bs = eff[1][0]; a.k_hs = eff[1][1]; a.k_rs = (int)eff[1][2];
        a.v_bs = eff[2][0]; a.v_hs = eff[2][1]; a.v_rs = (int)eff[2][2];
        a.o_bs = eff[3][0]; a.o_hs = eff[3][1]; a.o_rs = (int)eff[3][2];
    }
    const int waves = waves_of(p);
    const int block_rows = 32 * waves;
    a.n_qblocks = a.pack > 1 ? 1 : (p->S + block_rows - 1) / block_rows;
    const int s_max = a.Sk > p->S ? a.Sk : p->S;        // stands in for "unbounded"
    fa_mask_bounds(s_max, p->is_causal, p->window_size_left, p->window_size_right, &a.L, &a.R);
    // (a sequence that ends inside a 64-key tile needs the element mask on that tile, whatever the mask)
    const int masked = (a.L < s_max || a.R < s_max || a.Sk % kBlockKeysHost != 0) ? 1 : 0;
    a.descending = (a.L < s_max || a.R < s_max) ? 1 : 0;
    a.scale = p->softmax_scale;
    a.scale_log2e = p->softmax_scale * 1.44269504088896340736f;
    a.n_items = (long long)(a.BH / a.pack) * a.n_qblocks * a.n_splits;

    a.merge = nullptr;
    const Launch launch = launch_of(p, ds->compute_units);
    auto launch_decode = [&]() {
        a.pack = p->N / a.Hk;
        const long long heads = (long long)p->B * a.Hk;
        a.n_items = heads * a.n_splits;
        a.merge = nullptr;
        if (a.n_splits > 1 && merge_inside(heads, (long long)a.pack * p->S, (long long)p->S + a.L < a.Sk ? (long long)p->S + a.L : a.Sk, p->d, a.n_splits))
            a.merge = merge_counters_for_launch(ds, static_cast<hipStream_t>(stream));
        hipError_t e = fa_launch_forward_decode(a, p->dtype == FA_DTYPE_BF16, p->d, a.pack * p->S, launch.streaming ? 1 : 0, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "decode launch");
        if (a.n_splits > 1 && a.merge == nullptr) {
            e = fa_launch_combine_splits(a, p->dtype == FA_DTYPE_BF16, p->d, static_cast<hipStream_t>(stream));
            if (e != hipSuccess) return device_fail(e, "combine launch");
        }
        return (int)FA_OK;
    };
#ifndef FA_CHECK_RING
    if (launch.decode) return launch_decode();      // (before a work queue is asked for: this kernel uses none)
#endif      // (the checking build runs the tile kernels, whose ring it checks, on these problems as well, in front)
    a.exact_first_rows = p->exact_first_rows != 0;
    auto launch_small = [&]() {
        a.pack = 1;
        a.n_qblocks = (p->S + 31) / 32;
        a.n_items = (long long)a.BH * a.n_qblocks;
        a.first_parts = launch.small_parts;
        const hipError_t e = fa_launch_forward_small(a, p->dtype == FA_DTYPE_BF16, p->d, launch.small_waves, static_cast<hipStream_t>(stream));
        return e != hipSuccess ? device_fail(e, "small launch") : (int)FA_OK;
    };
#ifndef FA_CHECK_RING
    if (launch.small_waves > 0) return launch_small();      // (the checking build: as with the decoding kernel)
#endif
    // Dispatch mode launches one workgroup per item, in list order; the hardware hands them to CUs as these
    // free up, which is a longest-first greedy schedule.  Persistent mode launches one resident set of
    // workgroups that walk the list themselves.
    long long grid = a.n_items;
    a.queue = nullptr;
    if (launch.sched == FA_SCHED_PERSISTENT || launch.sched == FA_SCHED_QUEUE) {
        const long long resident = resident_groups(ds->compute_units, waves);
        if (grid > resident) grid = resident;
        if (launch.sched == FA_SCHED_QUEUE) a.queue = work_queue_for_launch(ds, static_cast<hipStream_t>(stream));
    }
    const int shape = waves == 8 ? 0 : 1;
    // dropout: p in units of 1/256 (a key is kept iff its random byte is >= the threshold)
    a.drop_threshold = (unsigned)fa_dropout_threshold(p->dropout_prob);
    a.drop_scale = 256.0f / (256.0f - (float)a.drop_threshold);
    a.seed_lo = (unsigned)(p->seed & 0xffffffffull);
    a.seed_hi = (unsigned)(p->seed >> 32);
    a.first_parts = launch.first_parts;
#ifdef FA_CHECK_RING
    a.ring_check = ds->ring_check;
#endif
    hipError_t e = (a.drop_threshold != 0 ? (general ? fa_launch_forward_dropout : fa_launch_forward_dropout_regular)
                    : general ? fa_launch_forward_general
                    : strided ? fa_launch_forward_strided : fa_launch_forward_contiguous)(
        a, p->dtype == FA_DTYPE_BF16, p->d, masked, shape, (unsigned)grid, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "forward launch");
    if (a.n_splits > 1) {
        e = fa_launch_combine_splits(a, p->dtype == FA_DTYPE_BF16, p->d, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "combine launch");
    }
#ifdef FA_CHECK_RING
    if (launch.decode) return launch_decode();
    if (launch.small_waves > 0) return launch_small();
#endif
    return FA_OK;
}
}  // namespace

int fa_init(void)
{
    const FaDeviceState *ds = nullptr;
    hipError_t e = fa_device_state(&ds);
    if (e != hipSuccess) return device_fail(e, "device set-up");
    // everything a first launch would otherwise do besides the launch itself: after this call no entry point makes
    // a HIP call on this device that is not a stream operation (which is what a stream capture needs)
    hipError_t (*const configure[])() = {fa_configure_forward_contiguous, fa_configure_forward_strided, fa_configure_forward_general, fa_configure_forward_decode, fa_configure_forward_small,
                                         fa_configure_forward_dropout, fa_configure_forward_dropout_regular, fa_configure_backward, fa_configure_backward_dropout,
                                         fa_configure_backward_strided, fa_configure_backward_dropout_regular, fa_configure_backward_alibi_regular};
    for (auto fn : configure) {
        e = fn();
        if (e != hipSuccess) return device_fail(e, "kernel set-up");
    }
    return FA_OK;
}

int fa_fwd(const fa_fwd_params *p, void *stream)
{
    const int st = fa_fwd_validate(p);
    if (st != FA_OK) return st;
    const FaDeviceState *ds = nullptr;
    const hipError_t e = fa_device_state(&ds);
    if (e != hipSuccess) return device_fail(e, "device set-up");
    return forward(p, p->workspace, ds, stream);
}

unsigned long long fa_fwd_static_scratch_bytes(void) { return kFaStaticScratchBytes; }

int fa_fwd_split_static(const fa_fwd_params *p, void *stream)
{
    const int st = validate_no_workspace(p);
    if (st != FA_OK) return st;
    if (fa_fwd_workspace_bytes(p) > kFaStaticScratchBytes) return FA_ERR_SCRATCH_LIMIT;
    const FaDeviceState *ds = nullptr;
    const hipError_t e = fa_device_state(&ds);      // first call on a device: looks the two arrays up, no allocation
    if (e != hipSuccess) return device_fail(e, "device set-up");
    // the kernels get the array's device address, exactly as they get a caller's workspace in fa_fwd
    return forward(p, ds->scratch, ds, stream);
}

#ifdef FA_CHECK_RING
// Checking build only (libfa_fwd_gfx950_check.so): waits for the device, returns how many 16-byte comparisons the
// forward kernels' ring checks have made and how many of them found other bytes in LDS than the tile the
// iteration expected, and sets both counters back to zero.
int fa_debug_ring_counts(unsigned long long *checks, unsigned long long *violations)
{
    const FaDeviceState *ds = nullptr;
    hipError_t e = fa_device_state(&ds);
    if (e != hipSuccess) return device_fail(e, "device set-up");
    unsigned long long host[2] = {0, 0};
    e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(host, ds->ring_check, sizeof(host), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemset(ds->ring_check, 0, sizeof(host));
    if (e != hipSuccess) return device_fail(e, "ring check counters");
    if (checks) *checks = host[0];
    if (violations) *violations = host[1];
    return FA_OK;
}
#endif

int fa_reset_work_queues(void)
{
    const FaDeviceState *ds = nullptr;
    hipError_t e = fa_device_state(&ds);
    if (e != hipSuccess) return device_fail(e, "device set-up");
    e = hipDeviceSynchronize();
    if (e != hipSuccess) return device_fail(e, "synchronize");
    e = hipMemset(ds->queues, 0, (size_t)kFaQueueSlots * 16 * sizeof(unsigned));
    if (e == hipSuccess) e = hipMemset(ds->merges, 0, sizeof(unsigned) * kFaMergeSlots * kFaMergeHeads * kFaMergeStride);
    if (e != hipSuccess) return device_fail(e, "work queue reset");
    // (nothing is in flight after the synchronisation: streams may claim their sets anew)
    std::lock_guard<std::mutex> lock(g_slot_mutex);
    for (int i = 0; i < kFaEagerQueueSlots; ++i) g_slot_owner[fa_launch_device()][i] = SlotOwner{0, 0};
    for (int i = 0; i < kFaEagerMergeSlots; ++i) g_merge_owner[fa_launch_device()][i] = SlotOwner{0, 0};
    return FA_OK;
}

int fa_release_work_queue(void *stream_handle)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);
    const FaDeviceState *ds = nullptr;
    hipError_t e = fa_device_state(&ds);
    if (e != hipSuccess) return device_fail(e, "device set-up");
    if (stream == hipStreamPerThread) return FA_OK;             // never owns a set
    const bool legacy = stream == nullptr || stream == hipStreamLegacy;
    const uintptr_t handle = legacy ? (uintptr_t)1 : reinterpret_cast<uintptr_t>(stream);
    unsigned long long id = 0;
    if (!legacy && !stream_id(stream, &id)) return device_fail(hipErrorInvalidHandle, "hipStreamGetId");
    // the stream's last launch must have left the set rewound before another stream may take it
    e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return device_fail(e, "synchronize");
    std::lock_guard<std::mutex> lock(g_slot_mutex);
    auto release = [&](SlotOwner *owners, int n) {
        for (int i = 0; i < n; ++i)
            if (owners[i].handle == handle && owners[i].id == id) owners[i] = SlotOwner{0, 0};
    };
    release(g_slot_owner[fa_launch_device()], kFaEagerQueueSlots);
    release(g_merge_owner[fa_launch_device()], kFaEagerMergeSlots);
    return FA_OK;
}

int run_flash_attention(int B, int N, int S, int d, void *Q, void *K, void *V, void *O, void *L, void *M,
                        int Is_dropout, int Is_causal, int Is_local, int Has_alibi, int window_size,
                        float *alibi_slopes, float dropout_prob, void *states)
{
    (void)M;
    (void)states;
    if (Has_alibi && alibi_slopes == nullptr) return FA_ERR_NULL_POINTER;
    if (d <= 0) return FA_ERR_HEAD_DIM;
    fa_fwd_params p;
    memset(&p, 0, sizeof(p));
    p.Q = Q; p.K = K; p.V = V; p.O = O;
    p.L = static_cast<float *>(L);
    p.B = B; p.N = N; p.S = S; p.d = d;
    p.softmax_scale = (float)(1.0 / sqrt((double)d));      // flash_forward.h:639
    p.dropout_prob = Is_dropout ? dropout_prob : 0.0f;
    p.seed = 48;                                             // the seed main() gives its curand states, main.cu:93
    p.alibi_slopes_ptr = Has_alibi ? alibi_slopes : nullptr;      // [N] device floats, main.cu:36-45
    p.window_size_left = Is_local ? window_size : -1;      // flash_forward.h:640-641, mask.h:55
    p.window_size_right = Is_local ? window_size : -1;
    if (Is_local && window_size < 0) { p.window_size_left = p.window_size_right = 0; }
    p.dtype = FA_DTYPE_F16;
    p.is_causal = Is_causal ? 1 : 0;
    const int st = fa_fwd(&p, nullptr);
    if (st != FA_OK) return st;
    hipError_t e = hipStreamSynchronize(nullptr);           // flash_forward.h:655
    if (e != hipSuccess) return device_fail(e, "synchronize");
    return FA_OK;
}

/* ---------------- thin device layer ---------------- */
int fa_dev_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int fa_dev_name(char *buf, size_t len, int *compute_units, int *clock_khz)
{
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, 0);
    if (e != hipSuccess) return device_fail(e, "hipGetDeviceProperties");
    if (buf && len) { snprintf(buf, len, "%s (%s)", prop.name, prop.gcnArchName); }
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (clock_khz) *clock_khz = prop.clockRate;
    return FA_OK;
}

#define FA_DEV(call, what) do { hipError_t e_ = (call); if (e_ != hipSuccess) return device_fail(e_, what); } while (0)

int fa_dev_malloc(void **ptr, size_t bytes) { if (!ptr) return FA_ERR_NULL_POINTER; FA_DEV(hipMalloc(ptr, bytes), "hipMalloc"); return FA_OK; }
int fa_dev_free(void *ptr) { FA_DEV(hipFree(ptr), "hipFree"); return FA_OK; }
int fa_dev_h2d(void *dst, const void *src, size_t bytes) { FA_DEV(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy H2D"); return FA_OK; }
int fa_dev_d2h(void *dst, const void *src, size_t bytes) { FA_DEV(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "hipMemcpy D2H"); return FA_OK; }
int fa_dev_memset(void *dst, int value, size_t bytes) { FA_DEV(hipMemset(dst, value, bytes), "hipMemset"); return FA_OK; }
int fa_dev_sync(void) { FA_DEV(hipDeviceSynchronize(), "hipDeviceSynchronize"); return FA_OK; }
int fa_event_create(void **ev)
{
    if (!ev) return FA_ERR_NULL_POINTER;
    hipEvent_t e;
    FA_DEV(hipEventCreate(&e), "hipEventCreate");
    *ev = e;
    return FA_OK;
}
int fa_event_record(void *ev, void *stream) { FA_DEV(hipEventRecord(static_cast<hipEvent_t>(ev), static_cast<hipStream_t>(stream)), "hipEventRecord"); return FA_OK; }
int fa_event_sync(void *ev) { FA_DEV(hipEventSynchronize(static_cast<hipEvent_t>(ev)), "hipEventSynchronize"); return FA_OK; }
int fa_event_elapsed_ms(void *start, void *stop, float *ms)
{
    if (!ms) return FA_ERR_NULL_POINTER;
    FA_DEV(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)), "hipEventElapsedTime");
    return FA_OK;
}
int fa_event_destroy(void *ev) { FA_DEV(hipEventDestroy(static_cast<hipEvent_t>(ev)), "hipEventDestroy"); return FA_OK; }

// ---- backward pass (include/fa_bwd.h); the reference has none ----
unsigned long long fa_bwd_workspace_bytes(const fa_bwd_params *p)
{
    if (!p || p->B <= 0 || p->N <= 0 || p->S <= 0) return 0;
    return 2ull * (unsigned long long)p->B * p->N * p->S * 4ull;       // delta and the rescaled logsumexp
}

namespace {
// as many keys as queries, in any storage order and with any grouping of K/V heads; lengths that are a multiple of
// 128 also with dropout or with ALiBi (not both), other lengths without either
bool five_product_shape(const fa_bwd_params *p)
{
    if (p->S_kv != 0 && p->S_kv != p->S) return false;
    const bool alibi = p->alibi_slopes_ptr != nullptr, drop = fa_dropout_threshold(p->dropout_prob) != 0;
    return p->S % 128 == 0 ? !(alibi && drop) : !(alibi || drop);
}
unsigned long long ds_blocks_offset(const fa_bwd_params *p)
{
    return (fa_bwd_workspace_bytes(p) + 255ull) & ~255ull;
}
// K/V heads (counted through the batch) and the bytes of dS blocks that belong to one of them: those of its group
// of query heads
long long kv_heads_total(const fa_bwd_params *p) { return (long long)p->B * (p->n_kv_heads > 0 ? p->n_kv_heads : p->N); }
unsigned long long ds_bytes_per_kv_head(const fa_bwd_params *p)
{
    const int group = p->n_kv_heads > 0 ? p->N / p->n_kv_heads : 1;
    return (unsigned long long)group * (unsigned long long)fa_ds_blocks_per_head(p->S) * 2048ull;
}
// The fewest K/V heads a chunk of the five-product form may hold: enough key blocks for two rounds of a full chip,
// a multiple of eight (one head per XCD); all of them when the problem has no more.
long long min_chunk_kv_heads(const fa_bwd_params *p)
{
    const long long key_blocks = (p->S + 255) / 256, all = kv_heads_total(p);
    long long n = (2LL * kComputeUnits + key_blocks - 1) / key_blocks;
    n = (n + 7) / 8 * 8;
    return n < all ? n : all;
}
}  // namespace

unsigned long long fa_bwd_min_fast_workspace_bytes(const fa_bwd_params *p)
{
    if (fa_bwd_fast_workspace_bytes(p) == 0) return 0;
    return ds_blocks_offset(p) + (unsigned long long)min_chunk_kv_heads(p) * ds_bytes_per_kv_head(p);
}

unsigned long long fa_bwd_fast_workspace_bytes(const fa_bwd_params *p)
{
    if (!p || p->B <= 0 || p->N <= 0 || p->S <= 0 || (p->d != 64 && p->d != 128) || !five_product_shape(p)) return 0;
    return ds_blocks_offset(p) + (unsigned long long)p->B * p->N * (unsigned long long)fa_ds_blocks_per_head(p->S) * 2048ull;
}

int fa_bwd_validate(const fa_bwd_params *p)
{
    if (!p || !p->Q || !p->K || !p->V || !p->O || !p->dO || !p->L || !p->dQ || !p->dK || !p->dV) return FA_ERR_NULL_POINTER;
    if (p->B <= 0 || p->N <= 0 || p->S <= 0 || p->S_kv < 0) return FA_ERR_BAD_SHAPE;
    if (p->d != 64 && p->d != 128) return FA_ERR_HEAD_DIM;
    if (p->dtype != FA_DTYPE_F16 && p->dtype != FA_DTYPE_BF16) return FA_ERR_DTYPE;
    if (!(p->softmax_scale > 0.0f) || !isfinite(p->softmax_scale)) return FA_ERR_SCALE;
    if (p->n_kv_heads < 0 || (p->n_kv_heads > 0 && p->N % p->n_kv_heads != 0)) return FA_ERR_LAYOUT;
    if (!(p->dropout_prob >= 0.0f) || !(p->dropout_prob < 1.0f)) return FA_ERR_UNSUPPORTED;
    const long long s_kv = p->S_kv > 0 ? p->S_kv : p->S;
    if ((long long)p->B * p->N * ((p->S + 255) / 256) > 0x7fffffffLL || (long long)p->B * p->N * ((s_kv + 255) / 256) > 0x7fffffffLL ||
        (long long)p->S + s_kv > 0x3fffffffLL) return FA_ERR_TOO_LARGE;
    const void *ptrs[8] = {p->Q, p->K, p->V, p->O, p->dO, p->dQ, p->dK, p->dV};
    const long long *strides[8] = {p->q_strides, p->k_strides, p->v_strides, p->o_strides, p->do_strides,
                                   p->dq_strides, p->dk_strides, p->dv_strides};
    for (int t = 0; t < 8; ++t) {
        if (reinterpret_cast<uintptr_t>(ptrs[t]) % 16 != 0) return FA_ERR_LAYOUT;
        const long long *st = strides[t];
        if (st[0] == 0 && st[1] == 0 && st[2] == 0) continue;       // contiguous
        for (int k = 0; k < 3; ++k)
            if (st[k] < 0 || st[k] % 8 != 0) return FA_ERR_LAYOUT;
        if (st[2] < p->d) return FA_ERR_LAYOUT;
        if (st[2] > (1LL << 24)) return FA_ERR_TOO_LARGE;           // per-lane byte offsets inside a tile are 32-bit
        // a gradient whose batch or head stride is zero would have several writers per element
        if (t >= 5) {
            const int heads = t == 5 ? p->N : (p->n_kv_heads > 0 ? p->n_kv_heads : p->N);
            if ((p->B > 1 && st[0] == 0) || (heads > 1 && st[1] == 0)) return FA_ERR_LAYOUT;
        }
    }
    if (p->workspace == nullptr || reinterpret_cast<uintptr_t>(p->workspace) % 16 != 0 ||
        p->workspace_bytes < fa_bwd_workspace_bytes(p)) return FA_ERR_WORKSPACE;
    return FA_OK;
}

namespace {
// The K/V heads whose dS blocks fit a workspace of this size (whole chunks), 0 when it does not select the five-product form
int ds_heads_for(const fa_bwd_params *p, unsigned long long workspace_bytes)
{
    if (fa_bwd_fast_workspace_bytes(p) == 0 || workspace_bytes < fa_bwd_min_fast_workspace_bytes(p)) return 0;
    const long long all = kv_heads_total(p);
    long long fit = (long long)((workspace_bytes - ds_blocks_offset(p)) / ds_bytes_per_kv_head(p));
    if (fit < all) fit = fit / 8 * 8;
    return (int)(fit < all ? fit : all);
}
// pairs in the walks of one K/V head's key blocks (0: too many to count in 31 bits)
int walk_pairs_per_head(int S, int G, int L, int R)
{
    long long pairs = 0;
    for (int kb = 0; kb < (S + 255) / 256; ++kb) pairs += (long long)G * fa_bwd_walk_tiles(S, S, R, L, kb);
    return pairs <= 0x3fffffffLL ? (int)pairs : 0;
}
// fp32 dK and dV parts of one share
unsigned long long bytes_per_share(const fa_bwd_params *p) { return FA_BWD_PARTS_PER_SHARE * 2ull * 256ull * (unsigned long long)p->d * 4ull; }
}  // namespace

unsigned long long fa_bwd_share_bytes(const fa_bwd_params *p)
{
    if (!p) return 0;
    const int heads = ds_heads_for(p, p->workspace_bytes);
    if (heads == 0 || !fa_bwd_can_share(p->d, fa_dropout_threshold(p->dropout_prob) != 0)) return 0;
    const int G = p->n_kv_heads > 0 ? p->N / p->n_kv_heads : 1;
    int L, R;
    fa_mask_bounds(2 * p->S, p->is_causal, p->window_size_left, p->window_size_right, &L, &R);
    const int per_head = walk_pairs_per_head(p->S, G, L, R);
    // the launches: whole chunks and a smaller last one
    const int rest = (int)(kv_heads_total(p) % heads);
    const int slots = fa_bwd_share_slots(p->d, heads, rest, G, p->S, R, L, per_head);
    return (unsigned long long)slots * bytes_per_share(p);
}

int fa_bwd(const fa_bwd_params *p, void *stream) { return fa_bwd_shared(p, nullptr, 0, stream); }

int fa_bwd_shared(const fa_bwd_params *p, void *partials, unsigned long long partials_bytes, void *stream)
{
    const int st = fa_bwd_validate(p);
    if (st != FA_OK) return st;
    const unsigned long long share_bytes = partials != nullptr ? fa_bwd_share_bytes(p) : 0;
    if (partials != nullptr && (reinterpret_cast<uintptr_t>(partials) % 16 != 0 || partials_bytes < share_bytes)) return FA_ERR_WORKSPACE;
    const FaDeviceState *ds = nullptr;
    {
        const hipError_t de = fa_device_state(&ds);
        if (de != hipSuccess) return device_fail(de, "device set-up");
    }
    FaBwdArgs a;
    a.Q = static_cast<const uint16_t *>(p->Q);
    a.K = static_cast<const uint16_t *>(p->K);
    a.V = static_cast<const uint16_t *>(p->V);
    a.O = static_cast<const uint16_t *>(p->O);
    a.dO = static_cast<const uint16_t *>(p->dO);
    a.lse = p->L;
    a.delta = static_cast<float *>(p->workspace);
    a.lse2 = a.delta + (size_t)p->B * p->N * p->S;
    // a workspace large enough for the dS blocks selects the five-product form
    // (all of them at once when it holds fa_bwd_fast_workspace_bytes, else for as many K/V heads' groups at a time as
    // fit, a multiple of eight and not fewer than fa_bwd_min_fast_workspace_bytes allows)
    a.ds_heads = ds_heads_for(p, p->workspace_bytes);
    a.ds_blocks = a.ds_heads > 0 ? reinterpret_cast<uint16_t *>(static_cast<char *>(p->workspace) + ds_blocks_offset(p)) : nullptr;
    a.head0 = 0;
    a.heads = (int)kv_heads_total(p);
    a.partials = share_bytes != 0 ? static_cast<float *>(partials) : nullptr;
    a.share_slots = a.partials != nullptr ? (int)(share_bytes / bytes_per_share(p)) : 0;
    a.walk_head = a.walk_total = 0;
    a.dQ = static_cast<uint16_t *>(p->dQ);
    a.dK = static_cast<uint16_t *>(p->dK);
    a.dV = static_cast<uint16_t *>(p->dV);
    a.alibi = p->alibi_slopes_ptr;
    a.B = p->B;
    a.H = p->N;
    a.Hk = p->n_kv_heads > 0 ? p->n_kv_heads : p->N;
    a.S = p->S;
    a.Sk = p->S_kv > 0 ? p->S_kv : p->S;
    // general: any lengths, ALiBi, dropout; strided: the reference's lengths with other strides or grouped K/V heads
    // (drop_threshold is set further down: the same function of the probability)
    const bool general = a.S % 128 != 0 || a.Sk != a.S || (a.alibi != nullptr && fa_dropout_threshold(p->dropout_prob) != 0);
    bool strided = a.Hk != a.H;
    {
        const long long *strides[8] = {p->q_strides, p->k_strides, p->v_strides, p->o_strides, p->do_strides,
                                       p->dq_strides, p->dk_strides, p->dv_strides};
        FaBwdTensor *out[8] = {&a.q, &a.k, &a.v, &a.o, &a.dO_, &a.dq, &a.dk, &a.dv};
        for (int t = 0; t < 8; ++t) {
            const bool kv = t == 1 || t == 2 || t == 6 || t == 7;
            const long long heads = kv ? a.Hk : a.H, len = kv ? a.Sk : a.S;
            const long long dense[3] = {heads * len * p->d, len * p->d, p->d};
            const long long *st = strides[t];
            const bool given = st[0] != 0 || st[1] != 0 || st[2] != 0;
            long long eff[3];
            for (int k = 0; k < 3; ++k) {
                eff[k] = given ? st[k] : dense[k];
                if (eff[k] != dense[k]) strided = true;
            }
            out[t]->bs = eff[0]; out[t]->hs = eff[1]; out[t]->rs = (int)eff[2];
        }
    }
    // "unbounded" must stay unbounded after the shift by Sk - S that the key-owning kernel applies
    const int far = a.S + a.Sk;
    fa_mask_bounds(far, p->is_causal, p->window_size_left, p->window_size_right, &a.L, &a.R);
    if (a.partials != nullptr) a.walk_head = walk_pairs_per_head(a.S, a.H / a.Hk, a.L, a.R);
    a.scale = p->softmax_scale;
    a.key_scale = a.scale < kTinyScale ? a.scale / kTinyScaleKeys : a.scale;
    a.drop_threshold = (unsigned)fa_dropout_threshold(p->dropout_prob);
    a.drop_scale = 256.0f / (256.0f - (float)a.drop_threshold);
    a.drop_log = logf(a.drop_scale);
    a.seed_lo = (unsigned)(p->seed & 0xffffffffull);
    a.seed_hi = (unsigned)(p->seed >> 32);
    const int masked = (general || a.L < far || a.R < far) ? 1 : 0;
    hipError_t e = (a.drop_threshold != 0 && !general)
        ? fa_launch_backward_dropout_regular(a, p->dtype == FA_DTYPE_BF16, p->d, masked, strided ? 1 : 0, ds->compute_units,
                                             static_cast<hipStream_t>(stream))
        : (a.alibi != nullptr && !general)
        ? fa_launch_backward_alibi_regular(a, p->dtype == FA_DTYPE_BF16, p->d, masked, strided ? 1 : 0, ds->compute_units,
                                           static_cast<hipStream_t>(stream))
        : a.drop_threshold != 0
        ? fa_launch_backward_dropout(a, p->dtype == FA_DTYPE_BF16, p->d, a.alibi != nullptr ? 1 : 0, ds->compute_units,
                                     static_cast<hipStream_t>(stream))
        : (strided && !general)
        ? fa_launch_backward_strided(a, p->dtype == FA_DTYPE_BF16, p->d, masked, ds->compute_units, static_cast<hipStream_t>(stream))
        : fa_launch_backward(a, p->dtype == FA_DTYPE_BF16, p->d, masked, general || strided ? 1 : 0, a.alibi != nullptr ? 1 : 0,
                             ds->compute_units, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? FA_OK : device_fail(e, "backward launch");
}

void fa_bwd_sched_query_tile_range(int S, int S_kv, int is_causal, int window_left, int window_right,
                                   int k_begin, int rows, int *tile_lo, int *tile_hi)
{
    const int Sk = S_kv > 0 ? S_kv : S, off = Sk - S;
    int L, R;
    fa_mask_bounds(S + Sk, is_causal, window_left, window_right, &L, &R);
    fa_tile_range(S, 64, R + off, L - off, k_begin, rows, tile_lo, tile_hi);
}

int fa_bwd_sched_classify(int S, int S_kv, int is_causal, int window_left, int window_right,
                          int k_begin, int rows, int tile)
{
    const int Sk = S_kv > 0 ? S_kv : S, off = Sk - S;
    int L, R;
    fa_mask_bounds(S + Sk, is_causal, window_left, window_right, &L, &R);
    return fa_tile_class(64, R + off, L - off, k_begin, rows, tile);
}

// Five products over the unmasked pairs (the forward has two).  Square problems only, like fa_algorithmic_flops.
double fa_bwd_algorithmic_flops(int B, int N, int S, int d, int is_causal, int window_left, int window_right)
{
    return 2.5 * fa_algorithmic_flops(B, N, S, d, is_causal, window_left, window_right);
}

}  // extern "C"
