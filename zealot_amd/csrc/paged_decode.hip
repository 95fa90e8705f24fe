// paged_decode.hip -- split-K paged decode attention for gfx950.
//
// One query row per (sequence, q-head) attends to the sequence's pages
// (src/attention/kernels/paged_attention.cu:13-291 computes the same thing
// with one serial thread per workgroup).  The context of every (sequence,
// kv-head) is cut into partitions of `part_pages` pages; one wavefront owns
// one partition of one kv-head and serves all G = H/Hkv query heads that share
// it, so every K/V byte is read from HBM exactly once.  Sequences forked from
// one prefix (the KV cache passes their subgroups) read the shared pages once
// per subgroup as well.  Partials (running max m, sum l, unnormalised o) of
// sequences with more than one partition are merged by a log-sum-exp reduce.
//
// Kernels
//   seq_info_kernel   effective length: the page walk stops at the first table
//                     entry that is < 0 or >= num_blocks (paged_attention.cu:66-67)
//   plan_kernel       partitions -> work-item descriptors, longest first;
//                     resets the queue
//   decode_mfma_kernel  bf16 / fp8 / f32 pools, D in {64,128}, G in {1,2,4,8}:
//       persistent one-wave workgroups take (sequence or subgroup, partition,
//       kv-head) items from an atomic queue (no tail of short waves), stream
//       each page through LDS with global_load_lds, and run QK^T and PV on
//       MFMA with a lazily rescaled softmax (details at the kernel).
//       Small and mid-sized batches run it without plan and queue (DIRECT): one
//       workgroup per (kv-head, partition, sequence).  f32 pools use the f32
//       MFMA (no precision is given up).
//   decode_generic_kernel  any dtype / D <= 256 / G <= 16:
//       one wavefront per (partition, kv-head, sequence); token-per-lane QK on
//       the VALU, readlane-broadcast PV.
//   decode_reduce_kernel  log-sum-exp merge of the partitions.
// Softmax runs in the log2 domain: scores are pre-multiplied by
// scale * log2(e) and exponentiated with exp2 (the FlashAttention trick).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <string>
#include <type_traits>
#include <utility>

#include "zk_common.h"

using namespace zk;

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kWave = 64;

// Pages per work item.  ZEALOT_DECODE_PART_PAGES (1..64) overrides; otherwise
// an item covers ~128 KiB of K+V: 16 pages of bf16 D=128, 32 of fp8 D=128.
int part_pages_env() {
    static int v = [] {
        const char *e = std::getenv("ZEALOT_DECODE_PART_PAGES");
        int p = e ? std::atoi(e) : 0;
        return p < 0 ? 0 : (p > 64 ? 64 : p);
    }();
    return v;
}
int part_pages_for(int kv_dtype, int head_dim, int block_size) {
    if (int e = part_pages_env()) return e;
    const long page_bytes = (long)block_size * head_dim * (kv_dtype == ZK_FP8_E4M3 ? 1 : 2);
    long p = (128 * 1024) / (2 * page_bytes);
    return (int)(p < 16 ? 16 : (p > 64 ? 64 : p));
}
// Smallest partition any path uses (sizes the workspace): every path uses at
// least 16 pages unless ZEALOT_DECODE_PART_PAGES asks for fewer.
int min_part_pages(int head_dim, int block_size) {
    (void)head_dim;
    (void)block_size;
    const int e = part_pages_env();
    return e ? e : 16;
}

constexpr int kSgStride = 32;  // member slots per prefix subgroup (query rows of one shared item)

// Work queues of the persistent MFMA decode (Params::queues of them, 1 or
// kQueues): item i belongs to queue i % queues, and workgroup w takes its
// items from queue w % queues (with 8 queues, the XCD it runs on when
// workgroups are dispatched round-robin over the 8 XCDs).  Each head sits on
// its own 128-byte line.  One queue balances best (a global
// longest-first order); batches of shared-prefix items, many of equal length
// that finish at the same moment, use eight, so their claims go to eight
// lines instead of one, whose atomics the L2 serialises.
constexpr int kQueues = 8;
constexpr int kQueueStride = 32;  // int32 slots between heads
// Two sets of queue heads: a launch takes its items through set
// Params::head_set and puts the other set back to its start values, which
// the launch after it (same workspace, same stream) then uses; the plan
// kernel sets both.  So launches that reuse a plan (the layers of one step)
// need no kernel of their own to reset the heads.
constexpr size_t kWorkBytes = sizeof(int32_t) * kQueueStride * (2 * kQueues + 1);

struct Params {
    const void *q;        // [rows, H, D]; sequence n's row is q_rows[n] (n when q_rows is null)
    const char *k_pool;
    const char *v_pool;
    void *out;
    const int32_t *bt;
    const int32_t *seq_lens;
    const float *k_scales;
    const float *v_scales;
    const int32_t *q_rows;  // optional: q / out row of each sequence
    int64_t q_stride;       // elements between consecutive q rows (out rows: H * D)
    int trusted;            // tables hold valid ids up to every length: no page walk
    int32_t *eff_len;     // [N] length after the page walk
    int4 *items;          // [N * MP][2] work-item descriptors, longest first (MFMA path):
                          //   {n, part, first page, pages} of a sequence's own pages or
                          //   {-1 - g, part, member 0, pages} of subgroup g's shared pages,
                          //   then the block ids of the item's first kDescPages pages
    int32_t *work;        // total items at [0]; the head of queue j of set s at
                          // [kQueueStride * (1 + j + s * kQueues)] (MFMA path)
    int num_waves;        // persistent grid: wave w starts with item w
    int queues;           // work queues in use (1 or kQueues)
    int head_set;         // the set of queue heads this launch claims from (0 or 1)
    // Fused append (MFMA bf16 path; null when unused): the step's K / V row
    // of sequence n, kv-head h, at new_k / new_v + n * new_row_bytes + h * D * 2,
    // is the token at position len - 1; the item holding the sequence's last
    // page stores it into the pools and attends it from registers.
    const char *new_k;
    const char *new_v;
    int64_t new_row_bytes;
    float2 *ml;   // [N][H][MP] (m, l), log2 domain
    float *po;    // [N][H][MP][D]
    // Shared prefixes (MFMA bf16 path; all null when unused): sequence n's
    // first seq_pb[n] pages are the same blocks as every other member of its
    // prefix subgroup.  Subgroup g has members sg_members[g * kSgStride + i]
    // (batch indices, at most 32 / G, padded with -1) and sg_pages[g] shared
    // full pages.  Partial slots of a member: shared parts first, then its
    // private parts.
    const int32_t *seq_pb;
    const int32_t *sg_members;
    const int32_t *sg_pages;
    int num_sg, shared_part_pages;
    int shared_parts;  // planless: partitions of the longest shared prefix
    int num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_blocks, part_pages, max_parts;
    int64_t num_blocks;
    float scale_log2;  // softmax scale * log2(e)
    int grouped;       // 1: kv = h / G, 0: kv = h % Hkv
    int q_f32;         // Q / out dtype: 1 f32, 0 bf16
    // Chunk rows (RowGroups in zk_common.h; null otherwise): "sequence" n of the
    // partials and of the reduce is token n % (32 / G) of group n / (32 / G).
    const int4 *groups;
};

// Tokens of a row group: its tile of 32 rows holds the G heads of each.
__device__ __forceinline__ int group_tokens(const Params &p) { return 32 * p.num_kv_heads / p.num_heads; }

// PLANLESS launches alone have groups.
template <bool PLANLESS = false>
__device__ __forceinline__ size_t qrow(const Params &p, int n) {
    if (PLANLESS && p.groups) return (size_t)p.groups[n / group_tokens(p)].y + n % group_tokens(p);
    return p.q_rows ? (size_t)p.q_rows[n] : (size_t)n;
}

__device__ __forceinline__ int qhead_of(const Params &p, int kvh, int j, int G) {
    return p.grouped ? kvh * G + j : kvh + j * p.num_kv_heads;
}

__device__ __forceinline__ float load_q(const Params &p, size_t i) {
    return p.q_f32 ? ((const float *)p.q)[i]
                   : __uint_as_float((uint32_t)((const uint16_t *)p.q)[i] << 16);
}
__device__ __forceinline__ void store_out(const Params &p, size_t i, float x) {
    if (p.q_f32) ((float *)p.out)[i] = x;
    else ((uint16_t *)p.out)[i] = (uint16_t)f32_to_bf16_bits(x);
}

__device__ __forceinline__ int num_parts_for(const Params &p, int len) {
    int pages = (len + p.block_size - 1) / p.block_size;
    return (pages + p.part_pages - 1) / p.part_pages;
}
__device__ __forceinline__ int prefix_pages_of(const Params &p, int n) { return p.seq_pb ? p.seq_pb[n] : 0; }
// Partitions of sequence n's shared prefix (computed by its subgroup's items).
__device__ __forceinline__ int shared_parts_of(const Params &p, int n) {
    const int pb = prefix_pages_of(p, n);
    return pb > 0 ? (pb + p.shared_part_pages - 1) / p.shared_part_pages : 0;
}
// Partitions of the pages after the shared prefix (the sequence's own items).
// PLANLESS launches have no eff_len: the length is the caller's.
template <bool PLANLESS = false>
__device__ __forceinline__ int private_parts_of(const Params &p, int n) {
    int len;
    if (PLANLESS && p.groups) {
        const int4 g = p.groups[n / group_tokens(p)];
        const int i = n % group_tokens(p);
        len = i < g.z ? g.w + i : 0;  // 0: no such token
    } else {
        len = PLANLESS ? min(max(p.seq_lens[n], 0), p.max_blocks * p.block_size) : p.eff_len[n];
    }
    const int pages = (len + p.block_size - 1) / p.block_size;
    const int rest = pages - prefix_pages_of(p, n);
    return rest > 0 ? (rest + p.part_pages - 1) / p.part_pages : 0;
}

// ------------------------------------------------------------ seq info
__global__ void __launch_bounds__(kWave) seq_info_kernel(Params p) {
    int n = blockIdx.x;
    int len = p.seq_lens[n];
    if (len < 0) len = 0;
    int cap = p.max_blocks * p.block_size;
    if (len > cap) len = cap;
    int pages = (len + p.block_size - 1) / p.block_size;
    const int32_t *row = p.bt + (size_t)n * p.max_blocks;
    int first_bad = pages;
    for (int i0 = 0; i0 < pages && first_bad == pages; i0 += 8 * kWave) {
        int32_t b[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {  // eight independent loads in flight per lane
            const int i = i0 + j * kWave + (int)threadIdx.x;
            b[j] = i < pages ? row[i] : 0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = i0 + j * kWave + (int)threadIdx.x;
            if (i < pages && (b[j] < 0 || (int64_t)b[j] >= p.num_blocks)) first_bad = min(first_bad, i);
        }
        for (int o = 32; o > 0; o >>= 1) first_bad = min(first_bad, __shfl_xor(first_bad, o));
    }
    if (threadIdx.x == 0) p.eff_len[n] = min(len, first_bad * p.block_size);
}

// ------------------------------------------------------------ helpers
// Lane l ^ 16 / l ^ 32's value, on the VALU: v_permlane16_swap exchanges the
// odd 16-lane rows of its first operand with the even rows of its second, and
// v_permlane32_swap the upper half of the first with the lower half of the
// second; with both operands v, a lane's partner value lands in the second
// result on the even rows (lower half) and in the first elsewhere.  (Unlike
// ds_swizzle / ds_bpermute they are not LDS instructions, so they never wait
// behind outstanding LDS or scalar loads.)
__device__ __forceinline__ float xor16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float((threadIdx.x & 16) ? r[0] : r[1]);
}
__device__ __forceinline__ float xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Two f32 -> packed bf16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t bf16x2_rne(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2_t));
}

// scale / l for a row of maximum m: 0 where it saw no keys (m = -inf), NaN where
// all their scores were -inf (l = 0 at the lowest finite m).
__device__ __forceinline__ float inverse_sum(float l, float m, float scale = 1.0f) {
    return l > 0.0f ? scale / l : m == -INFINITY ? 0.0f : NAN;
}

// Lazy-rescale slack of the shared-prefix softmax, in log2 units.
constexpr float kRescaleSlack = 8.0f;

// ------------------------------------------------------------ work plan
// A work item is (sequence or prefix subgroup, partition, kv-head).  The host
// picks the partition length (part_pages, up to kMaxItemPages) so the queue
// holds a few items per wave; plan_kernel sizes pairs from the effective
// lengths of seq_info_kernel and lists them longest first (counting sort on
// the page count) as self-contained descriptors (first page and page count
// included), so that the persistent waves, which take items in queue order,
// perform greedy longest-processing-time-first scheduling and start an item
// with one descriptor load.  Item i is pair i / Hkv, kv-head i % Hkv; wave w
// takes item w first, then pulls from the queue, whose head the kernel sets.
constexpr int kMaxItemPages = 1024;
// Block ids carried in a work-item descriptor (the first pages of the item).
constexpr int kDescPages = 4;

// Pages in flight per wave in the MFMA decode (LDS stages of K + V).
#ifndef ZK_DECODE_STAGES
#define ZK_DECODE_STAGES 2
#endif
constexpr int kStages = ZK_DECODE_STAGES;

// Planless launches (DIRECT): most pages of a partition (one table entry per
// lane).
constexpr int kDirectPages = 64;

__device__ __forceinline__ int pair_pages(const Params &p, int n, int k) {
    const int pages = (p.eff_len[n] + p.block_size - 1) / p.block_size - prefix_pages_of(p, n);
    return max(0, min(p.part_pages, pages - k * p.part_pages));
}
// Items of sequence n: its private partitions; a sequence with neither shared
// nor private pages still gets one (it writes the zero row).
__device__ __forceinline__ int private_items_of(const Params &p, int n) {
    const int np = private_parts_of(p, n);
    return shared_parts_of(p, n) == 0 ? max(1, np) : np;
}
__device__ __forceinline__ int shared_pair_pages(const Params &p, int g, int k) {
    return max(0, min(p.shared_part_pages, p.sg_pages[g] - k * p.shared_part_pages));
}

// At most 64 VGPRs a lane, so that its 16 waves fit beside attention waves
// already resident (four a SIMD beside one decode or prefill wave).
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8)))
plan_kernel(Params p, int num_seqs) {
    __shared__ int hist[2048];  // bin j = kMaxItemPages - pages (longest first)
    __shared__ int wsum[16];
    const int t = threadIdx.x;
    hist[2 * t] = 0;
    hist[2 * t + 1] = 0;
    if (p.trusted) {  // the caller built the tables: the walk would reach every length
        const int cap = p.max_blocks * p.block_size;
        for (int n = t; n < num_seqs; n += 1024) p.eff_len[n] = min(max(p.seq_lens[n], 0), cap);
        __threadfence_block();
    }
    __syncthreads();
    for (int n = t; n < num_seqs; n += 1024) {
        const int np = private_items_of(p, n);
        for (int k = 0; k < np; ++k) atomicAdd(&hist[kMaxItemPages - pair_pages(p, n, k)], 1);
    }
    for (int g = t; g < p.num_sg; g += 1024) {
        const int np = (p.sg_pages[g] + p.shared_part_pages - 1) / p.shared_part_pages;
        for (int k = 0; k < np; ++k) atomicAdd(&hist[kMaxItemPages - shared_pair_pages(p, g, k)], 1);
    }
    __syncthreads();
    // exclusive scan of the bins, two per thread (each thread rewrites only
    // its own two, so no barrier between reading and writing them)
    const int a = hist[2 * t], b = hist[2 * t + 1];
    int total_pairs;
    const int base = zk::block_exclusive_scan_1024(a + b, wsum, &total_pairs);
    hist[2 * t] = base;
    hist[2 * t + 1] = base + a;
    __syncthreads();
    // an item's descriptor carries the block ids of its first pages, so the
    // decode issues them without waiting for the item's table entries
    auto first_blocks = [&](const int32_t *row, int pages) {
        int b[kDescPages];
#pragma unroll
        for (int j = 0; j < kDescPages; ++j) b[j] = j < pages ? row[j] : 0;
        return make_int4(b[0], b[1], b[2], b[3]);
    };
    for (int n = t; n < num_seqs; n += 1024) {
        const int np = private_items_of(p, n);
        for (int k = 0; k < np; ++k) {
            const int np = pair_pages(p, n, k);
            const int pos = atomicAdd(&hist[kMaxItemPages - np], 1);
            const int first = prefix_pages_of(p, n) + k * p.part_pages;
            p.items[2 * pos] = make_int4(n, k, first, np);
            p.items[2 * pos + 1] = first_blocks(p.bt + (size_t)n * p.max_blocks + first, np);
        }
    }
    for (int g = t; g < p.num_sg; g += 1024) {
        const int np = (p.sg_pages[g] + p.shared_part_pages - 1) / p.shared_part_pages;
        const int n0 = p.sg_members[(size_t)g * kSgStride];
        // pages member 0's walk reaches (all unless its table is cut inside the prefix)
        const int valid = min(p.sg_pages[g], p.eff_len[n0] / p.block_size);
        for (int k = 0; k < np; ++k) {
            const int pos = atomicAdd(&hist[kMaxItemPages - shared_pair_pages(p, g, k)], 1);
            const int pages = max(0, min(p.shared_part_pages, valid - k * p.shared_part_pages));
            p.items[2 * pos] = make_int4(-1 - g, k, n0, pages);  // negative: subgroup item
            p.items[2 * pos + 1] =
                first_blocks(p.bt + (size_t)n0 * p.max_blocks + (size_t)k * p.shared_part_pages, pages);
        }
    }
    if (t == 0) {
        p.work[0] = total_pairs * p.num_kv_heads;  // total items
    }
    if (t < p.queues) {  // queue heads, both sets: wave w takes item w statically, w < num_waves
        p.work[kQueueStride * (1 + t)] = (p.num_waves - t + p.queues - 1) / p.queues;
        p.work[kQueueStride * (1 + t + kQueues)] = (p.num_waves - t + p.queues - 1) / p.queues;
    }
}

// ------------------------------------------------------------ MFMA kernel
typedef __attribute__((address_space(3))) void lds_void;

// 16 bytes per lane from global memory straight into LDS at lds + 16 * lane
// (global_load_lds_dwordx4; no VGPRs, counted by vmcnt).  Cache policy NT
// (nontemporal, aux bit 1): every K/V byte is read exactly once, and the
// streaming hint measured ~9% faster than the default policy on C2.
constexpr int kCachePolicyNT = 2;
__device__ __forceinline__ void g2l16(const void *g, lds_void *l) {
    __builtin_amdgcn_global_load_lds(g, l, 16, 0, kCachePolicyNT);
}
// s_waitcnt vmcnt(N) alone (gfx9 encoding: expcnt 7 and lgkmcnt 15 mean "no wait").
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N <= 63, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xc07f); }

template <int BYTES>
struct LdsVec;
template <>
struct LdsVec<16> { typedef u32x4 T; };
template <>
struct LdsVec<8> { typedef u32x2 T; };
template <>
struct LdsVec<4> { typedef uint32_t T; };

// Persistent split-K decode for bf16 / fp8 / f32 pools, D in {64, 128},
// block_size 16, G = H/Hkv in {1, 2, 4, 8}.  The grid holds a fixed number of one-wave
// workgroups; each loops over work items.  Per item, the partition's pages
// stream through kStages LDS stages per wave: every page (K and V, 16 rows of
// D elements each) arrives by global_load_lds_dwordx4, 1 KiB contiguous per
// instruction, so the next page is in flight while this one is computed.
//   K stage layout: 16-byte chunk c of row r sits at chunk slot
//     r * CPR + (c ^ (r % CPR)), so the MFMA fragment reads (16 rows, same c)
//     hit distinct LDS banks.
//   V stage layout: natural [row][D].
// An item computes the query rows held in the columns of T 16-column MFMA
// tiles: a sequence's own partition has the G heads of one kv-head (T = 1,
// columns >= G idle); a prefix subgroup's shared partition has member-major
// rows, G heads per member (T = 2, up to 32 rows), so one read of a shared
// page serves every member.
//   QK^T  v_mfma_f32_16x16x32_bf16, A = the page's 16 K rows (tokens), B = the
//         tile's query rows; lane (grp, col) gets tokens 4*grp+i of row col.
//   softmax  one reference max per row, shared by the 4 lane groups and moved
//         lazily: only when a score exceeds it by kRescaleSlack (always on the
//         first page), so weights stay <= 2^kRescaleSlack, the 16 tokens of a
//         page share a scale, and most pages leave the accumulators alone.
//   PV    O^T[dims x rows] += V^T[dims x 16 tokens] * P^T[16 tokens x rows] on
//         v_mfma_f32_16x16x16_bf16: P^T is the score fragment in bf16; lane
//         (grp, col) reads DT = D/16 consecutive dims of the token rows
//         4*grp+i (fp8 pools: converted to bf16, exactly) and v_perm
//         transposes them into DT A operands, so A row m of tile dt is dim
//         DT*m + dt.
// fp8 pools: the K scale folds into the softmax scale, the V scale into the
// result.
// f32 pools: QK^T and PV on v_mfma_f32_16x16x4_f32, four k-steps per 16-byte
// chunk, with V's dims of a lane chosen so that its LDS reads are contiguous
// over 16 lanes; the scores' fragment is P^T's, as above.  64 MFMAs of 32 cycles
// a page are 0.85 us, hidden behind the 2.3 us that a page takes at the HBM rate
// with one wave a SIMD.  48 x 128..4096 tokens, 32 / 8 heads of 128: 2500 us in
// decode_generic_kernel (a row per lane: uncoalesced, serial), 155 us here
// (5.6 TB/s).
// DIRECT: no plan and no queue; workgroup (kvh, part, n) is partition `part` of
// sequence n (at most kDirectPages pages), derives its pages from the length
// and the table itself and ends.  A partition whose pages end at an invalid
// table entry marks its partial (sign bit of l), and the reduce drops the
// partitions after it.
// ROWS (with DIRECT): workgroup (kvh, part, g) is partition `part` of row group g,
// up to 32 / G consecutive tokens of one chunk: their 32 (token, head) rows are
// two tiles, every page is read once for all of them, and each row masks the
// tokens past its own position.  f32 pools only; bound by the f32 MFMA (128 of
// 32 cycles a page, 1.7 us, against 0.85 for one row tile).  A 150-token chunk
// behind 0..600 tokens, 32 / 8 heads of 128: 57 us as 150 one-row decodes, 31
// here, and its tables no longer displace the decode half's (four uploads of a
// step gone): the step of it and 12 decodes 113 -> 59 us.  Pages with tokens that
// only some of the rows see come last (SOME below).
// SHARED (with DIRECT): the first num_sg * shared_parts workgroups of a kv-head
// are the shared-prefix partitions, the others the sequences' own.
template <int KV, int D, int G, bool DIRECT, bool ROWS = false, bool SHARED = false>
__global__ void __launch_bounds__(kWave) decode_mfma_kernel(Params p) {
    constexpr int BS = 16;
    constexpr int BIDS = DIRECT && !ROWS ? kDirectPages : kMaxItemPages;
    constexpr bool F32 = KV == ZK_F32;
    // The maximum starts finite, so that keys whose scores are -inf have weight
    // 0 and not NaN wherever a partition begins (fp8 keys are finite).
    constexpr bool LOWEST = DIRECT || KV != ZK_FP8_E4M3;
    constexpr int ELT = F32 ? 4 : KV == ZK_BF16 ? 2 : 1;
    constexpr int DG = D / 4;            // head dims per lane group in QK
    constexpr int KK = F32 ? D / 16 : DG / 8;  // 16-byte Q chunks per lane (bf16: MFMA k-steps)
    constexpr int DT = D / 16;           // PV dim tiles = dims per lane per V row
    constexpr int RB = D * ELT;          // bytes per token row
    constexpr int CPR = RB / 16;         // 16-byte chunks per row
    constexpr int PAGE = BS * RB;        // bytes per (block, kv-head) page
    constexpr int LPK = PAGE / 1024;     // global_load_lds per page of K (or V)
    constexpr int LPP = 2 * LPK;         // per page, K and V
    constexpr int KBYTES = DG * ELT;     // K fragment bytes per lane per page
    constexpr int KCH = KBYTES / 16;     // ... in 16-byte chunks
    constexpr int VTB = DT * ELT;        // V bytes per lane per token row
    static_assert(PAGE % 1024 == 0 && KBYTES % 16 == 0 && DT % 2 == 0, "page shape");
    typedef typename LdsVec<F32 ? 16 : VTB>::T vtrow_t;
    constexpr int VR = F32 ? VTB / 16 : 1;  // V reads per lane and token row
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef typename std::conditional<F32, f32x4, bf16x8>::type qfrag_t;  // 16 bytes of a query row
    const qfrag_t qzero = __builtin_bit_cast(qfrag_t, u32x4{0u, 0u, 0u, 0u});
    __shared__ __attribute__((aligned(16))) char lds[kStages][2][PAGE];  // [stage][K|V]
    __shared__ int32_t bids[BIDS];                              // this item's block ids

    const int lane = threadIdx.x, col = lane & 15, grp = lane >> 4;
    const int H = p.num_heads, Hkv = p.num_kv_heads;

    // per-lane byte offsets, fixed for the whole kernel
    uint32_t kg[LPK], vg[LPK];  // global offsets inside a page
#pragma unroll
    for (int j = 0; j < LPK; ++j) {
        const int q = 64 * j + lane, row = q / CPR, c = (q % CPR) ^ (row % CPR);
        kg[j] = row * RB + c * 16;
        vg[j] = q * 16;
    }
    uint32_t kl[KCH];  // LDS offsets of this lane's K fragment chunks
#pragma unroll
    for (int f = 0; f < KCH; ++f) {
        // bf16 / fp8: lane group grp holds dims DG grp .. of the row; f32: dims
        // 16 f + 4 grp .. of chunk f, so consecutive chunks feed consecutive k-steps
        const int row = col, c = F32 ? 4 * f + grp : grp * KCH + f;
        kl[f] = (row * CPR + (c ^ (row % CPR))) * 16;
    }
    // + i * RB; f32: + 256 h, dims 64 h + 4 col .. + 3 (16 lanes read one
    // contiguous 256-byte piece)
    const uint32_t vt_off = (uint32_t)((4 * grp) * RB + col * (F32 ? 16 : VTB));

    // Wait until page pi of an np-page item has landed in LDS: the pages
    // issued after it (up to kStages - 1) may still be in flight.
    auto wait_page = [&](int pi, int np) {
        const int ahead = min(kStages - 1, np - 1 - pi);
        static_assert(kStages >= 2 && kStages <= 4, "pipeline depth");
        if (ahead <= 0) wait_vmcnt<0>();
        else if (ahead == 1) wait_vmcnt<LPP>();
        else if (ahead == 2) wait_vmcnt<(kStages > 2 ? 2 * LPP : 0)>();
        else wait_vmcnt<(kStages > 3 ? 3 * LPP : 0)>();
    };

    int next = 0;
    // Claims the next item.  Called once per item, in the iteration that
    // issues the item's last page (right after the first issues for items of
    // at most kStages pages), so the atomic's round trip overlaps the item's
    // last pages.  (Claiming at the start of an item instead lets every wave
    // holding a long item reserve a short one it only starts much later,
    // while waves that finish their short items find the queue empty: with
    // mixed item lengths that left a tail of late short items.)
    const int nq = DIRECT ? 1 : p.queues, xq = blockIdx.x % nq;
    auto head = [&](int q) { return p.work + kQueueStride * (1 + q + p.head_set * kQueues); };
    // the other set of heads back to its start for the next launch on this
    // workspace (no wave of this launch touches it)
    if (!DIRECT && blockIdx.x == 0 && lane < nq)
        p.work[kQueueStride * (1 + lane + (1 - p.head_set) * kQueues)] = (p.num_waves - lane + nq - 1) / nq;
    auto claim_next = [&]() {
        if (lane == 0) next = atomicAdd(head(xq), 1);
    };

    // Data the kernel only reads (descriptors, subgroup members, lengths,
    // scales) goes through constant-space views: scalar loads, counted by
    // lgkmcnt, so they never hold up the page stream's vmcnt waits.
    typedef const __attribute__((address_space(4))) int32_t *cint_t;
    typedef const __attribute__((address_space(4))) float *cfloat_t;
    const cint_t citems = (cint_t)p.items;
    // descriptor of pair k: 8 ints (two int4)
    auto load_desc = [&](int k, int4 &a, int4 &b) {
        const cint_t c = citems + 8 * (size_t)k;
        a = make_int4(c[0], c[1], c[2], c[3]);
        b = make_int4(c[4], c[5], c[6], c[7]);
    };

    // Block ids of an item's pages kStages .. np-1 into LDS (bids[i] = table
    // entry i; the first pages' ids come with the descriptor), eight
    // independent loads in flight per lane.  The LDS writes wait for their
    // loads, which retires every earlier load of the item (Q fragments, the
    // first pages) too, so the page loop starts with nothing pending in the
    // compiler's view.  (LDS-DMA staging of the ids, or register loads still
    // pending at the loop, make the compiler wait for vmcnt(0) inside the
    // page loop, which drains the page stream every page.)
    auto stage_bids = [&](const int32_t *row, int np) {
        for (int i0 = kStages; i0 < np; i0 += 8 * kWave) {
            int32_t b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = i0 + j * kWave + lane;
                b[j] = i < np ? row[i] : 0;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = i0 + j * kWave + lane;
                if (i < np) bids[i] = b[j];
            }
        }
        wait_lgkmcnt0();  // this wave's LDS writes are visible to its own reads
    };

    // B fragment of query row (n, qh): this lane group's DG dims as KK bf16x8.
    auto load_q = [&](size_t qr, int qh, qfrag_t *qf) {
        if constexpr (F32) {
            const size_t qb = qr * (size_t)p.q_stride + (size_t)qh * D + 4 * grp;
#pragma unroll
            for (int j = 0; j < KK; ++j) {
                if (p.q_f32) {
                    qf[j] = *reinterpret_cast<const f32x4 *>((const float *)p.q + qb + 16 * j);
                } else {
                    const u32x2 w = *reinterpret_cast<const u32x2 *>((const uint16_t *)p.q + qb + 16 * j);
                    qf[j] = f32x4{bf16lo(w[0]), bf16hi(w[0]), bf16lo(w[1]), bf16hi(w[1])};
                }
            }
            return;
        } else {
            const size_t qb = qr * (size_t)p.q_stride + (size_t)qh * D + (size_t)grp * DG;
            if (p.q_f32) {
                const float *qq = (const float *)p.q + qb;
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    u32x4 w;
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j] = pack_bf16x2(qq[8 * kk + 2 * j], qq[8 * kk + 2 * j + 1]);
                    qf[kk] = __builtin_bit_cast(bf16x8, w);
                }
            } else {
                const uint16_t *qq = (const uint16_t *)p.q + qb;
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) qf[kk] = *reinterpret_cast<const bf16x8 *>(qq + 8 * kk);
            }
        }
    };

    const int total = DIRECT ? 0 : *(cint_t)p.work;
    // The next item and its descriptor, loaded while the current item's last
    // page is computed (the claim has returned by then).  The scalar load is
    // issued by inline asm: a plain load, whose result is only used after the
    // page loop, is moved past the loop by the compiler; the asm keeps it in
    // the last iteration, and desc_ready() waits for it (lgkmcnt) and hands
    // the registers on.
    typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
    int nx = 0;
    i32x8 nraw = {0, 0, 0, 0, 0, 0, 0, 0};
    bool have_next = false;
    // (claims past the last item read a descriptor the item loop then
    // ignores: the index is clamped to the descriptor array)
    const int desc_cap = p.num_seqs * p.max_parts;
    auto fetch_next = [&]() {
        nx = __builtin_amdgcn_readfirstlane(next) * nq + xq;
        if (nx >= total) {
            // own queue done: take from the others (a plain load first, so
            // exhausted queues cost no atomic)
            int got = total;
            if (lane == 0)
                for (int j = 1; j < nq && got >= total; ++j) {
                    const int q = (xq + j) % nq;
                    if (__hip_atomic_load(head(q), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * nq + q >= total)
                        continue;
                    const int idx = atomicAdd(head(q), 1) * nq + q;
                    if (idx < total) got = idx;
                }
            nx = __builtin_amdgcn_readfirstlane(got);
        }
        const int k = __builtin_amdgcn_readfirstlane(min(nx / Hkv, desc_cap - 1));
        asm volatile("s_load_dwordx8 %0, %1, 0x0" : "=s"(nraw) : "s"(p.items + 2 * (size_t)k) : "memory");
        have_next = true;
    };
    auto desc_ready = [&](int4 &a, int4 &b) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(nraw)::"memory");
        a = make_int4(nraw[0], nraw[1], nraw[2], nraw[3]);
        b = make_int4(nraw[4], nraw[5], nraw[6], nraw[7]);
    };

    // q / out row of sequence n
    auto q_row = [&](int n) -> size_t { return p.q_rows ? (size_t)((cint_t)p.q_rows)[n] : (size_t)n; };

    // Attention of T tiles of query rows (qf) over pages [page0, page0 + np)
    // of table `trow` for kv-head kvh; tokens at positions >= row_len[t] are
    // masked for this lane's row of tile t, and V rows at or past len (the
    // longest) are zeroed; every row sees the tokens before `open`.
    // trow points at the table entry of page page0; blk0 holds the block ids
    // of the first kDescPages pages.
    // Leaves O^T (o), the rows' reference max (m) and sum (l, all 4 lane
    // groups) for the caller to write.  fuse_tib >= 0 (fused append): the
    // last page's row fuse_tib is the step's token, nrow in this wave's
    // registers (lane c < CPR: chunk c of K, CPR <= lane < 2 CPR: of V); it is
    // written into the page's LDS copy once that has landed, and to the pools
    // at byte offset row_dst of the K / V pool.
    auto attend = [&]<int T>(const qfrag_t (&qf)[T][KK], const int32_t *trow, int4 blk0, int page0, int np, int len,
                             const int (&row_len)[T], int open, int kvh, float sl2, f32x4 (&o)[DT][T], float (&m)[T], float (&l)[T], int fuse_tib,
                             u32x4 nrow, size_t row_dst) {
        const char *kbase = p.k_pool + ((size_t)kvh * PAGE);
        const char *vbase = p.v_pool + ((size_t)kvh * PAGE);
        const size_t block_bytes = (size_t)PAGE * Hkv;
        auto issue_blk = [&](int blk, int s) {
            const char *kp = kbase + (size_t)blk * block_bytes;
            const char *vp = vbase + (size_t)blk * block_bytes;
#pragma unroll
            for (int j = 0; j < LPK; ++j) g2l16(kp + kg[j], (lds_void *)(lds[s][0] + 1024 * j));
#pragma unroll
            for (int j = 0; j < LPK; ++j) g2l16(vp + vg[j], (lds_void *)(lds[s][1] + 1024 * j));
        };
#pragma unroll
        for (int t = 0; t < T; ++t) {
            m[t] = LOWEST ? -FLT_MAX : -INFINITY;
            l[t] = 0.0f;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // SOME: a row group's page with tokens that only some of its rows see
        auto page = [&]<bool SOME>(int pi, int s) {
            wait_page(pi, np);
            if constexpr (KV == ZK_BF16) {
                if (fuse_tib >= 0 && pi == np - 1) {  // the step's token over the page's stale row
                    if (lane < CPR)
                        *reinterpret_cast<u32x4 *>(lds[s][0] + (fuse_tib * CPR + (lane ^ (fuse_tib % CPR))) * 16) =
                            nrow;
                    else if (lane < 2 * CPR)
                        *reinterpret_cast<u32x4 *>(lds[s][1] + fuse_tib * RB + (lane - CPR) * 16) = nrow;
                    if (lane < 2 * CPR)
                        __builtin_nontemporal_store(
                            nrow, reinterpret_cast<u32x4 *>((char *)(lane < CPR ? p.k_pool : p.v_pool) + row_dst));
                }
            }
            uint32_t kw[KBYTES / 4];
#pragma unroll
            for (int f = 0; f < KCH; ++f) {
                const u32x4 c4 = *reinterpret_cast<const u32x4 *>(lds[s][0] + kl[f]);
#pragma unroll
                for (int j = 0; j < 4; ++j) kw[4 * f + j] = c4[j];
            }
            // token rows 4*grp+i, dims DT*col .. DT*col+DT-1 (f32: see vt_off)
            vtrow_t vt[4][VR];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int h = 0; h < VR; ++h)
                    vt[i][h] = *reinterpret_cast<const vtrow_t *>(lds[s][1] + vt_off + i * RB + 256 * h);
            const int nb = bids[min(pi + kStages, BIDS - 1)];
            // The stage is free once its reads are done: the empty asm needs
            // their results, so the compiler's own lgkmcnt wait lands here
            // (it does not count an explicit s_waitcnt as completing them and
            // would wait again at the MFMAs, behind the prefetch below).
#pragma unroll
            for (int j = 0; j < KBYTES / 4; ++j) asm volatile("" ::"v"(kw[j]));
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int h = 0; h < VR; ++h) asm volatile("" ::"v"(vt[i][h]));
            asm volatile("" ::"v"(nb));
            if (pi + kStages < np) issue_blk(__builtin_amdgcn_readfirstlane(nb), s);
            if constexpr (!DIRECT) {
                if (pi == np - 1 - kStages) claim_next();
                if (pi == np - 1) fetch_next();
            }

            f32x4 sacc[T];
#pragma unroll
            for (int t = 0; t < T; ++t) sacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (F32) {
                // k-step (f, e): lane group grp holds dim 16 f + 4 grp + e of
                // its K row (A) and query row (B); two chains a tile
                f32x4 s2[T];
#pragma unroll
                for (int t = 0; t < T; ++t) s2[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int f = 0; f < KCH; ++f)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int t = 0; t < T; ++t) {
                            f32x4 &a = e & 1 ? s2[t] : sacc[t];
                            a = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(kw[4 * f + e]), qf[t][f][e], a, 0, 0, 0);
                        }
#pragma unroll
                for (int t = 0; t < T; ++t) sacc[t] += s2[t];
            } else {
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    u32x4 w;
                    if constexpr (KV == ZK_BF16) {
                        w = u32x4{kw[4 * kk], kw[4 * kk + 1], kw[4 * kk + 2], kw[4 * kk + 3]};
                    } else {
                        const u32x2 lo2 = e4m3x4_to_bf16x4(kw[2 * kk]), hi2 = e4m3x4_to_bf16x4(kw[2 * kk + 1]);
                        w = u32x4{lo2[0], lo2[1], hi2[0], hi2[1]};
                    }
#pragma unroll
                    for (int t = 0; t < T; ++t)
                        sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), qf[t][kk],
                                                                          sacc[t], 0, 0, 0);
                }
            }
            // V rows as bf16 pairs: w[i][j] = dims (2j, 2j+1) of token row
            // 4*grp+i; f32: the DT values themselves
            constexpr int VW = F32 ? DT : DT / 2;
            uint32_t w[4][VW];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (KV != ZK_FP8_E4M3) {
                    __builtin_memcpy(w[i], &vt[i], 4 * VW);
                } else {
                    uint32_t b8[DT / 4];
                    __builtin_memcpy(b8, &vt[i], DT);
#pragma unroll
                    for (int j = 0; j < DT / 4; ++j) {
                        const u32x2 c2 = e4m3x4_to_bf16x4(b8[j]);
                        w[i][2 * j] = c2[0];
                        w[i][2 * j + 1] = c2[1];
                    }
                }
            }
            const int tok0 = (page0 + pi) * BS + 4 * grp;
            if (tok0 + 4 > len) {  // partial last page: stale rows must not reach O
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (tok0 + i >= len)
#pragma unroll
                        for (int j = 0; j < VW; ++j) w[i][j] = 0u;
            }
            // V of a token must not reach the rows that do not see it, whose
            // weight of 0 times an infinity would be NaN: a page with a value that
            // is not finite takes its tokens one by one.
            bool one_by_one = false;
            if constexpr (SOME) {
                uint32_t top = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < VW; ++j) top = max(top, w[i][j] & 0x7f800000u);
                one_by_one = __builtin_amdgcn_ballot_w64(top == 0x7f800000u) != 0;
            }
            s16x4 va[F32 ? 1 : DT];  // element i of tile dt = V[4*grp+i][DT*col+dt]
            if constexpr (!F32)
#pragma unroll
            for (int j = 0; j < DT / 2; ++j) {
                const u32x2 lo{__builtin_amdgcn_perm(w[1][j], w[0][j], 0x05040100u),
                               __builtin_amdgcn_perm(w[3][j], w[2][j], 0x05040100u)};
                const u32x2 hi{__builtin_amdgcn_perm(w[1][j], w[0][j], 0x07060302u),
                               __builtin_amdgcn_perm(w[3][j], w[2][j], 0x07060302u)};
                va[2 * j] = __builtin_bit_cast(s16x4, lo);
                va[2 * j + 1] = __builtin_bit_cast(s16x4, hi);
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                float sc[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[i] = tok0 + i < row_len[t] ? sacc[t][i] * sl2 : -INFINITY;
                const float mx = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
                // lazy rescale (wave-uniform branch): the new reference is the
                // row max over the page's 16 tokens (all four lane groups)
                if (__builtin_amdgcn_ballot_w64(mx > m[t] + kRescaleSlack)) {
                    float cm = fmaxf(mx, xor16(mx));
                    cm = fmaxf(cm, xor32(cm));
                    const float m_new = fmaxf(m[t], cm);
                    const float alpha = m_new == -INFINITY ? 1.0f : exp2_fast(m[t] - m_new);
                    l[t] *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[dt][t] *= alpha;
                    m[t] = m_new;
                }
                float pr[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) pr[i] = exp2_fast(sc[i] - m[t]);
                l[t] += (pr[0] + pr[1]) + (pr[2] + pr[3]);
                if constexpr (SOME) {
                    if (one_by_one) {
#pragma unroll 1
                        for (int g = 0; g < 4; ++g)
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const bool sees = (page0 + pi) * BS + 4 * g + i < row_len[t];
#pragma unroll
                                for (int dt = 0; dt < DT; ++dt) {
                                    const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                        grp == g ? __uint_as_float(w[i][dt]) : 0.0f, pr[i], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                                    if (sees) o[dt][t] += c;
                                }
                            }
                        continue;
                    }
                }
                if constexpr (F32) {
                    // k-step i: V^T column token 4*grp+i (A) and its weight (B)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt)
                            o[dt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[i][dt]), pr[i], o[dt][t], 0, 0, 0);
                    continue;
                }
                const s16x4 pb = __builtin_bit_cast(s16x4, u32x2{bf16x2_rne(pr[0], pr[1]), bf16x2_rne(pr[2], pr[3])});
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    o[dt][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[F32 ? 0 : dt], pb, o[dt][t], 0, 0, 0);
            }
        };
        // the first pages straight from the descriptor, then the other ids
        static_assert(kStages <= kDescPages, "descriptor carries the first kStages block ids");
        const int b0[4] = {blk0.x, blk0.y, blk0.z, blk0.w};
#pragma unroll
        for (int j = 0; j < kStages; ++j)
            if (j < np) issue_blk(b0[j], j);
        if constexpr (!DIRECT) stage_bids(trow, np);  // (DIRECT: staged by the caller)
        // Q is complete before the loop on every path (see stage_bids)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) asm volatile("" ::"v"(qf[t][kk]));
        // and so is the fused row
        asm volatile("" ::"v"(nrow[0]), "v"(nrow[1]), "v"(nrow[2]), "v"(nrow[3]));
        if constexpr (!DIRECT)
            if (np <= kStages) claim_next();
        // one page per iteration (a single loop-carried accumulator set)
        // (row groups: the pages that every row sees whole first)
        const int whole = ROWS ? min(np, max(0, open / BS - page0)) : np;
        int pi = 0, st = 0;
        for (; pi < whole; ++pi, st = (st + 1 == kStages ? 0 : st + 1)) page.template operator()<false>(pi, st);
        if constexpr (ROWS)
            for (; pi < np; ++pi, st = (st + 1 == kStages ? 0 : st + 1)) page.template operator()<true>(pi, st);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            l[t] += xor16(l[t]);
            l[t] += xor32(l[t]);
            if (LOWEST && np == 0) m[t] = -INFINITY;
        }
    };

    // Lane (grp, col) holds dims DT*(4*grp+i)+dt, i < 4, dt < DT, of row col:
    // four runs of DT consecutive floats.  f32 pools: tile dt = 4 h + e is dims
    // 64 h + 4*(4*grp+i) + e, runs of four.
    auto store_row_f32 = [&](float *dst, const f32x4 (&o)[DT][2], int t, float scale) {
        if constexpr (F32) {
#pragma unroll
            for (int h = 0; h < DT / 4; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 v = f32x4{o[4 * h][t][i], o[4 * h + 1][t][i], o[4 * h + 2][t][i], o[4 * h + 3][t][i]} * scale;
                    __builtin_memcpy(dst + 64 * h + 16 * grp + 4 * i, &v, sizeof(v));
                }
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v[DT];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) v[dt] = o[dt][t][i] * scale;
            __builtin_memcpy(dst + DT * (4 * grp + i), v, sizeof(v));
        }
    };
    // a partial slot and its (m, l), for decode_reduce_kernel
    auto store_partial = [&](size_t slot, const f32x4 (&o)[DT][2], int t, float scale, float m_, float l_) {
        store_row_f32(p.po + slot * D, o, t, scale);
        if (grp == 0) p.ml[slot] = make_float2(m_, l_);
    };
    const u32x4 no_row = {0u, 0u, 0u, 0u};

    // shared-prefix partition `part` of subgroup sg (np pages of member 0's table)
    auto shared_part = [&](int sg, int kvh, int part, int n0, int np, int4 d1) {
        // shared-prefix partition of subgroup sg: up to 32 rows, member-major
        const int page0 = part * p.shared_part_pages;
        // members (batch indices) of the subgroup, by scalar loads; lane
        // (grp, col) serves row r = 16 t + col, member r / G
        constexpr int NM = kSgStride / G;
        const cint_t cmem = (cint_t)(p.sg_members + (size_t)sg * kSgStride);
        int mem_s[NM];
#pragma unroll
        for (int j = 0; j < NM; ++j) mem_s[j] = cmem[j];
        qfrag_t qf[2][KK];
        int nm[2];  // member of this lane's row in tile t, or -1
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int r = 16 * t + col;
            int v = mem_s[0];
#pragma unroll
            for (int j = 1; j < NM; ++j) v = r / G == j ? mem_s[j] : v;
            nm[t] = v;
            if (nm[t] >= 0) load_q(q_row(nm[t]), qhead_of(p, kvh, r % G, G), qf[t]);
            else
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) qf[t][kk] = qzero;
        }
        f32x4 o[DT][2];
        float m[2], l[2];
        const int all[2] = {0x7fffffff, 0x7fffffff};
        attend.template operator()<2>(qf, p.bt + (size_t)n0 * p.max_blocks + page0, d1, page0, np, 0x7fffffff, all,
                                      0x7fffffff, kvh, p.scale_log2, o, m, l, -1, no_row, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int r = 16 * t + col;
            if (nm[t] >= 0) {
                const size_t slot = ((size_t)nm[t] * H + qhead_of(p, kvh, r % G, G)) * p.max_parts + part;
                store_partial(slot, o, t, 1.0f, m[t], l[t]);
            }
        }
    };

    // a sequence's own partition: rows 0..G-1 are its heads of kv-head kvh
    // (ns shared and nparts own partitions in all; cut: the partition's pages
    // end at an invalid table entry)
    auto own_part = [&](int n, int kvh, int part, int page0, int np, int len, int ns, int nparts, int4 d1, bool cut) {
        const int qh = qhead_of(p, kvh, col % G, G);
        const size_t qr = q_row(n);
        qfrag_t qf[1][KK];
        if (col < G) load_q(qr, qh, qf[0]);
        else
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) qf[0][kk] = qzero;
        float sl2 = p.scale_log2, vscale = 1.0f;
        if constexpr (KV == ZK_FP8_E4M3) {
            sl2 *= ((cfloat_t)p.k_scales)[(size_t)n * Hkv + kvh];
            vscale = ((cfloat_t)p.v_scales)[(size_t)n * Hkv + kvh];
        }
        // fused append: the item holding the sequence's last page
        int fuse_tib = -1;
        u32x4 nrow = no_row;
        size_t row_dst = 0;
        if constexpr (KV == ZK_BF16) {
            if (p.new_k && len > 0 && np > 0 && page0 + np == (len + BS - 1) / BS) {
                fuse_tib = (len - 1) % BS;
                const int blk = ((cint_t)p.bt)[(size_t)n * p.max_blocks + (len - 1) / BS];
                const int c = lane % CPR;
                row_dst = ((size_t)blk * Hkv + kvh) * PAGE + (size_t)fuse_tib * RB + (size_t)c * 16;
                if (lane < 2 * CPR)
                    nrow = *reinterpret_cast<const u32x4 *>((lane < CPR ? p.new_k : p.new_v) +
                                                            (size_t)n * p.new_row_bytes + (size_t)kvh * RB + c * 16);
            }
        }
        f32x4 o[DT][1];
        const int own_len[1] = {len};
        float m[1], l[1];
        attend.template operator()<1>(qf, p.bt + (size_t)n * p.max_blocks + page0, d1, page0, np, len, own_len, len, kvh, sl2,
                                      o, m, l, fuse_tib, nrow, row_dst);
        if (col < G) {
            if (ns == 0 && nparts <= 1) {  // the whole context: write the output row
                const float inv = inverse_sum(l[0], m[0], vscale);
                const size_t ob = (qr * H + qh) * D;
                if (p.q_f32) {
                    f32x4 o2[DT][2];
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o2[dt][0] = o[dt][0];
                    store_row_f32((float *)p.out + ob, o2, 0, inv);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uint32_t v[DT / 2];
#pragma unroll
                        for (int j = 0; j < DT / 2; ++j)
                            v[j] = bf16x2_rne(o[2 * j][0][i] * inv, o[2 * j + 1][0][i] * inv);
                        if constexpr (F32) {
#pragma unroll
                            for (int h = 0; h < DT / 4; ++h)
                                __builtin_memcpy((uint16_t *)p.out + ob + 64 * h + 16 * grp + 4 * i, v + 2 * h, 8);
                        } else {
                            __builtin_memcpy((uint16_t *)p.out + ob + DT * (4 * grp + i), v, sizeof(v));
                        }
                    }
                }
            } else {
                const size_t slot = ((size_t)n * H + qh) * p.max_parts + ns + part;
                f32x4 o2[DT][2];
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o2[dt][0] = o[dt][0];
                store_partial(slot, o2, 0, vscale, m[0], cut ? -l[0] : l[0]);
            }
        }
    };

    if constexpr (ROWS) {
        constexpr int NT = 32 / G;  // tokens of a group
        const int kvh = blockIdx.x, part = blockIdx.y, g = blockIdx.z;
        const int page0 = part * p.part_pages;
        const cint_t gd = (cint_t)(p.groups + g);
        const int4 d = make_int4(gd[0], gd[1], gd[2], gd[3]);
        const int len = d.w + d.z - 1;  // the longest row's
        const int want = min(p.part_pages, (len + BS - 1) / BS - page0);
        if (want <= 0) return;
        const int32_t *row = p.bt + (size_t)d.x * p.max_blocks + page0;
        int np = want;  // (the caller's tables are valid up to every length; an id outside the pool still ends the walk)
        int4 first = make_int4(0, 0, 0, 0);
        for (int i0 = 0; i0 < want && np == want; i0 += kWave) {
            const int e = row[min(i0 + lane, want - 1)];
            const uint64_t bad = __builtin_amdgcn_ballot_w64(i0 + lane < want && (e < 0 || (int64_t)e >= p.num_blocks));
            if (bad) np = i0 + (int)__builtin_ctzll(bad);
            bids[i0 + lane] = e;
            if (i0 == 0)
                first = make_int4(__builtin_amdgcn_readlane(e, 0), __builtin_amdgcn_readlane(e, 1),
                                  __builtin_amdgcn_readlane(e, 2), __builtin_amdgcn_readlane(e, 3));
        }
        wait_lgkmcnt0();  // visible to this wave's own reads
        qfrag_t qf[2][KK];
        int row_len[2];  // context of this lane's row of tile t; 0: no row
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int r = 16 * t + col;
            row_len[t] = r / G < d.z ? d.w + r / G : 0;
            if (row_len[t] > 0) load_q((size_t)d.y + r / G, qhead_of(p, kvh, r % G, G), qf[t]);
            else
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) qf[t][kk] = qzero;
        }
        f32x4 o[DT][2];
        float m[2], l[2];
        attend.template operator()<2>(qf, row, first, page0, np, len, row_len, d.w, kvh, p.scale_log2, o, m, l, -1, no_row, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int r = 16 * t + col, qh = qhead_of(p, kvh, r % G, G);
            const int parts = ((row_len[t] + BS - 1) / BS + p.part_pages - 1) / p.part_pages;
            if (part >= parts) continue;  // no row, or none of its tokens here
            if (parts > 1) {
                store_partial(((size_t)(g * NT + r / G) * H + qh) * p.max_parts + part, o, t, 1.0f, m[t], l[t]);
                continue;
            }
            const float inv = inverse_sum(l[t], m[t]);
            const size_t ob = ((size_t)(d.y + r / G) * H + qh) * D;
            if (p.q_f32) {
                store_row_f32((float *)p.out + ob, o, t, inv);
            } else {
#pragma unroll
                for (int h = 0; h < DT / 4; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t v[2] = {bf16x2_rne(o[4 * h][t][i] * inv, o[4 * h + 1][t][i] * inv),
                                               bf16x2_rne(o[4 * h + 2][t][i] * inv, o[4 * h + 3][t][i] * inv)};
                        __builtin_memcpy((uint16_t *)p.out + ob + 64 * h + 16 * grp + 4 * i, v, 8);
                    }
            }
        }
        return;
    }
    if constexpr (SHARED) {
        const int kvh = blockIdx.x, items = p.num_sg * p.shared_parts;
        int y = blockIdx.y;
        const bool sh = y < items;
        int n, part, page0, pages, len = 0, ns = 0, nparts = 0, sg = 0;  // pages of the partition
        if (sh) {
            sg = y / p.shared_parts;
            part = y % p.shared_parts;
            n = ((cint_t)p.sg_members)[(size_t)sg * kSgStride];
            page0 = part * p.shared_part_pages;
            pages = min(p.shared_part_pages, ((cint_t)p.sg_pages)[sg] - page0);
            if (pages <= 0) return;
        } else {
            y -= items;
            const int own = p.max_parts - p.shared_parts;
            n = y / own;
            part = y % own;
            len = min(max(((cint_t)p.seq_lens)[n], 0), p.max_blocks * BS);
            const int pb = ((cint_t)p.seq_pb)[n], rest = (len + BS - 1) / BS - pb;
            ns = pb > 0 ? (pb + p.shared_part_pages - 1) / p.shared_part_pages : 0;
            nparts = rest > 0 ? (rest + p.part_pages - 1) / p.part_pages : 0;
            if (part >= (ns == 0 ? max(1, nparts) : nparts)) return;
            page0 = pb + part * p.part_pages;
            pages = max(0, min(p.part_pages, rest - part * p.part_pages));
        }
        // (the cache's tables: valid up to every length; an id outside the pool
        // still ends the walk)
        const int e = pages > 0 ? p.bt[(size_t)n * p.max_blocks + page0 + min(lane, pages - 1)] : 0;
        const uint64_t bad = __builtin_amdgcn_ballot_w64(lane < pages && (e < 0 || (int64_t)e >= p.num_blocks));
        const int np = bad ? (int)__builtin_ctzll(bad) : pages;
        bids[lane] = e;
        wait_lgkmcnt0();
        const int4 first = make_int4(__builtin_amdgcn_readlane(e, 0), __builtin_amdgcn_readlane(e, 1),
                                     __builtin_amdgcn_readlane(e, 2), __builtin_amdgcn_readlane(e, 3));
        if (sh) shared_part(sg, kvh, part, n, np, first);
        else own_part(n, kvh, part, page0, np, len, ns, nparts, first, bad != 0);
        return;
    }
    if constexpr (DIRECT && !ROWS && !SHARED) {
        const int kvh = blockIdx.x, part = blockIdx.y, n = blockIdx.z;
        const int page0 = part * p.part_pages;
        const int32_t *row = p.bt + (size_t)n * p.max_blocks;
        // this lane's page id beside the length: one round trip
        const int e = page0 + lane < p.max_blocks ? row[page0 + lane] : -1;
        const int len = min(max(((cint_t)p.seq_lens)[n], 0), p.max_blocks * BS);
        const int pages = (len + BS - 1) / BS, nparts = (pages + p.part_pages - 1) / p.part_pages;
        if (part >= max(1, nparts)) return;
        const int want = min(p.part_pages, pages - page0);
        const uint64_t bad = __builtin_amdgcn_ballot_w64(lane < want && (e < 0 || (int64_t)e >= p.num_blocks));
        const int np = bad ? min(want, (int)__builtin_ctzll(bad)) : want;
        bids[lane] = e;
        static_assert(kDirectPages == kWave, "one table entry per lane");
        wait_lgkmcnt0();  // visible to this wave's own reads
        const int4 first = make_int4(__builtin_amdgcn_readlane(e, 0), __builtin_amdgcn_readlane(e, 1),
                                     __builtin_amdgcn_readlane(e, 2), __builtin_amdgcn_readlane(e, 3));
        own_part(n, kvh, part, page0, np, len, 0, nparts, first, bad != 0);
        return;
    }

    int item = blockIdx.x;  // first item static, the rest from the queue
    int4 d0 = make_int4(0, 0, 0, 0), d1 = make_int4(0, 0, 0, 0);
    if (item < total) load_desc(item / Hkv, d0, d1);
    while (item < total) {
        const int kvh = item % Hkv;
        have_next = false;
        bool own = true;
        if constexpr (KV == ZK_BF16) own = d0.x >= 0;
        if (!own) {
            shared_part(-1 - d0.x, kvh, d0.y, d0.z, d0.w, d1);
        } else {
            const int n = d0.x, part = d0.y, page0 = d0.z, np = d0.w;
            const int len = ((cint_t)p.eff_len)[n];  // walk already cut at the first invalid entry
            const int pb = p.seq_pb ? ((cint_t)p.seq_pb)[n] : 0;
            const int ns = pb > 0 ? (pb + p.shared_part_pages - 1) / p.shared_part_pages : 0;
            const int rest = (len + p.block_size - 1) / p.block_size - pb;
            const int nparts = rest > 0 ? (rest + p.part_pages - 1) / p.part_pages : 0;
            own_part(n, kvh, part, page0, np, len, ns, nparts, d1, false);
        }
        if (!have_next) fetch_next();  // an item without pages
        item = nx;
        desc_ready(d0, d1);
        // consumed: a constant until the next fetch, so the descriptor's
        // scalar registers are not kept across the next item's prologue
        nraw = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
}

// ------------------------------------------------------------ generic kernel
// One wavefront per (partition, kv-head, sequence).  Lane = token for QK
// (64-token chunks), lane = dim for PV with readlane broadcasts of p.
constexpr int kMaxG = 16;
constexpr int kMaxDSlots = 4;  // D <= 256

template <int KV>
__device__ __forceinline__ float load_kv(const char *pool, size_t i) {
    if constexpr (KV == ZK_F32) return ((const float *)pool)[i];
    else if constexpr (KV == ZK_BF16) return __uint_as_float((uint32_t)((const uint16_t *)pool)[i] << 16);
    else {
        f32x2 r = __builtin_amdgcn_cvt_pk_f32_fp8((int)((const uint8_t *)pool)[i], false);
        return r[0];
    }
}

template <int KV>
__global__ void __launch_bounds__(kWave) decode_generic_kernel(Params p) {
    __shared__ float q_s[kMaxG * 256];
    const int part = blockIdx.x, kvh = blockIdx.y, n = blockIdx.z;
    const int lane = threadIdx.x;
    const int len = p.eff_len[n];
    const int nparts = num_parts_for(p, len);
    if (part >= (nparts > 0 ? nparts : 1)) return;
    const int H = p.num_heads, Hkv = p.num_kv_heads, D = p.head_dim, BS = p.block_size;
    const int G = H / Hkv;

    for (int i = lane; i < G * D; i += kWave) {
        int j = i / D, d = i % D;
        q_s[i] = load_q(p, qrow(p, n) * (size_t)p.q_stride + (size_t)qhead_of(p, kvh, j, G) * D + d);
    }
    __syncthreads();
    float ks = 1.0f, vs = 1.0f;
    if constexpr (KV == ZK_FP8_E4M3) {
        ks = p.k_scales[(size_t)n * Hkv + kvh];
        vs = p.v_scales[(size_t)n * Hkv + kvh];
    }
    const float sl2 = p.scale_log2 * ks;

    float m[kMaxG], l[kMaxG], o[kMaxG][kMaxDSlots];
#pragma unroll
    for (int j = 0; j < kMaxG; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.0f;
#pragma unroll
        for (int c = 0; c < kMaxDSlots; ++c) o[j][c] = 0.0f;
    }
    const int t_begin = part * p.part_pages * BS;
    const int t_end = min(len, t_begin + p.part_pages * BS);
    const int32_t *btrow = p.bt + (size_t)n * p.max_blocks;
    const size_t rows_per_block = (size_t)Hkv * BS;

    for (int t0 = t_begin; t0 < t_end; t0 += kWave) {
        const int t = t0 + lane;
        const bool valid = t < t_end;
        size_t row = 0;
        if (valid) row = ((size_t)btrow[t / BS] * rows_per_block + (size_t)kvh * BS + t % BS);
        float s[kMaxG];
#pragma unroll
        for (int j = 0; j < kMaxG; ++j) s[j] = 0.0f;
        if (valid) {
            for (int d = 0; d < D; ++d) {
                float kd = load_kv<KV>(p.k_pool, row * D + d);
#pragma unroll
                for (int j = 0; j < kMaxG; ++j)
                    if (j < G) s[j] = fmaf(q_s[j * D + d], kd, s[j]);
            }
        }
        float pj[kMaxG];
#pragma unroll
        for (int j = 0; j < kMaxG; ++j) {
            if (j >= G) break;
            float sj = valid ? s[j] * sl2 : -INFINITY;
            float mx = sj;
            for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
            float m_new = fmaxf(m[j], mx);  // at least one valid token: finite
            float alpha = exp2f(m[j] - m_new);
            float pv = valid ? exp2f(sj - m_new) : 0.0f;
            float ps = pv;
            for (int off = 32; off > 0; off >>= 1) ps += __shfl_xor(ps, off);
            l[j] = l[j] * alpha + ps;
            m[j] = m_new;
#pragma unroll
            for (int c = 0; c < kMaxDSlots; ++c) o[j][c] *= alpha;
            pj[j] = pv;
        }
        const int nvalid = min(kWave, t_end - t0);
        for (int i = 0; i < nvalid; ++i) {
            size_t row_i = ((size_t)(uint32_t)__builtin_amdgcn_readlane((int)(row & 0xffffffffu), i)) |
                           ((size_t)(uint32_t)__builtin_amdgcn_readlane((int)(row >> 32), i) << 32);
            float vd[kMaxDSlots];
#pragma unroll
            for (int c = 0; c < kMaxDSlots; ++c) {
                int d = lane + c * kWave;
                vd[c] = d < D ? load_kv<KV>(p.v_pool, row_i * D + d) : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < kMaxG; ++j) {
                if (j >= G) break;
                float pi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pj[j]), i));
#pragma unroll
                for (int c = 0; c < kMaxDSlots; ++c) o[j][c] = fmaf(pi, vd[c], o[j][c]);
            }
        }
    }

#pragma unroll
    for (int j = 0; j < kMaxG; ++j) {
        if (j >= G) break;
        const int qh = qhead_of(p, kvh, j, G);
        if (nparts <= 1) {
            const float inv = l[j] > 0.0f ? 1.0f / l[j] : 0.0f;
#pragma unroll
            for (int c = 0; c < kMaxDSlots; ++c) {
                int d = lane + c * kWave;
                if (d < D) store_out(p, (qrow(p, n) * H + qh) * D + d, o[j][c] * vs * inv);
            }
        } else {
            const size_t slot = ((size_t)n * H + qh) * p.max_parts + part;
#pragma unroll
            for (int c = 0; c < kMaxDSlots; ++c) {
                int d = lane + c * kWave;
                if (d < D) p.po[slot * D + d] = o[j][c] * vs;
            }
            if (lane == 0) p.ml[slot] = make_float2(m[j], l[j]);
        }
    }
}

// ------------------------------------------------------------ reduce
// One wavefront per (q-head, sequence): o = sum_p w_p o_p / sum_p w_p l_p with
// w_p = 2^(m_p - M).  Lane i owns partition i's weight; the weighted sum walks
// the partitions eight at a time so 16 loads per lane are in flight.
__global__ void __launch_bounds__(kWave) decode_reduce_kernel(Params p) {
    const int h = blockIdx.x, n = blockIdx.y, lane = threadIdx.x;
    const int ns = shared_parts_of(p, n);
    const int nparts = ns + private_parts_of(p, n);
    if (ns == 0 && nparts <= 1) return;  // written by the partition kernel
    const int D = p.head_dim;
    const size_t base = ((size_t)n * p.num_heads + h) * p.max_parts;
    float M = -INFINITY;
    for (int i = lane; i < nparts; i += kWave) M = fmaxf(M, p.ml[base + i].x);
    for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
    float L = 0.0f;
    for (int i = lane; i < nparts; i += kWave) {
        const float2 v = p.ml[base + i];
        L += v.x == -INFINITY ? 0.0f : v.y * exp2f(v.x - M);
    }
    for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off);
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};  // d = lane + 64 * c, D <= 256
    for (int c0 = 0; c0 < nparts; c0 += kWave) {
        float w = 0.0f;
        if (c0 + lane < nparts) {
            const float2 v = p.ml[base + c0 + lane];
            w = v.x == -INFINITY ? 0.0f : exp2f(v.x - M);
        }
        const int cnt = min(kWave, nparts - c0);
        for (int i0 = 0; i0 < cnt; i0 += 8) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u;
                if (i < cnt) {
                    const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i));
                    const float *src = p.po + (base + c0 + i) * D;
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (lane + 64 * c < D) acc[c] = fmaf(wi, src[lane + 64 * c], acc[c]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < D) store_out(p, (qrow(p, n) * p.num_heads + h) * D + lane + 64 * c, acc[c] * inv);
}

// The same merge for D = 4 * LP (D in {64, 128, 256}): LP lanes hold a
// partition's partial output as one float4 each, so one load instruction
// covers 64 / LP partitions and all of a sequence's partitions are in flight
// at once (the loop above waits for each group of eight).  Lane i reads
// partition i's (m, l) once for the maximum, the sum and its weight; the
// first 64 * U0 / LP partials are loaded beside the (m, l), so after the
// lengths a row of up to that many partitions needs one more memory round
// trip, not two.
template <int D>
__global__ void __launch_bounds__(kWave) decode_reduce_vec_kernel(Params p) {
    constexpr int LP = D / 4, P = kWave / LP, U = 16;  // lanes per partition, partitions per load, loads per lane
    constexpr int U0 = 4;  // loads per lane issued with the (m, l): few, so that four waves fit a SIMD
    static_assert(D % 4 == 0 && kWave % LP == 0, "partition layout");
    const int h = blockIdx.x, n = blockIdx.y, lane = threadIdx.x;
    const int ns = shared_parts_of(p, n);
    const int nparts = ns + private_parts_of(p, n);
    if (ns == 0 && nparts <= 1) return;  // written by the partition kernel
    const size_t base = ((size_t)n * p.num_heads + h) * p.max_parts;
    const float2 none = make_float2(-INFINITY, 0.0f);
    const int sub = lane / LP, j = lane % LP;  // partition slot within a load, float4 index
    // the first P * U0 partials go out with the (m, l) loads: one round trip
    // instead of two (they do not depend on the maximum)
    const int cnt0 = min(kWave, nparts);
    f32x4 x0[U0];
#pragma unroll
    for (int u = 0; u < U0; ++u) {
        const int i = P * u + sub;
        x0[u] = i < cnt0 ? *reinterpret_cast<const f32x4 *>(p.po + (base + i) * D + 4 * j) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float2 ml0 = lane < nparts ? p.ml[base + lane] : none;
    float M = ml0.x;
    for (int i = lane + kWave; i < nparts; i += kWave) M = fmaxf(M, p.ml[base + i].x);
    for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
    auto weight = [&](float2 v) { return v.x == -INFINITY ? 0.0f : exp2f(v.x - M); };
    float L = ml0.y * weight(ml0);
    for (int i = lane + kWave; i < nparts; i += kWave) {
        const float2 v = p.ml[base + i];
        L += v.y * weight(v);
    }
    for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off);
    const float inv = inverse_sum(L, M);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < nparts; c0 += kWave) {  // weights of partitions c0 .. c0 + 63 in lanes
        const float w = weight(c0 == 0 ? ml0 : (c0 + lane < nparts ? p.ml[base + c0 + lane] : none));
        const int cnt = min(kWave, nparts - c0);
        for (int i0 = 0; i0 < cnt; i0 += P * U) {
            f32x4 x[U];
            float wi[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + P * u + sub;
                wi[u] = __shfl(w, min(i, kWave - 1));
                if (c0 == 0 && i0 == 0 && u < U0) x[u] = x0[u];
                else x[u] = i < cnt ? *reinterpret_cast<const f32x4 *>(p.po + (base + c0 + i) * D + 4 * j)
                                    : f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + P * u + sub < cnt)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[c] = fmaf(wi[u], x[u][c], acc[c]);
        }
    }
    // the P partition slots of a load sit LP lanes apart
#pragma unroll
    for (int off = LP; off < kWave; off <<= 1)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] += __shfl_xor(acc[c], off);
    if (sub == 0)
#pragma unroll
        for (int c = 0; c < 4; ++c) store_out(p, (qrow(p, n) * p.num_heads + h) * D + 4 * j + c, acc[c] * inv);
}

// One wave per (kv-head, sequence): the G query heads of the kv-head at once
// (LPH = 64 / G lanes a head, F = G * D / 64 floats a lane), so a launch has
// Hkv / H of the waves of decode_reduce_vec_kernel.  Each lane reads its
// head's (m, l) of every partition itself (no cross-lane reductions) and the
// first C partitions' partials with them, one memory round trip; partitions
// are added in slot order.
// MARKS: a partition marked by the sign of its l (planless launches) is the
// context's last.
template <int D, int G, bool MARKS>
__global__ void __launch_bounds__(kWave) decode_reduce_kv_kernel(Params p) {
    constexpr int LPH = kWave / G, F = G * D / kWave, F4 = F / 4;
    constexpr int C = 8;  // partitions loaded with the (m, l)
    static_assert(F % 4 == 0 && kWave % G == 0, "lane layout");
    const int kvh = blockIdx.x, n = blockIdx.y, lane = threadIdx.x;
    const int ns = shared_parts_of(p, n);
    int nparts = ns + private_parts_of<MARKS>(p, n);
    if (ns == 0 && nparts <= 1) return;  // written by the partition kernel
    const int hh = lane / LPH, d0 = (lane % LPH) * F;
    const int qh = qhead_of(p, kvh, hh, G);
    const size_t base = ((size_t)n * p.num_heads + qh) * p.max_parts;
    float2 ml[C];
    f32x4 x[C][F4];
#pragma unroll
    for (int i = 0; i < C; ++i) {
        if (i < nparts) {
            ml[i] = p.ml[base + i];
#pragma unroll
            for (int k = 0; k < F4; ++k) x[i][k] = *reinterpret_cast<const f32x4 *>(p.po + (base + i) * D + d0 + 4 * k);
        } else {
            ml[i] = make_float2(-INFINITY, 0.0f);
        }
    }
    float M = -INFINITY;
    if constexpr (MARKS) {
#pragma unroll
        for (int i = C - 1; i >= 0; --i)
            if (i < nparts && signbit(ml[i].y)) nparts = i + 1;
#pragma unroll
        for (int i = 0; i < C; ++i) {
            M = i < nparts ? fmaxf(M, ml[i].x) : M;
            ml[i].y = fabsf(ml[i].y);
        }
        for (int i = C; i < nparts; ++i) {
            const float2 v = p.ml[base + i];
            M = fmaxf(M, v.x);
            if (signbit(v.y)) nparts = i + 1;
        }
    } else {
#pragma unroll
        for (int i = 0; i < C; ++i) M = fmaxf(M, ml[i].x);
        for (int i = C; i < nparts; ++i) M = fmaxf(M, p.ml[base + i].x);
    }
    auto weight = [&](float2 v) { return v.x == -INFINITY ? 0.0f : exp2f(v.x - M); };
    float L = 0.0f;
    f32x4 acc[F4];
#pragma unroll
    for (int k = 0; k < F4; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < C; ++i)
        if (i < nparts) {
            const float w = weight(ml[i]);
            L += ml[i].y * w;
#pragma unroll
            for (int k = 0; k < F4; ++k)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[k][c] = fmaf(w, x[i][k][c], acc[k][c]);
        }
    for (int i = C; i < nparts; ++i) {
        const float2 v = p.ml[base + i];
        const float w = weight(v);
        L += (MARKS ? fabsf(v.y) : v.y) * w;
#pragma unroll
        for (int k = 0; k < F4; ++k) {
            const f32x4 y = *reinterpret_cast<const f32x4 *>(p.po + (base + i) * D + d0 + 4 * k);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[k][c] = fmaf(w, y[c], acc[k][c]);
        }
    }
    const float inv = inverse_sum(L, M);
    const size_t ob = (qrow<MARKS>(p, n) * p.num_heads + qh) * D + d0;
    if (p.q_f32) {
#pragma unroll
        for (int k = 0; k < F4; ++k) {
            const f32x4 y = acc[k] * inv;
            __builtin_memcpy((float *)p.out + ob + 4 * k, &y, sizeof(y));
        }
    } else {
        uint32_t v[F / 2];
#pragma unroll
        for (int k = 0; k < F4; ++k) {
            v[2 * k] = bf16x2_rne(acc[k][0] * inv, acc[k][1] * inv);
            v[2 * k + 1] = bf16x2_rne(acc[k][2] * inv, acc[k][3] * inv);
        }
        __builtin_memcpy((uint16_t *)p.out + ob, v, sizeof(v));
    }
}

// The merge for sequences of many partitions (long contexts in small batches):
// one 256-thread workgroup per (q-head, sequence), LP = D / 4 lanes a
// partition, so 256 / LP partitions a load and U loads in flight per thread;
// each wave reads all (m, l) itself, and the groups' sums meet in LDS.
template <int D>
__global__ void __launch_bounds__(256) decode_reduce_many_kernel(Params p) {
    constexpr int LP = D / 4, PG = 256 / LP, U = 8;
    __shared__ f32x4 part_sum[256];
    const int h = blockIdx.x, n = blockIdx.y, t = threadIdx.x, lane = t & 63;
    const int ns = shared_parts_of(p, n);
    int nparts = ns + (p.eff_len ? private_parts_of(p, n) : private_parts_of<true>(p, n));
    if (ns == 0 && nparts <= 1) return;  // written by the partition kernel
    const size_t base = ((size_t)n * p.num_heads + h) * p.max_parts;
    const int g = t / LP, d0 = 4 * (t % LP);
    auto load = [&](int i) { return *reinterpret_cast<const f32x4 *>(p.po + (base + i) * D + d0); };
    f32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = load(min(u * PG + g, nparts - 1));  // beside the (m, l)
    // the first marked partition (sign of l) ends the context
    int last = nparts - 1;
    for (int i = lane; i < nparts; i += kWave)
        if (signbit(p.ml[base + i].y)) last = min(last, i);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) last = min(last, __shfl_xor(last, o));
    nparts = last + 1;
    float M = -INFINITY;
    for (int i = lane; i < nparts; i += kWave) M = fmaxf(M, p.ml[base + i].x);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
    auto weight = [&](float m) { return m == -INFINITY ? 0.0f : exp2f(m - M); };
    float L = 0.0f;
    for (int i = lane; i < nparts; i += kWave) {
        const float2 v = p.ml[base + i];
        L += fabsf(v.y) * weight(v.x);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) L += __shfl_xor(L, o);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < nparts; i0 += PG * U) {
        float w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * PG + g;
            if (i0 > 0) x[u] = load(min(i, nparts - 1));
            w[u] = weight(p.ml[base + min(i, nparts - 1)].x);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * PG + g < nparts)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[c] = fmaf(w[u], x[u][c], acc[c]);
    }
    part_sum[t] = acc;
    __syncthreads();
    if (t >= LP) return;
    acc = part_sum[t];
#pragma unroll
    for (int q = 1; q < PG; ++q) acc += part_sum[q * LP + t];
    const float inv = inverse_sum(L, M);
    const size_t ob = (qrow<true>(p, n) * p.num_heads + h) * D + d0;
#pragma unroll
    for (int c = 0; c < 4; ++c) store_out(p, ob + c, acc[c] * inv);
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct WsLayout {
    size_t eff, items, map, work, ml, po, total;
};
WsLayout ws_layout(int num_seqs, int num_heads, int head_dim, int max_parts) {
    WsLayout w;
    w.eff = 0;
    w.items = align256(sizeof(int32_t) * (size_t)num_seqs);
    w.map = w.items;
    w.work = w.map + align256(2 * sizeof(int4) * (size_t)num_seqs * max_parts);
    w.ml = w.work + align256(kWorkBytes);
    size_t slots = (size_t)num_seqs * num_heads * max_parts;
    w.po = w.ml + align256(sizeof(float2) * slots);
    w.total = w.po + align256(sizeof(float) * slots * head_dim);
    return w;
}

int max_parts_for(int max_blocks, int part_pages) { return (max_blocks + part_pages - 1) / part_pages; }

int waves_per_simd_config() {
    static int v = [] {
        const char *e = std::getenv("ZEALOT_DECODE_WAVES_PER_SIMD");
        int w = e ? std::atoi(e) : 1;
        return w < 1 ? 1 : (w > 8 ? 8 : w);
    }();
    return v;
}

// Persistent grid: waves_per_simd one-wave workgroups per SIMD (4 SIMDs per CU).
// Partition length for the persistent kernel: enough (sequence, partition)
// pairs for ~ZEALOT_DECODE_ITEMS_PER_WAVE (default 6) items per wave, at least
// 16 pages, at most kMaxItemPages.
int items_per_wave_config() {
    static int v = [] {
        const char *e = std::getenv("ZEALOT_DECODE_ITEMS_PER_WAVE");
        int w = e ? std::atoi(e) : 6;
        return w < 1 ? 1 : (w > 64 ? 64 : w);
    }();
    return v;
}

int persistent_grid();

int mfma_part_pages(int num_seqs, int num_kv_heads, int max_blocks, long waves) {
    if (int e = part_pages_env()) return e;
    const long pairs = (items_per_wave_config() * waves + num_kv_heads - 1) / num_kv_heads;
    const long per_seq = (pairs + num_seqs - 1) / num_seqs;
    long pp = (max_blocks + per_seq - 1) / per_seq;
    pp = (pp + 15) / 16 * 16;
    return (int)(pp < 16 ? 16 : (pp > kMaxItemPages ? kMaxItemPages : pp));
}

int persistent_grid() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus * 4 * waves_per_simd_config();
}

template <int KV, int D, int G>
void launch_mfma_k(const Params &p, hipStream_t s) {
    if (p.num_waves == 0 && p.num_sg > 0) {
        if constexpr (KV == ZK_BF16) {
            const int own = p.max_parts - p.shared_parts;
            const dim3 grid(p.num_kv_heads, p.num_sg * p.shared_parts + p.num_seqs * own);
            decode_mfma_kernel<KV, D, G, true, false, true><<<grid, kWave, 0, s>>>(p);
        }
    } else if (p.num_waves > 0) {
        decode_mfma_kernel<KV, D, G, false><<<p.num_waves, kWave, 0, s>>>(p);
    } else {
        // Not a multiple of four partitions a sequence: a table wider than the
        // contexts leaves a sequence's later workgroups without work, and at a
        // stride of 20, say, those with work go to 8 of an XCD's 32 CUs (40 x
        // 100..1000 tokens, tables of 1024 pages: 50 us, 33.6 with 21; 128 x
        // 200..2000 in their own tables 121 and 109; two partitions as three, six
        // as seven, and f32's one wave a SIMD, lose as often as they win).
        const int parts = p.max_parts + (KV != ZK_F32 && p.max_parts % 4 == 0);
        decode_mfma_kernel<KV, D, G, true><<<dim3(p.num_kv_heads, parts, p.num_seqs), kWave, 0, s>>>(p);
    }
}

template <int KV, int D>
void launch_mfma_g(const Params &p, hipStream_t s, int G) {
    switch (G) {
        case 1: launch_mfma_k<KV, D, 1>(p, s); break;
        case 2: launch_mfma_k<KV, D, 2>(p, s); break;
        case 4: launch_mfma_k<KV, D, 4>(p, s); break;
        default: launch_mfma_k<KV, D, 8>(p, s); break;
    }
}

template <int KV>
void launch_mfma(const Params &p, hipStream_t s, int G) {
    if (p.head_dim == 128) launch_mfma_g<KV, 128>(p, s, G);
    else launch_mfma_g<KV, 64>(p, s, G);
}

// Partitions from which one workgroup a q-head merges them: eight lines of a
// wave's loads in flight instead of a serial walk (2 sequences of 125
// partitions: 35 -> 5 us).
constexpr int kManyParts = 16;

template <int G>
void launch_reduce_kv(const Params &p, bool planless, hipStream_t s) {
    const dim3 grid(p.num_kv_heads, p.num_seqs);
    if (planless) decode_reduce_kv_kernel<128, G, true><<<grid, kWave, 0, s>>>(p);
    else decode_reduce_kv_kernel<128, G, false><<<grid, kWave, 0, s>>>(p);
}

// The merge for head_dim 64 or 128 (planless: partials may be marked).
void launch_reduce(const Params &p, int G, bool planless, hipStream_t s) {
    const dim3 rgrid(p.num_heads, p.num_seqs);
    const bool kv = p.head_dim == 128 && (G == 2 || G == 4 || G == 8);
    // (with shared prefixes max_parts is the stride of the slots, not their number)
    if ((planless && !kv) || (p.max_parts > kManyParts && p.num_sg == 0)) {
        if (p.head_dim == 128) decode_reduce_many_kernel<128><<<rgrid, 256, 0, s>>>(p);
        else decode_reduce_many_kernel<64><<<rgrid, 256, 0, s>>>(p);
    } else if (kv) {
        if (G == 4) launch_reduce_kv<4>(p, planless, s);
        else if (G == 8) launch_reduce_kv<8>(p, planless, s);
        else launch_reduce_kv<2>(p, planless, s);
    } else if (p.head_dim == 128) {
        decode_reduce_vec_kernel<128><<<rgrid, kWave, 0, s>>>(p);
    } else {
        decode_reduce_vec_kernel<64><<<rgrid, kWave, 0, s>>>(p);
    }
}

bool mfma_supported(int kv_dtype, int head_dim, int block_size, int G) {
    return valid_dtype(kv_dtype) && block_size == 16 &&
           (head_dim == 128 || head_dim == 64) && (G == 1 || G == 2 || G == 4 || G == 8);
}

int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(ZK_ERR_HIP, std::string("Internal error: ") + what + ": " + hipGetErrorString(e));
    return ZK_OK;
}

// Pages per shared-prefix item: about one item per two waves over all
// subgroups' pages, so half the waves stream the shared pages (two query-row
// tiles each) while the rest run the sequences' own items; measured best on
// forked-prefix batches.  ZEALOT_DECODE_SHARED_PART_PAGES (16..1024) overrides.
int shared_part_pages_for(long total_shared_pages, int num_kv_heads, long waves) {
    static const int env = [] {
        const char *e = std::getenv("ZEALOT_DECODE_SHARED_PART_PAGES");
        const int v = e ? std::atoi(e) : 0;
        return v <= 0 ? 0 : (v < 16 ? 16 : (v > kMaxItemPages ? kMaxItemPages : v));
    }();
    if (env) return env;
    const long half = waves / 2;
    long pp = (total_shared_pages * num_kv_heads + half - 1) / half;
    pp = (pp + 15) / 16 * 16;
    return (int)(pp < 16 ? 16 : (pp > kMaxItemPages ? kMaxItemPages : pp));
}

// Planless launches: partitions of a sequence for `units` (capacity) pages
// over all sequences and kv-heads, of page_bytes of K and V each; 0: too much
// work for one.  The host knows the tables' capacity, not the lengths.
//
// Against the planned persistent grid a planless launch saves the table walk
// and plan kernels (7-50 us) and hides an item's prologue behind other
// resident waves, but starts items in table order, not longest first.
// Measured (planned / planless, us): 2 x 26000 bf16 tokens 94 / 38, 4 x 17..1000
// 22 / 15, 64 x 512..8192 bf16 177 / 165, fp8 116 / 89, f32 324 / 313; 40 x
// 1024..16384 206 / 193; then 192 x 300..4000 bf16 264 / 278 and 256 x 512..8192
// 643 / 708: the line lies at 3 GB of capacity.
// Where one plan serves the layers of a step (plan_launches) and the tables need
// no walk, nothing of that is saved, and the line lies where the kernels' own
// times cross (planned / planless, us a layer with the merge; 8 layers): bf16 96 x
// 200..2000 (0.8 GB) 94 / 83, 48 x 512..8192 (1.6) 135 / 127, 256 x 100..1000 (1.1)
// 117 / 119, 64 x 512..8192 (2.1) 176.4 / 178.9, 88 x (3.0) 237 / 246; fp8 48 x
// 4000..16000 (1.6) 188 / 176, 110 x 512..8192 (1.8) 171 / 170; f32 24 x 512..4096
// (0.8) 88 / 75, 64 x 100..2000 (1.0) 101 / 113, 8 x 4000..16000 (1.0) 122 / 133.
//
// The partition length P balances the items' fixed cost, (units / P) a / waves,
// against the tail of one item, P b: P ~ sqrt(units), with page_bytes for the
// page time.  sqrt(bytes) / 1000 is within 5 % of the best of 4, 8, 16, 24, 32,
// 48, 64 on bf16, fp8 and f32, 128 and 64 dims, 8000 to 260000 pages.  Fewer
// than 8 pages do not pay for the reduce; the count is rounded to the nearest
// so that a table a little over P stays one partition (no reduce at all).
constexpr double kDirectBytes = 3e9;
constexpr int kPlanLaunches = 4;  // a plan over fewer launches still costs each 5 us and more
double direct_limit(int kv_dtype, int plan_launches) {
    if (plan_launches < kPlanLaunches) return kDirectBytes;
    return kv_dtype == ZK_F32 ? 0.9e9 : kv_dtype == ZK_BF16 ? 1.6e9 : 2.0e9;
}
// Shared prefixes without a plan: about this many shared items over all
// kv-heads (each streams its pages for up to 32 rows, beside the sequences' own
// one- and two-page items, all resident at once), of at least 10 pages.  Against
// the planned launch (eight queues, 32-page items), four layers of a step, us: 16
// x 8 forks of 2050 tokens 152 / 139 (134 with the merge a kv-head), 12 x 8 of 3900
// 187 / 172, 5 x 11 of 2420 117 / 107, 8 x 2 of 700 76 / 62, 1 x 2 of 400 70 / 45;
// 256, 512, 640 and 1024 items 171, 146, 147 and 161 on the first.  Over 8 layers
// with one plan, us a layer: 8 x 8 of 4000 (131 MB of shared pages) 40.5 / 36, 24 x
// 8 of 4000 (393) 97 / 97, 16 x 8 of 8000 (525) 125 / 132, 8 x 8 of 16000 (523) 121 /
// 130, 200 x 4 of 1000 (817) 196 / 211 (but 4 x 32 of 16000, 1018, whose subgroups
// read the same pages: 162 / 138).
constexpr long kSharedItems = 384, kSharedMinPages = 10;
constexpr double kDirectSharedBytes = 0.45e9;
int direct_parts(double units, double page_bytes, int max_blocks, double limit = kDirectBytes) {
    const double bytes = units * page_bytes;
    if (bytes > limit) return 0;
    const double pp = std::min((double)kDirectPages, std::max(8.0, std::sqrt(bytes) * 1e-3));
    return std::max((max_blocks + kDirectPages - 1) / kDirectPages, std::max(1, (int)(max_blocks / pp + 0.5)));
}

}  // namespace

size_t zk::paged_decode_workspace(int num_seqs, int num_heads, int head_dim, int max_blocks_per_seq,
                                  int block_size, bool shared) {
    if (num_seqs <= 0 || num_heads <= 0 || head_dim <= 0 || max_blocks_per_seq <= 0) return 256;
    // the planned paths' partitions, or (16-token blocks of 64 or 128 dims) the
    // planless one's at the fewest bytes a page and the most heads a kv-head
    int parts = max_parts_for(max_blocks_per_seq, min_part_pages(head_dim, block_size)) + (shared ? 1 : 0);
    if (block_size == 16 && (head_dim == 64 || head_dim == 128))
        parts = std::max(parts, direct_parts((double)num_seqs * max_blocks_per_seq * std::max(1, num_heads / 8),
                                             2.0 * block_size * head_dim, max_blocks_per_seq));
    return ws_layout(num_seqs, num_heads, head_dim, parts).total;
}

bool zk::paged_decode_shares_prefixes(int kv_dtype, int head_dim, int block_size, int num_heads, int num_kv_heads) {
    return kv_dtype == ZK_BF16 && num_kv_heads > 0 && num_heads % num_kv_heads == 0 &&
           mfma_supported(kv_dtype, head_dim, block_size, num_heads / num_kv_heads);
}

bool zk::paged_decode_fuses_append(int kv_dtype, int head_dim, int block_size, int num_heads, int num_kv_heads) {
    return zk::paged_decode_shares_prefixes(kv_dtype, head_dim, block_size, num_heads, num_kv_heads);
}

namespace {

// Host-side argument checks of zk_paged_decode (no device work).
int check_decode_args(zk_dtype q_dtype, zk_dtype kv_dtype, int num_seqs, int num_heads, int num_kv_heads,
                      int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                      zk_gqa_mapping mapping) {
    if (q_dtype != ZK_F32 && q_dtype != ZK_BF16)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: q dtype must be f32 or bf16");
    if (!valid_dtype(kv_dtype))
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: unsupported kv dtype");
    if (num_seqs < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
        max_blocks_per_seq <= 0 || num_blocks <= 0)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: bad shape");
    if (num_heads % num_kv_heads != 0)
        return set_error(ZK_ERR_INVALID_ARGUMENT,
                         "Internal error: zk_paged_decode: num_heads must be a multiple of num_kv_heads");
    if (mapping != ZK_GQA_GROUPED && mapping != ZK_GQA_MODULO)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: bad gqa mapping");
    if (head_dim > 256 || num_heads / num_kv_heads > kMaxG)
        return set_error(ZK_ERR_INVALID_ARGUMENT,
                         "Internal error: zk_paged_decode: head_dim <= 256 and H/Hkv <= 16 required");
    if ((int64_t)max_blocks_per_seq * block_size > 0x7fffffff)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: context too long");
    return ZK_OK;
}

// Which kernel a call runs, how it cuts the contexts and the workspace it
// needs (arguments already checked).
struct DecodeShape {
    bool use_mfma, shared, direct;
    int shared_parts;
    size_t need;  // workspace a caller must give: the planned launch's, also where the planless one takes less
    int part_pages, shared_pages, max_parts, waves;
    WsLayout w;
};
// max_waves > 0 caps the MFMA path's persistent grid (partitions are sized
// for the waves that run them); plan_launches: see direct_limit.
DecodeShape decode_shape(zk_dtype kv_dtype, int num_seqs, int num_heads, int num_kv_heads, int head_dim,
                         int block_size, int max_blocks_per_seq, const PrefixGroups *pg, bool aligned,
                         size_t workspace_bytes, int max_waves = 0, int plan_launches = 1) {
    DecodeShape d;
    const int G = num_heads / num_kv_heads;
    // f32 pools: any alignment was and is accepted, the 16-byte accesses of
    // the MFMA kernel need theirs
    d.use_mfma = mfma_supported(kv_dtype, head_dim, block_size, G) && (kv_dtype != ZK_F32 || aligned);
    d.waves = persistent_grid();
    if (max_waves > 0 && max_waves < d.waves) d.waves = max_waves;
    d.part_pages = d.use_mfma ? mfma_part_pages(num_seqs, num_kv_heads, max_blocks_per_seq, d.waves)
                              : part_pages_for(ZK_F32, head_dim, block_size);
    // (no smaller than the generic kernel's: one workspace serves both)
    if (kv_dtype == ZK_F32) d.part_pages = std::max(d.part_pages, part_pages_for(ZK_F32, head_dim, block_size));
    d.shared = pg && pg->num_sg > 0 &&
               paged_decode_shares_prefixes(kv_dtype, head_dim, block_size, num_heads, num_kv_heads);
    d.shared_pages = d.shared ? shared_part_pages_for(pg->total_shared_pages, num_kv_heads, d.waves) : 0;
    // slot stride: a sequence's shared and private partitions together
    d.max_parts = d.shared ? max_parts_for(max_blocks_per_seq, min_part_pages(head_dim, block_size)) + 1
                           : max_parts_for(max_blocks_per_seq, d.part_pages);
    d.w = ws_layout(num_seqs, num_heads, head_dim, d.max_parts);
    d.need = d.w.total;
    if (d.use_mfma && kv_dtype == ZK_F32)  // (as the generic kernel, which takes the unaligned calls, needs)
        d.need = std::max(d.need, ws_layout(num_seqs, num_heads, head_dim,
                                            max_parts_for(max_blocks_per_seq, part_pages_for(ZK_F32, head_dim, block_size)))
                                      .total);
    d.direct = false;
    d.shared_parts = 0;
    if (workspace_bytes < d.need) return d;  // refused
    const double limit = direct_limit(kv_dtype, plan_launches);
    if (d.use_mfma && d.shared && max_waves == 0 && !part_pages_env() && pg->max_pages > 0) {
        // shared prefixes without a plan: see kSharedItems
        const double page_bytes = 2.0 * block_size * head_dim * elt_size(kv_dtype);
        const double own_units = (double)num_seqs * std::max(1, pg->max_rest) * num_kv_heads;
        const int own = direct_parts(own_units, page_bytes, std::max(1, pg->max_rest), limit);
        const double shared_bytes = (double)pg->total_shared_pages * num_kv_heads * page_bytes;
        const int sp = (int)std::min<long>(kDirectPages, std::max<long>(kSharedMinPages, (pg->total_shared_pages * num_kv_heads + kSharedItems - 1) / kSharedItems));
        const int parts = (pg->max_pages + sp - 1) / sp;
        const WsLayout w = ws_layout(num_seqs, num_heads, head_dim, parts + own);
        if (own > 0 && own_units * page_bytes + shared_bytes <= limit &&
            (plan_launches < kPlanLaunches || shared_bytes <= kDirectSharedBytes) &&
            (long)pg->num_sg * parts + (long)num_seqs * own <= 65535 && w.total <= workspace_bytes) {
            d.direct = true;
            d.waves = 0;
            d.shared_parts = parts;
            d.shared_pages = sp;
            d.part_pages = (std::max(1, pg->max_rest) + own - 1) / own;
            d.max_parts = parts + own;
            d.w = w;
        }
    }
    if (d.use_mfma && !d.shared && max_waves == 0 && !part_pages_env()) {
        const int parts = direct_parts((double)num_seqs * max_blocks_per_seq * num_kv_heads,
                                       2.0 * block_size * head_dim * elt_size(kv_dtype), max_blocks_per_seq, limit);
        const WsLayout w = ws_layout(num_seqs, num_heads, head_dim, parts);
        if (parts > 0 && num_seqs <= 65535 && w.total <= workspace_bytes) {
            d.direct = true;
            d.waves = 0;
            d.part_pages = (max_blocks_per_seq + parts - 1) / parts;
            d.max_parts = parts;
            d.w = w;
        }
    }
    d.need = std::max(d.need, d.w.total);
    return d;
}

}  // namespace

int zk::paged_decode(const void *q, zk_dtype q_dtype, const void *k_pool, const void *v_pool, zk_dtype kv_dtype,
                     void *out, const int32_t *block_tables, const int32_t *seq_lens, int num_seqs, int num_heads,
                     int num_kv_heads, int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                     float scale, zk_gqa_mapping mapping, const float *k_scales, const float *v_scales,
                     void *workspace, size_t workspace_bytes, void *stream, const PrefixGroups *pg,
                     const int32_t *q_rows, int64_t q_stride, bool trusted_tables, bool reuse_plan,
                     const AppendRows *append, int *head_set, int max_waves, int plan_launches) {
    if (int rc = check_decode_args(q_dtype, kv_dtype, num_seqs, num_heads, num_kv_heads, head_dim, block_size,
                                   max_blocks_per_seq, num_blocks, mapping))
        return rc;
    if (num_seqs == 0) return ZK_OK;
    if (!q || !k_pool || !v_pool || !out || !block_tables || !seq_lens || !workspace)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode: NULL pointer");
    const bool fp8 = kv_dtype == ZK_FP8_E4M3;
    if (fp8 != (k_scales != nullptr && v_scales != nullptr))
        return set_error(ZK_ERR_INVALID_ARGUMENT,
                         "Internal error: zk_paged_decode: fp8 pools need k/v scales, other pools none");
    const int G = num_heads / num_kv_heads;
    if (pg && pg->num_sg > 0 && (!pg->seq_pb || !pg->sg_members || !pg->sg_pages) &&
        paged_decode_shares_prefixes(kv_dtype, head_dim, block_size, num_heads, num_kv_heads))
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: paged decode: NULL prefix-group array");
    const bool aligned = (((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool | (uintptr_t)out) & 15u) == 0 &&
                         q_stride % 4 == 0;
    const DecodeShape ds = decode_shape(kv_dtype, num_seqs, num_heads, num_kv_heads, head_dim, block_size,
                                        max_blocks_per_seq, pg, aligned, workspace_bytes, max_waves, plan_launches);
    const bool use_mfma = ds.use_mfma, shared = ds.shared;
    if (append && (!use_mfma || kv_dtype != ZK_BF16 || !trusted_tables || !append->k || !append->v ||
                   append->row_bytes < (int64_t)num_kv_heads * head_dim * 2 || (append->row_bytes & 15) ||
                   (((uintptr_t)append->k | (uintptr_t)append->v) & 15u)))
        return set_error(ZK_ERR_INVALID_ARGUMENT,
                         "Internal error: paged decode: fused append needs the bf16 MFMA path, trusted tables and "
                         "16-byte aligned rows");
    const int part_pages = ds.part_pages, shared_pages = ds.shared_pages, max_parts = ds.max_parts;
    const WsLayout &w = ds.w;
    if (workspace_bytes < ds.need || ((uintptr_t)workspace & 255u))
        return set_error(ZK_ERR_INVALID_ARGUMENT,
                         "Internal error: zk_paged_decode: workspace too small or not 256-B aligned (need " +
                             std::to_string(ds.need) + " bytes)");

    Params p{};
    p.q = q;
    p.k_pool = (const char *)k_pool;
    p.v_pool = (const char *)v_pool;
    p.out = out;
    p.bt = block_tables;
    p.seq_lens = seq_lens;
    p.k_scales = k_scales;
    p.v_scales = v_scales;
    p.q_rows = q_rows;
    p.q_stride = q_stride > 0 ? q_stride : (int64_t)num_heads * head_dim;
    p.trusted = trusted_tables ? 1 : 0;
    char *ws = (char *)workspace;
    p.eff_len = ds.direct ? nullptr : (int32_t *)(ws + w.eff);
    p.items = (int4 *)(ws + w.map);
    p.work = (int32_t *)(ws + w.work);
    p.num_waves = use_mfma ? ds.waves : 0;
    p.queues = shared ? kQueues : 1;
    p.ml = (float2 *)(ws + w.ml);
    p.po = (float *)(ws + w.po);
    p.num_seqs = num_seqs;
    p.num_heads = num_heads;
    p.num_kv_heads = num_kv_heads;
    p.head_dim = head_dim;
    p.block_size = block_size;
    p.max_blocks = max_blocks_per_seq;
    p.part_pages = part_pages;
    p.max_parts = max_parts;
    p.num_blocks = num_blocks;
    p.seq_pb = shared ? pg->seq_pb : nullptr;
    p.sg_members = shared ? pg->sg_members : nullptr;
    p.sg_pages = shared ? pg->sg_pages : nullptr;
    p.num_sg = shared ? pg->num_sg : 0;
    p.shared_part_pages = shared ? shared_pages : 1;
    p.shared_parts = ds.shared_parts;
    p.scale_log2 = scale * kLog2e;
    p.grouped = mapping == ZK_GQA_GROUPED ? 1 : 0;
    p.q_f32 = q_dtype == ZK_F32 ? 1 : 0;
    if (append) {
        p.new_k = (const char *)append->k;
        p.new_v = (const char *)append->v;
        p.new_row_bytes = append->row_bytes;
    }

    hipStream_t s = (hipStream_t)stream;
    reuse_plan = reuse_plan && use_mfma;
    if (!ds.direct && !(use_mfma && (trusted_tables || reuse_plan))) {  // trusted MFMA launches: the plan sets the lengths
        {
            KernelTimer timer("decode_seq_info", s);
            seq_info_kernel<<<num_seqs, kWave, 0, s>>>(p);
        }
        if (int rc = check_launch("zk_paged_decode seq_info")) return rc;
    }
    const bool reduce = max_parts > 1 || shared;
    if (ds.direct) {
        KernelTimer timer("decode_partials", s);
        if (kv_dtype == ZK_F32) launch_mfma<ZK_F32>(p, s, G);
        else if (kv_dtype == ZK_BF16) launch_mfma<ZK_BF16>(p, s, G);
        else launch_mfma<ZK_FP8_E4M3>(p, s, G);
    } else if (use_mfma) {
        // a launch reusing the plan claims from the head set the launch
        // before it put back
        reuse_plan = reuse_plan && head_set;
        p.head_set = reuse_plan ? (*head_set & 1) : 0;
        if (!reuse_plan) {
            {
                KernelTimer timer("decode_plan", s);
                plan_kernel<<<1, 1024, 0, s>>>(p, num_seqs);
            }
            if (int rc = check_launch("zk_paged_decode plan")) return rc;
        }
        {
            KernelTimer timer("decode_partials", s);
            if (kv_dtype == ZK_F32) launch_mfma<ZK_F32>(p, s, G);
            else if (kv_dtype == ZK_BF16) launch_mfma<ZK_BF16>(p, s, G);
            else launch_mfma<ZK_FP8_E4M3>(p, s, G);
        }
        if (int rc = check_launch("zk_paged_decode partials")) return rc;
        if (head_set) *head_set = p.head_set ^ 1;
    } else {
        KernelTimer timer("decode_partials", s);
        dim3 grid(max_parts, num_kv_heads, num_seqs);
        if (kv_dtype == ZK_F32) decode_generic_kernel<ZK_F32><<<grid, kWave, 0, s>>>(p);
        else if (kv_dtype == ZK_BF16) decode_generic_kernel<ZK_BF16><<<grid, kWave, 0, s>>>(p);
        else decode_generic_kernel<ZK_FP8_E4M3><<<grid, kWave, 0, s>>>(p);
    }
    if (int rc = check_launch("zk_paged_decode partials")) return rc;
    if (reduce) {
        KernelTimer timer("decode_reduce", s);
        if (use_mfma) {
            launch_reduce(p, G, ds.direct, s);
        } else {
            const dim3 rgrid(num_heads, num_seqs);
            if (head_dim == 128 && (G == 2 || G == 4 || G == 8)) launch_reduce(p, G, false, s);
            else if (head_dim == 128) decode_reduce_vec_kernel<128><<<rgrid, kWave, 0, s>>>(p);
            else if (head_dim == 64) decode_reduce_vec_kernel<64><<<rgrid, kWave, 0, s>>>(p);
            else if (head_dim == 256) decode_reduce_vec_kernel<256><<<rgrid, kWave, 0, s>>>(p);
            else decode_reduce_kernel<<<rgrid, kWave, 0, s>>>(p);
        }
        if (int rc = check_launch("zk_paged_decode reduce")) return rc;
    }
    return ZK_OK;
}

// ------------------------------------------------------------ chunk rows on f32 pools
bool zk::paged_rows_supported(int kv_dtype, int head_dim, int block_size, int num_heads, int num_kv_heads) {
    return kv_dtype == ZK_F32 && num_kv_heads > 0 && num_heads % num_kv_heads == 0 &&
           mfma_supported(kv_dtype, head_dim, block_size, num_heads / num_kv_heads);
}

namespace {

// Partitions of a group's pages: two waves a SIMD over all groups.  Of at least
// 4 pages while the merge reads them in one round (eight partials), else of 8
// (a partial row costs as much as two of its pages), and not 9 to 16 of them,
// which the merge would walk one by one (150 rows behind 600 tokens: 11
// partitions 61 us a step, 5 partitions 51).
int rows_parts(long groups, int num_kv_heads, int max_blocks) {
    const long want = std::max<long>(1, 2048 / std::max<long>(1, groups * num_kv_heads));
    long parts = std::min<long>(want, max_blocks / 4);
    if (parts > 8) {
        parts = std::min<long>(want, max_blocks / 8);
        if (parts <= kManyParts) parts = std::min<long>(parts, 8);
    }
    return (int)std::max<long>(std::max<long>(1, parts), (max_blocks + kMaxItemPages - 1) / kMaxItemPages);
}
WsLayout rows_layout(int groups, int num_heads, int num_kv_heads, int head_dim, int max_blocks) {
    return ws_layout(groups * (32 * num_kv_heads / num_heads), num_heads, head_dim, rows_parts(groups, num_kv_heads, max_blocks));
}

template <int D>
void launch_rows(const Params &p, int groups, hipStream_t s, int G) {
    const dim3 grid(p.num_kv_heads, p.max_parts, groups);
    switch (G) {
        case 1: decode_mfma_kernel<ZK_F32, D, 1, true, true><<<grid, kWave, 0, s>>>(p); break;
        case 2: decode_mfma_kernel<ZK_F32, D, 2, true, true><<<grid, kWave, 0, s>>>(p); break;
        case 4: decode_mfma_kernel<ZK_F32, D, 4, true, true><<<grid, kWave, 0, s>>>(p); break;
        default: decode_mfma_kernel<ZK_F32, D, 8, true, true><<<grid, kWave, 0, s>>>(p); break;
    }
}

}  // namespace

size_t zk::paged_rows_workspace(int groups, int num_heads, int num_kv_heads, int head_dim, int max_blocks_per_seq) {
    if (rows_parts(groups, num_kv_heads, max_blocks_per_seq) == 1) return 256;  // every row is written by its own item
    return rows_layout(groups, num_heads, num_kv_heads, head_dim, max_blocks_per_seq).total;
}

// The attention's grid holds a group and the merge's a row per z / y: 65535 at most.
int zk::paged_rows_max_groups(int num_heads, int num_kv_heads) { return 65535 / (32 * num_kv_heads / num_heads); }

int zk::paged_rows(const void *q, zk_dtype q_dtype, const void *k_pool, const void *v_pool, void *out,
                   const int32_t *block_tables, const int4 *row_groups, int groups, int num_heads, int num_kv_heads,
                   int head_dim, int max_blocks_per_seq, int64_t num_blocks, float scale, zk_gqa_mapping mapping,
                   void *workspace, size_t workspace_bytes, void *stream, int64_t q_stride) {
    if (int rc = check_decode_args(q_dtype, ZK_F32, groups, num_heads, num_kv_heads, head_dim, 16, max_blocks_per_seq,
                                   num_blocks, mapping))
        return rc;
    if (groups == 0) return ZK_OK;
    if (!q || !k_pool || !v_pool || !out || !block_tables || !row_groups || !workspace)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: paged rows: NULL pointer");
    const WsLayout w = rows_layout(groups, num_heads, num_kv_heads, head_dim, max_blocks_per_seq);
    if (groups > paged_rows_max_groups(num_heads, num_kv_heads) ||
        workspace_bytes < paged_rows_workspace(groups, num_heads, num_kv_heads, head_dim, max_blocks_per_seq) ||
        ((uintptr_t)workspace & 255u))
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: paged rows: too many groups or workspace too small");
    const int G = num_heads / num_kv_heads;
    Params p{};
    p.q = q;
    p.k_pool = (const char *)k_pool;
    p.v_pool = (const char *)v_pool;
    p.out = out;
    p.bt = block_tables;
    p.groups = row_groups;
    p.q_stride = q_stride > 0 ? q_stride : (int64_t)num_heads * head_dim;
    char *ws = (char *)workspace;
    p.ml = (float2 *)(ws + w.ml);
    p.po = (float *)(ws + w.po);
    p.num_seqs = groups * (32 / G);
    p.num_heads = num_heads;
    p.num_kv_heads = num_kv_heads;
    p.head_dim = head_dim;
    p.block_size = 16;
    p.max_blocks = max_blocks_per_seq;
    p.max_parts = rows_parts(groups, num_kv_heads, max_blocks_per_seq);
    p.part_pages = (max_blocks_per_seq + p.max_parts - 1) / p.max_parts;
    p.num_blocks = num_blocks;
    p.shared_part_pages = 1;
    p.scale_log2 = scale * kLog2e;
    p.grouped = mapping == ZK_GQA_GROUPED ? 1 : 0;
    p.q_f32 = q_dtype == ZK_F32 ? 1 : 0;
    hipStream_t s = (hipStream_t)stream;
    {
        KernelTimer timer("prefill_attention", s);
        if (head_dim == 128) launch_rows<128>(p, groups, s, G);
        else launch_rows<64>(p, groups, s, G);
    }
    if (int rc = check_launch("paged rows")) return rc;
    if (p.max_parts > 1) {
        KernelTimer timer("decode_reduce", s);
        launch_reduce(p, G, /*planless=*/true, s);
        if (int rc = check_launch("paged rows reduce")) return rc;
    }
    return ZK_OK;
}

// ------------------------------------------------------------ no-allocation decode
// zk_paged_decode_noalloc's workspace is the device array of
// noalloc_scratch.hip (zk::noalloc_scratch), reserved on a GPU by the first
// call there.

extern "C" {

size_t zk_paged_decode_workspace_size(int num_seqs, int num_heads, int head_dim, int max_blocks_per_seq,
                                      int block_size) {
    return zk::paged_decode_workspace(num_seqs, num_heads, head_dim, max_blocks_per_seq, block_size, false);
}

int zk_paged_decode(const void *q, zk_dtype q_dtype, const void *k_pool, const void *v_pool,
                    zk_dtype kv_dtype, void *out, const int32_t *block_tables, const int32_t *seq_lens,
                    int num_seqs, int num_heads, int num_kv_heads, int head_dim, int block_size,
                    int max_blocks_per_seq, int64_t num_blocks, float scale, zk_gqa_mapping mapping,
                    const float *k_scales, const float *v_scales, void *workspace, size_t workspace_bytes,
                    void *stream) {
    return zk::paged_decode(q, q_dtype, k_pool, v_pool, kv_dtype, out, block_tables, seq_lens, num_seqs,
                            num_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, num_blocks, scale,
                            mapping, k_scales, v_scales, workspace, workspace_bytes, stream, nullptr, nullptr);
}

int zk_paged_decode_noalloc(const void *q, zk_dtype q_dtype, const void *k_pool, const void *v_pool,
                            zk_dtype kv_dtype, void *out, const int32_t *block_tables, const int32_t *seq_lens,
                            int num_seqs, int num_heads, int num_kv_heads, int head_dim, int block_size,
                            int max_blocks_per_seq, int64_t num_blocks, float scale, zk_gqa_mapping mapping,
                            const float *k_scales, const float *v_scales, void *stream) {
    if (int rc = check_decode_args(q_dtype, kv_dtype, num_seqs, num_heads, num_kv_heads, head_dim, block_size,
                                   max_blocks_per_seq, num_blocks, mapping))
        return rc;
    if (num_seqs == 0) return ZK_OK;
    const size_t need =
        decode_shape(kv_dtype, num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, nullptr,
                     (((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool | (uintptr_t)out) & 15u) == 0,
                     (size_t)ZK_DECODE_SCRATCH_BYTES)
            .need;
    if (need > (size_t)ZK_DECODE_SCRATCH_BYTES)
        return set_error(ZK_ERR_INVALID_ARGUMENT, "Internal error: zk_paged_decode_noalloc: the call needs " +
                                                      std::to_string(need) + " bytes of scratch, the maximum is " +
                                                      std::to_string((size_t)ZK_DECODE_SCRATCH_BYTES));
    void *ws = nullptr;
    if (int rc = zk::noalloc_scratch(&ws)) return rc;
    zk::TimingSuspend no_events;  // per-kernel timing would create hipEvents
    return zk::paged_decode(q, q_dtype, k_pool, v_pool, kv_dtype, out, block_tables, seq_lens, num_seqs, num_heads,
                            num_kv_heads, head_dim, block_size, max_blocks_per_seq, num_blocks, scale, mapping,
                            k_scales, v_scales, ws, (size_t)ZK_DECODE_SCRATCH_BYTES, stream, nullptr, nullptr);
}

}  // extern "C"
